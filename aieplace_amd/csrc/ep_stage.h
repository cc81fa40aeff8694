// ep_stage.h -- transfers between device arrays and the caller's host arrays.
//
// The caller's arrays are pageable.  hipMemcpy moves those at 2 GB/s up to half a
// megabyte (0.25 MB: 110 us each way) and at 17 GB/s beyond.  Here they pass
// through two pinned slots in turn, so that one chunk is on its way to the
// host (50 GB/s) while the host copies the one before it, and a kernel puts the
// cells into the caller's order on the way: 0.25 MB takes 20 us.  What fits a slot
// moves by a kernel both ways, which starts sooner than the copy engine: positions
// of 6400 cells go in in 30 us (copy engine 43, hipMemcpy 37).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "ep_common.h"

namespace ep {

constexpr size_t kStageSlot = (size_t)1 << 20;  // bytes of a slot, at most

// Two pinned slots of one context, used on its stream.
struct Stage {
    hipStream_t stream = nullptr;
    char *pin[2] = {nullptr, nullptr};
    hipEvent_t done[2] = {nullptr, nullptr};
    size_t bytes = 0;              // of one slot
    int up = 0;                    // slot of the next upload
    int32_t *flag = nullptr;       // pinned word that kernels set
};
// Slots for transfers of up to `most` bytes at a time (kStageSlot at most).
ep_status stage_init(Stage &st, hipStream_t stream, size_t most);
void stage_free(Stage &st);

// Device to host; the arrays are complete after finish().  A call's output
// pointers may be null.
class StageOut {
public:
    explicit StageOut(Stage &st) : st_(st) {}
    // x[o] = src[k].x, y[o] = src[k].y with k = stored[o] for o < n_stored, else o
    // (stored may be null)
    ep_status pairs(const float2 *src, const int32_t *stored, int64_t n_stored, int64_t n, float *x, float *y);
    ep_status flat(const void *src, int64_t n, void *out);  // n words of 4 bytes
    ep_status finish();

private:
    struct Piece {
        float *dst[2] = {nullptr, nullptr};
        size_t n = 0;
        bool busy = false;
    };
    ep_status take();  // frees the next slot
    ep_status drain(int k);
    ep_status queued();
    Stage &st_;
    Piece piece_[2];
    int next_ = 0;
};

// Host to device; the host array is read before the call returns, the copy to
// the device is queued on the stage's stream.
ep_status stage_in(Stage &st, float *dst, const float *src, int64_t n);

// pos[k] = u[k] = clamp((x[o], y[o])) into the die for the stored cells k < n, o =
// order[k] for k < n_order (order may be null), else k; *flag is set when a
// coordinate is not finite.  All device arrays (flag may be pinned).
void launch_place_cells(const float *x, const float *y, const int32_t *order, int64_t n_order, const float2 *wh,
                        int64_t n, float4 die, float2 *pos, float2 *u, int32_t *flag, hipStream_t s);

}  // namespace ep
