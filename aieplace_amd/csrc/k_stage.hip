// k_stage.hip -- kernels and pinned slots of the host transfers (ep_stage.h).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>

#include "ep_stage.h"

namespace ep {

namespace {

constexpr int kStageBlock = 256;

// One coalesced store per lane and coordinate straight into the pinned slot;
// bound by the link (50 GB/s), so the gather by `stored` costs nothing.
__global__ __launch_bounds__(kStageBlock) void k_unpack(const float2 *__restrict__ src,
                                                        const int32_t *__restrict__ stored, int64_t n_stored,
                                                        int64_t o0, int64_t m, float *__restrict__ x,
                                                        float *__restrict__ y)
{
    for (int64_t i = (int64_t)blockIdx.x * kStageBlock + threadIdx.x; i < m; i += (int64_t)gridDim.x * kStageBlock) {
        const int64_t o = o0 + i;
        const float2 v = src[stored && o < n_stored ? (int64_t)stored[o] : o];
        if (x) x[i] = v.x;
        if (y) y[i] = v.y;
    }
}

// n floats, whole float4s while they last where both ends are 16-byte aligned; one end is
// a slot.
__global__ __launch_bounds__(kStageBlock) void k_move(const float *__restrict__ src, int64_t n,
                                                      float *__restrict__ out)
{
    const int64_t t = (int64_t)blockIdx.x * kStageBlock + threadIdx.x, step = (int64_t)gridDim.x * kStageBlock;
    const int64_t v = (reinterpret_cast<uintptr_t>(src) | reinterpret_cast<uintptr_t>(out)) % 16 ? 0 : n / 4;
    for (int64_t i = t; i < v; i += step)
        reinterpret_cast<float4 *>(out)[i] = reinterpret_cast<const float4 *>(src)[i];
    for (int64_t i = v * 4 + t; i < n; i += step) out[i] = src[i];
}

__global__ __launch_bounds__(kStageBlock) void k_place_cells(const float *__restrict__ x, const float *__restrict__ y,
                                                             const int32_t *__restrict__ order, int64_t n_order,
                                                             const float2 *__restrict__ wh, int64_t n, float4 die,
                                                             float2 *__restrict__ pos, float2 *__restrict__ u,
                                                             int32_t *__restrict__ flag)
{
    const int64_t k = (int64_t)blockIdx.x * kStageBlock + threadIdx.x;
    if (k >= n) return;
    const int64_t o = order && k < n_order ? (int64_t)order[k] : k;
    const float px = x[o], py = y[o];
    const float2 s = wh[k];
    if (!isfinite(px) || !isfinite(py)) *flag = 1;  // every writer writes the same value
    const float2 p = make_float2(fminf(fmaxf(px, die.x), die.z - s.x), fminf(fmaxf(py, die.y), die.w - s.y));
    pos[k] = p;
    u[k] = p;
}

void launch_move(const float *src, int64_t n, float *out, hipStream_t s)
{
    hipLaunchKernelGGL(k_move, dim3((unsigned)((n / 4 + kStageBlock) / kStageBlock)), dim3(kStageBlock), 0, s, src, n,
                       out);
}

ep_status hip_ok(hipError_t e, const char *what)
{
    return e == hipSuccess ? EP_OK : fail(EP_EDEVICE, "%s: %s", what, hipGetErrorString(e));
}

}  // namespace

ep_status stage_init(Stage &st, hipStream_t stream, size_t most)
{
    st.stream = stream;
    st.bytes = std::min(kStageSlot, (std::max<size_t>(most, 256) + 255) / 256 * 256);
    char *p = nullptr;
    if (hipHostMalloc((void **)&p, 2 * st.bytes + 256, hipHostMallocDefault) != hipSuccess)
        return fail(EP_ENOMEM, "pinned host allocation failed");
    // the host's first touch of a megabyte's pages takes 110 us: here, not in the first transfer
    std::memset(p, 0, 2 * st.bytes + 256);
    st.pin[0] = p;
    st.pin[1] = p + st.bytes;
    st.flag = reinterpret_cast<int32_t *>(p + 2 * st.bytes);
    for (hipEvent_t &e : st.done)
        if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess)
            return fail(EP_EDEVICE, "event creation failed");
    return EP_OK;
}

void stage_free(Stage &st)
{
    for (hipEvent_t &e : st.done)
        if (e) (void)hipEventDestroy(e);
    if (st.pin[0]) (void)hipHostFree(st.pin[0]);
    st = Stage();
}

ep_status StageOut::drain(int k)
{
    Piece &p = piece_[k];
    if (!p.busy) return EP_OK;
    p.busy = false;
    ep_status s = hip_ok(hipEventSynchronize(st_.done[k]), "download");
    if (s != EP_OK) return s;
    const char *at = st_.pin[k];
    for (float *d : p.dst)
        if (d) {
            std::memcpy(d, at, p.n * sizeof(float));
            at += p.n * sizeof(float);
        }
    return EP_OK;
}

ep_status StageOut::take() { return drain(next_); }

ep_status StageOut::queued()
{
    ep_status s = hip_ok(hipGetLastError(), "download");
    // the end of a launch itself (hipExtLaunchKernel) as the event saves 2.5 us of a call,
    // but then the next work on another stream takes 100 us more
    if (s == EP_OK) s = hip_ok(hipEventRecord(st_.done[next_], st_.stream), "download");
    if (s != EP_OK) return s;
    piece_[next_].busy = true;
    next_ ^= 1;
    return EP_OK;
}

ep_status StageOut::pairs(const float2 *src, const int32_t *stored, int64_t n_stored, int64_t n, float *x, float *y)
{
    if (!x && !y) return EP_OK;
    const int64_t per = (int64_t)(st_.bytes / (2 * sizeof(float)));
    for (int64_t o = 0; o < n; o += per) {
        ep_status s = take();
        if (s != EP_OK) return s;
        const int64_t m = std::min(per, n - o);
        float *at = reinterpret_cast<float *>(st_.pin[next_]);
        float *px = x ? at : nullptr, *py = y ? (x ? at + m : at) : nullptr;
        const unsigned blocks = (unsigned)std::min<int64_t>((m + kStageBlock - 1) / kStageBlock, 1024);
        hipLaunchKernelGGL(k_unpack, dim3(blocks), dim3(kStageBlock), 0, st_.stream, src, stored, n_stored, o, m, px,
                           py);
        piece_[next_].dst[0] = x ? x + o : nullptr;
        piece_[next_].dst[1] = y ? y + o : nullptr;
        piece_[next_].n = (size_t)m;
        if ((s = queued()) != EP_OK) return s;
    }
    return EP_OK;
}

ep_status StageOut::flat(const void *from, int64_t n, void *to)
{
    const float *src = static_cast<const float *>(from);
    float *out = static_cast<float *>(to);
    if (!out) return EP_OK;
    const int64_t per = (int64_t)(st_.bytes / sizeof(float));
    for (int64_t o = 0; o < n; o += per) {
        ep_status s = take();
        if (s != EP_OK) return s;
        const int64_t m = std::min(per, n - o);
        float *pin = reinterpret_cast<float *>(st_.pin[next_]);
        if (n <= per) {
            // a kernel starts sooner than the copy engine (three maps of 128^2, 224^2, 480^2:
            // 92 / 104 / 186 us a call, 103 / 120 / 199 with copies), but chunks that follow
            // each other are slower with it (three of 1024^2: 826, 764 with copies)
            launch_move(src, m, pin, st_.stream);
        } else {
            s = hip_ok(hipMemcpyAsync(pin, src + o, (size_t)m * sizeof(float), hipMemcpyDeviceToHost, st_.stream),
                       "download");
            if (s != EP_OK) return s;
        }
        piece_[next_].dst[0] = out + o;
        piece_[next_].dst[1] = nullptr;
        piece_[next_].n = (size_t)m;
        if ((s = queued()) != EP_OK) return s;
    }
    return EP_OK;
}

ep_status StageOut::finish()
{
    ep_status s = drain(next_);  // the older of the two
    const ep_status t = drain(next_ ^ 1);
    return s != EP_OK ? s : t;
}

ep_status stage_in(Stage &st, float *dst, const float *src, int64_t n)
{
    const int64_t per = (int64_t)(st.bytes / sizeof(float));
    for (int64_t o = 0; o < n; o += per, st.up ^= 1) {
        const int64_t m = std::min(per, n - o);
        const int k = st.up;
        // the slot's last use, in this call or an earlier one
        ep_status s = hip_ok(hipEventSynchronize(st.done[k]), "upload");
        if (s != EP_OK) return s;
        std::memcpy(st.pin[k], src + o, (size_t)m * sizeof(float));
        if (n <= per) {
            launch_move(reinterpret_cast<const float *>(st.pin[k]), m, dst, st.stream);
            s = hip_ok(hipGetLastError(), "upload");
        } else {
            s = hip_ok(hipMemcpyAsync(dst + o, st.pin[k], (size_t)m * sizeof(float), hipMemcpyHostToDevice, st.stream),
                       "upload");
        }
        if (s == EP_OK) s = hip_ok(hipEventRecord(st.done[k], st.stream), "upload");
        if (s != EP_OK) return s;
    }
    return EP_OK;
}

void launch_place_cells(const float *x, const float *y, const int32_t *order, int64_t n_order, const float2 *wh,
                        int64_t n, float4 die, float2 *pos, float2 *u, int32_t *flag, hipStream_t s)
{
    hipLaunchKernelGGL(k_place_cells, dim3((unsigned)((n + kStageBlock - 1) / kStageBlock)), dim3(kStageBlock), 0, s, x,
                       y, order, n_order, wh, n, die, pos, u, flag);
}

}  // namespace ep
