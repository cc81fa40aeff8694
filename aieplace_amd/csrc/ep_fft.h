// ep_fft.h -- the field solve's FFT path (k_fft.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <vector>

namespace ep {

// Stages of an FFT whose length is no power of two (Stockham, radix r after a product
// ns of radices), with the reciprocals for the index divisions.
struct FftPlan {
    int stages;
    struct Stage {
        int r, ns;
        float inv_ns, inv_span;  // 1 / ns, 1 / (r ns)
    } st[8];
};

// One solve; every pointer is device memory.
struct FftArgs {
    const float *map;      // [Mx][My] density map
    const float *mean;     // its mean, subtracted
    const int32_t *skip;   // nonzero: the solve is skipped (finished run or instance)
    const float2 *tab_x, *tab_y;  // fft_table(Mx), fft_table(My)
    float *t1;             // scratch, Mx My floats
    float2 *pq;            // scratch, Mx My pairs
    float2 *exy;           // [Mx][My] field
    int Mx, My;
    float scale, wxs, wys;  // spectral scaling, as GemmArgs
    FftPlan px, py;         // fft_plan(Mx), fft_plan(My)
};

// What the overflow pass (k_overflow) does, done by the rows kernel as it reads the map:
// scatter accumulators -> maps, overflow numerator, accumulators and tile counts cleared.
struct FftMaps {
    unsigned long long *acc_field, *acc_mov;
    const float *map_fix;
    float *map_field, *map_mov;
    double unit;
    float rho_t, cap;
    double *part;        // overflow partials, [part_blocks] of four (the first is used)
    int part_blocks;     // at least fft_row_blocks; the rest is zeroed
    int32_t *count;      // sort counts and cursors
};

// Grid sides are multiples of 16.  The FFT path takes powers of two up to 8192 (the
// columns of two FFTs of 16384 points do not fit the LDS) and any other side up to
// 4080 (40 bytes of LDS per point in the columns kernel).
constexpr int kFftPow2Max = 8192, kFftMixedMax = 4080;
inline bool fft_pow2(int n) { return (n & (n - 1)) == 0; }
inline bool fft_side(int n) { return n >= 16 && n % 16 == 0 && n <= (fft_pow2(n) ? kFftPow2Max : kFftMixedMax); }

// Rows of 8192 points leave the overflow pass to its own kernel: their blocks of 1024
// threads hold 128 registers a thread and spill 31 beside the bins.  us per evaluation, in
// the rows / by itself: 16 x 8192 134 / 124 (100k cells), 64 x 8192 157 / 147, 1024 x 8192 4480 /
// 4400; 16 x 4096 105.7 / 104.7, 64 x 4096 106 / 106, 256 x 4096 141 / 143 (400k), 16 x 2048
// 89.5 / 89.6, 16 x 1008 78.5 / 81.8.
constexpr int kFftMapsMax = 4096;

// Constants of length-n transforms, made in FP64.
void fft_table(int n, std::vector<float2> &tab);
// Stages of a length that is no power of two (none for one that is).
FftPlan fft_plan(int n);
// Blocks of the rows kernel.
int fft_row_blocks(int Mx, int My);
// `maps`: the overflow pass goes with the rows (null: the map is there), which are no
// longer than kFftMapsMax.
void launch_field_fft(const FftArgs &a, const FftMaps *maps, hipStream_t s);

// Batched solves: one launch per stage (rows, columns, field) and class covers
// the tiles (instance, block of the instance's stage) of every instance.  The
// classes: powers of two up to 1024 and above (128 and 1024 threads), other sides.
constexpr int kFftClasses = 3;
struct FftBatchTiles {
    int2 *d[3];
    int n[3];
    int longest;  // side among the tiles' instances
};
int fft_class(int M);
// Appends instance i's tiles (side M) to the lists of its class.
void fft_batch_tiles(int i, int M, std::vector<int2> (&tiles)[kFftClasses][3]);
void launch_field_fft_batch(const FftArgs *args, const FftBatchTiles (&t)[kFftClasses], hipStream_t s);

}  // namespace ep
