// ep_fft.h -- the field solve's FFT path (k_fft.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <vector>

namespace ep {

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
};

// Grid sides that the FFT path takes: powers of two from 16 (the smallest grid)
// to 8192 (the columns of two FFTs of 16384 points do not fit the LDS).
inline bool fft_side(int n) { return n >= 16 && n <= 8192 && (n & (n - 1)) == 0; }

// Constants of length-n transforms (n a power of two), made in FP64.
void fft_table(int n, std::vector<float2> &tab);
void launch_field_fft(const FftArgs &a, hipStream_t s);

// Batched solves: one launch per stage (rows, columns, field) and class covers
// the tiles (instance, block of the instance's stage) of every instance.  The
// classes are block sizes: 128 threads for sides up to 1024, 1024 above.
constexpr int kFftClasses = 2;
struct FftBatchTiles {
    int2 *d[3];
    int n[3];
};
// Appends instance i's tiles (side M) to the lists of its class.
void fft_batch_tiles(int i, int M, std::vector<int2> (&tiles)[kFftClasses][3]);
void launch_field_fft_batch(const FftArgs *args, const FftBatchTiles (&t)[kFftClasses], hipStream_t s);

}  // namespace ep
