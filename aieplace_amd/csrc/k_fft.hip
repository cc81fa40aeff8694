// k_fft.hip -- Poisson field solve as FP32 FFTs in LDS.
//
// The same field as the transform products of k_field.hip (RePlAce scaling,
// python/AIEmath/fft_replace/fft.cpp:118-212), in three kernels instead of four:
//   rows     T1[i][v] = sum_j cos(pi v (j+1/2)/My) (rho[i][j] - mean)       every row i
//   columns  A[u][v]  = sum_i cos(pi u (i+1/2)/Mx) T1[i][v] -> spectral scaling ->
//            P[i][v] = sum_u A wx/k^2 sin(pi u (i+1/2)/Mx),
//            Q[i][v] = sum_u A wy/k^2 cos(pi u (i+1/2)/Mx)                  every column v
//   fields   Ex[i][j] = sum_v P[i][v] cos(pi v (j+1/2)/My),
//            Ey[i][j] = sum_v Q[i][v] sin(pi v (j+1/2)/My)                  every row i
// The x transform, the scaling and the inverse x transforms of one column stay
// in LDS.  A real transform of length N is half of an N-point complex FFT
// (J. Makhoul, "A fast cosine transform in one and two dimensions", 1980): with
// z[n] = x[2n], z[N-1-n] = x[2n+1], the DCT is C[k] = Re(e^{-i pi k/2N} Z[k]).
// Two real rows (or columns) share one complex FFT as its real and imaginary
// part; in the inverse direction P and Q do, so the last kernel's complex
// output is the interleaved field itself.  The sine sums are cosine sums of the
// reversed spectrum with alternating sign.
//
// Why FFTs: the products execute 6.4 GFLOP per 1024^2 solve, the FFTs 0.16 GFLOP
// over 36 MB of L2/MALL traffic.  One solve alone, FP32 products -> FFTs: 32^2
// 14.8 -> 9.2 us, 128^2 23.6 -> 14.9, 256^2 31.5 -> 15.3, 512^2 48 -> 17.5, 1024^2
// 108 -> 32 (split-BF16 products 72), 2048^2 585 -> 70; max-norm error at most
// 5e-7 (products: FP32 3e-6, split-BF16 1.1e-5).  What bounds them is latency:
// one wave per SIMD at 1024^2, where a kernel without its butterflies takes 5-10
// us, without its stores 1.5-3 us less, and with free twiddles or LDS exchanges
// about 1.5 us less each.  The columns' second half of threads (H = 2) takes them
// from 7.1 to 6.5 us at 256^2; at 1024^2 it changes nothing.  Padding the layout
// groups against channel conflicts changed nothing either.
//
// Layout of T1 (float) and PQ (float2): [v/4][i][v%4].  The column kernel reads
// and writes whole runs; a block of the row kernels touches two consecutive
// rows, runs of 32 and 64 bytes of lines that the XCD's next blocks complete.
#include <hip/hip_runtime.h>

#include <cmath>
#include <vector>

#include "ep_device.h"
#include "ep_fft.h"

// Multiply-adds only where they are written: the single and the batched kernels
// then round alike, so a batch reproduces its instances' own runs bit for bit.
#pragma clang fp contract(off)

namespace ep {

namespace {

constexpr float kSqrtHalf = 0.70710678118654752f;

// Radix of stage s of a 2^l-point FFT: 8, then one or two stages of 4 where 3
// does not divide l (8 4 4 has as many stages as 8 8 2 and fewer operations).
constexpr int radix_of(int l, int s) { return s < (l - 2 * ((3 - l % 3) % 3)) / 3 ? 8 : 4; }

// Stockham plan of a 2^L-point FFT with eight points per thread.
template <int L>
struct Plan {
    static constexpr int N = 1 << L, T = N / 8;  // points, threads
    static constexpr int stages = (L + 2) / 3;
    static constexpr int radix(int s) { return radix_of(L, s); }
    static constexpr int ns(int s) { return s == 0 ? 1 : ns(s - 1) * radix(s - 1); }  // product of the radices before s
    // twiddles of stage s: (radix - 1) * ns values, after those of the stages before
    static constexpr int tw_off(int s) { return s <= 1 ? 0 : tw_off(s - 1) + (radix(s - 1) - 1) * ns(s - 1); }
    static constexpr int buf = N + N / 8;  // LDS points with padding
};

// LDS slot of point i: one spare slot per eight keeps the strided stage writes
// (runs of eight points per thread) off each other's banks.
__device__ inline int slot(int i) { return i + (i >> 3); }

__device__ inline float2 cadd(float2 a, float2 b) { return make_float2(a.x + b.x, a.y + b.y); }
__device__ inline float2 csub(float2 a, float2 b) { return make_float2(a.x - b.x, a.y - b.y); }
// a * w, or a * conj(w)
template <bool INV>
__device__ inline float2 cmul(float2 a, float2 w)
{
    const float s = INV ? -w.y : w.y;
    return make_float2(fmaf(a.x, w.x, -(a.y * s)), fmaf(a.x, s, a.y * w.x));
}
// a * (-i), or a * i
template <bool INV>
__device__ inline float2 crot(float2 a)
{
    return INV ? make_float2(-a.y, a.x) : make_float2(a.y, -a.x);
}

template <bool INV>
__device__ inline void bfly2(float2 &a, float2 &b)
{
    const float2 t = a;
    a = cadd(t, b);
    b = csub(t, b);
}

template <bool INV>
__device__ inline void bfly4(float2 &a, float2 &b, float2 &c, float2 &d)
{
    bfly2<INV>(a, c);
    bfly2<INV>(b, d);
    d = crot<INV>(d);
    bfly2<INV>(a, b);
    bfly2<INV>(c, d);
    const float2 t = b;  // natural order
    b = c;
    c = t;
}

template <bool INV>
__device__ inline void bfly8(float2 (&v)[8])
{
    bfly4<INV>(v[0], v[2], v[4], v[6]);
    bfly4<INV>(v[1], v[3], v[5], v[7]);
    const float h = kSqrtHalf;
    // odd half times e^{-+ i pi r / 4}
    v[3] = cmul<INV>(v[3], make_float2(h, -h));
    v[5] = crot<INV>(v[5]);
    v[7] = cmul<INV>(v[7], make_float2(-h, -h));
    bfly2<INV>(v[0], v[1]);
    bfly2<INV>(v[2], v[3]);
    bfly2<INV>(v[4], v[5]);
    bfly2<INV>(v[6], v[7]);
    // v[0..7] = X0 X4 X1 X5 X2 X6 X3 X7
    float2 x[8] = {v[0], v[2], v[4], v[6], v[1], v[3], v[5], v[7]};
#pragma unroll
    for (int r = 0; r < 8; ++r) v[r] = x[r];
}

// A thread's twiddles: the stages' (slots of stage s from 7 (s - 1) on) and the
// half-sample shifts e^{-i pi k/2N} of its k = t + m T.
template <int L>
struct Twiddles {
    float2 st[7 * (Plan<L>::stages > 1 ? Plan<L>::stages - 1 : 1)];
    float2 half[4];
};

// Table layout: N/2 half-sample shifts, then the stages' twiddles (r - 1, k).
template <int L>
__device__ inline void load_twiddles(const float2 *__restrict__ tab, int t, Twiddles<L> &w)
{
    using P = Plan<L>;
#pragma unroll
    for (int m = 0; m < 4; ++m) w.half[m] = tab[t + m * P::T];
    const float2 *__restrict__ st = tab + P::N / 2;
#pragma unroll
    for (int s = 1; s < P::stages; ++s) {
        const int R = P::radix(s), ns = P::ns(s), nb = 8 / R;
#pragma unroll
        for (int b = 0; b < nb; ++b) {
            const int k = (t + b * P::T) & (ns - 1);
#pragma unroll
            for (int r = 1; r < R; ++r) w.st[7 * (s - 1) + b * (R - 1) + r - 1] = st[P::tw_off(s) + (r - 1) * ns + k];
        }
    }
}

// Registers -> LDS in natural order, visible to the block.
template <int L>
__device__ inline void put_points(const float2 (&v)[8], float2 *buf, int t)
{
#pragma unroll
    for (int m = 0; m < 8; ++m) buf[slot(t + m * Plan<L>::T)] = v[m];
}

template <int L>
__device__ inline void get_points(float2 (&v)[8], const float2 *buf, int t)
{
#pragma unroll
    for (int m = 0; m < 8; ++m) v[m] = buf[slot(t + m * Plan<L>::T)];
}

// C complex FFTs at once (their stages share the barriers): in and out,
// v[c][m] is point t + m T of FFT c; buf[c] is its LDS, whose content the
// block may still be reading on entry.  A thread without `on` only takes part
// in the barriers.
template <int L, bool INV, int C>
__device__ inline void fft(float2 (&v)[C][8], const Twiddles<L> &w, float2 *const *buf, int t, bool on = true)
{
    using P = Plan<L>;
#pragma unroll
    for (int s = 0; s < P::stages; ++s) {
        const int R = P::radix(s), ns = P::ns(s), nb = 8 / R;
#pragma unroll
        for (int c = 0; c < C; ++c) {
            if (!on) break;
            if (s > 0)
#pragma unroll
                for (int b = 0; b < nb; ++b)
#pragma unroll
                    for (int r = 1; r < R; ++r)
                        v[c][b + r * nb] = cmul<INV>(v[c][b + r * nb], w.st[7 * (s - 1) + b * (R - 1) + r - 1]);
            if (R == 8) bfly8<INV>(v[c]);
            else
#pragma unroll
                for (int b = 0; b < 2; ++b) bfly4<INV>(v[c][b], v[c][b + 2], v[c][b + 4], v[c][b + 6]);
        }
        if (s + 1 < P::stages) {
            __syncthreads();
#pragma unroll
            for (int c = 0; c < C; ++c)
#pragma unroll
                for (int b = 0; b < nb && on; ++b) {
                    const int j = t + b * P::T, k = j & (ns - 1), o = (j - k) * R + k;
#pragma unroll
                    for (int r = 0; r < R; ++r) buf[c][slot(o + r * ns)] = v[c][b + r * nb];
                }
            __syncthreads();
#pragma unroll
            for (int c = 0; c < C; ++c)
                if (on) get_points<L>(v[c], buf[c], t);
        }
    }
}

// DCT values k and N - k of the two real sequences packed in Z, for 0 < k < N/2
// (w = e^{-i pi k/2N}).
struct DctPair {
    float a_k, a_n, b_k, b_n;
};
__device__ inline DctPair dct_pair(float2 zk, float2 zn, float2 w)
{
    const float c = w.x, s = -w.y;
    const float ax = 0.5f * (zk.x + zn.x), ay = 0.5f * (zk.y - zn.y);
    const float bx = 0.5f * (zk.y + zn.y), by = 0.5f * (zn.x - zk.x);
    return {fmaf(c, ax, s * ay), fmaf(s, ax, -(c * ay)), fmaf(c, bx, s * by), fmaf(s, bx, -(c * by))};
}

// Spectrum points k and N - k of the complex inverse FFT whose real and
// imaginary parts are the cosine sums of a and b, for 0 < k < N/2.
__device__ inline void idct_pair(float a_k, float a_n, float b_k, float b_n, float2 w, float2 &zk, float2 &zn)
{
    const float c = w.x, s = -w.y;
    const float p = fmaf(c, a_k, s * a_n), q = fmaf(s, a_k, -(c * a_n));
    const float r = fmaf(c, b_k, s * b_n), u = fmaf(s, b_k, -(c * b_n));
    zk = make_float2(0.5f * (p - u), 0.5f * (q + r));
    zn = make_float2(0.5f * (p + u), 0.5f * (r - q));
}

// FFTs per block: one where that is a wave or more, so that a 512^2 map occupies every
// CU; neighbouring blocks, which share the layout groups' cache lines, then go to one
// XCD.  One solve with two FFTs per block and four rows per field block / as now: 512^2
// 18.7 / 17.5 us, 1024^2 32.9 / 32.0, 2048^2 81 / 70.
template <int L>
constexpr int ffts_of()
{
    return Plan<L>::T >= 64 ? 1 : Plan<L>::T >= 32 ? 2 : 64 / Plan<L>::T;
}
template <int L>
__device__ inline int fft_block()
{
    return Plan<L>::T >= 64 ? dev::xcd_block(blockIdx.x, gridDim.x) : blockIdx.x;
}
// The column kernel's threads per FFT point set (see columns_pass).
template <int L>
constexpr int col_halves_of()
{
    return Plan<L>::T >= 1024 ? 1 : 2;
}
// The last kernel's: one row each, so two (four of 128).
template <int L>
constexpr int field_ffts_of()
{
    return Plan<L>::T >= 1024 ? 1 : Plan<L>::T >= 32 ? 2 : Plan<L>::T >= 16 ? 4 : 64 / Plan<L>::T;
}

// Bins o and o + 1 of the map (o even) from their accumulators, which are cleared; adds
// their overflow.  Bins of a row that is another block's (`mine` unset) are only read.
struct MapBins {
    ulonglong2 field, mov;
    float2 fix;
};
__device__ inline MapBins load_bins(const FftMaps &mp, size_t o)
{
    return {*reinterpret_cast<const ulonglong2 *>(mp.acc_field + o), *reinterpret_cast<const ulonglong2 *>(mp.acc_mov + o),
            *reinterpret_cast<const float2 *>(mp.map_fix + o)};
}
__device__ inline float2 store_bins(const FftMaps &mp, size_t o, const MapBins &b, bool mine, double &ovf)
{
    const float2 fd = make_float2(dev::field_bin(b.fix.x, b.field.x, mp.unit, mp.rho_t),
                                  dev::field_bin(b.fix.y, b.field.y, mp.unit, mp.rho_t));
    const float2 mv = make_float2(dev::mov_bin(b.mov.x, mp.unit), dev::mov_bin(b.mov.y, mp.unit));
    if (mine) {
        const ulonglong2 zero = {0ull, 0ull};
        *reinterpret_cast<ulonglong2 *>(mp.acc_field + o) = zero;
        *reinterpret_cast<ulonglong2 *>(mp.acc_mov + o) = zero;
        *reinterpret_cast<float2 *>(mp.map_mov + o) = mv;
        *reinterpret_cast<float2 *>(mp.map_field + o) = fd;
        ovf += fmax((double)dev::ovf_bin(mv.x, b.fix.x, mp.rho_t, mp.cap), 0.0);
        ovf += fmax((double)dev::ovf_bin(mv.y, b.fix.y, mp.rho_t, mp.cap), 0.0);
    }
    return fd;
}
// The tile counts, and the overflow partials of the launch (NT threads per block).
template <int NT>
__device__ inline void finish_maps(const FftMaps &mp, int blk, int blocks, double ovf)
{
    for (int t = blk * NT + (int)threadIdx.x; t < 2 * kSortTiles; t += blocks * NT) mp.count[t] = 0;
    for (int p = blocks + blk * NT + (int)threadIdx.x; p < mp.part_blocks; p += blocks * NT) mp.part[4 * p] = 0.0;
    double v[1] = {ovf};
    dev::block_reduce<1, 0, NT>(v, mp.part + 4 * blk);
}

// Rows 2 F blk ... of the map (row length N, `rows` rows, an even number).
// F * T threads, F * buf points of LDS.  With MAPS the map is made on the way.
template <int L, int F, bool MAPS>
__device__ inline void rows_pass(const FftArgs &a, const FftMaps &mp, int blk, float2 *lds)
{
    using P = Plan<L>;
    constexpr int N = P::N, T = P::T;
    const int f = threadIdx.x / T, t = threadIdx.x % T, rows = a.Mx;
    const int r0 = min((blk * F + f) * 2, rows - 2);
    const float2 *__restrict__ x0 = reinterpret_cast<const float2 *>(a.map + (size_t)r0 * N);
    const float2 *__restrict__ x1 = x0 + N / 2;
    float2 *buf = lds + f * P::buf;
    const int halt = *a.skip;
    const float mean = *a.mean;
    float2 xa[4], xb[4];
    [[maybe_unused]] MapBins ma[4], mb[4];
#pragma unroll
    for (int m = 0; m < 4; ++m) {
        if constexpr (MAPS) {
            const size_t o = (size_t)r0 * N + 2 * (t + m * T);
            ma[m] = load_bins(mp, o);
            mb[m] = load_bins(mp, o + N);
        } else {
            xa[m] = x0[t + m * T];
            xb[m] = x1[t + m * T];
        }
    }
    Twiddles<L> w;
    if constexpr (!MAPS) load_twiddles<L>(a.tab_y, t, w);
    if (halt) return;
    [[maybe_unused]] double ovf = 0.0;
    if constexpr (MAPS) {
        const bool mine = (blk * F + f) * 2 < rows;
#pragma unroll
        for (int m = 0; m < 4; ++m) {
            const size_t o = (size_t)r0 * N + 2 * (t + m * T);
            xa[m] = store_bins(mp, o, ma[m], mine, ovf);
            xb[m] = store_bins(mp, o + N, mb[m], mine, ovf);
        }
        // not before: with the bins' registers they would not fit (256 and spills)
        __builtin_amdgcn_sched_barrier(0);
        load_twiddles<L>(a.tab_y, t, w);
    }
#pragma unroll
    for (int m = 0; m < 4; ++m) {
        const int n = t + m * T;
        buf[slot(n)] = make_float2(xa[m].x - mean, xb[m].x - mean);
        buf[slot(N - 1 - n)] = make_float2(xa[m].y - mean, xb[m].y - mean);
    }
    __syncthreads();
    float2 v[1][8];
    float2 *const bufs[1] = {buf};
    get_points<L>(v[0], buf, t);
    fft<L, false, 1>(v, w, bufs, t);
    __syncthreads();
    put_points<L>(v[0], buf, t);
    __syncthreads();
#pragma unroll
    for (int m = 0; m < 4; ++m) {
        const int k = t + m * T;
        if (k == 0) {  // and N/2
            const float2 h = buf[slot(N / 2)];
            buf[slot(N / 2)] = make_float2(h.x * kSqrtHalf, h.y * kSqrtHalf);
        } else {
            const DctPair d = dct_pair(buf[slot(k)], buf[slot(N - k)], w.half[m]);
            buf[slot(k)] = make_float2(d.a_k, d.b_k);
            buf[slot(N - k)] = make_float2(d.a_n, d.b_n);
        }
    }
    __syncthreads();
    // four columns of one row per store; consecutive lanes take the block's rows
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int e = threadIdx.x + q * F * T, r = e % (2 * F), g = e / (2 * F);
        const int row = blk * 2 * F + r;
        const float2 *b = lds + (r >> 1) * P::buf;
        float o[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const float2 z = b[slot(4 * g + c)];
            o[c] = (r & 1) ? z.y : z.x;
        }
        if (row < rows)
            *reinterpret_cast<float4 *>(a.t1 + ((size_t)g * rows + row) * 4) = make_float4(o[0], o[1], o[2], o[3]);
    }
    if constexpr (MAPS) finish_maps<F * T>(mp, blk, gridDim.x, ovf);
}

// One value of the spectral scaling: A -> (A wx / k^2, A wy / k^2), the halved
// weights of u = 0 and v = 0 included; the mean (u = v = 0) carries no field.
__device__ inline float2 spectral(const FftArgs &a, int u, int v, float A)
{
    float val = A * a.scale;
    if (u == 0) val *= 0.5f;
    if (v == 0) val *= 0.5f;
    const float wx = a.wxs * (float)u, wy = a.wys * (float)v;
    const float p = (u == 0 && v == 0) ? 0.0f : val / fmaf(wx, wx, wy * wy);
    return make_float2(p * wx, p * wy);
}

// Columns 2 F blk ... (column length N, `cols` columns, a multiple of 16).
// H * F * T threads, 2 F * buf points of LDS.  With H = 2 a second half of the
// threads takes the second column of every pair from the spectral scaling on
// (one inverse FFT per thread group), with H = 1 each thread does both.
template <int L, int F, int H>
__device__ inline void columns_pass(const FftArgs &a, int blk, float2 *lds)
{
    using P = Plan<L>;
    constexpr int N = P::N, T = P::T, C = 2 / H;  // C: columns per thread after the forward FFT
    const int h = H == 1 ? 0 : threadIdx.x / (F * T), id = threadIdx.x - h * F * T;
    const int f = id / T, t = id % T, cols = a.My;
    const int col = (blk * F + f) * 2, ca = min(col, cols - 2);
    float2 *b0 = lds + 2 * f * P::buf, *b1 = b0 + P::buf;
    const int halt = *a.skip;
    const size_t at = (size_t)(ca >> 2) * N * 4 + (ca & 3);
    float2 x[8 / H];
#pragma unroll
    for (int m = 0; m < 8 / H; ++m)
        x[m] = *reinterpret_cast<const float2 *>(a.t1 + at + (size_t)(t + (H * m + h) * T) * 4);
    Twiddles<L> w;
    load_twiddles<L>(a.tab_x, t, w);
    if (halt) return;
#pragma unroll
    for (int m = 0; m < 8 / H; ++m) {
        const int i = t + (H * m + h) * T;
        b0[slot((i & 1) ? N - 1 - (i >> 1) : i >> 1)] = x[m];
    }
    __syncthreads();
    {
        float2 v[1][8] = {};
        float2 *const bufs[1] = {b0};
        const bool on = h == 0;
        if (on) get_points<L>(v[0], b0, t);
        fft<L, false, 1>(v, w, bufs, t, on);
        __syncthreads();
        if (on) put_points<L>(v[0], b0, t);
        __syncthreads();
    }
    // DCT values, their spectral scaling and the inverse FFTs' inputs.  Points k
    // and N - k of a column belong to one thread; the first column's inputs
    // replace the DCT values.
    float2 ik[C][4], in[C][4];
#pragma unroll
    for (int m = 0; m < 4; ++m) {
        const int k = t + m * T;
        const float2 zk = b0[slot(k)], zn = b0[slot(k == 0 ? N / 2 : N - k)];
#pragma unroll
        for (int c = 0; c < C; ++c) {
            const bool second = H == 1 ? c == 1 : h == 1;
            const int v = ca + (second ? 1 : 0);
            if (k == 0) {  // and N/2
                const float2 e = spectral(a, 0, v, second ? zk.y : zk.x);
                const float2 q = spectral(a, N / 2, v, (second ? zn.y : zn.x) * kSqrtHalf);
                ik[c][m] = make_float2(0.0f, e.y);
                in[c][m] = make_float2(q.x * kSqrtHalf, q.y * kSqrtHalf);
            } else {
                const DctPair d = dct_pair(zk, zn, w.half[m]);
                const float2 ek = spectral(a, k, v, second ? d.b_k : d.a_k);
                const float2 en = spectral(a, N - k, v, second ? d.b_n : d.a_n);
                idct_pair(en.x, ek.x, ek.y, en.y, w.half[m], ik[c][m], in[c][m]);  // sine sum: reversed spectrum
            }
        }
    }
    if (H == 2) __syncthreads();  // both halves have read the DCT values
#pragma unroll
    for (int c = 0; c < C; ++c) {
        float2 *b = (H == 1 ? c : h) ? b1 : b0;
#pragma unroll
        for (int m = 0; m < 4; ++m) {
            const int k = t + m * T;
            b[slot(k)] = ik[c][m];
            b[slot(k == 0 ? N / 2 : N - k)] = in[c][m];
        }
    }
    __syncthreads();
    float2 v[C][8];
    float2 *bufs[C];
#pragma unroll
    for (int c = 0; c < C; ++c) {
        bufs[c] = (H == 1 ? c : h) ? b1 : b0;
        get_points<L>(v[c], bufs[c], t);
    }
    fft<L, true, C>(v, w, bufs, t);
    __syncthreads();
#pragma unroll
    for (int c = 0; c < C; ++c) put_points<L>(v[c], bufs[c], t);
    __syncthreads();
    if (col < cols)
#pragma unroll
        for (int m = 0; m < 8 / H; ++m) {
            const int i = t + (H * m + h) * T, n = (i & 1) ? N - 1 - (i >> 1) : i >> 1;
            const float2 z0 = b0[slot(n)], z1 = b1[slot(n)];
            const float sg = (i & 1) ? -1.0f : 1.0f;
            *reinterpret_cast<float4 *>(a.pq + at + (size_t)i * 4) = make_float4(sg * z0.x, z0.y, sg * z1.x, z1.y);
        }
}

// Rows F blk ... of the field (row length N, `rows` rows).  F * T threads,
// F * buf points of LDS.
template <int L, int F>
__device__ inline void field_pass(const FftArgs &a, int blk, float2 *lds)
{
    using P = Plan<L>;
    constexpr int N = P::N, T = P::T;
    const int f = threadIdx.x / T, t = threadIdx.x % T, rows = a.Mx;
    float2 *buf = lds + f * P::buf;
    const int halt = *a.skip;
    // two columns of one row per load; consecutive lanes take the block's rows
    float4 x[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int e = threadIdx.x + q * F * T, r = (e >> 1) % F, g = (e >> 1) / F;
        const int row = min(blk * F + r, rows - 1);
        x[q] = *reinterpret_cast<const float4 *>(a.pq + ((size_t)g * rows + row) * 4 + 2 * (e & 1));
    }
    Twiddles<L> w;
    load_twiddles<L>(a.tab_y, t, w);
    if (halt) return;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int e = threadIdx.x + q * F * T, r = (e >> 1) % F, k = (e >> 1) / F * 4 + 2 * (e & 1);
        float2 *b = lds + r * P::buf;
        b[slot(k)] = make_float2(x[q].x, x[q].y);
        b[slot(k + 1)] = make_float2(x[q].z, x[q].w);
    }
    __syncthreads();
#pragma unroll
    for (int m = 0; m < 4; ++m) {
        const int k = t + m * T;
        if (k == 0) {  // and N/2
            const float2 h = buf[slot(N / 2)];
            buf[slot(0)] = make_float2(buf[slot(0)].x, 0.0f);
            buf[slot(N / 2)] = make_float2(h.x * kSqrtHalf, h.y * kSqrtHalf);
        } else {
            const float2 ek = buf[slot(k)], en = buf[slot(N - k)];
            float2 zk, zn;
            idct_pair(ek.x, en.x, en.y, ek.y, w.half[m], zk, zn);
            buf[slot(k)] = zk;
            buf[slot(N - k)] = zn;
        }
    }
    __syncthreads();
    float2 v[1][8];
    float2 *const bufs[1] = {buf};
    get_points<L>(v[0], buf, t);
    fft<L, true, 1>(v, w, bufs, t);
    __syncthreads();
    put_points<L>(v[0], buf, t);
    __syncthreads();
    const int row = blk * F + f;
    if (row < rows)
#pragma unroll
        for (int m = 0; m < 4; ++m) {
            const int n = t + m * T;
            const float2 z0 = buf[slot(n)], z1 = buf[slot(N - 1 - n)];
            *reinterpret_cast<float4 *>(a.exy + (size_t)row * N + 2 * n) = make_float4(z0.x, z0.y, z1.x, -z1.y);
        }
}

extern __shared__ __attribute__((aligned(16))) float2 fft_lds[];

template <int L, bool MAPS>
__global__ __launch_bounds__(ffts_of<L>() * Plan<L>::T) void k_fft_rows(FftArgs a, FftMaps mp)
{
    rows_pass<L, ffts_of<L>(), MAPS>(a, mp, fft_block<L>(), fft_lds);
}
template <int L>
__global__ __launch_bounds__(col_halves_of<L>() * ffts_of<L>() * Plan<L>::T) void k_fft_columns(FftArgs a)
{
    columns_pass<L, ffts_of<L>(), col_halves_of<L>()>(a, fft_block<L>(), fft_lds);
}
template <int L>
__global__ __launch_bounds__(field_ffts_of<L>() * Plan<L>::T) void k_fft_field(FftArgs a)
{
    field_pass<L, field_ffts_of<L>()>(a, fft_block<L>(), fft_lds);
}

// ------------------------------------------------------------------ other lengths
// Lengths that are no power of two: the same three passes over a plan of stages, the odd
// factors first, then radices 8 and 4.  A long odd radix is a plain sum (61 is a plan like
// 3 is), and a block's threads share every stage's points, so that a length of 240 keeps
// eight waves busy.  One solve alone in us, products (FP32 / split BF16 / split FP16) -> FFTs:
// 48^2 17.8 / 16.0 / 23.0 -> 14.8, 96 x 80 23.3 / 19.6 / 26.0 -> 15.9, 400 x 240 37.3 /
// 29.1 / 34.6 -> 18.8, 544^2 (17) 54 / 46 / 52 -> 24, 976^2 (61) 105 / 82 / 92 -> 43, 1008^2
// 104 / 75 / 89 -> 44, 2000^2 588 / 497 / 560 -> 144; max-norm error at most 9e-7 (products:
// 7e-6 / 1.4e-5 / 1.8e-6).  Small sides are bound by latency (a barrier and an LDS round
// trip per stage), large ones by LDS bandwidth.  512 threads: 256 and 1024 take 20.2 and
// 18.7 at 400 x 240 (512: 19.3), 55 and 56 at 976^2 (49).

// o / d for 0 <= o < 2^12 and inv = 1 / d rounded: (o + 1/2) / d is further from a whole
// number than its error.
__device__ inline int quotient(int o, float inv) { return (int)(((float)o + 0.5f) * inv); }

constexpr int kMixedThreads = 512;

// First stage, r odd, ns = 1, so no twiddles: outputs q and r - q of a butterfly share the
// sums of cosines and sines over the pairs (i, r - i).  Lanes run over the butterflies:
// they read consecutive points and the same root (one output per item and lanes over the
// outputs, which reads the roots with bank conflicts, took 203 us for 61 at 976^2).
template <bool INV, int R>
__device__ __forceinline__ void mixed_first(const float2 *__restrict__ in, float2 *__restrict__ out, const float2 *root, int N,
                                   int C, int r_any)
{
    const int r = R ? R : r_any, half = (r - 1) / 2, jump = N / r, items = jump * (half + 1);
    const float inv = 1.0f / (float)jump;
    for (int e = threadIdx.x; e < C * items; e += blockDim.x) {
        const int c = e >= items ? 1 : 0, w = e - c * items;
        const int q = quotient(w, inv), g = w - q * jump;
        const float2 *x = in + c * N + g;
        float2 cs = x[0], sn = make_float2(0.0f, 0.0f);
        int k = 0;
        auto pair = [&](int i) {
            k += q;
            k -= k >= r ? r : 0;
            const float2 a = x[i * jump], b = x[(r - i) * jump], t = root[k * jump];  // (cos, -sin)
            cs = make_float2(fmaf(t.x, a.x + b.x, cs.x), fmaf(t.x, a.y + b.y, cs.y));
            sn = make_float2(fmaf(t.y, a.x - b.x, sn.x), fmaf(t.y, a.y - b.y, sn.y));
        };
        if (R) {
#pragma unroll
            for (int i = 1; i <= (R - 1) / 2; ++i) pair(i);
        } else {
#pragma unroll 4
            for (int i = 1; i <= half; ++i) pair(i);
        }
        const float2 d = INV ? make_float2(sn.y, -sn.x) : make_float2(-sn.y, sn.x);
        float2 *y = out + c * N + g * r;
        y[q] = cadd(cs, d);
        if (q) y[r - q] = csub(cs, d);
    }
}

// The same with a long radix, outputs 2 p and 2 p + 1 per item: they share the sums and
// differences of a pair, so that LDS, which bounds the stage, is read four times for two
// terms and not six.  Same operations per output.  One and two outputs per item, us per
// solve: 4016 x 16 (251) 114 / 92 (split-BF16 products 107), 4016^2 1690 / 1317, 2032^2
// (127) 191 / 162, 1808^2 (113) 169 / 164.
template <bool INV>
__device__ __forceinline__ void mixed_first_two(const float2 *__restrict__ in, float2 *__restrict__ out,
                                                const float2 *root, int N, int C, int r)
{
    const int half = (r - 1) / 2, jump = N / r, items = jump * (half / 2 + 1);
    const float inv = 1.0f / (float)jump;
    for (int e = threadIdx.x; e < C * items; e += blockDim.x) {
        const int c = e >= items ? 1 : 0, w = e - c * items;
        const int p = quotient(w, inv), g = w - p * jump;
        const float2 *x = in + c * N + g;
        float2 cs[2] = {x[0], x[0]}, sn[2] = {};
        int k[2] = {0, 0};
#pragma unroll 4
        for (int i = 1; i <= half; ++i) {
            const float2 a = x[i * jump], b = x[(r - i) * jump];
#pragma unroll
            for (int o = 0; o < 2; ++o) {
                k[o] += 2 * p + o;
                k[o] -= k[o] >= r ? r : 0;
                const float2 t = root[k[o] * jump];  // (cos, -sin)
                cs[o] = make_float2(fmaf(t.x, a.x + b.x, cs[o].x), fmaf(t.x, a.y + b.y, cs[o].y));
                sn[o] = make_float2(fmaf(t.y, a.x - b.x, sn[o].x), fmaf(t.y, a.y - b.y, sn[o].y));
            }
        }
        float2 *y = out + c * N + g * r;
#pragma unroll
        for (int o = 0; o < 2; ++o) {
            const int q = 2 * p + o;
            if (q > half) break;
            const float2 d = INV ? make_float2(sn[o].y, -sn[o].x) : make_float2(-sn[o].y, sn[o].x);
            y[q] = cadd(cs[o], d);
            if (q) y[r - q] = csub(cs[o], d);
        }
    }
}

// A later stage with an odd radix: point o = (j / ns) r ns + j % ns + q ns is the sum over
// i < r of in[j + i N/r] e^{-2 pi i (o mod r ns) i / (r ns)}, one point per item.
template <bool INV, int R>
__device__ __forceinline__ void mixed_stage(const float2 *__restrict__ in, float2 *__restrict__ out,
                                            const float2 *root, int N, int C, int r_any, const FftPlan::Stage &st)
{
    const int r = R ? R : r_any, span = r * st.ns, step = N / span, jump = N / r;
    for (int e = threadIdx.x; e < C * N; e += blockDim.x) {
        const int c = e >= N ? 1 : 0, o = e - c * N;
        const int g = quotient(o, st.inv_span), m = o - g * span;
        const int k = m - quotient(m, st.inv_ns) * st.ns;
        const float2 *x = in + c * N + g * st.ns + k;
        const int turn = m * step;  // < N
        float2 acc = x[0];
        int w = 0;
        auto term = [&](int i) {
            w += turn;
            w -= w >= N ? N : 0;
            const float2 z = x[i * jump], t = root[w];
            const float s = INV ? -t.y : t.y;
            acc = make_float2(fmaf(-z.y, s, fmaf(z.x, t.x, acc.x)), fmaf(z.y, t.x, fmaf(z.x, s, acc.y)));
        };
        if (R) {
#pragma unroll
            for (int i = 1; i < R; ++i) term(i);
        } else {
#pragma unroll 4
            for (int i = 1; i < r; ++i) term(i);
        }
        out[e] = acc;
    }
}

// A later stage of radix 4 or 8: one butterfly per item (one output per item: 47.5 us at
// 976^2, 20.5 at 480 x 352; 43.0 and 19.0 so).
template <bool INV, int R>
__device__ __forceinline__ void mixed_butterflies(const float2 *__restrict__ in, float2 *__restrict__ out,
                                                  const float2 *root, int N, int C, const FftPlan::Stage &st)
{
    const int jump = N / R, step = jump / st.ns;
    for (int e = threadIdx.x; e < C * jump; e += blockDim.x) {
        const int c = e >= jump ? 1 : 0, j = e - c * jump, k = j - quotient(j, st.inv_ns) * st.ns;
        float2 v[R];
#pragma unroll
        for (int i = 0; i < R; ++i) v[i] = in[c * N + j + i * jump];
#pragma unroll
        for (int i = 1; i < R; ++i) v[i] = cmul<INV>(v[i], root[i * k * step]);  // i k < R ns
        if constexpr (R == 8) bfly8<INV>(v);
        else bfly4<INV>(v[0], v[1], v[2], v[3]);
        float2 *y = out + c * N + (j - k) * R + k;
#pragma unroll
        for (int i = 0; i < R; ++i) y[i * st.ns] = v[i];
    }
}

// C FFTs of N points in a ([c][N]) with b as the other buffer; returns the one that
// holds the result, visible to the block.
template <bool INV>
__device__ __forceinline__ float2 *mixed_fft(float2 *a, float2 *b, const float2 *root, int N, int C, const FftPlan &p)
{
    __syncthreads();
    switch (p.st[0].r) {
    case 3: mixed_first<INV, 3>(a, b, root, N, C, 3); break;
    case 5: mixed_first<INV, 5>(a, b, root, N, C, 5); break;
    case 7: mixed_first<INV, 7>(a, b, root, N, C, 7); break;
    default: {
        const int r = p.st[0].r, jump = N / r;
        // two outputs per item where that leaves every thread one
        if (C * jump * ((r + 3) / 4) >= (int)blockDim.x) mixed_first_two<INV>(a, b, root, N, C, r);
        else mixed_first<INV, 0>(a, b, root, N, C, r);
        break;
    }
    }
    for (int s = 1; s < p.stages; ++s) {
        float2 *t = a;
        a = b;
        b = t;
        __syncthreads();
        const FftPlan::Stage &st = p.st[s];
        switch (st.r) {
        case 3: mixed_stage<INV, 3>(a, b, root, N, C, 3, st); break;
        case 4: mixed_butterflies<INV, 4>(a, b, root, N, C, st); break;
        case 5: mixed_stage<INV, 5>(a, b, root, N, C, 5, st); break;
        case 7: mixed_stage<INV, 7>(a, b, root, N, C, 7, st); break;
        case 8: mixed_butterflies<INV, 8>(a, b, root, N, C, st); break;
        default: mixed_stage<INV, 0>(a, b, root, N, C, st.r, st); break;
        }
    }
    __syncthreads();
    return b;
}

// Table of such a length: the N/2 half-sample shifts, then the N roots.
__device__ __forceinline__ void load_roots(const float2 *__restrict__ tab, float2 *root, int N)
{
    for (int i = threadIdx.x; i < N; i += blockDim.x) root[i] = tab[N / 2 + i];
}

// A thread's first half-sample shift, loaded ahead of the FFT, and that of any k.
__device__ inline float2 first_half(const float2 *__restrict__ tab, int N) { return tab[min((int)threadIdx.x, N / 2 - 1)]; }
__device__ inline float2 half_at(const float2 *__restrict__ tab, float2 first, int k)
{
    return k == (int)threadIdx.x ? first : tab[k];
}

// Rows 2 blk and 2 blk + 1.  3 N points of LDS.
template <bool MAPS>
__device__ __forceinline__ void mixed_rows(const FftArgs &a, const FftMaps &mp, const FftPlan &p, int blk, float2 *lds)
{
    const int N = a.My, rows = a.Mx;
    if (*a.skip) return;
    float2 *root = lds, *b0 = lds + N, *b1 = b0 + N;
    const float2 *__restrict__ x0 = reinterpret_cast<const float2 *>(a.map + (size_t)2 * blk * N);
    const float2 *__restrict__ x1 = x0 + N / 2;
    const float mean = *a.mean;
    const float2 half = first_half(a.tab_y, N);
    load_roots(a.tab_y, root, N);
    [[maybe_unused]] double ovf = 0.0;
    for (int n = threadIdx.x; n < N / 2; n += blockDim.x) {
        float2 xa, xb;
        if constexpr (MAPS) {
            const size_t o = (size_t)2 * blk * N + 2 * n;
            const MapBins ma = load_bins(mp, o), mb = load_bins(mp, o + N);
            xa = store_bins(mp, o, ma, true, ovf);
            xb = store_bins(mp, o + N, mb, true, ovf);
        } else {
            xa = x0[n];
            xb = x1[n];
        }
        b0[n] = make_float2(xa.x - mean, xb.x - mean);
        b0[N - 1 - n] = make_float2(xa.y - mean, xb.y - mean);
    }
    float2 *z = mixed_fft<false>(b0, b1, root, N, 1, p);
    for (int k = threadIdx.x; k < N / 2; k += blockDim.x) {
        if (k == 0) {  // and N/2
            const float2 h = z[N / 2];
            z[N / 2] = make_float2(h.x * kSqrtHalf, h.y * kSqrtHalf);
        } else {
            const DctPair d = dct_pair(z[k], z[N - k], half_at(a.tab_y, half, k));
            z[k] = make_float2(d.a_k, d.b_k);
            z[N - k] = make_float2(d.a_n, d.b_n);
        }
    }
    __syncthreads();
    for (int e = threadIdx.x; e < N / 2; e += blockDim.x) {
        const int r = e & 1, g = e >> 1;
        float o[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const float2 v = z[4 * g + c];
            o[c] = r ? v.y : v.x;
        }
        *reinterpret_cast<float4 *>(a.t1 + ((size_t)g * rows + 2 * blk + r) * 4) = make_float4(o[0], o[1], o[2], o[3]);
    }
    if constexpr (MAPS) finish_maps<kMixedThreads>(mp, blk, rows / 2, ovf);
}

// Columns 2 blk and 2 blk + 1.  5 N points of LDS.
__device__ __forceinline__ void mixed_columns(const FftArgs &a, const FftPlan &p, int blk, float2 *lds)
{
    const int N = a.Mx, ca = 2 * blk;
    if (*a.skip) return;
    float2 *root = lds, *b0 = lds + N, *b1 = b0 + 2 * N;
    const size_t at = (size_t)(ca >> 2) * N * 4 + (ca & 3);
    const float2 half = first_half(a.tab_x, N);
    load_roots(a.tab_x, root, N);
    for (int i = threadIdx.x; i < N; i += blockDim.x)
        b0[(i & 1) ? N - 1 - (i >> 1) : i >> 1] = *reinterpret_cast<const float2 *>(a.t1 + at + (size_t)i * 4);
    const float2 *z = mixed_fft<false>(b0, b1, root, N, 1, p);
    float2 *in = z == b0 ? b1 : b0, *other = z == b0 ? b0 : b1;  // the spectrum is read before `other` is written
    for (int k = threadIdx.x; k < N / 2; k += blockDim.x) {  // both columns' points k and N - k
        const float2 zk = z[k], zn = z[k == 0 ? N / 2 : N - k];
        if (k == 0) {  // and N/2
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                const float2 e = spectral(a, 0, ca + c, c ? zk.y : zk.x);
                const float2 q = spectral(a, N / 2, ca + c, (c ? zn.y : zn.x) * kSqrtHalf);
                in[c * N] = make_float2(0.0f, e.y);
                in[c * N + N / 2] = make_float2(q.x * kSqrtHalf, q.y * kSqrtHalf);
            }
        } else {
            const float2 w = half_at(a.tab_x, half, k);
            const DctPair d = dct_pair(zk, zn, w);
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                const float2 ek = spectral(a, k, ca + c, c ? d.b_k : d.a_k);
                const float2 en = spectral(a, N - k, ca + c, c ? d.b_n : d.a_n);
                idct_pair(en.x, ek.x, ek.y, en.y, w, in[c * N + k], in[c * N + N - k]);  // sine sum: reversed spectrum
            }
        }
    }
    z = mixed_fft<true>(in, other, root, N, 2, p);
    for (int i = threadIdx.x; i < N; i += blockDim.x) {
        const int n = (i & 1) ? N - 1 - (i >> 1) : i >> 1;
        const float2 z0 = z[n], z1 = z[N + n];
        const float sg = (i & 1) ? -1.0f : 1.0f;
        *reinterpret_cast<float4 *>(a.pq + at + (size_t)i * 4) = make_float4(sg * z0.x, z0.y, sg * z1.x, z1.y);
    }
}

// Row blk of the field.  3 N points of LDS.
__device__ __forceinline__ void mixed_field(const FftArgs &a, const FftPlan &p, int row, float2 *lds)
{
    const int N = a.My, rows = a.Mx;
    if (*a.skip) return;
    float2 *root = lds, *b0 = lds + N, *b1 = b0 + N;
    const float2 half = first_half(a.tab_y, N);
    load_roots(a.tab_y, root, N);
    for (int e = threadIdx.x; e < N / 2; e += blockDim.x) {
        const float4 x = *reinterpret_cast<const float4 *>(a.pq + ((size_t)(e >> 1) * rows + row) * 4 + 2 * (e & 1));
        b1[2 * e] = make_float2(x.x, x.y);
        b1[2 * e + 1] = make_float2(x.z, x.w);
    }
    __syncthreads();
    for (int k = threadIdx.x; k < N / 2; k += blockDim.x) {
        const float2 ek = b1[k], en = b1[k == 0 ? N / 2 : N - k];
        if (k == 0) {  // and N/2
            b0[0] = make_float2(ek.x, 0.0f);
            b0[N / 2] = make_float2(en.x * kSqrtHalf, en.y * kSqrtHalf);
        } else {
            float2 zk, zn;
            idct_pair(ek.x, en.x, en.y, ek.y, half_at(a.tab_y, half, k), zk, zn);
            b0[k] = zk;
            b0[N - k] = zn;
        }
    }
    const float2 *z = mixed_fft<true>(b0, b1, root, N, 1, p);
    for (int n = threadIdx.x; n < N / 2; n += blockDim.x) {
        const float2 z0 = z[n], z1 = z[N - 1 - n];
        *reinterpret_cast<float4 *>(a.exy + (size_t)row * N + 2 * n) = make_float4(z0.x, z0.y, z1.x, -z1.y);
    }
}

// Pass S (rows, columns, field).  Neighbouring rows and columns, which share the
// layout groups' cache lines, go to one XCD.
template <int S, bool MAPS>
__global__ __launch_bounds__(kMixedThreads) void k_fft_mixed(FftArgs a, FftMaps mp)
{
    const int blk = dev::xcd_block(blockIdx.x, gridDim.x);
    if (S == 0) mixed_rows<MAPS>(a, mp, a.py, blk, fft_lds);
    else if (S == 1) mixed_columns(a, a.px, blk, fft_lds);
    else mixed_field(a, a.py, blk, fft_lds);
}

template <int S>
__global__ __launch_bounds__(kMixedThreads) void k_fft_mixed_b(const FftArgs *__restrict__ args, const int2 *__restrict__ tiles)
{
    const int2 t = tiles[dev::xcd_block(blockIdx.x, gridDim.x)];
    const FftArgs a = args[t.x];  // a batch's grids are square
    __shared__ FftPlan p;         // indexed by stage: not in registers
    for (int i = threadIdx.x; i < (int)(sizeof(FftPlan) / 4); i += kMixedThreads)
        reinterpret_cast<int *>(&p)[i] = reinterpret_cast<const int *>(&args[t.x].px)[i];
    __syncthreads();
    if (S == 0) mixed_rows<false>(a, FftMaps{}, p, t.y, fft_lds);
    else if (S == 1) mixed_columns(a, p, t.y, fft_lds);
    else mixed_field(a, p, t.y, fft_lds);
}

template <int S>
void launch_mixed(const FftArgs &a, const FftMaps *maps, hipStream_t s)
{
    const int n = S == 1 ? a.Mx : a.My, blocks = S == 0 ? a.Mx / 2 : S == 1 ? a.My / 2 : a.Mx;
    const size_t lds = (S == 1 ? 5 : 3) * sizeof(float2) * (size_t)n;
    auto go = [&](auto kern, const FftMaps &mp) {
        hipLaunchKernelGGL(kern, dim3(blocks), dim3(kMixedThreads), lds, s, a, mp);
    };
    if (S == 0 && maps) go(k_fft_mixed<S, S == 0>, *maps);
    else go(k_fft_mixed<S, false>, FftMaps{});
}

// ------------------------------------------------------------------ batches

// Batched: block b runs tile tiles[b] = (instance, block) of stage S with
// blocks of NT threads; the instance's side picks the length.
template <int NT, int S, int L>
__device__ inline void batch_tile(const FftArgs &a, int blk)
{
    constexpr int F = NT / Plan<L>::T;
    if (S == 0) rows_pass<L, F, false>(a, FftMaps{}, blk, fft_lds);
    else if (S == 1) columns_pass<L, F, 1>(a, blk, fft_lds);
    else field_pass<L, F>(a, blk, fft_lds);
}

template <int NT, int S>
__global__ __launch_bounds__(NT) void k_fft_b(const FftArgs *__restrict__ args, const int2 *__restrict__ tiles)
{
    const int2 t = tiles[blockIdx.x];
    const FftArgs a = args[t.x];
    const int l = 31 - __builtin_clz((unsigned)a.Mx);
    if (NT == 128) {
        switch (l) {
        case 4: batch_tile<128, S, 4>(a, t.y); break;
        case 5: batch_tile<128, S, 5>(a, t.y); break;
        case 6: batch_tile<128, S, 6>(a, t.y); break;
        case 7: batch_tile<128, S, 7>(a, t.y); break;
        case 8: batch_tile<128, S, 8>(a, t.y); break;
        case 9: batch_tile<128, S, 9>(a, t.y); break;
        default: batch_tile<128, S, 10>(a, t.y); break;
        }
    } else {
        switch (l) {
        case 11: batch_tile<1024, S, 11>(a, t.y); break;
        case 12: batch_tile<1024, S, 12>(a, t.y); break;
        default: batch_tile<1024, S, 13>(a, t.y); break;
        }
    }
}

int log2_of(int n)
{
    int l = 0;
    while ((1 << l) < n) ++l;
    return l;
}

// go(L) for the length 2^L, as a template argument.
template <class Go>
void with_length(int l, Go go)
{
    switch (l) {
    case 4: go(std::integral_constant<int, 4>()); break;
    case 5: go(std::integral_constant<int, 5>()); break;
    case 6: go(std::integral_constant<int, 6>()); break;
    case 7: go(std::integral_constant<int, 7>()); break;
    case 8: go(std::integral_constant<int, 8>()); break;
    case 9: go(std::integral_constant<int, 9>()); break;
    case 10: go(std::integral_constant<int, 10>()); break;
    case 11: go(std::integral_constant<int, 11>()); break;
    case 12: go(std::integral_constant<int, 12>()); break;
    default: go(std::integral_constant<int, 13>()); break;
    }
}

}  // namespace

// Odd primes share a stage up to this product.  One solve in us, 1 / 9 / 25 / 63: 400 x 240
// 20.0 / 19.8 / 19.6 / 19.5, 1008^2 47.0 / 51.9 / 47.6 / 49.3, 2000^2 174 / 174 / 159 / 160.
constexpr int kMixedOdd = 25;

FftPlan fft_plan(int n)
{
    FftPlan p{};
    if (fft_pow2(n)) return p;
    int odd = n, twos = 0;
    for (; odd % 2 == 0; odd /= 2) ++twos;
    std::vector<int> primes, r;
    for (int f = 3; odd > 1; f += 2)
        for (; odd % f == 0; odd /= f) primes.insert(primes.begin(), f);  // the largest first
    while (!primes.empty()) {  // one stage of up to kMixedOdd saves a barrier and an exchange
        int f = 1;
        for (size_t i = 0; i < primes.size();)
            if (f == 1 || f * primes[i] <= kMixedOdd) {
                f *= primes[i];
                primes.erase(primes.begin() + i);
            } else {
                ++i;
            }
        r.push_back(f);
    }
    for (int s = 0; twos > 0; twos -= r.back() == 8 ? 3 : 2, ++s) r.push_back(radix_of(twos, 0));
    int ns = 1;
    for (int f : r) {
        p.st[p.stages++] = {f, ns, 1.0f / (float)ns, 1.0f / (float)(f * ns)};
        ns *= f;
    }
    return p;
}

void fft_table(int n, std::vector<float2> &tab)
{
    tab.clear();
    auto unit = [&](double turns) {  // e^{-2 pi i turns}
        tab.push_back(make_float2((float)std::cos(2.0 * M_PI * turns), (float)-std::sin(2.0 * M_PI * turns)));
    };
    for (int k = 0; k < n / 2; ++k) unit(k / (4.0 * n));
    if (!fft_pow2(n)) {
        for (int k = 0; k < n; ++k) unit((double)k / n);
        return;
    }
    const int l = log2_of(n);
    for (int s = 1, ns = radix_of(l, 0); ns < n; ns *= radix_of(l, s++)) {
        const int R = radix_of(l, s);
        for (int r = 1; r < R; ++r)
            for (int k = 0; k < ns; ++k) unit((double)r * k / ((double)R * ns));
    }
}

int fft_row_blocks(int Mx, int My)
{
    if (!fft_pow2(My)) return Mx / 2;
    int blocks = 0;
    with_length(log2_of(My), [&](auto c) {
        constexpr int F = ffts_of<decltype(c)::value>();
        blocks = (Mx + 2 * F - 1) / (2 * F);
    });
    return blocks;
}

void launch_field_fft(const FftArgs &a, const FftMaps *maps, hipStream_t s)
{
    const int lx = log2_of(a.Mx), ly = log2_of(a.My);
    if (!fft_pow2(a.My)) launch_mixed<0>(a, maps, s);
    else with_length(ly, [&](auto c) {
        constexpr int L = decltype(c)::value, F = ffts_of<L>();
        auto go = [&](auto kern, const FftMaps &mp) {
            hipLaunchKernelGGL(kern, dim3(fft_row_blocks(a.Mx, a.My)), dim3(F * Plan<L>::T),
                               F * Plan<L>::buf * sizeof(float2), s, a, mp);
        };
        constexpr bool can = Plan<L>::N <= kFftMapsMax;
        if (can && maps) go(k_fft_rows<L, can>, *maps);
        else go(k_fft_rows<L, false>, FftMaps{});
    });
    if (!fft_pow2(a.Mx)) launch_mixed<1>(a, nullptr, s);
    else with_length(lx, [&](auto c) {
        constexpr int L = decltype(c)::value, F = ffts_of<L>();
        hipLaunchKernelGGL(k_fft_columns<L>, dim3((a.My + 2 * F - 1) / (2 * F)),
                           dim3(col_halves_of<L>() * F * Plan<L>::T), 2 * F * Plan<L>::buf * sizeof(float2), s, a);
    });
    if (!fft_pow2(a.My)) launch_mixed<2>(a, nullptr, s);
    else with_length(ly, [&](auto c) {
        constexpr int L = decltype(c)::value, F = field_ffts_of<L>();
        hipLaunchKernelGGL(k_fft_field<L>, dim3((a.Mx + F - 1) / F), dim3(F * Plan<L>::T),
                           F * Plan<L>::buf * sizeof(float2), s, a);
    });
}

int fft_class(int M) { return !fft_pow2(M) ? 2 : M <= 1024 ? 0 : 1; }

void fft_batch_tiles(int i, int M, std::vector<int2> (&tiles)[kFftClasses][3])
{
    const int cls = fft_class(M);
    const int F = cls < 2 ? (cls ? 1024 : 128) / (M / 8) : 1;
    for (int stage = 0; stage < 3; ++stage) {
        const int per = stage == 2 ? F : 2 * F;  // rows or columns per block
        for (int b = 0; b < (M + per - 1) / per; ++b) tiles[cls][stage].push_back(make_int2(i, b));
    }
}

void launch_field_fft_batch(const FftArgs *args, const FftBatchTiles (&t)[kFftClasses], hipStream_t s)
{
    // Powers of two: 8 NT points per block (9 with their padding).  Others: the longest
    // of the class.  The columns hold both inverse FFTs of each.
    auto stage = [&](int k, int i, auto kern, int nt) {
        const size_t lds = sizeof(float2) * (k < 2 ? 9 * nt * (i == 1 ? 2 : 1) : (i == 1 ? 5 : 3) * t[k].longest);
        if (t[k].n[i]) hipLaunchKernelGGL(kern, dim3(t[k].n[i]), dim3(nt), lds, s, args, t[k].d[i]);
    };
    stage(0, 0, k_fft_b<128, 0>, 128);
    stage(1, 0, k_fft_b<1024, 0>, 1024);
    stage(2, 0, k_fft_mixed_b<0>, kMixedThreads);
    stage(0, 1, k_fft_b<128, 1>, 128);
    stage(1, 1, k_fft_b<1024, 1>, 1024);
    stage(2, 1, k_fft_mixed_b<1>, kMixedThreads);
    stage(0, 2, k_fft_b<128, 2>, 128);
    stage(1, 2, k_fft_b<1024, 2>, 1024);
    stage(2, 2, k_fft_mixed_b<2>, kMixedThreads);
}

}  // namespace ep
