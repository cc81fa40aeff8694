// k_fft.hip -- Poisson field solve on power-of-two grids as FP32 FFTs in LDS.
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
// 14.8 -> 9.2 us, 128^2 23.6 -> 14.9, 256^2 31.5 -> 15.4, 512^2 48 -> 18.4, 1024^2
// 108 -> 33 (split-BF16 products 72), 2048^2 585 -> 82; max-norm error at most
// 5e-7 (products: FP32 3e-6, split-BF16 1.1e-5).  What bounds them is latency:
// one wave per SIMD at 1024^2, where a kernel without its butterflies takes 5-10
// us, without its stores 1.5-3 us less, and with free twiddles or LDS exchanges
// about 1.5 us less each.  The columns' second half of threads (H = 2) takes them
// from 7.1 to 6.5 us at 256^2; at 1024^2 it changes nothing.  Padding the layout
// groups against channel conflicts changed nothing either.
//
// Layout of T1 (float) and PQ (float2): [v/4][i][v%4].  The column kernel reads
// and writes whole runs; a block of the row kernels touches 4 consecutive rows,
// runs of 64 and 128 bytes.
#include <hip/hip_runtime.h>

#include <cmath>
#include <vector>

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

// FFTs per block: two (so that the four rows or columns of a layout group stay
// together), more where one FFT is less than half a wave's threads.
template <int L>
constexpr int ffts_of()
{
    return Plan<L>::T >= 1024 ? 1 : Plan<L>::T >= 32 ? 2 : 64 / Plan<L>::T;
}
// The column kernel's FFTs and its threads per FFT point set (see columns_pass).
template <int L>
constexpr int col_halves_of()
{
    return Plan<L>::T >= 1024 ? 1 : 2;
}
template <int L>
constexpr int col_ffts_of()
{
    return Plan<L>::T >= 512 ? 1 : ffts_of<L>();
}
// The last kernel's: one row each, so four where the block stays below 1024 threads.
template <int L>
constexpr int field_ffts_of()
{
    return Plan<L>::T >= 1024 ? 1 : Plan<L>::T >= 512 ? 2 : Plan<L>::T >= 16 ? 4 : 64 / Plan<L>::T;
}

// Rows 2 F blk ... of the map (row length N, `rows` rows, an even number).
// F * T threads, F * buf points of LDS.
template <int L, int F>
__device__ inline void rows_pass(const FftArgs &a, int blk, float2 *lds)
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
#pragma unroll
    for (int m = 0; m < 4; ++m) {
        xa[m] = x0[t + m * T];
        xb[m] = x1[t + m * T];
    }
    Twiddles<L> w;
    load_twiddles<L>(a.tab_y, t, w);
    if (halt) return;
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

template <int L>
__global__ __launch_bounds__(ffts_of<L>() * Plan<L>::T) void k_fft_rows(FftArgs a)
{
    rows_pass<L, ffts_of<L>()>(a, blockIdx.x, fft_lds);
}
template <int L>
__global__ __launch_bounds__(col_halves_of<L>() * col_ffts_of<L>() * Plan<L>::T) void k_fft_columns(FftArgs a)
{
    columns_pass<L, col_ffts_of<L>(), col_halves_of<L>()>(a, blockIdx.x, fft_lds);
}
template <int L>
__global__ __launch_bounds__(field_ffts_of<L>() * Plan<L>::T) void k_fft_field(FftArgs a)
{
    field_pass<L, field_ffts_of<L>()>(a, blockIdx.x, fft_lds);
}

// Batched: block b runs tile tiles[b] = (instance, block) of stage S with
// blocks of NT threads; the instance's side picks the length.
template <int NT, int S, int L>
__device__ inline void batch_tile(const FftArgs &a, int blk)
{
    constexpr int F = NT / Plan<L>::T;
    if (S == 0) rows_pass<L, F>(a, blk, fft_lds);
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

void fft_table(int n, std::vector<float2> &tab)
{
    const int l = log2_of(n);
    tab.clear();
    auto unit = [&](double turns) {  // e^{-2 pi i turns}
        tab.push_back(make_float2((float)std::cos(2.0 * M_PI * turns), (float)-std::sin(2.0 * M_PI * turns)));
    };
    for (int k = 0; k < n / 2; ++k) unit(k / (4.0 * n));
    for (int s = 1, ns = radix_of(l, 0); ns < n; ns *= radix_of(l, s++)) {
        const int R = radix_of(l, s);
        for (int r = 1; r < R; ++r)
            for (int k = 0; k < ns; ++k) unit((double)r * k / ((double)R * ns));
    }
}

void launch_field_fft(const FftArgs &a, hipStream_t s)
{
    const int lx = log2_of(a.Mx), ly = log2_of(a.My);
    with_length(ly, [&](auto c) {
        constexpr int L = decltype(c)::value, F = ffts_of<L>();
        hipLaunchKernelGGL(k_fft_rows<L>, dim3((a.Mx + 2 * F - 1) / (2 * F)), dim3(F * Plan<L>::T),
                           F * Plan<L>::buf * sizeof(float2), s, a);
    });
    with_length(lx, [&](auto c) {
        constexpr int L = decltype(c)::value, F = col_ffts_of<L>();
        hipLaunchKernelGGL(k_fft_columns<L>, dim3((a.My + 2 * F - 1) / (2 * F)),
                           dim3(col_halves_of<L>() * F * Plan<L>::T), 2 * F * Plan<L>::buf * sizeof(float2), s, a);
    });
    with_length(ly, [&](auto c) {
        constexpr int L = decltype(c)::value, F = field_ffts_of<L>();
        hipLaunchKernelGGL(k_fft_field<L>, dim3((a.Mx + F - 1) / F), dim3(F * Plan<L>::T),
                           F * Plan<L>::buf * sizeof(float2), s, a);
    });
}

void fft_batch_tiles(int i, int M, std::vector<int2> (&tiles)[kFftClasses][3])
{
    const int cls = M <= 1024 ? 0 : 1, nt = cls ? 1024 : 128, F = nt / (M / 8);
    for (int stage = 0; stage < 3; ++stage) {
        const int per = stage == 2 ? F : 2 * F;  // rows or columns per block
        for (int b = 0; b < (M + per - 1) / per; ++b) tiles[cls][stage].push_back(make_int2(i, b));
    }
}

void launch_field_fft_batch(const FftArgs *args, const FftBatchTiles (&t)[kFftClasses], hipStream_t s)
{
    // 8 NT points per block; the columns hold both inverse FFTs of each
    const size_t pt = 9 * sizeof(float2);
    auto stage = [&](int k, int i, auto kern, int nt) {
        if (t[k].n[i])
            hipLaunchKernelGGL(kern, dim3(t[k].n[i]), dim3(nt), nt * pt * (i == 1 ? 2 : 1), s, args, t[k].d[i]);
    };
    stage(0, 0, k_fft_b<128, 0>, 128);
    stage(1, 0, k_fft_b<1024, 0>, 1024);
    stage(0, 1, k_fft_b<128, 1>, 128);
    stage(1, 1, k_fft_b<1024, 1>, 1024);
    stage(0, 2, k_fft_b<128, 2>, 128);
    stage(1, 2, k_fft_b<1024, 2>, 1024);
}

}  // namespace ep
