// fft_blue.hpp -- Bluestein's algorithm in registers (FP64 / FP32): lengths len
// with a prime factor above 61, as a chirp convolution of power-of-two length
// L = 2^8 .. 2^13 (FP64) / 2^14 (FP32), L >= 2 len - 1:
//   X[k] = c[k] sum_j (x[j] c[j]) conj(c[k-j]),  c[j] = w_{2 len}^{j^2},
//        = c[k] conj(DFT_L(conj(DFT_L(x c) Bh)))[k],  Bh = DFT_L(conj c) / L.
//
// What bounds it: instruction issue and the LDS exchanges; each row or column
// crosses HBM once each way, at well below its rate.  The in-LDS form
// (gen_blue_ip, fft_general.hpp) makes 7 passes of radix 8 over the LDS for
// L = 4096, each with run-time index arithmetic.  Here a sequence stays in
// registers (16 NB points per thread), with the radix-16 stages and the split
// exchanges of the long columns (fft_col_long.hpp).  The outputs of the last
// stage of DFT_L are, thread by thread, the inputs of the next transform's first
// stage, so the product with Bh takes no exchange: 2 exchanges in all for 2^8
// points, 4 for 2^9 .. 2^12, 6 for 2^13 and 2^14.  len <= L/2, so the first stage's upper
// inputs are zero, and its upper outputs are never formed.
// In-LDS form -> this one (us, whole transform): FP64 2039 x 4078 206 -> 106, 1021 x
// 1024 48 -> 28, 1024 x 8186 168 -> 95, 67 x 1024 30 -> 14; FP32 2039 x 1024 58 -> 34,
// 8191 x 1024 190 -> 141 (the small grids' figures hold about 10 us of phase events
// that the in-LDS side still recorded).
#pragma once

#include "fft_col_long.hpp"

namespace hpxfft_dev {

constexpr int BLUE_MIN_LG = 8, BLUE_MAX_LG_F64 = 13, BLUE_MAX_LG_F32 = 14;

// COL: W adjacent columns per workgroup, LDS [pad(e)][w]; else W rows, one LDS
// block each.  Columns: a row segment of 128 bytes where NT <= 512 covers it, down
// to 32 (L = 2^13, FP64) and 16 bytes.
template <typename T, int LG, bool COL> struct bluecfg
{
    using real = T;
    static constexpr int L = 1 << LG;
    // two butterflies per thread where the workgroup would otherwise be too wide
    static constexpr int NB = sizeof(T) == 8 ? 1 : (COL ? (LG >= 10 ? 2 : 1) : (LG >= 13 ? 2 : 1));
    static constexpr int JT = L / (16 * NB);                     // threads per sequence
    static constexpr int WMAX = 128 / (2 * (int)sizeof(T));      // columns of a 128-byte segment
    // (L = 2^12: 512 threads, two workgroups per CU; FP32 with 1024: 2039 x 1024 61 us, not 33)
    static constexpr int NTMAX = LG >= 13 ? 1024 : 512;
    static constexpr int W = COL ? (JT * WMAX <= NTMAX ? WMAX : NTMAX / JT) : (JT >= 128 ? 1 : 128 / JT);
    static constexpr int NT = JT * W;
    static constexpr int M = L / 16;
    static constexpr int NR16 = LG / 4;
    static constexpr int RL = 1 << (LG % 4);
    static constexpr int NSL = L / RL;
    static constexpr int LP = L + L / 16;
    static constexpr int ES = COL ? W : 1;
    static constexpr int ns(int s) { return s == 0 ? 1 : 16 * ns(s - 1); }
    __device__ static __forceinline__ int pad(int e) { return e + (e >> 4); }
    // element of register u before a first stage, and after the last one
    __device__ static __forceinline__ int in_e(int u, int jj) { return jj + (u / 16) * JT + (u % 16) * M; }
    __device__ static __forceinline__ int out_e(int u, int jj)
    {
        constexpr int R = RL > 1 ? RL : 16, STR = RL > 1 ? NSL : M;
        return jj + (u / R) * JT + (u % R) * STR;
    }
    // waves per SIMD that the registers are cut to: 4 (128 VGPRs, no spills), which
    // lets two 512-thread workgroups share a CU (FP64 2039 x 1024 at 2: 51 us, at 4:
    // 43).  Two FP32 butterflies per thread spill 20 VGPRs there and take 2 (2039 x 1024
    // 38.4 -> 34.7), but rows of 2^14 points still gain by two workgroups (1024 x 16382
    // 171 -> 138)
    static constexpr int WAVES = NB == 2 && LG < 14 ? 2 : 4;
    static_assert(W >= 1 && JT * NB == M, "threads cover the butterflies");
};

struct BlueArgs
{
    int len;                       // the DFT's length
    const cpx<double> *stw64;      // radix-16 stage twiddles (stage_tw_off)
    const void *tw_L;              // w_L^m, m < L, compute precision
    const cpx<double> *chirp;      // c[j], j < len
    const cpx<double> *bh;         // Bh, natural order
    const cpx<double> *tab2;       // rows: w_{2 len}^m (the r2c split)
};

// table loads four at a time: all at once they would take more registers than the
// data (spills of up to 650 bytes a thread)
__device__ __forceinline__ void blue_chunk(int u)
{
    if (u % 4 == 0) __builtin_amdgcn_sched_barrier(0);
}

// v: the sequence by in_e (element e >= len: 0, and 8..15 of each butterfly not
// read); on return its DFT by out_e, for e < len
template <typename C>
__device__ __forceinline__ void blue_fft(cpx<typename C::real> *v, typename C::real *lds, const BlueArgs &g, int jj, int w)
{
    using T = typename C::real;
    const cpx<T> *tw = reinterpret_cast<const cpx<T> *>(g.tw_L);
#pragma unroll
    for (int u = 0; u < 16 * C::NB; ++u)
    {
        if (u % 16 >= 8) continue;
        blue_chunk(u);
        const int e = C::in_e(u, jj), ec = e < g.len ? e : g.len - 1;
        const cpx<T> z = cmul(v[u], tabv<T>(g.chirp, ec));
        v[u] = e < g.len ? z : cpx<T>{T(0), T(0)};
    }
    col_long_stages<C, 0, true>(v, lds, g.stw64, jj, w);
    if constexpr (C::RL > 1) col_long_last<C>(v, lds, tw, jj, w);
#pragma unroll
    for (int u = 0; u < 16 * C::NB; ++u)
    {
        blue_chunk(u);
        v[u] = conjc(cmul(v[u], tabv<T>(g.bh, C::out_e(u, jj))));
    }
    if constexpr (C::RL > 1)
    {
        // register i RL + q of the last stage is input r = i / NB + (16 / RL) q of butterfly i % NB
        cpx<T> x[16 * C::NB];
#pragma unroll
        for (int u = 0; u < 16 * C::NB; ++u)
        {
            const int i = u / C::RL, q = u % C::RL;
            x[16 * (i % C::NB) + i / C::NB + (16 / C::RL) * q] = v[u];
        }
#pragma unroll
        for (int u = 0; u < 16 * C::NB; ++u) v[u] = x[u];
    }
    __syncthreads();   // the last exchange's reads
    // the inverse's twiddles and chirp are the forward's: without this the compiler
    // keeps them all from one to the other (up to 60 registers, spilled)
    asm volatile("" : "+v"(jj));
    col_long_stages<C, 0>(v, lds, g.stw64, jj, w);
    if constexpr (C::RL > 1) col_long_last<C>(v, lds, tw, jj, w);
    // the outputs are formed here: else the last stage sinks into the callers' guarded
    // stores, below the chirp's loads
#pragma unroll
    for (int u = 0; u < 16 * C::NB; ++u)
        if (C::out_e(u, 0) < C::L / 2) asm volatile("" : "+v"(v[u].x), "+v"(v[u].y));
#pragma unroll
    for (int u = 0; u < 16 * C::NB; ++u)
    {
        blue_chunk(u);
        const int e = C::out_e(u, jj), ec = e < g.len ? e : g.len - 1;
        if (C::out_e(u, 0) < C::L / 2) v[u] = cmul(conjc(v[u]), tabv<T>(g.chirp, ec));
    }
}

// Row r2c (as gen_row_r2c_kernel): blockIdx.x = group of W rows (XCD order), .y = grid
template <typename T, int LG>
__global__ void __launch_bounds__((bluecfg<T, LG, false>::NT), (bluecfg<T, LG, false>::WAVES)) blue_row_r2c_kernel(RowArgs a, BlueArgs g)
{
    using C = bluecfg<T, LG, false>;
    __shared__ __align__(16) T lds[C::LP * C::W];
    const unsigned long long t_start = stamp_now(a.ts, a.nrows);
    const int t = threadIdx.x, s = t / C::JT, jj = t % C::JT, len = g.len;
    const long long b = blockIdx.y;
    const int row = xcd_order((int)blockIdx.x, (int)gridDim.x) * C::W + s, rowc = min(row, a.nrows - 1);
    const T *in = reinterpret_cast<const T *>(a.in) + b * a.dist_in + (long long)rowc * a.ld_in;
    cpx<T> v[16 * C::NB];
#pragma unroll
    for (int u = 0; u < 16 * C::NB; ++u)
    {
        if (u % 16 >= 8) continue;
        v[u] = stor<T>::ld(in + 2 * min(C::in_e(u, jj), len - 1));
    }
    blue_fft<C>(v, lds, g, jj, s * C::LP);
    // the split: Z[e], e < len <= L/2, as complex values in the row's block
    __syncthreads();
    cpx<T> *Z = reinterpret_cast<cpx<T> *>(lds + s * C::LP);
#pragma unroll
    for (int u = 0; u < 16 * C::NB; ++u)
    {
        const int e = C::out_e(u, jj);
        if (C::out_e(u, 0) < C::L / 2 && e < len) Z[e] = v[u];
    }
    __syncthreads();
    if (row < a.nrows)
    {
        T *o = reinterpret_cast<T *>(a.out) + b * a.dist_out + (long long)row * a.ld_out;
        for (int k = jj; 2 * k <= len; k += C::JT)
        {
            const cpx<T> A = Z[k];
            if (k == 0)
            {
                stor<T>::st(o, cpx<T>{A.x + A.y, T(0)});
                stor<T>::st(o + 2 * len, cpx<T>{A.x - A.y, T(0)});
            }
            else if (2 * k == len) stor<T>::st(o + 2 * k, conjc(A));
            else
            {
                cpx<T> x0, x1;
                r2c_val(A, Z[len - k], tabv<T>(g.tab2, k), x0, x1);
                stor<T>::st(o + 2 * k, x0);
                stor<T>::st(o + 2 * (len - k), x1);
            }
        }
    }
    stamp_first(a.ts, t_start);
}

// Row c2r (as gen_row_c2r_kernel); hs: 0.5 halves the interior bins (the adjoint), else 1
template <typename T, int LG>
__global__ void __launch_bounds__((bluecfg<T, LG, false>::NT), (bluecfg<T, LG, false>::WAVES)) blue_row_c2r_kernel(RowArgs a, BlueArgs g, T hs)
{
    using C = bluecfg<T, LG, false>;
    __shared__ T lds[C::LP * C::W];
    const unsigned long long t_start = stamp_now(a.ts, a.nrows);
    const int t = threadIdx.x, s = t / C::JT, jj = t % C::JT, len = g.len;
    const long long b = blockIdx.y;
    const int row = xcd_order((int)blockIdx.x, (int)gridDim.x) * C::W + s, rowc = min(row, a.nrows - 1);
    const T *in = reinterpret_cast<const T *>(a.in) + b * a.dist_in + (long long)rowc * a.ld_in;
    cpx<T> v[16 * C::NB];
#pragma unroll
    for (int u = 0; u < 16 * C::NB; ++u)
    {
        if (u % 16 >= 8) continue;
        blue_chunk(u);
        const int k = min(C::in_e(u, jj), len - 1);
        const cpx<T> gk = stor<T>::ld(in + 2 * k), gl = stor<T>::ld(in + 2 * (len - k)), w = tabv<T>(g.tab2, k);
        const cpx<T> hk = scal(gk, hs), hl = scal(gl, hs);
        const cpx<T> s0 = hk + conjc(hl), d0 = cmul(hk - conjc(hl), conjc(w));
        v[u] = k == 0 ? cpx<T>{gk.x + gl.x, -(gk.x - gl.x)} : cpx<T>{s0.x - d0.y, -(s0.y + d0.x)};   // conj Z[k]
    }
    blue_fft<C>(v, lds, g, jj, s * C::LP);
    if (row < a.nrows)
    {
        T *o = reinterpret_cast<T *>(a.out) + b * a.dist_out + (long long)row * a.ld_out;
#pragma unroll
        for (int u = 0; u < 16 * C::NB; ++u)
        {
            const int e = C::out_e(u, jj);
            if (C::out_e(u, 0) < C::L / 2 && e < len) stor<T>::st(o + 2 * e, conjc(v[u]));
        }
    }
    stamp(a.ts, t_start);
}

// Columns (as gen_col_kernel): blockIdx.x = strip of W columns (XCD order), .y = grid;
// sg: -1 for the inverse transform, conj(DFT(conj .)), else 1
template <typename T, int LG>
__global__ void __launch_bounds__((bluecfg<T, LG, true>::NT), (bluecfg<T, LG, true>::WAVES)) blue_col_kernel(ColArgs a, BlueArgs g, T sg)
{
    using C = bluecfg<T, LG, true>;
    __shared__ T lds[C::LP * C::W];
    const unsigned long long t_start = stamp_now(a.ts, a.ncols);
    const int t = threadIdx.x, w = t % C::W, jj = t / C::W, len = g.len;
    const int c = xcd_order((int)blockIdx.x, (int)gridDim.x) * C::W + w;
    const bool valid = c < a.ncols;
    const long long base = (long long)blockIdx.y * a.dist + (valid ? c : a.ncols - 1);
    const T *in = reinterpret_cast<const T *>(a.in) + 2 * base;
    T *out = reinterpret_cast<T *>(a.out) + 2 * base;
    cpx<T> v[16 * C::NB];
#pragma unroll
    for (int u = 0; u < 16 * C::NB; ++u)
    {
        if (u % 16 >= 8) continue;
        const cpx<T> z = stor<T>::ld(in + 2 * a.pitch * min(C::in_e(u, jj), len - 1));
        v[u] = cpx<T>{z.x, sg * z.y};
    }
    blue_fft<C>(v, lds, g, jj, w);
    if (valid)
    {
#pragma unroll
        for (int u = 0; u < 16 * C::NB; ++u)
        {
            const int e = C::out_e(u, jj);
            if (C::out_e(u, 0) < C::L / 2 && e < len) stor<T>::st(out + 2 * a.pitch * e, cpx<T>{v[u].x, sg * v[u].y});
        }
    }
    stamp(a.ts, t_start);
}

}   // namespace hpxfft_dev
