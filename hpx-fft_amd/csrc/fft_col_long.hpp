// fft_col_long.hpp -- columns of 2^11 and 2^12 points (FP64 / FP32 storage)
// in one launch: a workgroup of NT threads holds W adjacent columns over all
// Nx rows in VGPRs, so the spectrum crosses HBM once in each direction instead
// of twice through the four-step's scratch.
//
// What bounds it: HBM, at the rate of its row segments, plus the transform
// itself (one or two workgroups share a CU, so little of it is hidden).  512
// threads hold 2^13 FP64 or 2^14 FP32 points (64 VGPRs of data each), two
// workgroups per CU: 64-byte segments at 2^11 rows, 32 bytes at 2^12; 1024
// threads hold twice that, one per CU: 64 bytes at 2^12.  Moving 2 GiB in place
// in 64-byte segments with no arithmetic runs at 4.3 TB/s of read + write (32
// bytes 3.2, 16 bytes 1.9), against the four-step's two launches at 5.2, 2.6 per
// byte of spectrum.  Column pass, four-step -> one launch (us): FP64 2^11 rows x
// 512, 2048, 8192 reals 20.8 -> 14.7, 32.2 -> 24.1, 109 -> 63, 16 x 2048^2
// 461 -> 287; FP64 4096^2 115 -> 83, 4 x 4096^2 458 -> 384; FP32 16 x 2048^2
// 221 -> 160, 16 x 4096^2 857 -> 750.  At 2^13 rows (32-byte segments, 1024
// threads) it was even with the four-step (8192^2 FP64 465 against 478, FP32
// slower), so those columns keep the four-step.
//
// Radix-16 Stockham stages with one LDS exchange each, then (2^11) a last stage
// of radix 8.  LDS rows are [pad(e)][w], real and imaginary halves exchanged
// separately.  Stage twiddles come from the radix-16 stage tables of the long
// rows (fft_row_big.hpp).
#pragma once

#include "fft_row_big.hpp"

namespace hpxfft_dev {

constexpr int COL_LONG_MIN_LG = 11, COL_LONG_MAX_LG = 12;

template <typename T, int LG, int NTH> struct collong
{
    using real = T;
    static constexpr int L = 1 << LG;
    static constexpr int NB = 8 / (int)sizeof(T);               // radix-16 butterflies per thread and stage
    static constexpr int NT = NTH;                               // threads
    static constexpr int W = NT * 16 * NB / L;          // adjacent columns
    static constexpr int ES = W;                                 // LDS distance of consecutive elements of a column
    static constexpr int M = L / 16;                             // butterflies per column
    static constexpr int JT = NT / W;                   // threads per column
    static constexpr int NR16 = LG / 4;
    static constexpr int RL = 1 << (LG % 4);                     // last radix (1: none)
    static constexpr int NSL = L / RL;
    static constexpr int LP = L + L / 16;
    static constexpr int ns(int s) { return s == 0 ? 1 : 16 * ns(s - 1); }
    __device__ static __forceinline__ int pad(int e) { return e + (e >> 4); }
    static_assert(W >= 1 && JT * NB == M, "threads cover the butterflies");
};

// dft16 of inputs whose upper half is zero: the first four 4-point DFTs have two
template <typename T> __device__ __forceinline__ void dft16_half(cpx<T> *a)
{
    const T c = kconst<T>::c8, s = kconst<T>::s8;
    cpx<T> y[16];
#pragma unroll
    for (int n1 = 0; n1 < 4; ++n1)
    {
        const cpx<T> b0 = a[n1], b1 = a[n1 + 4], r1 = mul_mi(b1);
        y[n1 * 4 + 0] = b0 + b1;
        y[n1 * 4 + 1] = b0 + r1;
        y[n1 * 4 + 2] = b0 - b1;
        y[n1 * 4 + 3] = b0 - r1;
    }
    y[5] = cmul(y[5], cpx<T>{c, -s});
    y[6] = mul_w8_1(y[6]);
    y[7] = cmul(y[7], cpx<T>{s, -c});
    y[9] = mul_w8_1(y[9]);
    y[10] = mul_mi(y[10]);
    y[11] = mul_w8_3(y[11]);
    y[13] = cmul(y[13], cpx<T>{s, -c});
    y[14] = mul_w8_3(y[14]);
    y[15] = cmul(y[15], cpx<T>{-c, s});
#pragma unroll
    for (int k2 = 0; k2 < 4; ++k2)
    {
        cpx<T> b0 = y[k2], b1 = y[4 + k2], b2 = y[8 + k2], b3 = y[12 + k2];
        dft4v(b0, b1, b2, b3);
        a[k2] = b0;
        a[4 + k2] = b1;
        a[8 + k2] = b2;
        a[12 + k2] = b3;
    }
}

// exchange: this thread's outputs of radix-16 stage S to LDS, then the inputs of
// the next stage of radix R2 (element j + r L/R2 of butterfly j = jj + i JT).
// Element e lies at lds[pad(e) C::ES + w].
template <typename C, int S, int R2>
__device__ __forceinline__ void col_long_exchange(cpx<typename C::real> *v, typename C::real *lds, int jj, int w)
{
    constexpr int NS = C::ns(S), WS = NS == 1 ? 1 : NS + NS / 16, STR = C::L / R2, RS = STR + STR / 16;
    int wb[C::NB];
#pragma unroll
    for (int b = 0; b < C::NB; ++b)
    {
        const int j = jj + b * C::JT, k = j & (NS - 1);
        wb[b] = C::pad((j / NS) * 16 * NS + k) * C::ES + w;
    }
#pragma unroll
    for (int h = 0; h < 2; ++h)
    {
#pragma unroll
        for (int b = 0; b < C::NB; ++b)
#pragma unroll
            for (int q = 0; q < 16; ++q) lds[wb[b] + q * WS * C::ES] = h ? v[16 * b + q].y : v[16 * b + q].x;
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 16 * C::NB / R2; ++i)
        {
            const int rb = C::pad(jj + i * C::JT) * C::ES + w;
#pragma unroll
            for (int r = 0; r < R2; ++r)
            {
                if (h) v[i * R2 + r].y = lds[rb + r * RS * C::ES];
                else v[i * R2 + r].x = lds[rb + r * RS * C::ES];
            }
        }
        if (h == 0) __syncthreads();
    }
}

// HALF: the inputs 8..15 of each stage-0 butterfly are zero
template <typename C, int S, bool HALF = false>
__device__ __forceinline__ void col_long_stages(cpx<typename C::real> *v, typename C::real *lds,
                                                const cpx<double> *__restrict__ stw64, int jj, int w)
{
    using T = typename C::real;
    constexpr int NS = C::ns(S);
#pragma unroll
    for (int b = 0; b < C::NB; ++b)
    {
        if constexpr (NS > 1) twiddle16<T, NS>(v + 16 * b, stw64, (jj + b * C::JT) & (NS - 1));
        if constexpr (HALF) dft16_half(v + 16 * b);
        else dft16(v + 16 * b);
    }
    if constexpr (S + 1 < C::NR16)
    {
        if constexpr (S > 0) __syncthreads();   // the last exchange's reads
        col_long_exchange<C, S, 16>(v, lds, jj, w);
        col_long_stages<C, S + 1>(v, lds, stw64, jj, w);
    }
}

// the last stage, radix RL > 1, after its exchange: butterfly j reads
// j + r NSL, outputs j + q NSL (v[i RL + q], j = jj + i JT); twiddles w_L^{r j}
template <typename C>
__device__ __forceinline__ void col_long_last(cpx<typename C::real> *v, typename C::real *lds,
                                              const cpx<typename C::real> *__restrict__ tw, int jj, int w)
{
    using T = typename C::real;
    constexpr int RL = C::RL;
    __syncthreads();
    col_long_exchange<C, C::NR16 - 1, RL>(v, lds, jj, w);
#pragma unroll
    for (int i = 0; i < 16 * C::NB / RL; ++i)
    {
#pragma unroll
        for (int r = 1; r < RL; ++r) v[i * RL + r] = cmul(v[i * RL + r], tw[r * (jj + i * C::JT)]);
        dftR<T, RL>(v + i * RL);
    }
}

// one strip of W columns of grid b, from a.in to a.out in the same layout (in place
// for the forward transform).  CONJ: the inverse, conj(DFT(conj .)).  Shared with the
// batched column-phase kernel.
template <typename C, bool CONJ>
__device__ __forceinline__ void col_long_body(const ColArgs &a, long long b, int strip, typename C::real *lds, int t)
{
    using T = typename C::real;
    constexpr int W = C::W, JT = C::JT, M = C::M, RL = C::RL, NSL = C::NSL, NB = C::NB;
    const int w = t % W, jj = t / W;
    const int c = strip * W + w;
    const bool valid = c < a.ncols;
    const int cl = valid ? c : a.ncols - 1;   // lanes past the last column load it and store nothing
    const T *in = reinterpret_cast<const T *>(a.in) + 2 * (b * a.dist + cl + (long long)jj * a.pitch);
    cpx<T> v[16 * NB];
#pragma unroll
    for (int u = 0; u < 16 * NB; ++u)
    {
        cpx<T> z = stor<T>::ld(in + 2 * a.pitch * ((u / 16) * JT + (u % 16) * M));
        v[u] = CONJ ? conjc(z) : z;
    }
    col_long_stages<C, 0>(v, lds, reinterpret_cast<const cpx<double> *>(a.stw64), jj, w);
    if constexpr (RL > 1) col_long_last<C>(v, lds, reinterpret_cast<const cpx<T> *>(a.tw_L), jj, w);
    // FP64: the outputs are formed here, before the guard (the last stage else sinks
    // below it): 4096 x 2048 77.0 -> 73.8 us, 16 x 2048^2 530 -> 520; FP32 4096^2 lost 1%
    if constexpr (sizeof(T) == 8)
    {
#pragma unroll
        for (int u = 0; u < 16 * NB; ++u) asm volatile("" : "+v"(v[u].x), "+v"(v[u].y));
    }
    if (!valid) return;
    // the stores' addresses are formed after the stages (in place they are the loads',
    // which the batched kernel else kept, spilled)
    int js = jj;
    asm volatile("" : "+v"(js));
    T *out = reinterpret_cast<T *>(a.out) + 2 * (b * a.dist + cl + (long long)js * a.pitch);
    constexpr int R = RL > 1 ? RL : 16, STR = RL > 1 ? NSL : M;
#pragma unroll
    for (int u = 0; u < 16 * NB; ++u)
    {
        const cpx<T> z = v[u];
        stor<T>::st(out + 2 * a.pitch * ((u / R) * JT + (u % R) * STR), CONJ ? conjc(z) : z);
    }
}

// blockIdx.x = strip, .z = grid
template <typename T, int LG, int NTH, bool CONJ>
__global__ void __launch_bounds__(NTH, 4) col_long_kernel(ColArgs a)
{
    using C = collong<T, LG, NTH>;
    __shared__ T lds[C::LP * C::W];
    const unsigned long long t_start = stamp_now(a.ts, a.ncols);
    const blk3 bk = xcd_block();   // neighbouring strips share lines: one XCD
    col_long_body<C, CONJ>(a, bk.z, bk.x, lds, threadIdx.x);
    stamp(a.ts, t_start);
}

}   // namespace hpxfft_dev
