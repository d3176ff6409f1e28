// launch.hpp -- host-side dispatch from runtime sizes to kernel instantiations.
#pragma once

#include "fft_kernels.hpp"
#include "fft_row_big.hpp"
#include "fft_row_pair.hpp"
#include "fft_tile.hpp"
#include "fft_col_long.hpp"
#include <algorithm>

namespace hpxfft_host {

using hpxfft_dev::ColArgs;
using hpxfft_dev::RowArgs;

enum prec_id { P_F64 = 0, P_F32 = 1, P_F16 = 2, P_BF16 = 3 };

constexpr int ROW_MAX_LG = 14;       // Ny <= 32768
constexpr int COL_TILE_MIN_LG = 5;   // four-step sub-FFT lengths 32..256
constexpr int COL_TILE_MAX_LG = 8;

struct geom
{
    int nt;     // threads per workgroup
    int nseq;   // rows (row kernels) or columns W (column kernels) per workgroup
    int E;      // elements per thread
    bool split; // LDS exchange by real/imag halves
};

// per precision (defined in inst_<prec>.hip)
#define HPXFFT_DECL_LAUNCH(sfx)                                                                                    \
    hipError_t row_r2c_##sfx(int lg, const RowArgs &a, unsigned gx, unsigned gy, hipStream_t s);                   \
    hipError_t row_r2c_pair_##sfx(int lg, const RowArgs &a, unsigned total, hipStream_t s);                       \
    hipError_t row_c2r_##sfx(int lg, bool halve, const RowArgs &a, unsigned gx, unsigned gy, hipStream_t s);       \
    hipError_t col_##sfx(int lg, int mode, bool conj, const ColArgs &a, unsigned gx, unsigned gy, unsigned gz,    \
                         hipStream_t s);                                                                           \
    geom row_geom_##sfx(int lg);                                                                                   \
    geom col_geom_##sfx(int lg);                                                                                   \
    geom tile_geom_##sfx(int lg);                                                                                  \
    int col_direct_max_lg_##sfx();

HPXFFT_DECL_LAUNCH(f64)
HPXFFT_DECL_LAUNCH(f32)
HPXFFT_DECL_LAUNCH(f16)
HPXFFT_DECL_LAUNCH(bf16)

// columns of 2^11 and 2^12 points in one launch (fft_col_long.hpp; FP64 / FP32):
// gx strips of col_long_width columns, gz grids, nt threads per workgroup
hipError_t col_long_f64(int lg, bool conj, const ColArgs &a, unsigned gx, unsigned gz, int nt, hipStream_t s);
hipError_t col_long_f32(int lg, bool conj, const ColArgs &a, unsigned gx, unsigned gz, int nt, hipStream_t s);
inline hipError_t col_long(int p, int lg, bool conj, const ColArgs &a, unsigned gx, unsigned gz, int nt, hipStream_t s)
{
    switch (p)
    {
    case P_F64: return col_long_f64(lg, conj, a, gx, gz, nt, s);
    case P_F32: return col_long_f32(lg, conj, a, gx, gz, nt, s);
    default: return hipErrorInvalidValue;
    }
}
inline bool col_long_covers(int prec, int lg)
{
    return (prec == P_F64 || prec == P_F32) && lg >= hpxfft_dev::COL_LONG_MIN_LG && lg <= hpxfft_dev::COL_LONG_MAX_LG;
}
// adjacent columns per workgroup of nt threads (64 VGPRs of data per thread)
inline int col_long_width(int prec, int lg, int nt) { return (nt * (prec == P_F64 ? 16 : 32)) >> lg; }
// threads per workgroup.  2^11 rows: 512 (64-byte row segments, two workgroups
// per CU; 1024 threads with 128-byte segments were slower up to 4096 reals per
// row and even beyond).  2^12 rows: 1024 (64-byte segments, one workgroup per CU),
// except where the last of one or two rounds over the CUs is at most half full: there
// the narrow form, with half the columns and twice the workgroups, has one of them per
// CU where the wide one leaves CUs idle.  In a second round its 32-byte segments have
// to be made up for: FP64 gains only while that round is an eighth full; FP32, whose
// wide kernel spills 32 bytes per lane, as long as in the first.  Whole transforms out
// of place, buffers beyond the caches, narrow against wide (us, forward / c2r):
//   strips   64            112           128           136           272           304           384           400
//   FP64  -4.0 -5.7     -3.4 -5.4     -1.0 -4.0     +2.6 +1.2     -2.8 +0.2     -1.3 +2.7     +1.3 +3.5     +9.6 +13.9
//   FP32  -4.8 -7.8     -4.0 -7.6     -3.2 -6.9     +3.7 -2.6     -6.2 -4.8     -5.8 -2.7     -4.1 -4.2     +3.4 +8.0
// (FP64 4096 x 1000, 126 strips, 41.7 -> 38.7; FP32 4096 x 4800, 301, 122.6 -> 118.7.)
// In a third round it depends on more than the fill (513 strips: FP64 +9.2 +5.5, FP32
// -4.2 -1.1), and from four on the wide form wins (1025: FP64 columns 101 against 119).
inline int col_long_threads(int prec, int lg, size_t ncols, size_t batch)
{
    constexpr size_t CUS = 256;   // MI355X
    if (lg == 11) return 512;
    const size_t w = (size_t)col_long_width(prec, lg, 1024), strips = (ncols + w - 1) / w * batch;
    const size_t second = prec == P_F64 ? CUS / 8 : CUS / 2;
    return strips <= CUS / 2 || (strips > CUS && strips <= CUS + second) ? 512 : 1024;
}

// rows of 2^13 / 2^14 complex points with lane-pair radix-32 stages
// (fft_row_pair.hpp; FP32 arithmetic: FP32 and 16-bit storage); `total` rows
inline hipError_t row_r2c_pair(int p, int lg, const RowArgs &a, unsigned total, hipStream_t s)
{
    switch (p)
    {
    case P_F32: return row_r2c_pair_f32(lg, a, total, s);
    case P_F16: return row_r2c_pair_f16(lg, a, total, s);
    case P_BF16: return row_r2c_pair_bf16(lg, a, total, s);
    default: return hipErrorInvalidValue;
    }
}
inline bool row_pair_covers(int prec, int lg) { return prec != P_F64 && (lg == 13 || lg == 14); }

inline hipError_t row_r2c(int p, int lg, const RowArgs &a, unsigned gx, unsigned gy, hipStream_t s)
{
    switch (p)
    {
    case P_F64: return row_r2c_f64(lg, a, gx, gy, s);
    case P_F32: return row_r2c_f32(lg, a, gx, gy, s);
    case P_F16: return row_r2c_f16(lg, a, gx, gy, s);
    default: return row_r2c_bf16(lg, a, gx, gy, s);
    }
}
// halve: adjoint (interior bins halved); otherwise the unnormalised inverse c2r
inline hipError_t row_c2r(int p, int lg, bool halve, const RowArgs &a, unsigned gx, unsigned gy, hipStream_t s)
{
    switch (p)
    {
    case P_F64: return row_c2r_f64(lg, halve, a, gx, gy, s);
    case P_F32: return row_c2r_f32(lg, halve, a, gx, gy, s);
    default: return hipErrorInvalidValue;
    }
}
inline hipError_t col(int p, int lg, int mode, bool conj, const ColArgs &a, unsigned gx, unsigned gy, unsigned gz,
                      hipStream_t s)
{
    switch (p)
    {
    case P_F64: return col_f64(lg, mode, conj, a, gx, gy, gz, s);
    case P_F32: return col_f32(lg, mode, conj, a, gx, gy, gz, s);
    case P_F16: return col_f16(lg, mode, conj, a, gx, gy, gz, s);
    default: return col_bf16(lg, mode, conj, a, gx, gy, gz, s);
    }
}
inline geom row_geom(int p, int lg)
{
    switch (p)
    {
    case P_F64: return row_geom_f64(lg);
    case P_F32: return row_geom_f32(lg);
    case P_F16: return row_geom_f16(lg);
    default: return row_geom_bf16(lg);
    }
}
inline geom col_geom(int p, int lg)
{
    switch (p)
    {
    case P_F64: return col_geom_f64(lg);
    case P_F32: return col_geom_f32(lg);
    case P_F16: return col_geom_f16(lg);
    default: return col_geom_bf16(lg);
    }
}
inline geom tile_geom(int p, int lg)
{
    switch (p)
    {
    case P_F64: return tile_geom_f64(lg);
    case P_F32: return tile_geom_f32(lg);
    case P_F16: return tile_geom_f16(lg);
    default: return tile_geom_bf16(lg);
    }
}
inline int col_direct_max_lg(int p)
{
    switch (p)
    {
    case P_F64: return col_direct_max_lg_f64();
    case P_F32: return col_direct_max_lg_f32();
    case P_F16: return col_direct_max_lg_f16();
    default: return col_direct_max_lg_bf16();
    }
}

}   // namespace hpxfft_host

// ---------------------------------------------------------------------------
// instantiation helpers, used by inst_<prec>.hip only
#ifdef HPXFFT_INSTANTIATE
namespace hpxfft_host {
namespace detail {
using namespace hpxfft_dev;

template <typename T, typename S, int LG> constexpr bool use_big_row()
{
    return LG == 11 || LG == 13 || LG == 14;
}
template <typename T, typename S, int LG>
hipError_t launch_row_r2c(const RowArgs &a, unsigned gx, unsigned gy, hipStream_t s)
{
    if constexpr (use_big_row<T, S, LG>())
    {
        (void)gx;
        const unsigned total = (unsigned)a.nrows * gy;
        hipLaunchKernelGGL((row_r2c_big_kernel<T, S, S, LG>), dim3(total), dim3((1 << LG) / (16 * big_nb<T, LG>())), 0,
                           s, a);
    }
    else
    {
        hipLaunchKernelGGL((row_r2c_kernel<T, S, S, LG>), dim3(gx, gy), dim3(cfg<T, S>::row_NT(LG)), 0, s, a);
    }
    return hipGetLastError();
}

template <typename T, typename S>
hipError_t launch_row_r2c_pair(int lg, const RowArgs &a, unsigned total, hipStream_t s)
{
    if constexpr (sizeof(T) == 8) return hipErrorInvalidValue;   // FP64 rows keep the radix-16 kernel
    else if (lg == 13) hipLaunchKernelGGL((row_r2c_pair_kernel<T, S, S, 13>), dim3(total), dim3(256), 0, s, a);
    else if (lg == 14) hipLaunchKernelGGL((row_r2c_pair_kernel<T, S, S, 14>), dim3(total), dim3(512), 0, s, a);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}

template <typename T, typename S, int LG>
hipError_t launch_row_c2r(bool halve, const RowArgs &a, unsigned gx, unsigned gy, hipStream_t s)
{
    if constexpr (use_big_row<T, S, LG>())
    {
        // long rows: the radix-16 stages of the forward kernel, one row per workgroup
        (void)gx;
        const unsigned total = (unsigned)a.nrows * gy;
        const dim3 nt((1 << LG) / (16 * big_nb<T, LG>()));
        if (halve) hipLaunchKernelGGL((row_c2r_big_kernel<T, S, LG, true>), dim3(total), nt, 0, s, a);
        else hipLaunchKernelGGL((row_c2r_big_kernel<T, S, LG, false>), dim3(total), nt, 0, s, a);
    }
    else if (halve)
        hipLaunchKernelGGL((row_c2r_kernel<T, S, S, LG, true>), dim3(gx, gy), dim3(cfg<T, S>::row_NT(LG)), 0, s, a);
    else
        hipLaunchKernelGGL((row_c2r_kernel<T, S, S, LG, false>), dim3(gx, gy), dim3(cfg<T, S>::row_NT(LG)), 0, s, a);
    return hipGetLastError();
}
template <typename T, typename S, int LG, int MODE, bool CONJ>
hipError_t launch_col(const ColArgs &a, unsigned gx, unsigned gy, unsigned gz, hipStream_t s)
{
    if constexpr (MODE != 0)
    {
        // four-step tiles: specialised two-stage kernel (scratch in the compute type), gz = grids
        hipLaunchKernelGGL((tile_kernel<T, S, LG, MODE, CONJ>), dim3(gx, gy, gz), dim3((cfg<T, S>::TW << LG) / 16), 0,
                           s, a);
    }
    else
    {
        hipLaunchKernelGGL((col_kernel<T, S, LG, CONJ>), dim3(gx, gy, gz), dim3(cfg<T, S>::col_NT(LG)), 0, s, a);
    }
    return hipGetLastError();
}

template <typename T, int LG, int NT>
void launch_col_long_nt(bool conj, const ColArgs &a, unsigned gx, unsigned gz, hipStream_t s)
{
    if (conj) hipLaunchKernelGGL((col_long_kernel<T, LG, NT, true>), dim3(gx, 1, gz), dim3(NT), 0, s, a);
    else hipLaunchKernelGGL((col_long_kernel<T, LG, NT, false>), dim3(gx, 1, gz), dim3(NT), 0, s, a);
}
template <typename T>
hipError_t launch_col_long(int lg, bool conj, const ColArgs &a, unsigned gx, unsigned gz, int nt, hipStream_t s)
{
    if (lg == 11 && nt == 512) launch_col_long_nt<T, 11, 512>(conj, a, gx, gz, s);
    else if (lg == 12 && nt == 512) launch_col_long_nt<T, 12, 512>(conj, a, gx, gz, s);
    else if (lg == 12 && nt == 1024) launch_col_long_nt<T, 12, 1024>(conj, a, gx, gz, s);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}

template <typename T, typename S, int LG = 0>
hipError_t row_r2c_sw(int lg, const RowArgs &a, unsigned gx, unsigned gy, hipStream_t s)
{
    if constexpr (LG > ROW_MAX_LG) return hipErrorInvalidValue;
    else return lg == LG ? launch_row_r2c<T, S, LG>(a, gx, gy, s) : row_r2c_sw<T, S, LG + 1>(lg, a, gx, gy, s);
}
template <typename T, typename S, int LG = 0>
hipError_t row_c2r_sw(int lg, bool halve, const RowArgs &a, unsigned gx, unsigned gy, hipStream_t s)
{
    if constexpr (LG > ROW_MAX_LG) return hipErrorInvalidValue;
    else
        return lg == LG ? launch_row_c2r<T, S, LG>(halve, a, gx, gy, s)
                        : row_c2r_sw<T, S, LG + 1>(lg, halve, a, gx, gy, s);
}
template <typename T, typename S, bool ADJ, int LG = 0>
hipError_t col_sw(int lg, int mode, bool conj, const ColArgs &a, unsigned gx, unsigned gy, unsigned gz, hipStream_t s)
{
    constexpr int DMAX = cfg<T, S>::col_direct_max_lg;
    if constexpr (LG > DMAX && LG > COL_TILE_MAX_LG) return hipErrorInvalidValue;
    else
    {
        if (lg == LG)
        {
            if (mode == 0)
            {
                if constexpr (LG <= DMAX)
                {
                    if (!conj) return launch_col<T, S, LG, 0, false>(a, gx, gy, gz, s);
                    if constexpr (ADJ) return launch_col<T, S, LG, 0, true>(a, gx, gy, gz, s);
                }
                return hipErrorInvalidValue;
            }
            if constexpr (LG >= COL_TILE_MIN_LG && LG <= COL_TILE_MAX_LG)
            {
                if (!conj)
                    return mode == 1 ? launch_col<T, S, LG, 1, false>(a, gx, gy, gz, s)
                                     : launch_col<T, S, LG, 2, false>(a, gx, gy, gz, s);
                if constexpr (ADJ)
                    return mode == 1 ? launch_col<T, S, LG, 1, true>(a, gx, gy, gz, s)
                                     : launch_col<T, S, LG, 2, true>(a, gx, gy, gz, s);
            }
            return hipErrorInvalidValue;
        }
        return col_sw<T, S, ADJ, LG + 1>(lg, mode, conj, a, gx, gy, gz, s);
    }
}

template <typename T, typename S, bool ADJ>
hipError_t row_c2r_maybe(int lg, bool halve, const RowArgs &a, unsigned gx, unsigned gy, hipStream_t s)
{
    if constexpr (ADJ) return row_c2r_sw<T, S>(lg, halve, a, gx, gy, s);
    else return hipErrorInvalidValue;
}

template <typename T, typename S> geom row_geom_t(int lg)
{
    using C = cfg<T, S>;
    if (lg == 11 || lg == 13 || lg == 14)
    {
        const int nb = sizeof(T) == 4 && lg >= 13 ? 2 : 1;   // as big_nb<T, LG>()
        return geom{(1 << lg) / (16 * nb), 1, 16 * nb, (long)((1 << lg) + (1 << lg) / 16) * 2 * (long)sizeof(T) > 40 * 1024};
    }
    return geom{C::row_NT(lg), C::row_NSEQ(lg), C::row_E(lg), C::row_SPLIT(lg)};
}
template <typename T, typename S> geom col_geom_t(int lg)
{
    using C = cfg<T, S>;
    return geom{C::col_NT(lg), C::W, C::col_E(lg), C::col_SPLIT(lg)};
}
template <typename T, typename S> geom tile_geom_t(int lg)
{
    using C = cfg<T, S>;
    return geom{C::tile_NT(lg), C::TW, C::tile_E(lg), C::tile_SPLIT(lg)};
}
}   // namespace detail
}   // namespace hpxfft_host

#define HPXFFT_DEFINE_COL_LONG(sfx, T)                                                                             \
    namespace hpxfft_host {                                                                                        \
    hipError_t col_long_##sfx(int lg, bool conj, const ColArgs &a, unsigned gx, unsigned gz, int nt,               \
                              hipStream_t s)                                                                       \
    {                                                                                                              \
        return detail::launch_col_long<T>(lg, conj, a, gx, gz, nt, s);                                             \
    }                                                                                                              \
    }
#define HPXFFT_DEFINE_LAUNCH(sfx, T, S, ADJ)                                                                         \
    namespace hpxfft_host {                                                                                        \
    hipError_t row_r2c_##sfx(int lg, const RowArgs &a, unsigned gx, unsigned gy, hipStream_t s)                    \
    {                                                                                                              \
        return detail::row_r2c_sw<T, S>(lg, a, gx, gy, s);                                                         \
    }                                                                                                              \
    hipError_t row_r2c_pair_##sfx(int lg, const RowArgs &a, unsigned total, hipStream_t s)                        \
    {                                                                                                              \
        return detail::launch_row_r2c_pair<T, S>(lg, a, total, s);                                                 \
    }                                                                                                              \
    hipError_t row_c2r_##sfx(int lg, bool halve, const RowArgs &a, unsigned gx, unsigned gy, hipStream_t s)        \
    {                                                                                                              \
        return detail::row_c2r_maybe<T, S, ADJ>(lg, halve, a, gx, gy, s);                                          \
    }                                                                                                              \
    hipError_t col_##sfx(int lg, int mode, bool conj, const ColArgs &a, unsigned gx, unsigned gy, unsigned gz,     \
                         hipStream_t s)                                                                            \
    {                                                                                                              \
        return detail::col_sw<T, S, ADJ>(lg, mode, conj, a, gx, gy, gz, s);                                        \
    }                                                                                                              \
    geom row_geom_##sfx(int lg) { return detail::row_geom_t<T, S>(lg); }                                           \
    geom col_geom_##sfx(int lg) { return detail::col_geom_t<T, S>(lg); }                                           \
    geom tile_geom_##sfx(int lg) { return detail::tile_geom_t<T, S>(lg); }                                         \
    int col_direct_max_lg_##sfx() { return hpxfft_dev::cfg<T, S>::col_direct_max_lg; }                             \
    }
#endif
