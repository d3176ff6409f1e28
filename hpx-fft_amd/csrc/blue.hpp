// blue.hpp -- host interface of the in-register Bluestein kernels (implemented
// in inst_blue_f64.hip and inst_blue_f32.hip): lg = log2 of the convolution length
#pragma once

#include "fft_blue.hpp"

namespace hpxfft_host {

using hpxfft_dev::BlueArgs;
using hpxfft_dev::ColArgs;
using hpxfft_dev::RowArgs;

#define HPXFFT_DECL_BLUE(sfx)                                                                                     \
    hipError_t blue_row_r2c_##sfx(int lg, const RowArgs &a, const BlueArgs &g, unsigned batch, hipStream_t s);    \
    hipError_t blue_row_c2r_##sfx(int lg, bool halve, const RowArgs &a, const BlueArgs &g, unsigned batch,        \
                                  hipStream_t s);                                                                 \
    hipError_t blue_col_##sfx(int lg, bool conj, const ColArgs &a, const BlueArgs &g, unsigned batch, hipStream_t s);
HPXFFT_DECL_BLUE(f64)
HPXFFT_DECL_BLUE(f32)


// rows or adjacent columns of a workgroup, and its threads
struct blue_geom { int w, nt; };
template <typename T, bool COL, int LG = hpxfft_dev::BLUE_MIN_LG> blue_geom blue_shape(int lg)
{
    using C = hpxfft_dev::bluecfg<T, LG, COL>;
    if constexpr (LG < (sizeof(T) == 8 ? hpxfft_dev::BLUE_MAX_LG_F64 : hpxfft_dev::BLUE_MAX_LG_F32))
        if (lg > LG) return blue_shape<T, COL, LG + 1>(lg);
    return {C::W, C::NT};
}

}   // namespace hpxfft_host

#ifdef HPXFFT_INSTANTIATE
namespace hpxfft_host {
namespace detail {
using namespace hpxfft_dev;

template <typename T> constexpr int blue_max_lg() { return sizeof(T) == 8 ? BLUE_MAX_LG_F64 : BLUE_MAX_LG_F32; }
// kind 0: row r2c (f ignored), 1: row c2r (f: halve), 2: columns (f: conjugate)
template <typename T, int LG = BLUE_MIN_LG>
hipError_t blue_sw(int kind, int lg, bool f, const RowArgs *r, const ColArgs *c, const BlueArgs &g, unsigned batch,
                   hipStream_t s)
{
    if constexpr (LG > blue_max_lg<T>()) return hipErrorInvalidValue;
    else
    {
        if (lg != LG) return blue_sw<T, LG + 1>(kind, lg, f, r, c, g, batch, s);
        using R = bluecfg<T, LG, false>;
        using C = bluecfg<T, LG, true>;
        if (g.len < 1 || 2 * g.len > R::L) return hipErrorInvalidValue;
        if (kind == 2)
        {
            const dim3 grid((unsigned)((c->ncols + C::W - 1) / C::W), batch);
            hipLaunchKernelGGL((blue_col_kernel<T, LG>), grid, dim3(C::NT), 0, s, *c, g, f ? T(-1) : T(1));
        }
        else
        {
            const dim3 grid((unsigned)((r->nrows + R::W - 1) / R::W), batch);
            if (kind == 0) hipLaunchKernelGGL((blue_row_r2c_kernel<T, LG>), grid, dim3(R::NT), 0, s, *r, g);
            else hipLaunchKernelGGL((blue_row_c2r_kernel<T, LG>), grid, dim3(R::NT), 0, s, *r, g, f ? T(0.5) : T(1));
        }
        return hipGetLastError();
    }
}
}   // namespace detail
}   // namespace hpxfft_host

#define HPXFFT_DEFINE_BLUE(sfx, T)                                                                                \
    namespace hpxfft_host {                                                                                       \
    hipError_t blue_row_r2c_##sfx(int lg, const RowArgs &a, const BlueArgs &g, unsigned batch, hipStream_t s)     \
    {                                                                                                             \
        return detail::blue_sw<T>(0, lg, false, &a, nullptr, g, batch, s);                                        \
    }                                                                                                             \
    hipError_t blue_row_c2r_##sfx(int lg, bool halve, const RowArgs &a, const BlueArgs &g, unsigned batch,        \
                                  hipStream_t s)                                                                  \
    {                                                                                                             \
        return detail::blue_sw<T>(1, lg, halve, &a, nullptr, g, batch, s);                                        \
    }                                                                                                             \
    hipError_t blue_col_##sfx(int lg, bool conj, const ColArgs &a, const BlueArgs &g, unsigned batch, hipStream_t s) \
    {                                                                                                             \
        return detail::blue_sw<T>(2, lg, conj, nullptr, &a, g, batch, s);                                         \
    }                                                                                                             \
    }   // namespace hpxfft_host
#endif
