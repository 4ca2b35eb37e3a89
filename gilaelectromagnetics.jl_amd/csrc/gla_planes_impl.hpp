// Launches of the plane kernels; included by gla_xy_c64.hip (R = float) and
// gla_xy_c128.hip (R = double).
#pragma once
#include "gla_launch.hpp"
#include "gla_planes.hpp"

// the list again, for the nested expansion of (axis 1, axis 2) pairs
#define GLA_FOR_EACH_PLANE2(X) X(8) X(12) X(16) X(20) X(24) X(32) X(40) X(48) X(64)

namespace gla {

template <typename K>
static hipError_t plane_lds(K kernel, size_t lds)
{
    return lds > 65536 ? hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds)
                       : hipSuccess;
}

template <typename R, int N1, int N2>
static hipError_t fwd_plane(const Geom& g, const DevTab& tb, const void* X, void* W2, int slots, hipStream_t st)
{
    const auto kernel = streams(g.w2s * slots * (int)sizeof(cpx<R>))
                            ? k_fwd_xy<R, N1, N2, true>
                            : k_fwd_xy<R, N1, N2, false>;
    const size_t lds = plane_bytes(g, (int)sizeof(cpx<R>), false);
    const hipError_t e = plane_lds(kernel, lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(kernel, dim3(g.S[2] * 3, 2, slots), dim3(PlaneK<R, N1, N2>::NTF), lds, st, (const cpx<R>*)X,
                       (cpx<R>*)W2, g.S[0], g.S[1], g.S[2], g.Z, g.xs, g.w2s, (const cpx<R>*)tb.phz[0],
                       (const cpx<R>*)tb.tw[0], (const cpx<R>*)tb.phz[1], (const cpx<R>*)tb.tw[1], g.xp);
    return hipGetLastError();
}

template <typename R, int N1, int N2>
static hipError_t inv_plane(const Geom& g, const DevTab& tb, const void* W2, void* Y, int slots, cpx<R> al, cpx<R> be,
                            int axpby, const Epi& epi, hipStream_t st)
{
    const auto kernel = streams(g.w2s * slots * (int)sizeof(cpx<R>))
                            ? k_inv_yx<R, N1, N2, true>
                            : k_inv_yx<R, N1, N2, false>;
    const size_t lds = plane_bytes(g, (int)sizeof(cpx<R>), true);
    const hipError_t e = plane_lds(kernel, lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(kernel, dim3(g.T[2] * 3, slots), dim3(PlaneK<R, N1, N2>::NTI), lds, st, (const cpx<R>*)W2,
                       (cpx<R>*)Y, g.T[0], g.T[1], g.T[2], g.Z, g.w2s, g.ys, (const cpx<R>*)tb.phz[0],
                       (const cpx<R>*)tb.tw[0], (const cpx<R>*)tb.phz[1], (const cpx<R>*)tb.tw[1], al, be, axpby,
                       (const cpx<R>*)epi.x, epi.xs, (const cpx<R>*)epi.chi, epi.chis, g.yp);
    return hipGetLastError();
}

template <typename R>
hipError_t run_fwd_planes(const Geom& g, const DevTab& tb, const void* X, void* W2, int slots, hipStream_t st)
{
#define GLA_Y(n2) case n2: return fwd_plane<R, N1, n2>(g, tb, X, W2, slots, st);
#define GLA_X(n1) case n1: { constexpr int N1 = n1; switch (g.B[1]) { GLA_FOR_EACH_PLANE(GLA_Y) default: break; } break; }
    switch (g.B[0]) { GLA_FOR_EACH_PLANE2(GLA_X) default: break; }
#undef GLA_X
#undef GLA_Y
    return hipErrorInvalidValue;
}

template <typename R>
hipError_t run_inv_planes(const Geom& g, const DevTab& tb, const void* W2, void* Y, int slots, double ar, double ai,
                          double br, double bi, int axpby, const Epi& epi, hipStream_t st)
{
    const cpx<R> al{R(ar), R(ai)}, be{R(br), R(bi)};
#define GLA_Y(n2) case n2: return inv_plane<R, N1, n2>(g, tb, W2, Y, slots, al, be, axpby, epi, st);
#define GLA_X(n1) case n1: { constexpr int N1 = n1; switch (g.B[1]) { GLA_FOR_EACH_PLANE(GLA_Y) default: break; } break; }
    switch (g.B[0]) { GLA_FOR_EACH_PLANE2(GLA_X) default: break; }
#undef GLA_X
#undef GLA_Y
    return hipErrorInvalidValue;
}

}  // namespace gla
