// Passes 1 + 2 and 4 + 5 of the matvec as one kernel each, for small planes:
// a workgroup holds an (axis 1, axis 2) plane of one component and axis-3
// index in LDS between the two transforms, so W1 is neither written nor read
// and a matvec is three launches instead of five.
#pragma once
#include "gla_launch.hpp"

namespace gla {

// Branch lengths the plane kernels are built for (axis 1 and axis 2).  The
// line lies at 64 x 64, us a matvec in five launches / in three: 16^3 c64
// 17.0 / 12.8, 32^3 c64 23.7 / 19.1, c128 30.7 / 25.3, 48^3 c64 40.1 / 37.4,
// c128 53.6 / 53.2, 64^3 c64 47.7 / 43.7, c128 78.0 / 71.7, eight right-hand
// sides on 64x64x48 c64 212 / 172; 96x64x64 c64 65.8 / 69.5, 128x64x48 c64
// 68.5 / 71.3 (one plane a CU, its load, transform and store in a row).
#define GLA_FOR_EACH_PLANE(X) X(8) X(12) X(16) X(20) X(24) X(32) X(40) X(48) X(64)

// Shape of a plane kernel: TPX threads per row (inside one wave), TPY threads
// per column, CF / CI columns of the forward / inverse kernel side by side
// (a divisor of the plane's columns, so no column is masked).
__host__ __device__ constexpr int plane_div(int cols, int tpy, int lim)
{
    int best = 1;
    for (int d = 1; d <= cols; ++d)
        if (cols % d == 0 && d * tpy <= lim) best = d;
    return best;
}

template <typename R, int N1, int N2>
struct PlaneK {
    // up to 1024 threads: all columns in one sweep (64^3 c128 74 -> 72 us
    // against 512)
    static constexpr int CB = (int)sizeof(cpx<R>), LIM = 1024;
    static constexpr int EX = pick_e(N1, rtune(CB, N1).ex, 64, true, ptune(CB, N1)), TPX = N1 / EX;
    static constexpr int EY = pick_e(N2, rtune(CB, N2).ey, 64, false, ptune(CB, N2)), TPY = N2 / EY;
    static constexpr int CF = plane_div(N1, TPY, LIM), CI = plane_div(2 * N1, TPY, LIM);
    static constexpr int NTF = CF * TPY, NTI = CI * TPY;
    // both parities of a column through the stages together where the two
    // exchange buffers fit 64 KB, else one after the other
    static constexpr int KF = plane_k(CB, N1, N2), KI = plane_k(CB, 2 * N1, N2);
};

// --------------------------------------------------------------------------
// Passes 1 + 2.  One workgroup: axis-1 parity blockIdx.y of the plane (i3, c)
// = blockIdx.x of slot blockIdx.z.  plane[i2 N1 + m1]: rows are transformed
// in place (wave-local), then each column's slots are its exchange buffer.
// --------------------------------------------------------------------------
template <typename R, int N1, int N2, bool ONCE>
__global__ __launch_bounds__((PlaneK<R, N1, N2>::NTF)) void k_fwd_xy(
    const cpx<R>* __restrict__ X, cpx<R>* __restrict__ W2, int S1, int S2, int S3, int Z, int64_t xs, int64_t w2s,
    const cpx<R>* __restrict__ phz1, const cpx<R>* __restrict__ tw1, const cpx<R>* __restrict__ phz2,
    const cpx<R>* __restrict__ tw2, Part xp)
{
    using K = PlaneK<R, N1, N2>;
    constexpr int NT = K::NTF, EX = K::EX, TPX = K::TPX, EY = K::EY, TPY = K::TPY, RG = NT / TPX > 0 ? NT / TPX : 1;
    static_assert(NT >= TPX, "a row fits the workgroup");
    extern __shared__ __align__(16) unsigned char smem[];
    cpx<R>* const t1 = reinterpret_cast<cpx<R>*>(smem);   // roots and phases of axis 1, then of axis 2
    cpx<R>* const t2 = t1 + 2 * N1;
    cpx<R>* const plane = t2 + 2 * N2;
    const int i3 = blockIdx.x % S3, c = blockIdx.x / S3, p1 = blockIdx.y;
    int po[3];
    const int rhs = part_slot(xp, blockIdx.z, po);
    const cpx<R>* const xq =
        X + (int64_t)rhs * xs + (((int64_t)c * xp.f[2] + (int64_t)i3 * xp.d[2] + po[2]) * xp.f[1] + po[1]) * xp.f[0] + po[0];
    const int xd = xp.d[0];
    {
        const int t = threadIdx.x % TPX, grp = threadIdx.x / TPX;
        cpx<R> v[EX];
        auto load = [&](int i2) {
            const cpx<R>* const xr = xq + (int64_t)i2 * xp.d[1] * xp.f[0];
#pragma unroll
            for (int e = 0; e < EX; ++e) {
                const int n = t + TPX * e;
                cpx<R> a = {R(0), R(0)}, b = {R(0), R(0)};
                if (n < S1) a = xr[(int64_t)n * xd];
                if (n + N1 < S1) b = xr[(int64_t)(n + N1) * xd];
                v[e] = p1 ? a - b : a + b;
            }
        };
        // the first rows are on their way while the tables are staged
        const bool any = grp < RG && grp < S2;
        if (any) load(grp);
        for (int i = threadIdx.x; i < N1; i += NT) {
            t1[i] = tw1[i];
            t1[N1 + i] = phz1[i];
        }
        for (int i = threadIdx.x; i < N2; i += NT) {
            t2[i] = tw2[i];
            t2[N2 + i] = phz2[i];
        }
        __syncthreads();
        if (any)
            for (int i2 = grp; i2 < S2; i2 += RG) {
                if (i2 != grp) load(i2);
                if (p1) {
#pragma unroll
                    for (int e = 0; e < EX; ++e) v[e] = t1[N1 + t + TPX * e] * v[e];
                }
                PencilFft<R, N1, TPX, 1, N1, false, 1>::run(v, plane, t, i2, t1);
#pragma unroll
                for (int e = 0; e < EX; ++e) plane[i2 * N1 + t + TPX * e] = v[e];
            }
    }
    __syncthreads();
    const int xl = threadIdx.x % K::CF, t = threadIdx.x / K::CF;
    cpx<R>* const w = W2 + (int64_t)blockIdx.z * w2s + ((int64_t)c * Z + i3) * (int64_t)(4 * N1 * N2) + p1 * N1;
    for (int m = xl; m < N1; m += K::CF) {
        cpx<R> v[2][EY];
#pragma unroll
        for (int e = 0; e < EY; ++e) {
            const int n = t + TPY * e;
            const cpx<R> a = n < S2 ? plane[n * N1 + m] : cpx<R>{R(0), R(0)};
            const cpx<R> b = n + N2 < S2 ? plane[(n + N2) * N1 + m] : cpx<R>{R(0), R(0)};
            v[0][e] = a + b;
            v[1][e] = t2[N2 + n] * (a - b);
        }
        __syncthreads();
        if constexpr (K::KF == 2) {
            PencilFft<R, N2, TPY, N1, 1, false, 0, 2, N1 * N2>::run(v, plane, t, m, t2);
        } else {
#pragma unroll
            for (int p = 0; p < 2; ++p) PencilFft<R, N2, TPY, N1, 1, false>::run(v[p], plane, t, m, t2);
        }
#pragma unroll
        for (int p = 0; p < 2; ++p)
#pragma unroll
            for (int e = 0; e < EY; ++e) st<ONCE>(&w[(int64_t)(p * N2 + t + TPY * e) * (2 * N1) + m], v[p][e]);
    }
}

// --------------------------------------------------------------------------
// Passes 4 + 5.  One workgroup: the plane (i3, c) = blockIdx.x of slot
// blockIdx.y, both axis-1 parities (the merge needs them): plane[n2 2 N1 + m1].
// --------------------------------------------------------------------------
template <typename R, int N1, int N2, bool ONCE>
__global__ __launch_bounds__((PlaneK<R, N1, N2>::NTI)) void k_inv_yx(
    const cpx<R>* __restrict__ W2, cpx<R>* __restrict__ Y, int T1, int T2, int T3, int Z, int64_t w2s, int64_t ys,
    const cpx<R>* __restrict__ phz1, const cpx<R>* __restrict__ tw1, const cpx<R>* __restrict__ phz2,
    const cpx<R>* __restrict__ tw2, cpx<R> alpha, cpx<R> beta, int axpby, const cpx<R>* __restrict__ lsx, int64_t lsxs,
    const cpx<R>* __restrict__ chi, int64_t chis, Part yp)
{
    using K = PlaneK<R, N1, N2>;
    constexpr int NT = K::NTI, EX = K::EX, TPX = K::TPX, EY = K::EY, TPY = K::TPY, RG = NT / TPX > 0 ? NT / TPX : 1;
    static_assert(NT >= TPX, "a row fits the workgroup");
    constexpr int L1 = 2 * N1;
    extern __shared__ __align__(16) unsigned char smem[];
    cpx<R>* const t1 = reinterpret_cast<cpx<R>*>(smem);
    cpx<R>* const t2 = t1 + 2 * N1;
    cpx<R>* const plane = t2 + 2 * N2;
    const int i3 = blockIdx.x % T3, c = blockIdx.x / T3;
    {
        const int xl = threadIdx.x % K::CI, t = threadIdx.x / K::CI;
        const cpx<R>* const w = W2 + (int64_t)blockIdx.y * w2s + ((int64_t)c * Z + i3) * (int64_t)(2 * N2 * L1);
        cpx<R> v[2][EY];
        auto load = [&](int m) {
#pragma unroll
            for (int p = 0; p < 2; ++p)
#pragma unroll
                for (int e = 0; e < EY; ++e) v[p][e] = ld<ONCE>(&w[(int64_t)(p * N2 + t + TPY * e) * L1 + m]);
        };
        load(xl);   // on its way while the tables are staged
        for (int i = threadIdx.x; i < N1; i += NT) {
            t1[i] = tw1[i];
            t1[N1 + i] = phz1[i];
        }
        for (int i = threadIdx.x; i < N2; i += NT) {
            t2[i] = tw2[i];
            t2[N2 + i] = phz2[i];
        }
        __syncthreads();
        for (int m = xl; m < L1; m += K::CI) {
            if (m != xl) load(m);
            if constexpr (K::KI == 2) {
                PencilFft<R, N2, TPY, L1, 1, true, 0, 2, L1 * N2>::run(v, plane, t, m, t2);
            } else {
#pragma unroll
                for (int p = 0; p < 2; ++p) PencilFft<R, N2, TPY, L1, 1, true>::run(v[p], plane, t, m, t2);
            }
#pragma unroll
            for (int e = 0; e < EY; ++e) {
                const int n = t + TPY * e;
                const cpx<R> o = cmulc(v[1][e], t2[N2 + n]);
                if (n < T2) plane[n * L1 + m] = v[0][e] + o;
                if (n + N2 < T2) plane[(n + N2) * L1 + m] = v[0][e] - o;
            }
        }
    }
    __syncthreads();
    int po[3];
    const int rhs = part_slot(yp, blockIdx.y, po);
    cpx<R>* const yq =
        Y + (int64_t)rhs * ys + (((int64_t)c * yp.f[2] + (int64_t)i3 * yp.d[2] + po[2]) * yp.f[1] + po[1]) * yp.f[0] + po[0];
    const int yd = yp.d[0];
    const bool rd = axpby == 1 && !(beta.x == R(0) && beta.y == R(0));
    const int t = threadIdx.x % TPX, grp = threadIdx.x / TPX;
    if (grp >= RG) return;
    for (int i2 = grp; i2 < T2; i2 += RG) {
        cpx<R> v[2][EX];
#pragma unroll
        for (int p = 0; p < 2; ++p)
#pragma unroll
            for (int e = 0; e < EX; ++e) v[p][e] = plane[i2 * L1 + p * N1 + t + TPX * e];
        lds_sync<1>();
        PencilFft<R, N1, TPX, 1, L1, true, 1, 2, N1>::run(v, plane, t, i2, t1);
        cpx<R>* const yr = yq + (int64_t)i2 * yp.d[1] * yp.f[0];
        const int64_t row = ((int64_t)c * T3 + i3) * T2 + i2, cell0 = ((int64_t)i3 * T2 + i2) * T1;
        auto epilogue = [&](cpx<R> r, int n) {
            const int64_t ny = (int64_t)n * yd;
            if (axpby == 1) r = alpha * r + (rd ? beta * yr[ny] : cpx<R>{R(0), R(0)});
            else if (axpby == 2)
                r = lsx[(int64_t)blockIdx.y * lsxs + row * T1 + n] - chi[(int64_t)blockIdx.y * chis + cell0 + n] * r;
            st<ONCE>(&yr[ny], r);
        };
        const int top = T1 < N1 ? T1 : N1;
#pragma unroll
        for (int e = 0; e < EX; ++e) {
            const int n = t + TPX * e;
            const cpx<R> o = cmulc(v[1][e], t1[N1 + n]);
            if (n < top) epilogue(v[0][e] + o, n);
            if (n + N1 < T1) epilogue(v[0][e] - o, n + N1);
        }
    }
}

}  // namespace gla
