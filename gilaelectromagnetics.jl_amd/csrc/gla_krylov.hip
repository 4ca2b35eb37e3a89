// Krylov-basis kernels for the batched Lippmann-Schwinger GMRES: block dot
// products h[r][i] = sum_n conj(V[r][i][n]) w[r][n], block updates
// w[r] += s sum_i h[r][i] V[r][i] (with the squared norm of the result), and
// the row gather / scaled scatter between a basis slab and a batch, for r < k
// right-hand sides and i < nv basis vectors of length n.  A right-hand side
// may use fewer vectors (ncol[r] < nv: a request in the middle of its own
// restart cycle); the kernels then read only its first ncol[r] vectors and
// its coefficients beyond them are zero.  The reference has
// no solver (its examples use IterativeSolvers' gmres on the host,
// docs/src/usage.md:370-391); these are the reductions a library GEMM handles
// badly at this shape (two tiny dimensions and one of millions).
//
// Every reduction is two-stage: workgroups reduce fixed chunks of one
// right-hand side (FP64 accumulators, a fixed shuffle tree), and one wave per
// output sums the chunk partials in a fixed order.  A right-hand side's
// results therefore do not depend on how many share the launch.
#include <hip/hip_runtime.h>

#include "gla_fft.hpp"
#include "gla_krylov.hpp"

namespace gla {
namespace {

constexpr int KT = 256;          // threads per chunk workgroup
constexpr int KW = KT / 64;      // waves per chunk workgroup
constexpr int KG = 16;           // basis vectors per sweep over a chunk (2 KG sums, half a wave's lanes)

// the sums' step, written out in FP64: the kernels' variants round alike
__device__ __forceinline__ double fma(double a, double b, double c) { return __builtin_fma(a, b, c); }

__device__ __forceinline__ double wave_sum(double v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    return v;
}

// VW consecutive elements as one load (16 bytes where the addresses allow it,
// see wide_ok)
template <typename R, int VW>
struct alignas(sizeof(cpx<R>) * VW) vec {
    cpx<R> e[VW];
};

// Bytes of basis that the last-level cache still holds between the products
// and the update of one pass (192 MiB of its 256 MB).  A larger basis is read
// with hints that its lines are not needed again -- in the products where more
// than this follows, in the update, whose reads are a step's last, from twice
// this on -- so that the rest of it, w and the matvec's planes stay.
// 8 right-hand sides, 16 vectors of 3 x 64 x 64 x 48 ComplexF32 elements: the
// products 117 -> 98 us back to back, an Arnoldi step 490 -> 470; 2 x 20
// vectors of 6291456 ComplexF64: both 1627 -> 1500.  The update of half that basis, 302
// MB, with the hint 66 -> 68, and products and update in turn 115 -> 125.
constexpr int64_t KEEP_BYTES = 192 << 20;

template <bool ONCE, typename V>
__device__ __forceinline__ V load_vec(const V* p)
{
    if constexpr (ONCE) {
        typedef uint32_t W __attribute__((ext_vector_type(sizeof(V) / 4), aligned(alignof(V))));
        return __builtin_bit_cast(V, __builtin_nontemporal_load(reinterpret_cast<const W*>(p)));
    } else {
        return *p;
    }
}

// one sweep over a chunk for G basis vectors i0 .. i0 + G - 1 (G = 0: the
// norm of w alone).  Every load of a step (w and the G vectors) is issued
// before the first use; a thread visits units of VW elements q = lo + VW t,
// lo + VW (t + KT), ... in ascending order.  A last partial unit (n odd,
// VW == 2) goes element by element.
template <typename R, int G, int VW, bool ONCE>
__device__ __forceinline__ void dots_sweep(const cpx<R>* __restrict__ vp, int64_t vv, int i0,
                                           const cpx<R>* __restrict__ wp, int64_t lo, int64_t hi, bool first,
                                           double (&acc)[2 * KG + 1])
{
    auto add = [&](const cpx<R>& b, const cpx<R>* a) {
        if (first) acc[2 * KG] = fma(b.x, b.x, fma(b.y, b.y, acc[2 * KG]));
#pragma unroll
        for (int g = 0; g < G; ++g) {
            acc[2 * g] = fma(a[g].x, b.x, fma(a[g].y, b.y, acc[2 * g]));   // conj(a) b
            acc[2 * g + 1] = fma(a[g].x, b.y, fma(-a[g].y, b.x, acc[2 * g + 1]));
        }
    };
    const cpx<R>* const v0 = vp + (int64_t)i0 * vv;
    int64_t q = lo + (int64_t)VW * threadIdx.x;
    for (; q + VW <= hi; q += (int64_t)KT * VW) {
        using V = vec<R, VW>;
        const V b = *reinterpret_cast<const V*>(wp + q);
        V a[G > 0 ? G : 1];
#pragma unroll
        for (int g = 0; g < G; ++g) a[g] = load_vec<ONCE>(reinterpret_cast<const V*>(v0 + g * vv + q));
        __builtin_amdgcn_sched_barrier(0);   // keep the step's loads ahead of the arithmetic
#pragma unroll
        for (int e = 0; e < VW; ++e) {
            cpx<R> ae[G > 0 ? G : 1];
#pragma unroll
            for (int g = 0; g < G; ++g) ae[g] = a[g].e[e];
            add(b.e[e], ae);
        }
    }
    if (VW > 1 && q < hi) {
        cpx<R> ae[G > 0 ? G : 1];
#pragma unroll
        for (int g = 0; g < G; ++g) ae[g] = v0[g * vv + q];
        add(wp[q], ae);
    }
}

template <typename R, int VW, int G, bool ONCE>
__device__ __forceinline__ void dots_count(int count, const cpx<R>* __restrict__ vp, int64_t vv, int i0,
                                           const cpx<R>* __restrict__ wp, int64_t lo, int64_t hi, bool first,
                                           double (&acc)[2 * KG + 1])
{
    if (count == G) dots_sweep<R, G, VW, ONCE>(vp, vv, i0, wp, lo, hi, first, acc);
    else if constexpr (G > 0) dots_count<R, VW, G - 1, ONCE>(count, vp, vv, i0, wp, lo, hi, first, acc);
}

// Block products of one chunk.  part layout: [r][slot][chunk]; slots 0..nv-1
// the dots, slot nv the squared norm of w (when requested).  Bound by HBM:
// each right-hand side's basis is read once (8 right-hand sides, 16 vectors
// of 3 x 64 x 64 x 48 ComplexF32 elements, 640 MB: 97 to 98 us with its sums
// back to back, where the last-level cache still holds part of the basis; 112
// to 114 us, 5.6 TB/s, and 5 for the sums inside an Arnoldi step, after the
// matvec's planes went through that cache).  Before, with 8 vectors a sweep,
// 8-byte loads, one wave sum per value and 4096-element chunks, it took 129
// us back to back, and 8 x 98304 elements 34 us (now 21).
template <typename R, int VW, bool LARGE>
__global__ __launch_bounds__(KT) void k_dots(const cpx<R>* __restrict__ V, int64_t vr, int64_t vv,
                                             const cpx<R>* __restrict__ w, int64_t wr, int64_t n, int nv,
                                             const int64_t* __restrict__ ncol, int64_t chunk, int nchunk, int nslot,
                                             int self, double* __restrict__ part)
{
    __shared__ double red[2 * KG + 1][KW];
    const int r = blockIdx.y, c = blockIdx.x;
    const int nvr = ncol ? (int)(ncol[r] < 0 ? 0 : ncol[r] < nv ? ncol[r] : nv) : nv;
    const int64_t lo = (int64_t)c * chunk;
    const int64_t hi = lo + chunk < n ? lo + chunk : n;
    // more basis behind this chunk than stays in the last-level cache
    const bool once = LARGE && ((int64_t)(gridDim.y - r) * n - lo) * nv * (int64_t)sizeof(cpx<R>) > KEEP_BYTES;
    const cpx<R>* wp = w + r * wr;
    const cpx<R>* vp = V + r * vr;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    double* pr = part + (int64_t)r * nslot * 2 * nchunk;
    // coefficients of the vectors this right-hand side does not use
    for (int t = threadIdx.x; t < 2 * (nv - nvr); t += KT) pr[((int64_t)nvr * 2 + t) * nchunk + c] = 0.0;
    for (int i0 = 0; i0 < nvr || (i0 == 0 && self); i0 += KG) {
        double acc[2 * KG + 1];
#pragma unroll
        for (int g = 0; g < 2 * KG + 1; ++g) acc[g] = 0.0;
        const bool first = i0 == 0 && self;
        const int count = nvr - i0 < KG ? nvr - i0 : KG;
        if (once) dots_count<R, VW, KG, LARGE>(count, vp, vv, i0, wp, lo, hi, first, acc);
        else dots_count<R, VW, KG, false>(count, vp, vv, i0, wp, lo, hi, first, acc);
        // the wave's 2 KG sums, halving the values a lane carries at each step:
        // lane l ends with value l / 2 (37 exchanges where a sum per value
        // takes 192)
#pragma unroll
        for (int o = 32, hv = KG; o > 1; o >>= 1, hv >>= 1) {
            const bool up = (lane & o) != 0;
#pragma unroll
            for (int g = 0; g < hv; ++g) {
                const double keep = up ? acc[g + hv] : acc[g], give = up ? acc[g] : acc[g + hv];
                acc[g] = keep + __shfl_xor(give, o);
            }
        }
        acc[0] += __shfl_xor(acc[0], 1);
        if ((lane & 1) == 0) red[lane >> 1][wv] = acc[0];
        if (first) {
            const double v = wave_sum(acc[2 * KG]);
            if (lane == 0) red[2 * KG][wv] = v;
        }
        __syncthreads();
        if (threadIdx.x < 2 * KG + 1) {
            const int g = threadIdx.x;
            if (g < 2 * KG ? g < 2 * count : first) {
                double sum = 0.0;
#pragma unroll
                for (int u = 0; u < KW; ++u) sum += red[g][u];
                const int64_t slot = g < 2 * KG ? ((int64_t)i0 * 2 + g) : (int64_t)nv * 2;
                pr[slot * nchunk + c] = sum;
            }
        }
        __syncthreads();
    }
}

// basis vectors per step of the update loop (their loads issued together)
constexpr int KU = 4;

// w[r] += s sum_i h[r][i] V[r][i] over one chunk; the chunk's squared norm
// of the result goes to part[r][0][chunk] when norm is set.  Each element
// sums its nv terms in order i = 0, 1, ...; a thread visits its elements in
// ascending order (E units of VW elements at a time).  Right-hand sides run
// last to first: the products before it read the basis first to last, so the
// end of it is still in the last-level cache (products and update of the
// same case together: 264 us first to last, 231 last to first, 224 with the
// hints of KEEP_BYTES).
template <typename R, int VW, bool ONCE>
__global__ __launch_bounds__(KT) void k_axpy(const cpx<R>* __restrict__ V, int64_t vr, int64_t vv,
                                             const cpx<double>* __restrict__ h, int64_t hr,
                                             cpx<R>* __restrict__ w, int64_t wr, int64_t n, int nv,
                                             const int64_t* __restrict__ ncol, double s, int64_t chunk, int nchunk,
                                             int norm, double* __restrict__ part)
{
    constexpr int E = 2;
    using U = vec<R, VW>;
    __shared__ double red[KW];
    const int r = gridDim.y - 1 - blockIdx.y, c = gridDim.x - 1 - blockIdx.x;
    if (ncol) nv = (int)(ncol[r] < 0 ? 0 : ncol[r] < nv ? ncol[r] : nv);
    const int64_t lo = (int64_t)c * chunk;
    const int64_t hi = lo + chunk < n ? lo + chunk : n;
    const cpx<R>* vp = V + r * vr;
    const cpx<double>* hp = h + r * hr;
    cpx<R>* wp = w + r * wr;
    double nrm = 0.0;
    auto finish = [&](cpx<R> o, double ar, double ai) {
        const cpx<R> res{R(fma(s, ar, (double)o.x)), R(fma(s, ai, (double)o.y))};
        nrm = fma(res.x, res.x, fma(res.y, res.y, nrm));
        return res;
    };
    const int64_t whole = lo + (hi - lo) / VW * VW;   // end of the whole units
    for (int64_t q0 = lo + (int64_t)VW * threadIdx.x; q0 < whole; q0 += (int64_t)KT * E * VW) {
        int64_t qe[E];
        bool ok[E];
        double ar[E][VW], ai[E][VW];
#pragma unroll
        for (int e = 0; e < E; ++e) {
            ok[e] = q0 + (int64_t)e * KT * VW < whole;
            qe[e] = ok[e] ? q0 + (int64_t)e * KT * VW : q0;
#pragma unroll
            for (int k = 0; k < VW; ++k) ar[e][k] = ai[e][k] = 0.0;
        }
        U o[E];
#pragma unroll
        for (int e = 0; e < E; ++e) o[e] = *reinterpret_cast<const U*>(wp + qe[e]);
        auto mac = [&](const cpx<double>& cc, int e, const U& a) {
#pragma unroll
            for (int k = 0; k < VW; ++k) {
                ar[e][k] = fma(cc.x, a.e[k].x, fma(-cc.y, a.e[k].y, ar[e][k]));
                ai[e][k] = fma(cc.x, a.e[k].y, fma(cc.y, a.e[k].x, ai[e][k]));
            }
        };
        int i = 0;
        for (; i + KU <= nv; i += KU) {
            U a[KU][E];
#pragma unroll
            for (int u = 0; u < KU; ++u)
#pragma unroll
                for (int e = 0; e < E; ++e)
                    a[u][e] = load_vec<ONCE>(reinterpret_cast<const U*>(vp + (int64_t)(i + u) * vv + qe[e]));
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = 0; u < KU; ++u) {
                const cpx<double> cc = hp[i + u];
#pragma unroll
                for (int e = 0; e < E; ++e) mac(cc, e, a[u][e]);
            }
        }
        for (; i < nv; ++i) {
            U a[E];
#pragma unroll
            for (int e = 0; e < E; ++e) a[e] = load_vec<ONCE>(reinterpret_cast<const U*>(vp + (int64_t)i * vv + qe[e]));
            const cpx<double> cc = hp[i];
#pragma unroll
            for (int e = 0; e < E; ++e) mac(cc, e, a[e]);
        }
#pragma unroll
        for (int e = 0; e < E; ++e) {
            if (!ok[e]) continue;
            U res;
#pragma unroll
            for (int k = 0; k < VW; ++k) res.e[k] = finish(o[e].e[k], ar[e][k], ai[e][k]);
            *reinterpret_cast<U*>(wp + qe[e]) = res;
        }
    }
    if (VW > 1 && whole < hi && threadIdx.x == 0) {
        double ar = 0.0, ai = 0.0;
        for (int i = 0; i < nv; ++i) {
            const cpx<R> a = vp[(int64_t)i * vv + whole];
            const cpx<double> cc = hp[i];
            ar = fma(cc.x, a.x, fma(-cc.y, a.y, ar));
            ai = fma(cc.x, a.y, fma(cc.y, a.x, ai));
        }
        wp[whole] = finish(wp[whole], ar, ai);
    }
    if (!norm) return;   // uniform over the launch
    nrm = wave_sum(nrm);
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    if (lane == 0) red[wv] = nrm;
    __syncthreads();
    if (threadIdx.x == 0) {
        double sum = 0.0;
#pragma unroll
        for (int u = 0; u < KW; ++u) sum += red[u];
        part[(int64_t)r * nchunk + c] = sum;
    }
}

// The chunk sums of the products, one wave per output as k_chunk_sum, written
// where they belong: slot i < nv of right-hand side r to h[r nv + i] (re, im
// by row parity), slot nv to w2[r].
__global__ __launch_bounds__(64) void k_dots_sum(const double* __restrict__ part, int nchunk, int nv,
                                                 double* __restrict__ h, double* __restrict__ w2)
{
    const int row = blockIdx.x, r = blockIdx.y;
    if (row >= 2 * nv && (row > 2 * nv || !w2)) return;
    const double* const p = part + ((int64_t)r * (nv + 1) * 2 + row) * nchunk;
    double v = 0.0;
    for (int c = threadIdx.x; c < nchunk; c += 64) v += p[c];
    v = wave_sum(v);
    if (threadIdx.x != 0) return;
    if (row < 2 * nv) h[(int64_t)r * 2 * nv + row] = v;
    else w2[r] = v;
}

// out[j] = sum over chunks of part[j][chunk], one wave per output: lane l sums
// chunks l, l+64, ... in order, then a fixed shuffle tree
__global__ __launch_bounds__(64) void k_chunk_sum(const double* __restrict__ part, int nchunk, int64_t total,
                                                  double* __restrict__ out)
{
    const int64_t j = blockIdx.x;
    if (j >= total) return;
    double v = 0.0;
    for (int c = threadIdx.x; c < nchunk; c += 64) v += part[j * nchunk + c];
    v = wave_sum(v);
    if (threadIdx.x == 0) out[j] = v;
}

// out[r] = V[r][idx[r]] (row gather); with scale: V[r][idx[r]] = out[r] / scale[r]
template <typename R, bool SCATTER>
__global__ __launch_bounds__(256) void k_rows(cpx<R>* __restrict__ V, int64_t vr, int64_t vv,
                                              const int64_t* __restrict__ idx, cpx<R>* __restrict__ b,
                                              int64_t br, const double* __restrict__ scale, int64_t n)
{
    const int r = blockIdx.y;
    const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= n) return;
    cpx<R>* row = V + r * vr + idx[r] * vv;
    if constexpr (SCATTER) {
        const double inv = 1.0 / scale[r];
        const cpx<R> v = b[r * br + q];
        row[q] = cpx<R>{R(v.x * inv), R(v.y * inv)};
    } else {
        b[r * br + q] = row[q];
    }
}

// the next basis vector: V[r][idx[r]] = w[r] / max(sqrt(w2[r]), 1e-30), and
// the same into stage[r] (the next matvec's input) when stage is not null
template <typename R>
__global__ __launch_bounds__(256) void k_next(cpx<R>* __restrict__ V, int64_t vr, int64_t vv,
                                              const int64_t* __restrict__ idx, const cpx<R>* __restrict__ w,
                                              int64_t wr, const double* __restrict__ w2, cpx<R>* __restrict__ stage,
                                              int64_t sr, int64_t n)
{
    const int r = blockIdx.y;
    const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= n) return;
    double nrm = sqrt(w2[r]);
    nrm = nrm > 1e-30 ? nrm : 1e-30;
    const double inv = 1.0 / nrm;
    const cpx<R> v = w[r * wr + q];
    const cpx<R> o{R(v.x * inv), R(v.y * inv)};
    V[r * vr + idx[r] * vv + q] = o;
    if (stage) stage[r * sr + q] = o;
}

}  // namespace

int64_t krylov_chunk(int64_t n)
{
    // about 1024 workgroups per right-hand side for long vectors, at least
    // 2048 elements per workgroup; even, so that a chunk starts on a whole
    // 16-byte unit
    int64_t c = (n + 1023) / 1024;
    if (c < 2048) c = 2048;
    return c + (c & 1);
}

// Whether rows at these element strides allow 16-byte loads: ComplexF32
// pairs need even strides and aligned bases, ComplexF64 elements are 16
// bytes themselves.
template <typename R>
static bool wide_ok(const void* V, int64_t vr, int64_t vv, const void* w, int64_t wr)
{
    if (sizeof(cpx<R>) == 16) return false;   // one element is a whole unit
    return vr % 2 == 0 && vv % 2 == 0 && wr % 2 == 0 && (uintptr_t)V % 16 == 0 && (uintptr_t)w % 16 == 0;
}

int64_t krylov_part_doubles(int64_t k, int64_t nv, int64_t n)
{
    // chunk partials of 2 (nv + 1) rows per right-hand side, then their sums
    const int64_t chunk = krylov_chunk(n);
    const int64_t nchunk = (n + chunk - 1) / chunk;
    return k * 2 * (nv + 1) * (nchunk + 1);
}

template <typename R>
hipError_t run_krylov_dots(int64_t k, int nv, int64_t n, const void* V, int64_t vr, int64_t vv, const void* w,
                           int64_t wr, void* part, void* h, double* w2, const int64_t* ncol, hipStream_t st)
{
    const int64_t chunk = krylov_chunk(n);
    const int nchunk = (int)((n + chunk - 1) / chunk);
    const int self = w2 != nullptr;
    const int nslot = nv + 1;
    const bool large = k * nv * n * (int64_t)sizeof(cpx<R>) > KEEP_BYTES;
    const auto kernel = wide_ok<R>(V, vr, vv, w, wr)
                            ? (large ? k_dots<R, sizeof(cpx<R>) == 8 ? 2 : 1, true>
                                     : k_dots<R, sizeof(cpx<R>) == 8 ? 2 : 1, false>)
                            : (large ? k_dots<R, 1, true> : k_dots<R, 1, false>);
    hipLaunchKernelGGL(kernel, dim3(nchunk, (unsigned)k), dim3(KT), 0, st, (const cpx<R>*)V, vr, vv,
                       (const cpx<R>*)w, wr, n, nv, ncol, chunk, nchunk, nslot, self, (double*)part);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_dots_sum, dim3((unsigned)(2 * nv + self), (unsigned)k), dim3(64), 0, st, (const double*)part,
                       nchunk, nv, (double*)h, w2);
    return hipGetLastError();
}

template <typename R>
hipError_t run_krylov_axpy(int64_t k, int nv, int64_t n, const void* V, int64_t vr, int64_t vv, const void* h,
                           int64_t hr, void* w, int64_t wr, double s, void* part, double* w2, const int64_t* ncol,
                           hipStream_t st)
{
    const int64_t chunk = krylov_chunk(n);
    const int nchunk = (int)((n + chunk - 1) / chunk);
    const int norm = w2 != nullptr;
    const bool large = k * nv * n * (int64_t)sizeof(cpx<R>) > 2 * KEEP_BYTES;
    const auto kernel = wide_ok<R>(nv > 0 ? V : w, nv > 0 ? vr : 0, nv > 0 ? vv : 0, w, wr)
                            ? (large ? k_axpy<R, sizeof(cpx<R>) == 8 ? 2 : 1, true>
                                     : k_axpy<R, sizeof(cpx<R>) == 8 ? 2 : 1, false>)
                            : (large ? k_axpy<R, 1, true> : k_axpy<R, 1, false>);
    hipLaunchKernelGGL(kernel, dim3(nchunk, (unsigned)k), dim3(KT), 0, st, (const cpx<R>*)V, vr, vv,
                       (const cpx<double>*)h, hr, (cpx<R>*)w, wr, n, nv, ncol, s, chunk, nchunk, norm,
                       (double*)part);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || !norm) return e;
    hipLaunchKernelGGL(k_chunk_sum, dim3((unsigned)k), dim3(64), 0, st, (const double*)part, nchunk, k, w2);
    return hipGetLastError();
}

template <typename R>
hipError_t run_krylov_rows(int64_t k, int64_t n, void* V, int64_t vr, int64_t vv, const int64_t* idx, void* b,
                           int64_t br, const double* scale, hipStream_t st)
{
    dim3 grid((unsigned)((n + 255) / 256), (unsigned)k);
    if (scale)
        hipLaunchKernelGGL((k_rows<R, true>), grid, dim3(256), 0, st, (cpx<R>*)V, vr, vv, idx, (cpx<R>*)b, br,
                           scale, n);
    else
        hipLaunchKernelGGL((k_rows<R, false>), grid, dim3(256), 0, st, (cpx<R>*)V, vr, vv, idx, (cpx<R>*)b, br,
                           scale, n);
    return hipGetLastError();
}

template <typename R>
hipError_t run_krylov_next(int64_t k, int64_t n, void* V, int64_t vr, int64_t vv, const int64_t* idx, const void* w,
                           int64_t wr, const double* w2, void* stage, int64_t sr, hipStream_t st)
{
    dim3 grid((unsigned)((n + 255) / 256), (unsigned)k);
    hipLaunchKernelGGL(k_next<R>, grid, dim3(256), 0, st, (cpx<R>*)V, vr, vv, idx, (const cpx<R>*)w, wr, w2,
                       (cpx<R>*)stage, sr, n);
    return hipGetLastError();
}

template hipError_t run_krylov_dots<float>(int64_t, int, int64_t, const void*, int64_t, int64_t, const void*,
                                           int64_t, void*, void*, double*, const int64_t*, hipStream_t);
template hipError_t run_krylov_dots<double>(int64_t, int, int64_t, const void*, int64_t, int64_t, const void*,
                                            int64_t, void*, void*, double*, const int64_t*, hipStream_t);
template hipError_t run_krylov_axpy<float>(int64_t, int, int64_t, const void*, int64_t, int64_t, const void*,
                                           int64_t, void*, int64_t, double, void*, double*, const int64_t*,
                                           hipStream_t);
template hipError_t run_krylov_axpy<double>(int64_t, int, int64_t, const void*, int64_t, int64_t, const void*,
                                            int64_t, void*, int64_t, double, void*, double*, const int64_t*,
                                            hipStream_t);
template hipError_t run_krylov_next<float>(int64_t, int64_t, void*, int64_t, int64_t, const int64_t*, const void*,
                                           int64_t, const double*, void*, int64_t, hipStream_t);
template hipError_t run_krylov_next<double>(int64_t, int64_t, void*, int64_t, int64_t, const int64_t*, const void*,
                                            int64_t, const double*, void*, int64_t, hipStream_t);
template hipError_t run_krylov_rows<float>(int64_t, int64_t, void*, int64_t, int64_t, const int64_t*, void*,
                                           int64_t, const double*, hipStream_t);
template hipError_t run_krylov_rows<double>(int64_t, int64_t, void*, int64_t, int64_t, const int64_t*, void*,
                                            int64_t, const double*, hipStream_t);

}  // namespace gla
