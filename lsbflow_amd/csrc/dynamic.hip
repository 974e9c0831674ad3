// Dynamic Smagorinsky model of the step (sgsterm.f90:123-280) and the plane means of the
// plane-averaged coefficient.  Two passes read u' and g' (12 fields): k_dynm_test (stages 1
// and 2 with the test filter between them, 2 fields out), and k_dynm_avg3 or k_dynm_plane3
// (the average and stage 3, with what that takes of stage 1 again; 9 fields out).  The
// stages as passes of their own around the filter (what tests compare with) go over 34, 42,
// 23, 4 and 21 fields: the FP64 step at 512x193x256 took 11.86 ms so and takes 8.32, the
// mixed step at 256x129x128 1.26 and 1.00.
//
// The work fields are stored in FP32 in the mixed form and in FP64 otherwise; every
// expression is evaluated in FP64 registers.  The fields hold perturbation quantities only;
// the base flow U = (ubar(z), 0, 0) enters the kernels as FP64 profiles, so no FP32 field
// carries an O(1) part that later cancels:
//   stage 1  from u', g' (perturbation velocity and gradient): the advective term, the
//            perturbation products p_lm = u_l u_m - U_l U_m, the perturbation strain
//            S'_lm = (g'_lm + g'_ml)/2, |S| and L1_lm = delta^2 |S| S_lm of the full strain;
//   filter   S', L1, u', p with the (a, b) test filter;
//   stage 2  M_lm = 2 (L1^ - (2 delta)^2 |S^| S^_lm) with S^ = S'^ + (S^U)^ and
//            L_lm = (u_l u_m)^ - u^_l u^_m = p^_lm - (U^_l u'^_m + u'^_l U^_m + u'^_l u'^_m)
//                   + [(U^2)^ - (U^)^2] (0,0 only),
//            numerator M:L and denominator M:M;
//   <.>      (1, 1) filter of both, or their plane means;
//   stage 3  C = <M:L>/<M:M> clipped to [0, 0.04], tau = -2 C delta^2 |S| S, and
//            h_lm = p_lm/2 + tau_lm written over p (h_00 without its plane-constant ubar^2/2,
//            as the mixed form's other models store it).
// The z-filtered base profiles U^, (S^U)^_02 and (U^2)^ - (U^)^2 are precomputed in FP64.
// Symmetric tensors are stored once per distinct component in the order
// (0,0), (1,0), (2,0), (1,1), (2,1), (2,2).

#include <cmath>
#include <cstdlib>

#include "lsb_internal.h"
#include "physical.h"

namespace lsb {

namespace {

struct DDims {
    int nx, ny, nxpp, nzp;
};

DDims ddims(const lsb_ctx* c) { return DDims{c->nx, c->ny, c->nxpp, c->nzp}; }

constexpr int kL[6] = {0, 1, 2, 1, 2, 2};
constexpr int kM[6] = {0, 0, 0, 1, 1, 2};

// grid: x in blocks of 256 points, one (j, k) row per blockIdx.y (strided)
dim3 row_grid(const DDims& d) {
    const unsigned gx = (unsigned)((d.nx + 255) / 256);
    const long rows = (long)d.ny * d.nzp;
    return dim3(gx, (unsigned)(rows < 65535 ? rows : 65535));
}

// field element by byte offset: with a 32-bit offset the loads and stores take the
// scalar-base + vector-offset form (no 64-bit address arithmetic per field)
template <class T, class Off>
__device__ __forceinline__ T ldf(const T* p, Off bo) {
    return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(p) + bo);
}
template <class T, class Off>
__device__ __forceinline__ void stf(T* p, Off bo, T v) {
    *reinterpret_cast<T*>(reinterpret_cast<char*>(p) + bo) = v;
}

}  // namespace

// advective term -1/2 u_m du_l/dx_m with the full gradient (g'_02 + ubarp), and the sponge
template <class T>
__device__ __forceinline__ void dynm_adv(const DynMixArgs<T>& a, int k, int i, const double (&up)[3],
                                         const double (&g)[3][3], T (&nlt)[3]) {
    const double u[3] = {up[0] + a.ubar[k], up[1], up[2]};
    const double g02 = g[0][2] + a.ubarp[k];
    const double lam = a.lam ? a.lam[i] : 0.0;
#pragma unroll
    for (int l = 0; l < 3; ++l) {
        double s = 0.0;
#pragma unroll
        for (int m = 0; m < 3; ++m) s = s - 0.5 * u[m] * ((l == 0 && m == 2) ? g02 : g[l][m]);
        if (a.lam) s = s - lam * up[l];  // lambda (target - u): target = ubar for u, 0 for v, w
        nlt[l] = (T)s;
    }
}

// perturbation products: u_l u_m - U_l U_m (only U_0 = ubar is nonzero)
template <class T>
__device__ __forceinline__ void dynm_products(const DynMixArgs<T>& a, int k, const double (&up)[3], T (&p)[6]) {
    const double U = a.ubar[k];
    const double u0 = up[0] + U;
    p[0] = (T)(up[0] * (u0 + U));
    p[1] = (T)(up[1] * u0);
    p[2] = (T)(up[2] * u0);
    p[3] = (T)(up[1] * up[1]);
    p[4] = (T)(up[2] * up[1]);
    p[5] = (T)(up[2] * up[2]);
}

// strain S' of the perturbation, |S| and S of the full field (sf)
template <class T>
__device__ __forceinline__ void dynm_strain(const DynMixArgs<T>& a, int k, const double (&g)[3][3], T (&spo)[6],
                                            double (&sf)[6], double& sno) {
    double sp[6], sn = 0.0;
#pragma unroll
    for (int q = 0; q < 6; ++q) sp[q] = 0.5 * (g[kL[q]][kM[q]] + g[kM[q]][kL[q]]);
    const double su = 0.5 * a.ubarp[k];  // base strain S^U_20 = S^U_02
#pragma unroll
    for (int q = 0; q < 6; ++q) {
        sf[q] = sp[q] + (q == 2 ? su : 0.0);
        const double w = (kL[q] == kM[q]) ? 1.0 : 2.0;  // off-diagonals appear twice
        sn = sn + w * 2.0 * sf[q] * sf[q];
        spo[q] = (T)sp[q];
    }
    sno = sqrt(sn);
}

template <class T>
__device__ __forceinline__ void dynm_l1(const DynMixArgs<T>& a, int k, const double (&sf)[6], double sn,
                                        T (&l1)[6]) {
    const double dl = a.delta[k];
#pragma unroll
    for (int q = 0; q < 6; ++q) l1[q] = (T)(dl * dl * sn * sf[q]);
}

// u' and g' of a point (byte offset o)
template <class T, class Off>
__device__ __forceinline__ void dynm_load(const DynMixArgs<T>& a, Off o, double (&up)[3], double (&g)[3][3]) {
#pragma unroll
    for (int l = 0; l < 3; ++l) up[l] = (double)ldf(a.ui[l], o);
#pragma unroll
    for (int l = 0; l < 3; ++l)
#pragma unroll
        for (int m = 0; m < 3; ++m) g[l][m] = (double)ldf(a.g[l + 3 * m], o);
}

template <class T, class Off>
__global__ void __launch_bounds__(256) k_dynm_stage1(DDims d, DynMixArgs<T> a) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= d.nx) return;
    const int nrows = d.ny * d.nzp;
    for (int row = blockIdx.y; row < nrows; row += gridDim.y) {
        const int k = row / d.ny;
        const Off o = ((Off)row * (Off)d.nxpp + (Off)i) * (Off)sizeof(T);
        double up[3], g[3][3], sf[6], sn;
        dynm_load(a, o, up, g);
        T nlt[3], p[6], sp[6], l1[6];
        dynm_adv(a, k, i, up, g, nlt);
        dynm_products(a, k, up, p);
        dynm_strain(a, k, g, sp, sf, sn);
        dynm_l1(a, k, sf, sn, l1);
#pragma unroll
        for (int l = 0; l < 3; ++l) stf(a.nlt[l], o, nlt[l]);
        stf(a.snorm, o, (T)sn);
#pragma unroll
        for (int q = 0; q < 6; ++q) {
            stf(a.p[q], o, p[q]);
            stf(a.sp[q], o, sp[q]);
            stf(a.l1[q], o, l1[q]);
        }
    }
}

// stage 2 at one point of plane k from its 21 filtered values get(n), n: S' (6), L1 (6),
// u' (3), p (6), each taken once, when it is needed; returns M:L and M:M
template <class T, class Get>
__device__ __forceinline__ void dynm_stage2_math(const DynMixArgs<T>& a, int nzp, int k, Get get, T& num_o,
                                                 T& den_o) {
    const double Ub = a.base[k];
    const double SUh = a.base[nzp + k];
    const double LU = a.base[2 * nzp + k];
    double sh[6], snh = 0.0;
#pragma unroll
    for (int q = 0; q < 6; ++q) {
        sh[q] = get(q) + (q == 2 ? SUh : 0.0);
        const double w = (kL[q] == kM[q]) ? 1.0 : 2.0;
        snh = snh + w * 2.0 * sh[q] * sh[q];
    }
    snh = sqrt(snh);
    const double cd = 2.0 * a.delta[k];
    double uh[3];
#pragma unroll
    for (int l = 0; l < 3; ++l) uh[l] = get(12 + l);
    const double Uh[3] = {Ub, 0.0, 0.0};
    double num = 0.0, den = 0.0;
#pragma unroll
    for (int q = 0; q < 6; ++q) {
        const int l = kL[q], m = kM[q];
        const double mij = 2.0 * (get(6 + q) - cd * cd * snh * sh[q]);
        double lij = get(15 + q) - (Uh[l] * uh[m] + uh[l] * Uh[m] + uh[l] * uh[m]);
        if (q == 0) lij = lij + LU;
        const double w = (l == m) ? 1.0 : 2.0;
        num = num + w * mij * lij;
        den = den + w * mij * mij;
    }
    num_o = (T)num;
    den_o = (T)den;
}

template <class T>
__device__ __forceinline__ const T* dynm_stage2_src(const DynMixArgs<T>& a, int n) {
    return n < 6 ? a.sph[n] : n < 12 ? a.l1h[n - 6] : n < 15 ? a.uh[n - 12] : a.ph[n - 15];
}

template <class T, class Off>
__global__ void __launch_bounds__(256) k_dynm_stage2(DDims d, DynMixArgs<T> a) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= d.nx) return;
    const int nrows = d.ny * d.nzp;
    for (int row = blockIdx.y; row < nrows; row += gridDim.y) {
        const int k = row / d.ny;
        const Off o = ((Off)row * (Off)d.nxpp + (Off)i) * (Off)sizeof(T);
        T num, den;
        dynm_stage2_math(a, d.nzp, k, [&](int n) { return (double)ldf(dynm_stage2_src(a, n), o); }, num, den);
        stf(a.num, o, num);
        stf(a.den, o, den);
    }
}

// Value of the lane before / after (whole-wave shift by one; the first / last lane gets 0).
__device__ __forceinline__ float lane_prev(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x138, 0xf, 0xf, true));
}
__device__ __forceinline__ float lane_next(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x130, 0xf, 0xf, true));
}
__device__ __forceinline__ double lane_prev(double v) {
    return __hiloint2double(__builtin_amdgcn_update_dpp(0, __double2hiint(v), 0x138, 0xf, 0xf, true),
                            __builtin_amdgcn_update_dpp(0, __double2loint(v), 0x138, 0xf, 0xf, true));
}
__device__ __forceinline__ double lane_next(double v) {
    return __hiloint2double(__builtin_amdgcn_update_dpp(0, __double2hiint(v), 0x130, 0xf, 0xf, true),
                            __builtin_amdgcn_update_dpp(0, __double2loint(v), 0x130, 0xf, 0xf, true));
}

// M:L and M:M straight from u' and g': stage 1, the test filter of its 21 fields and
// stage 2 in one pass.  A block owns txo <= 62 columns by R rows and slides over KC planes;
// wave r holds row J0 - 1 + r (the first and the last are the y halo), lane t column
// i0 - 1 + t (lanes 0 and txo + 1 are the x halo), both periodic.  Per plane: stage 1 at the
// lane's point, the x pass with the neighbour lanes' values, one LDS store per field; then
// on the R inner rows the y pass from LDS and the z pass, with the last plane's values
// (zb) and the sum over the last two (za) in registers, and stage 2.  The loads of
// the next plane are in flight meanwhile.  The 21 values are rounded to T where the separate
// passes store them, in their expressions: the same bits.
// 14 field passes in place of 99, and the halo: at 512x193x256 the FP64 form reads 4.3 GB
// (12 fields are 2.5) and writes 0.4 in 1.10 ms, 4.3 TB/s, bound by HBM with the vector units
// 0.4 busy; the mixed form moves 2.7 GB in 0.88 ms, 3.1 TB/s, the vector units 0.56 busy (some
// 410 instructions per point and plane, 4/3 of the x phase for the halo rows), and waits at
// two waves a SIMD.  R = 6: 8 waves with up to 256 registers (42 FP64 values of the z pass
// each); R = 4 and R = 10 leave 168 and spill (FP64 step at that grid: 8.36 ms against 10.6
// and 13.3).  The FP64 1.10 ms are in place of 1.62 + 2.08 + 0.94 for stage 1, the filter and
// stage 2.
template <class T, int R, bool P2>
__global__ void __launch_bounds__(64 * (R + 2)) k_dynm_test(DDims d, DynMixArgs<T> A, const double* __restrict__ w,
                                                            double fa, double fb, int txo, int KC) {
    __shared__ double xs[21][R + 2][64];
    const int lane = threadIdx.x & 63;
    const int r = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int ntx = (d.nx + txo - 1) / txo;
    const int i0 = (blockIdx.x % ntx) * txo;
    const int J0 = (blockIdx.x / ntx) * R;
    const int k0 = blockIdx.y * KC;
    const int k1 = min(k0 + KC, d.nzp);
    // a sum a + b + a that is a power of two goes into the weights (exact)
    const double s = 2. * fa + fb;
    const double is = P2 ? 1.0 / s : 1.0;
    const double wa = fa * is, wb = fb * is;
    auto div = [&](double x) { return P2 ? x : x / s; };
    int i = (i0 - 1 + lane) % d.nx;
    i = (i < 0) ? i + d.nx : i;
    int j = (J0 - 1 + r) % d.ny;
    j = (j < 0) ? j + d.ny : j;
    const unsigned off = ((unsigned)j * (unsigned)d.nxpp + (unsigned)i) * (unsigned)sizeof(T);
    const size_t plane = (size_t)d.ny * d.nxpp;
    const bool live = lane >= 1 && lane <= txo && i0 + lane - 1 < d.nx && J0 + r - 1 < d.ny;
    T pre[12];
    auto load = [&](int k) {
        // scalar base + 32-bit lane offset, not 12 lane pointers (the asm keeps the widening
        // of the offset from being hoisted out of the loop)
        const size_t pl = (size_t)k * plane;
        unsigned o = off;
        asm("" : "+v"(o));
#pragma unroll
        for (int l = 0; l < 3; ++l) pre[l] = ldf(A.ui[l] + pl, o);
#pragma unroll
        for (int q = 0; q < 9; ++q) pre[3 + q] = ldf(A.g[q] + pl, o);
    };
    auto put = [&](int k, T num, T den) {
        if (live) {
            stf(A.num + k * plane, off, num);
            stf(A.den + k * plane, off, den);
        }
    };
    const int klast = min(k1, d.nzp - 1);
    const int kstart = (k0 > 0) ? k0 - 1 : k0;
    // stage 1 and the x pass of plane kk into LDS, the loads of the next plane behind them
    auto xphase = [&](int kk) {
        auto xpass = [&](int f, T v) {
            xs[f][r][lane] = div(wa * (double)lane_prev(v) + wb * (double)v + wa * (double)lane_next(v));
        };
        double up[3], g[3][3], sf[6], sn;
        T t6[6];
#pragma unroll
        for (int l = 0; l < 3; ++l) {
            up[l] = (double)pre[l];
            xpass(12 + l, pre[l]);
        }
        dynm_products(A, kk, up, t6);
#pragma unroll
        for (int q = 0; q < 6; ++q) xpass(15 + q, t6[q]);
#pragma unroll
        for (int l = 0; l < 3; ++l)
#pragma unroll
            for (int m = 0; m < 3; ++m) g[l][m] = (double)pre[3 + l + 3 * m];
        dynm_strain(A, kk, g, t6, sf, sn);
#pragma unroll
        for (int q = 0; q < 6; ++q) xpass(q, t6[q]);
        dynm_l1(A, kk, sf, sn, t6);
#pragma unroll
        for (int q = 0; q < 6; ++q) xpass(6 + q, t6[q]);
        if (kk < klast) load(kk + 1);
        __syncthreads();
    };
    load(kstart);
    if (r == 0 || r == R + 1) {  // the y halo rows
        for (int kk = kstart; kk <= klast; ++kk) {
            xphase(kk);
            __syncthreads();
        }
        return;
    }
    double za[21], zb[21];
#pragma unroll
    for (int f = 0; f < 21; ++f) za[f] = zb[f] = 0.0;
    auto ypass = [&](int f) {
        return div(wa * xs[f][r - 1][lane] + wb * xs[f][r][lane] + wa * xs[f][r + 1][lane]);
    };
    // a boundary plane keeps its xy-filtered values (no z pass: an infinite neighbour times
    // a weight of 0 would not leave it alone)
    auto edge = [&](int k) {
        T num, den;
        dynm_stage2_math(A, d.nzp, k, [&](int f) { return (double)(T)zb[f]; }, num, den);
        put(k, num, den);
    };
    int kk = kstart;
    if (k0 == 0) {
        xphase(0);
#pragma unroll
        for (int f = 0; f < 21; ++f) zb[f] = ypass(f);
        edge(0);
        __syncthreads();
        kk = 1;
    }
    for (; kk <= klast; ++kk) {
        xphase(kk);
        // weights of plane kk - 1 (w0) and kk (w1) in the output plane kk and of kk in kk - 1
        // (w2)
        const double w2 = is * w[2 * d.nzp + kk - 1];
        const double w1 = is * w[d.nzp + kk];
        const double w0 = is * w[kk];
        auto yz = [&](int f) {
            const double y = ypass(f);
            // z = za + w2 y, za = w0 zb + w1 y in the three-address form (the two-address one
            // costs copies of the sums on every plane)
            const double t = w1 * y;
            double z;
            asm("v_fma_f64 %0, %1, %2, %3" : "=v"(z) : "s"(w2), "v"(y), "v"(za[f]));
            asm("v_fma_f64 %0, %1, %2, %3" : "=v"(za[f]) : "s"(w0), "v"(zb[f]), "v"(t));
            zb[f] = y;
            if constexpr (!P2) z = z / s;
            return (double)(T)z;
        };
        T num, den;
        dynm_stage2_math(A, d.nzp, max(kk - 1, 0), yz, num, den);
        if (kk > max(k0, 1)) put(kk - 1, num, den);
        __syncthreads();
    }
    if (k1 == d.nzp) edge(d.nzp - 1);
}

// stage 3 at one point of plane k from the coefficient ratio ct = <M:L> / <M:M>
template <class T, class Off>
__device__ __forceinline__ void dynm_stage3_point(const DynMixArgs<T>& a, Off o, int k, double ct) {
    if (ct < 0.0 || isnan(ct)) ct = 0.0;
    if (ct > 0.2 * 0.2) ct = 0.2 * 0.2;
    const double dl = a.delta[k];
    const double nu = ct * dl * dl * (double)ldf(a.snorm, o);
    const double su = 0.5 * a.ubarp[k];
#pragma unroll
    for (int q = 0; q < 6; ++q) {
        const double s = (double)ldf(a.sp[q], o) + (q == 2 ? su : 0.0);
        const double tau = -2.0 * nu * s;
        stf(a.h[q], o, (T)(0.5 * (double)ldf(a.h[q], o) + tau));  // h holds p on entry
    }
}

template <class T, class Off>
__global__ void __launch_bounds__(256) k_dynm_stage3(DDims d, DynMixArgs<T> a) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= d.nx) return;
    const int nrows = d.ny * d.nzp;
    for (int row = blockIdx.y; row < nrows; row += gridDim.y) {
        const int k = row / d.ny;
        const Off o = ((Off)row * (Off)d.nxpp + (Off)i) * (Off)sizeof(T);
        const double ct =
            a.cplane ? a.cplane[k] / a.cplane[d.nzp + k] : (double)ldf(a.numf, o) / (double)ldf(a.denf, o);
        dynm_stage3_point(a, o, k, ct);
    }
}

// Stage 3 at one point from u' and g': what it takes of stage 1 (N pieces, products, |S|,
// S') again at the point, rounded to T where the separate stages store it.
template <class T>
__device__ __forceinline__ void dynm_tau_point(const DynMixArgs<T>& a, size_t pl, unsigned o, int k, int i,
                                               double ct) {
    if (ct < 0.0 || isnan(ct)) ct = 0.0;
    if (ct > 0.2 * 0.2) ct = 0.2 * 0.2;
    double up[3], g[3][3], sf[6], sn;
#pragma unroll
    for (int l = 0; l < 3; ++l) up[l] = (double)ldf(a.ui[l] + pl, o);
#pragma unroll
    for (int l = 0; l < 3; ++l)
#pragma unroll
        for (int m = 0; m < 3; ++m) g[l][m] = (double)ldf(a.g[l + 3 * m] + pl, o);
    T nlt[3], p[6], sp[6];
    dynm_adv(a, k, i, up, g, nlt);
    dynm_products(a, k, up, p);
    dynm_strain(a, k, g, sp, sf, sn);
#pragma unroll
    for (int l = 0; l < 3; ++l) stf(a.nlt[l] + pl, o, nlt[l]);
    const double dl = a.delta[k];
    const double nu = ct * dl * dl * (double)(T)sn;
    const double su = 0.5 * a.ubarp[k];
#pragma unroll
    for (int q = 0; q < 6; ++q) {
        const double tau = -2.0 * nu * ((double)sp[q] + (q == 2 ? su : 0.0));
        stf(a.h[q] + pl, o, (T)(0.5 * (double)p[q] + tau));
    }
}

// Stage 3 from u' and g' with the plane means.
template <class T>
__global__ void __launch_bounds__(256) k_dynm_plane3(DDims d, DynMixArgs<T> a) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= d.nx) return;
    const int nrows = d.ny * d.nzp;
    for (int row = blockIdx.y; row < nrows; row += gridDim.y) {
        const int k = row / d.ny;
        const unsigned o = ((unsigned)(row - k * d.ny) * (unsigned)d.nxpp + (unsigned)i) * (unsigned)sizeof(T);
        dynm_tau_point(a, (size_t)k * d.ny * d.nxpp, o, k, i, a.cplane[k] / a.cplane[d.nzp + k]);
    }
}

// The local (1, 1) average of M:L and M:M and stage 3 in one pass: k_filt3_lds's steps
// (a TX x R tile with periodic halos global -> registers -> LDS, the x pass into a second
// LDS array, the y pass, the z pass over three planes in registers, the next tile's loads
// in flight) for num and den in turn on every plane, and at each output point the two
// averages, rounded to T as stored averages would be, go into stage 3.  Same
// expressions and order as the filter followed by k_dynm_stage3: bit-identical to them.
template <class T, int R, int TX>
__global__ void __launch_bounds__(256) k_dynm_avg3(DDims d, DynMixArgs<T> A, const double* __restrict__ w, int KC) {
    constexpr int NT = (R + 2) * (TX + 2);  // tile elements
    constexpr int NL = (NT + 255) / 256;    // tile loads per thread
    constexpr int NP = (R * TX) / 256;      // output points per thread
    static_assert((R * TX) % 256 == 0, "R * TX must be a multiple of 256");
    __shared__ T tile[NT];
    __shared__ double xs[(R + 2) * TX];
    const int ntx = (d.nx + TX - 1) / TX;
    const int i0 = (blockIdx.x % ntx) * TX;
    const int J0 = (blockIdx.x / ntx) * R;
    const int k0 = blockIdx.y * KC;
    const int k1 = min(k0 + KC, d.nzp);
    const T* src[2] = {A.num, A.den};
    const double a = 1.0, b = 1.0;
    const double s = 2. * a + b;
    const double s2 = 2.00 * a + b;
    const bool p2 = pow2_exact(s);
    const double is = 1.0 / s;
    const long plane = (long)d.ny * d.nxpp;
    int toff[NL];
#pragma unroll
    for (int m = 0; m < NL; ++m) {
        const int e = threadIdx.x + 256 * m;
        int off = -1;
        if (e < NT) {
            const int rr = e / (TX + 2), cc = e - rr * (TX + 2);
            int j = (J0 - 1 + rr) % d.ny;
            j = (j < 0) ? j + d.ny : j;
            int i = (i0 - 1 + cc) % d.nx;
            i = (i < 0) ? i + d.nx : i;
            off = j * d.nxpp + i;
        }
        toff[m] = off;
    }
    T pre[NL];
    auto load = [&](int f, int k) {
        const T* qk = src[f] + (long)k * plane;
#pragma unroll
        for (int m = 0; m < NL; ++m) pre[m] = (toff[m] >= 0) ? qk[toff[m]] : (T)0;
    };
    // xy-filtered values of the tile in `pre`; then the loads of (fn, kn) (kn >= 0) in flight
    auto stage = [&](double (&y)[NP], int fn, int kn) {
#pragma unroll
        for (int m = 0; m < NL; ++m) {
            const int e = threadIdx.x + 256 * m;
            if (e < NT) tile[e] = pre[m];
        }
        __syncthreads();
        if (kn >= 0) load(fn, kn);
        for (int e = threadIdx.x; e < (R + 2) * TX; e += 256) {
            const int rr = e / TX, c = e - rr * TX;
            const T* t = tile + rr * (TX + 2) + c;
            xs[e] = fdiv(a * (double)t[0] + b * (double)t[1] + a * (double)t[2], s, is, p2);
        }
        __syncthreads();
#pragma unroll
        for (int m = 0; m < NP; ++m) {
            const int p = threadIdx.x + 256 * m;
            const int r = p / TX, c = p - r * TX;
            y[m] = fdiv(a * xs[r * TX + c] + b * xs[(r + 1) * TX + c] + a * xs[(r + 2) * TX + c], s2, is, p2);
        }
    };
    // planes k0 - 1 (if any) .. klast, num then den on each
    const int klast = min(k1, d.nzp - 1);
    const int kstart = (k0 > 0) ? k0 - 1 : k0;
    double Yp[2][NP], Yc[2][NP], Yn[2][NP];
    auto out = [&](int k, const double (&vn)[NP], const double (&vd)[NP]) {
#pragma unroll
        for (int m = 0; m < NP; ++m) {
            const int p = threadIdx.x + 256 * m;
            const int r = p / TX, c = p - r * TX;
            const int j = J0 + r, i = i0 + c;
            if (j < d.ny && i < d.nx) {
                const unsigned o = ((unsigned)j * (unsigned)d.nxpp + (unsigned)i) * (unsigned)sizeof(T);
                dynm_tau_point(A, (size_t)k * plane, o, k, i, (double)(T)vn[m] / (double)(T)vd[m]);
            }
        }
    };
    load(0, kstart);
    for (int kk = kstart; kk <= klast; ++kk) {
        double y[2][NP];
        stage(y[0], 1, kk);
        stage(y[1], 0, (kk + 1 <= klast) ? kk + 1 : -1);
#pragma unroll
        for (int f = 0; f < 2; ++f)
#pragma unroll
            for (int m = 0; m < NP; ++m) {
                if (kk < k0)
                    Yp[f][m] = y[f][m];
                else if (kk == k0)
                    Yc[f][m] = y[f][m];
                else
                    Yn[f][m] = y[f][m];
            }
        if (kk > k0) {
            const int k = kk - 1;
            const bool interior = (k > 0 && k < d.nzp - 1);
            const double w0 = w[k], w1 = w[d.nzp + k], w2 = w[2 * d.nzp + k];
            double v[2][NP];
#pragma unroll
            for (int f = 0; f < 2; ++f)
#pragma unroll
                for (int m = 0; m < NP; ++m) {
                    if (interior) {
                        double t = w0 * Yp[f][m] + w1 * Yc[f][m] + w2 * Yn[f][m];
                        v[f][m] = fdiv(t, s, is, p2);
                    } else {
                        v[f][m] = Yc[f][m];
                    }
                    Yp[f][m] = Yc[f][m];
                    Yc[f][m] = Yn[f][m];
                }
            out(k, v[0], v[1]);
        }
    }
    // the last plane of the grid keeps its xy-filtered value (no z pass)
    if (k1 == d.nzp) out(d.nzp - 1, Yc[0], Yc[1]);
}

// Planes per block of a pass that slides over z: each block takes two halo planes more, and a
// last round of blocks costs as much as a full one (at_once blocks run at a time).  Measured
// with 8 to 97 planes at 256x129x128 and 512x193x256: the choice was the fastest at both (the
// slowest of them 10% and 3% of the step behind).
static int slide_planes(long tiles, int nzp, long at_once) {
    int best = nzp;
    double cost = 1e300;
    for (int nb = 1; nb <= (nzp + 3) / 4; ++nb) {
        const int kc = (nzp + nb - 1) / nb;
        const long blocks = tiles * ((nzp + kc - 1) / kc);
        const double c = (double)((blocks + at_once - 1) / at_once) * (kc + 2);
        if (c < cost) {
            cost = c;
            best = kc;
        }
    }
    return best;
}

template <class T>
static void launch_dyn_test(lsb_ctx* c, const DDims& d, const DynMixArgs<T>& a, hipStream_t s) {
    constexpr int R = 6;
    const double* w = c->d_fz;  // the interpolating weights of the configured (a, b)
    const double fa = c->cfg.a, fb = c->cfg.b;
    int e = 0;
    const bool p2 = std::frexp(2. * fa + fb, &e) == 0.5;
    const int ntx = (d.nx + 61) / 62;
    const int txo = (d.nx + ntx - 1) / ntx;
    const long tiles = (long)ntx * ((d.ny + R - 1) / R);
    const int KC = slide_planes(tiles, d.nzp, 256);
    const dim3 g((unsigned)tiles, (unsigned)((d.nzp + KC - 1) / KC));
    if (p2)
        hipLaunchKernelGGL((k_dynm_test<T, R, true>), g, dim3(64 * (R + 2)), 0, s, d, a, w, fa, fb, txo, KC);
    else
        hipLaunchKernelGGL((k_dynm_test<T, R, false>), g, dim3(64 * (R + 2)), 0, s, d, a, w, fa, fb, txo, KC);
}

template <class T>
int ph_dyn_test(lsb_ctx* c, const DynMixArgs<T>& a, hipStream_t s) {
    const DDims d = ddims(c);
    int tok = -1;
    prof_mark_begin(c, PC_NL, s, &tok, 0.0, 14.0 * sizeof(T) * (double)d.nx * d.ny * d.nzp);
    launch_dyn_test(c, d, a, s);
    prof_mark_end(c, tok, s);
    LSB_HIP(hipGetLastError());
    return LSB_OK;
}
template int ph_dyn_test<float>(lsb_ctx*, const DynMixArgs<float>&, hipStream_t);
template int ph_dyn_test<double>(lsb_ctx*, const DynMixArgs<double>&, hipStream_t);

// Stage 3 from num and den (their local average, or the plane means in a.cplane) and u', g'.
template <class T>
int ph_dyn_tau(lsb_ctx* c, const DynMixArgs<T>& a, hipStream_t s) {
    const DDims d = ddims(c);
    int tok = -1;
    // num, den, u' and g' read; the N pieces and h written
    prof_mark_begin(c, PC_NL, s, &tok, 0.0, 23.0 * sizeof(T) * (double)d.nx * d.ny * d.nzp);
    if (a.cplane) {
        hipLaunchKernelGGL((k_dynm_plane3<T>), row_grid(d), dim3(256), 0, s, d, a);
    } else {
        const double* w = c->d_fz + 3 * c->nzp;  // the (1, 1) interpolating weights
        constexpr int R = 4, TX = 128;
        const int ntx = (d.nx + TX - 1) / TX;
        const long tiles = (long)ntx * ((d.ny + R - 1) / R);
        // 16 planes per block, fewer (each block recomputes two halo planes) until the grid
        // holds some 2048 blocks (8 per CU)
        int KC = 16;
        while (KC > 4 && tiles * ((d.nzp + KC - 1) / KC) < 2048) KC /= 2;
        const dim3 grid((unsigned)tiles, (unsigned)((d.nzp + KC - 1) / KC));
        hipLaunchKernelGGL((k_dynm_avg3<T, R, TX>), grid, dim3(256), 0, s, d, a, w, KC);
    }
    prof_mark_end(c, tok, s);
    LSB_HIP(hipGetLastError());
    return LSB_OK;
}
template int ph_dyn_tau<float>(lsb_ctx*, const DynMixArgs<float>&, hipStream_t);
template int ph_dyn_tau<double>(lsb_ctx*, const DynMixArgs<double>&, hipStream_t);

// Plane means of two fields over the nx physical points of every row: B partial sums per
// plane (one block each), then the B partials of each plane summed in a fixed order.
constexpr int kPlaneBlocks = 16;

template <class T>
__global__ void __launch_bounds__(256) k_plane_partial2(DDims d, const T* __restrict__ f0, const T* __restrict__ f1,
                                                        double* __restrict__ part) {
    const int k = blockIdx.y;
    const int b = blockIdx.x;
    const long n = (long)d.nx * d.ny;
    double s0 = 0.0, s1 = 0.0;
    for (long t = (long)b * blockDim.x + threadIdx.x; t < n; t += (long)gridDim.x * blockDim.x) {
        const int i = (int)(t % d.nx), j = (int)(t / d.nx);
        const long o = ((long)k * d.ny + j) * d.nxpp + i;
        s0 += (double)f0[o];
        s1 += (double)f1[o];
    }
    __shared__ double sh0[256], sh1[256];
    sh0[threadIdx.x] = s0;
    sh1[threadIdx.x] = s1;
    __syncthreads();
    for (int h = 128; h > 0; h >>= 1) {
        if ((int)threadIdx.x < h) {
            sh0[threadIdx.x] += sh0[threadIdx.x + h];
            sh1[threadIdx.x] += sh1[threadIdx.x + h];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        part[((long)k * kPlaneBlocks + b) * 2 + 0] = sh0[0];
        part[((long)k * kPlaneBlocks + b) * 2 + 1] = sh1[0];
    }
}

__global__ void k_plane_finish2(DDims d, const double* __restrict__ part, double* __restrict__ out) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= d.nzp) return;
    double s0 = 0.0, s1 = 0.0;
    for (int b = 0; b < kPlaneBlocks; ++b) {
        s0 += part[((long)k * kPlaneBlocks + b) * 2 + 0];
        s1 += part[((long)k * kPlaneBlocks + b) * 2 + 1];
    }
    const double n = (double)d.nx * (double)d.ny;
    out[k] = s0 / n;
    out[d.nzp + k] = s1 / n;
}

template <class T>
int ph_plane_mean2(lsb_ctx* c, const T* f0, const T* f1, double* scratch, double* out, hipStream_t s) {
    const DDims d = ddims(c);
    hipLaunchKernelGGL((k_plane_partial2<T>), dim3(kPlaneBlocks, (unsigned)d.nzp), dim3(256), 0, s, d, f0, f1,
                       scratch);
    LSB_HIP(hipGetLastError());
    hipLaunchKernelGGL(k_plane_finish2, dim3((unsigned)((d.nzp + 63) / 64)), dim3(64), 0, s, d, scratch, out);
    LSB_HIP(hipGetLastError());
    return LSB_OK;
}
template int ph_plane_mean2<double>(lsb_ctx*, const double*, const double*, double*, double*, hipStream_t);
template int ph_plane_mean2<float>(lsb_ctx*, const float*, const float*, double*, double*, hipStream_t);

size_t ph_plane_mean2_scratch(const lsb_ctx* c) { return (size_t)c->nzp * kPlaneBlocks * 2; }

template <class T>
int ph_dyn_mixed(lsb_ctx* c, int stage, const DynMixArgs<T>& a, hipStream_t s) {
    const DDims d = ddims(c);
    const dim3 g = row_grid(d);
    int tok = -1;
    // fields read + written per point by each stage
    const double per = (stage == 1) ? 12.0 + 22.0 : (stage == 2 ? 21.0 + 2.0 : 2.0 + 1.0 + 6.0 + 12.0);
    prof_mark_begin(c, PC_NL, s, &tok, 0.0, per * sizeof(T) * (double)d.nx * d.ny * d.nzp);
    // 32-bit byte offsets while a field is below 4 GiB
    const bool small = (double)d.ny * d.nzp * d.nxpp * sizeof(T) < 4294967296.0;
#define LSB_DYNM(K)                                                          \
    if (small)                                                               \
        hipLaunchKernelGGL((K<T, unsigned>), g, dim3(256), 0, s, d, a);      \
    else                                                                     \
        hipLaunchKernelGGL((K<T, size_t>), g, dim3(256), 0, s, d, a);
    switch (stage) {
        case 1: LSB_DYNM(k_dynm_stage1) break;
        case 2: LSB_DYNM(k_dynm_stage2) break;
        default: LSB_DYNM(k_dynm_stage3) break;
    }
#undef LSB_DYNM
    prof_mark_end(c, tok, s);
    LSB_HIP(hipGetLastError());
    return LSB_OK;
}
template int ph_dyn_mixed<float>(lsb_ctx*, int, const DynMixArgs<float>&, hipStream_t);
template int ph_dyn_mixed<double>(lsb_ctx*, int, const DynMixArgs<double>&, hipStream_t);

// z-filtered base profiles of the fused dynamic model (FP64, host): U^ = filter(ubar),
// (S^U)^_02 = filter(ubarp / 2), (U^2)^ - (U^)^2.  The x-y passes leave a function of z
// unchanged; the z pass uses the interpolating weights of interior planes (the boundary
// planes keep their value, filters.f90:450-453).
void dyn_base_profiles(const lsb_ctx* c, std::vector<double>& out) {
    const int n = c->nzp;
    const double s = 2.0 * c->cfg.a + c->cfg.b;
    const std::vector<double>& w = c->fz_ab;
    auto zf = [&](const std::vector<double>& v, int k) {
        if (k == 0 || k == n - 1) return v[k];
        return (w[k] * v[k - 1] + w[n + k] * v[k] + w[2 * n + k] * v[k + 1]) / s;
    };
    std::vector<double> u(n), su(n), u2(n);
    for (int k = 0; k < n; ++k) {
        u[k] = c->ubar[k];
        su[k] = 0.5 * c->ubarp[k];
        u2[k] = c->ubar[k] * c->ubar[k];
    }
    out.assign(3 * (size_t)n, 0.0);
    for (int k = 0; k < n; ++k) {
        const double ub = zf(u, k);
        out[k] = ub;
        out[n + k] = zf(su, k);
        out[2 * n + k] = zf(u2, k) - ub * ub;
    }
}

}  // namespace lsb
