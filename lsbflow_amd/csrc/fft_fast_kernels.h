// Kernels and launchers of the register-resident horizontal FFT passes (dispatch in
// fft_fast.hip; the lengths with a factor 3 or 5 are instantiated in fft_mixed_x64.hip,
// fft_mixed_y64.hip and their FP32 counterparts).  Lengths L = N1 * N2; the general
// mixed-radix path in fft.hip covers every other length.
//
// Index split n = N2*n1 + n2, k = k1 + N1*k2:
//   stage 1  each thread (one n2) loads its N1 points straight from HBM and does
//            a length-N1 DFT in registers, then multiplies by W_L^(n2*k1);
//   exchange one write/read through a padded LDS tile (the N1 x N2 transpose);
//   stage 2  length-N2 DFTs in registers, results stored with unit-stride lanes.
// Loads and stores are coalesced (consecutive lanes touch consecutive complex
// words of one row, or of one row of a tile of kx columns).  The r2c split /
// c2r merge of the x pass use the natural-order spectrum staged once more in
// the same LDS tile.  Semantics are those of fft.hip (scaling, Nyquist drop,
// zero pads).
//
// Every pass is templated on the arithmetic type R and on the element types of
// its input (TI) and output (TO): the FP64 form uses double throughout, the
// mixed form reads FP64 spectra and writes FP32 physical fields (and back), the
// conversion happening in registers at the load/store.  The inverse y pass can
// apply d/dx or d/dy (x i*kx, x i*ky, derivatives.f90:261-303) to a field as it
// loads it, so spectral derivative fields never round-trip through HBM.

#pragma once

#include <cstdlib>
#include <cstring>
#include <type_traits>

#include "lsb_internal.h"

namespace lsb {

// ------------------------------------------------------------- small DFTs
template <class R, int S>
__device__ __forceinline__ cpx<R> f_mul_si(cpx<R> a) {
    if (S < 0) return {a.im, -a.re};
    return {-a.im, a.re};
}

template <class R, int S>
__device__ __forceinline__ void f_dft4(cpx<R>& a0, cpx<R>& a1, cpx<R>& a2, cpx<R>& a3) {
    const cpx<R> s02 = cadd(a0, a2), d02 = csub(a0, a2), s13 = cadd(a1, a3), d13 = csub(a1, a3);
    const cpx<R> w = f_mul_si<R, S>(d13);
    a0 = cadd(s02, s13);
    a2 = csub(s02, s13);
    a1 = cadd(d02, w);
    a3 = csub(d02, w);
}

// exp(S*2*pi*i*m/16) for m = 0..15
template <class R, int S>
__device__ __forceinline__ cpx<R> w16(int m) {
    const R c[16] = {(R)1.0L,
                     (R)0.92387953251128675612818318939678829L,
                     (R)0.70710678118654752440084436210484904L,
                     (R)0.38268343236508977172845998403039887L,
                     (R)0.0L,
                     (R)-0.38268343236508977172845998403039887L,
                     (R)-0.70710678118654752440084436210484904L,
                     (R)-0.92387953251128675612818318939678829L,
                     (R)-1.0L,
                     (R)-0.92387953251128675612818318939678829L,
                     (R)-0.70710678118654752440084436210484904L,
                     (R)-0.38268343236508977172845998403039887L,
                     (R)0.0L,
                     (R)0.38268343236508977172845998403039887L,
                     (R)0.70710678118654752440084436210484904L,
                     (R)0.92387953251128675612818318939678829L};
    const int ms = (m + 12) & 15;  // sin(x) = cos(x - pi/2)
    return {c[m & 15], (R)S * c[ms]};
}

template <class R, int S, int N>
__device__ __forceinline__ void f_dft(cpx<R>* x);

// length A*B with A, B coprime: inputs n = (B a + A b) mod AB, outputs k with k = ka mod A
// and k = kb mod B, A- and B-point transforms between them and no twiddle factors (Good,
// 1958); the index maps fold to constants
constexpr int pfa_out(int A, int B, int ka, int kb) {
    for (int k = 0; k < A * B; ++k)
        if (k % A == ka && k % B == kb) return k;
    return 0;
}
template <class R, int S, int A, int B>
__device__ __forceinline__ void f_dft_coprime(cpx<R>* x) {
    cpx<R> t[A][B];
#pragma unroll
    for (int b = 0; b < B; ++b) {
        cpx<R> v[A];
#pragma unroll
        for (int a = 0; a < A; ++a) v[a] = x[(B * a + A * b) % (A * B)];
        f_dft<R, S, A>(v);
#pragma unroll
        for (int a = 0; a < A; ++a) t[a][b] = v[a];
    }
#pragma unroll
    for (int a = 0; a < A; ++a) {
        f_dft<R, S, B>(t[a]);
#pragma unroll
        for (int b = 0; b < B; ++b) x[pfa_out(A, B, a, b)] = t[a][b];
    }
}

template <class R, int S, int N>
__device__ __forceinline__ void f_dft(cpx<R>* x) {
    if constexpr (N == 3) {
        const R h = (R)0.86602540378443864676372317075293618L;  // sqrt(3)/2
        const cpx<R> a0 = x[0], t = cadd(x[1], x[2]), d = csub(x[1], x[2]);
        const cpx<R> m = {a0.re - (R)0.5 * t.re, a0.im - (R)0.5 * t.im};
        const cpx<R> w = f_mul_si<R, S>(cpx<R>{h * d.re, h * d.im});
        x[0] = cadd(a0, t);
        x[1] = cadd(m, w);
        x[2] = csub(m, w);
    } else if constexpr (N == 5) {
        const R c1 = (R)0.30901699437494742410229341718281906L;   // cos(2pi/5)
        const R c2 = (R)-0.80901699437494742410229341718281906L;  // cos(4pi/5)
        const R s1 = (R)0.95105651629515357211643933337938214L;   // sin(2pi/5)
        const R s2 = (R)0.58778525229247312916870595463907277L;   // sin(4pi/5)
        const cpx<R> a0 = x[0];
        const cpx<R> t1 = cadd(x[1], x[4]), t2 = cadd(x[2], x[3]), t3 = csub(x[1], x[4]), t4 = csub(x[2], x[3]);
        const cpx<R> b1 = {a0.re + c1 * t1.re + c2 * t2.re, a0.im + c1 * t1.im + c2 * t2.im};
        const cpx<R> b2 = {a0.re + c2 * t1.re + c1 * t2.re, a0.im + c2 * t1.im + c1 * t2.im};
        const cpx<R> e1 = f_mul_si<R, S>(cpx<R>{s1 * t3.re + s2 * t4.re, s1 * t3.im + s2 * t4.im});
        const cpx<R> e2 = f_mul_si<R, S>(cpx<R>{s2 * t3.re - s1 * t4.re, s2 * t3.im - s1 * t4.im});
        x[0] = cadd(a0, cadd(t1, t2));
        x[1] = cadd(b1, e1);
        x[4] = csub(b1, e1);
        x[2] = cadd(b2, e2);
        x[3] = csub(b2, e2);
    } else if constexpr (N == 6) {
        f_dft_coprime<R, S, 2, 3>(x);
    } else if constexpr (N == 10) {
        f_dft_coprime<R, S, 2, 5>(x);
    } else if constexpr (N == 12) {
        f_dft_coprime<R, S, 4, 3>(x);
    } else if constexpr (N == 15) {
        f_dft_coprime<R, S, 3, 5>(x);
    } else if constexpr (N == 18) {
        f_dft_coprime<R, S, 2, 9>(x);
    } else if constexpr (N == 20) {
        f_dft_coprime<R, S, 4, 5>(x);
    } else if constexpr (N == 9) {  // 3 x 3
        const R c1 = (R)0.76604444311897803520239265055541668L, s1 = (R)0.64278760968653932632264340990726343L;
        const R c2 = (R)0.17364817766693034885171662676931480L, s2 = (R)0.98480775301220805936674302458952301L;
        const R c4 = (R)-0.93969262078590838405410927732473147L, s4 = (R)0.34202014332566873304409961468225958L;
        const cpx<R> w1 = {c1, (R)S * s1}, w2 = {c2, (R)S * s2}, w4 = {c4, (R)S * s4};  // exp(S 2 pi i m/9)
        cpx<R> t[3][3];
#pragma unroll
        for (int b = 0; b < 3; ++b) {
            cpx<R> v[3] = {x[b], x[3 + b], x[6 + b]};
            f_dft<R, S, 3>(v);
#pragma unroll
            for (int a = 0; a < 3; ++a) t[a][b] = v[a];
        }
        t[1][1] = cmul(t[1][1], w1);
        t[1][2] = cmul(t[1][2], w2);
        t[2][1] = cmul(t[2][1], w2);
        t[2][2] = cmul(t[2][2], w4);
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            f_dft<R, S, 3>(t[a]);
#pragma unroll
            for (int b = 0; b < 3; ++b) x[a + 3 * b] = t[a][b];
        }
    } else if constexpr (N == 2) {
        const cpx<R> a = x[0], b = x[1];
        x[0] = cadd(a, b);
        x[1] = csub(a, b);
    } else if constexpr (N == 4) {
        f_dft4<R, S>(x[0], x[1], x[2], x[3]);
    } else if constexpr (N == 8) {
        cpx<R> e0 = x[0], e1 = x[2], e2 = x[4], e3 = x[6];
        cpx<R> o0 = x[1], o1 = x[3], o2 = x[5], o3 = x[7];
        f_dft4<R, S>(e0, e1, e2, e3);
        f_dft4<R, S>(o0, o1, o2, o3);
        const cpx<R> w1 = cmul(o1, w16<R, S>(2));
        const cpx<R> w2 = cmul(o2, w16<R, S>(4));
        const cpx<R> w3 = cmul(o3, w16<R, S>(6));
        x[0] = cadd(e0, o0);
        x[4] = csub(e0, o0);
        x[1] = cadd(e1, w1);
        x[5] = csub(e1, w1);
        x[2] = cadd(e2, w2);
        x[6] = csub(e2, w2);
        x[3] = cadd(e3, w3);
        x[7] = csub(e3, w3);
    } else {  // 16 = 4 x 4
        static_assert(N == 16, "transform length");
        cpx<R> t[16];
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            cpx<R> a0 = x[b], a1 = x[4 + b], a2 = x[8 + b], a3 = x[12 + b];
            f_dft4<R, S>(a0, a1, a2, a3);
            t[4 * b + 0] = a0;
            t[4 * b + 1] = a1;
            t[4 * b + 2] = a2;
            t[4 * b + 3] = a3;
        }
#pragma unroll
        for (int b = 1; b < 4; ++b)
#pragma unroll
            for (int c = 1; c < 4; ++c) t[4 * b + c] = cmul(t[4 * b + c], w16<R, S>(b * c));
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            cpx<R> a0 = t[c], a1 = t[4 + c], a2 = t[8 + c], a3 = t[12 + c];
            f_dft4<R, S>(a0, a1, a2, a3);
            x[c] = a0;
            x[c + 4] = a1;
            x[c + 8] = a2;
            x[c + 12] = a3;
        }
    }
}

// stage 1 twiddle: v[k1] *= W_L^(n2 k1) with W_L = exp(S 2 pi i / L), table tw[m] = exp(-2 pi i m/L)
// (n2 = 0 multiplies by tw[0] = 1 exactly: no branch, so the N1 - 1 loads issue
// together instead of each waiting inside a divergent region)
template <class R, int S, int N1>
__device__ __forceinline__ void f_twiddle(cpx<R>* v, int n2, const cpx<R>* __restrict__ tw) {
    cpx<R> w[N1];
#pragma unroll
    for (int k1 = 1; k1 < N1; ++k1) w[k1] = tw[n2 * k1];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int k1 = 1; k1 < N1; ++k1) {
        if (S > 0) w[k1].im = -w[k1].im;
        v[k1] = cmul(v[k1], w[k1]);
    }
}

// the same from a copy of the table in LDS (short latency: no batching needed)
template <class R, int S, int N1>
__device__ __forceinline__ void f_twiddle_lds(cpx<R>* v, int n2, const cpx<R>* tw) {
#pragma unroll
    for (int k1 = 1; k1 < N1; ++k1) {
        cpx<R> w = tw[n2 * k1];
        if (S > 0) w.im = -w.im;
        v[k1] = cmul(v[k1], w);
    }
}

// A stage-2 thread transforms columns k1 = n2, n2 + N2, ...: NQ of them, the last beyond
// N1 (and idle) where N2 does not divide N1.  Powers of two take N1 >= N2; the other
// lengths N1 <= N2 (one column a thread, as few registers as the balanced factors allow).
template <int N1, int N2>
constexpr int kNQ = (N1 + N2 - 1) / N2;
template <int N1, int N2>
__device__ __forceinline__ bool f_has_col(int k1) {
    return N1 % N2 == 0 || k1 < N1;
}
// lines of an x-pass block: 128 threads at the power-of-two lengths; elsewhere an even
// number (the staged copy's alignment) that leaves few lanes of the last wave idle
template <int N2>
constexpr int kXLines = N2 == 5 ? 24 : N2 == 6 ? 32 : N2 == 9 ? 14 : N2 == 10 ? 12 : N2 == 12 ? 16 : N2 == 15 ? 8
                        : N2 == 18 ? 14 : N2 == 20 ? 12 : 128 / N2;

// --------------------------------------------------------------- X passes
template <class R, class T>
__device__ __forceinline__ cpx<R> ld_c(const T* p, long i) {
    const T* q = p + 2 * i;
    return {(R)q[0], (R)q[1]};
}
template <class R, class T>
__device__ __forceinline__ void st_c(T* p, long i, cpx<R> v) {
    T* q = p + 2 * i;
    q[0] = (T)v.re;
    q[1] = (T)v.im;
}
template <>
__device__ __forceinline__ cpx<double> ld_c<double, double>(const double* p, long i) {
    return reinterpret_cast<const cpx<double>*>(p)[i];
}
template <>
__device__ __forceinline__ void st_c<double, double>(double* p, long i, cpx<double> v) {
    reinterpret_cast<cpx<double>*>(p)[i] = v;
}
template <>
__device__ __forceinline__ cpx<float> ld_c<float, float>(const float* p, long i) {
    return reinterpret_cast<const cpx<float>*>(p)[i];
}
template <>
__device__ __forceinline__ void st_c<float, float>(float* p, long i, cpx<float> v) {
    reinterpret_cast<cpx<float>*>(p)[i] = v;
}

// Forward r2c of rows: row r of field blockIdx.y, input stride istride reals (physical
// nxpp), output stride ostride reals (spectral nx).
template <class R, class TI, class TO, int N1, int N2>
__global__ void __launch_bounds__(kXLines<N2> * N2) k_xfwd_fast(FieldList<TI> in, FieldList<TO> out, int nrows,
                                                                int istride, int ostride,
                                                                const cpx<R>* __restrict__ tw,
                                                                const cpx<R>* __restrict__ twr) {
    constexpr int L = N1 * N2;
    constexpr int LPB = kXLines<N2>;       // lines per block
    constexpr int NQ = kNQ<N1, N2>;
    constexpr int TS = N1 * (N2 + 1);      // padded transpose tile per line (>= L)
    __shared__ cpx<R> T[LPB * TS];
    const int tid = threadIdx.x;
    const int l = tid / N2, n2 = tid % N2;
    const int f = blockIdx.y;
    const long r = (long)blockIdx.x * LPB + l;
    const bool valid = r < nrows;
    const long rr = valid ? r : nrows - 1;  // lines past the end read the last line, store nothing
    const TI* src = in.p[f] + rr * istride;
    TO* dst = out.p[f] + rr * ostride;
    cpx<R> v[N1];
#pragma unroll
    for (int n1 = 0; n1 < N1; ++n1) v[n1] = ld_c<R>(src, N2 * n1 + n2);
    f_dft<R, -1, N1>(v);
    f_twiddle<R, -1, N1>(v, n2, tw);
    cpx<R>* Tl = T + l * TS;
#pragma unroll
    for (int k1 = 0; k1 < N1; ++k1) Tl[k1 * (N2 + 1) + n2] = v[k1];
    __syncthreads();
    cpx<R> u[NQ][N2];
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        const int k1 = n2 + N2 * q;
        if (f_has_col<N1, N2>(k1)) {
#pragma unroll
            for (int j = 0; j < N2; ++j) u[q][j] = Tl[k1 * (N2 + 1) + j];
            f_dft<R, -1, N2>(u[q]);
        }
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < NQ; ++q)
        if (f_has_col<N1, N2>(n2 + N2 * q)) {
#pragma unroll
            for (int k2 = 0; k2 < N2; ++k2) Tl[(n2 + N2 * q) + N1 * k2] = u[q][k2];
        }
    __syncthreads();
    if (!valid) return;
    // X_k = 1/2 (Z_k + conj Z_{L-k}) - i/2 W^k (Z_k - conj Z_{L-k})
#pragma unroll
    for (int j = 0; j < N1; ++j) {
        const int k = n2 + N2 * j;
        const cpx<R> zk = Tl[k];
        const cpx<R> zc = cconj(Tl[k == 0 ? 0 : L - k]);
        const cpx<R> a = {(R)0.5 * (zk.re + zc.re), (R)0.5 * (zk.im + zc.im)};
        const cpx<R> d = {(R)0.5 * (zk.re - zc.re), (R)0.5 * (zk.im - zc.im)};
        const cpx<R> wd = cmul(twr[k], d);
        st_c<R>(dst, k, cpx<R>{a.re + wd.im, a.im - wd.re});
    }
}

// Inverse c2r of rows holding L complex coefficients (input row stride istride
// reals) into physical rows (stride nxpp, the two pad reals written as zero);
// in place when in == out and istride == nxpp.  STAGE: the block's rows, pads
// included, are one contiguous run of up to LPB*nxpp reals of one field; they are assembled in the LDS tile and stored as 16-byte vectors, so the
// stores fill whole 128-byte segments although the rows of stride nxpp = L*2 + 2 start
// off the segment grid.
template <class R, class TI, class TO, int N1, int N2, bool STAGE = false>
__global__ void __launch_bounds__(kXLines<N2> * N2) k_xinv_fast(FieldList<TI> in, FieldList<TO> out, int nrows,
                                                                int istride, int nxpp,
                                                                const cpx<R>* __restrict__ tw,
                                                                const cpx<R>* __restrict__ twr) {
    constexpr int L = N1 * N2;
    constexpr int LPB = kXLines<N2>;
    constexpr int NQ = kNQ<N1, N2>;
    constexpr int TS = N1 * (N2 + 1);
    __shared__ __align__(16) cpx<R> T[LPB * TS];  // 16-byte aligned for the staged vector copy
    const int tid = threadIdx.x;
    const int l = tid / N2, n2 = tid % N2;
    const int f = blockIdx.y;
    const long r = (long)blockIdx.x * LPB + l;
    const bool valid = r < nrows;
    // lines past the end read the last line (unconditional loads issue back to
    // back; a load under a per-element branch feeding the LDS store would wait
    // for each in turn) and store nothing
    const long rr = valid ? r : nrows - 1;
    const TI* rin = in.p[f] + rr * istride;
    TO* row = out.p[f] + rr * nxpp;
    cpx<R>* Tl = T + l * TS;
    {
        cpx<R> t[N1];
#pragma unroll
        for (int j = 0; j < N1; ++j) t[j] = ld_c<R>(rin, n2 + N2 * j);
#pragma unroll
        for (int j = 0; j < N1; ++j) Tl[n2 + N2 * j] = t[j];
    }
    __syncthreads();
    // Z'_n = (X_n + conj X_{L-n}) + i W^-n (X_n - conj X_{L-n}); X_L = 0, Im X_0 ignored
    cpx<R> v[N1];
#pragma unroll
    for (int n1 = 0; n1 < N1; ++n1) {
        const int n = N2 * n1 + n2;
        cpx<R> xk = Tl[n];
        cpx<R> xc;
        if (n == 0) {
            xk.im = 0;
            xc = {0, 0};
        } else {
            xc = cconj(Tl[L - n]);
        }
        const cpx<R> s = cadd(xk, xc);
        const cpx<R> d = csub(xk, xc);
        const cpx<R> wd = cmul(cconj(twr[n]), d);
        v[n1] = {s.re - wd.im, s.im + wd.re};
    }
    f_dft<R, 1, N1>(v);
    f_twiddle<R, 1, N1>(v, n2, tw);
    __syncthreads();
#pragma unroll
    for (int k1 = 0; k1 < N1; ++k1) Tl[k1 * (N2 + 1) + n2] = v[k1];
    __syncthreads();
    if constexpr (STAGE && sizeof(TO) <= sizeof(R)) {
        static_assert(LPB * TS * sizeof(cpx<R>) >= LPB * (2 * L + 2) * sizeof(TO), "staging tile");
        cpx<R> u[NQ][N2];
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            const int k1 = n2 + N2 * q;
            if (f_has_col<N1, N2>(k1)) {
#pragma unroll
                for (int j = 0; j < N2; ++j) u[q][j] = Tl[k1 * (N2 + 1) + j];
                f_dft<R, 1, N2>(u[q]);
            }
        }
        __syncthreads();
        // the block's rows in their memory layout (stride nxpp = 2L + 2 reals of TO)
        TO* S = reinterpret_cast<TO*>(T);
        TO* Sl = S + (long)l * (2 * L + 2);
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            const int k1 = n2 + N2 * q;
            if (!f_has_col<N1, N2>(k1)) continue;
#pragma unroll
            for (int k2 = 0; k2 < N2; ++k2) {
                Sl[2 * (k1 + N1 * k2)] = (TO)u[q][k2].re;
                Sl[2 * (k1 + N1 * k2) + 1] = (TO)u[q][k2].im;
            }
        }
        if (n2 == 0) {
            Sl[2 * L] = (TO)0;
            Sl[2 * L + 1] = (TO)0;
        }
        __syncthreads();
        // the valid rows of the block: one run of the field, 16-byte aligned (LPB is even)
        const long r0 = (long)blockIdx.x * LPB;
        const long nv = min((long)LPB, nrows - r0);
        TO* g = out.p[f] + r0 * nxpp;
        const long nreal = nv * nxpp;
        constexpr int VW = 16 / (int)sizeof(TO);
        using V = typename std::conditional<sizeof(TO) == 8, double2, float4>::type;
        const long nvec = nreal / VW;
        for (long e = tid; e < nvec; e += LPB * N2)
            reinterpret_cast<V*>(g)[e] = reinterpret_cast<const V*>(S)[e];
        for (long e = nvec * VW + tid; e < nreal; e += LPB * N2) g[e] = S[e];
        return;
    }
    if (!valid) return;
#pragma unroll
    for (int q = 0; q < kNQ<N1, N2>; ++q) {
        const int k1 = n2 + N2 * q;
        if (!f_has_col<N1, N2>(k1)) continue;
        cpx<R> u[N2];
#pragma unroll
        for (int j = 0; j < N2; ++j) u[j] = Tl[k1 * (N2 + 1) + j];
        f_dft<R, 1, N2>(u);
#pragma unroll
        for (int k2 = 0; k2 < N2; ++k2) st_c<R>(row, k1 + N1 * k2, u[k2]);
    }
    if (n2 == 0) st_c<R>(row, L, cpx<R>{0, 0});  // the two pad reals
}

// --------------------------------------------------------------- Y passes
// Tiles of C kx-columns x L ky-rows of one plane; lane index c fastest.
// Forward: input rows of lh complex (stride lh), output the same layout, scaled;
// in place when in == out.
template <class R, class TI, class TO, int N1, int N2, int C>
__global__ void __launch_bounds__(C * N2) k_yfwd_fast(FieldList<TI> in, FieldList<TO> out, int nplanes, int lh,
                                                      const cpx<R>* __restrict__ tw, R scale) {
    constexpr int TS = N1 * (N2 + 1) + 1;
    __shared__ cpx<R> T[C * TS];
    const int tid = threadIdx.x;
    const int c = tid % C, n2 = tid / C;
    const int ntile = (lh + C - 1) / C;
    const int tile = blockIdx.x % ntile;
    const long plane = blockIdx.x / ntile;
    const int f = (int)(plane / nplanes);
    const long pk = plane - (long)f * nplanes;
    const TI* src = in.p[f] + pk * (long)(N1 * N2) * (2 * lh);
    TO* dst = out.p[f] + pk * (long)(N1 * N2) * (2 * lh);
    const int m = tile * C + c;
    const bool valid = m < lh;
    const int mc = valid ? m : lh - 1;  // columns past the end read the last one, store nothing
    cpx<R> v[N1];
#pragma unroll
    for (int n1 = 0; n1 < N1; ++n1) v[n1] = ld_c<R>(src, (long)(N2 * n1 + n2) * lh + mc);
    f_dft<R, -1, N1>(v);
    f_twiddle<R, -1, N1>(v, n2, tw);
    cpx<R>* Tc = T + c * TS;
#pragma unroll
    for (int k1 = 0; k1 < N1; ++k1) Tc[k1 * (N2 + 1) + n2] = v[k1];
    __syncthreads();
    if (!valid) return;
#pragma unroll
    for (int q = 0; q < kNQ<N1, N2>; ++q) {
        const int k1 = n2 + N2 * q;
        if (!f_has_col<N1, N2>(k1)) continue;
        cpx<R> u[N2];
#pragma unroll
        for (int j = 0; j < N2; ++j) u[j] = Tc[k1 * (N2 + 1) + j];
        f_dft<R, -1, N2>(u);
#pragma unroll
        for (int k2 = 0; k2 < N2; ++k2)
            st_c<R>(dst, (long)(k1 + N1 * k2) * lh + m, cpx<R>{u[k2].re * scale, u[k2].im * scale});
    }
}

// Inverse: spectral rows (stride lh) in, rows of stride ph complex out.  ops.op[f]
// selects d/dx (x i*wavx) or d/dy (x i*wavy) applied to field f as it is loaded,
// in double before the conversion to R: (re, im) -> (-k im, k re).
template <class R, class TI, class TO, int N1, int N2, int C>
__global__ void __launch_bounds__(C * N2) k_yinv_fast(FieldList<TI> in, FieldList<TO> out, int nplanes, int lh,
                                                      int ph, const cpx<R>* __restrict__ tw, FftOps ops,
                                                      const double* __restrict__ wavx,
                                                      const double* __restrict__ wavy) {
    constexpr int TS = N1 * (N2 + 1) + 1;
    __shared__ cpx<R> T[C * TS];
    const int tid = threadIdx.x;
    const int c = tid % C, n2 = tid / C;
    const int ntile = (lh + C - 1) / C;
    const int tile = blockIdx.x % ntile;
    const long plane = blockIdx.x / ntile;
    const int f = (int)(plane / nplanes);
    const long pk = plane - (long)f * nplanes;
    const TI* src = in.p[f] + pk * (long)(N1 * N2) * (2 * lh);
    TO* dst = out.p[f] + pk * (long)(N1 * N2) * (2 * ph);
    const int m = tile * C + c;
    const bool valid = m < lh;
    const int mc = valid ? m : lh - 1;  // columns past the end read the last one, store nothing
    const int op = ops.op[f];
    TI qre[N1], qim[N1];
#pragma unroll
    for (int n1 = 0; n1 < N1; ++n1) {
        const TI* q = src + 2 * ((long)(N2 * n1 + n2) * lh + mc);
        qre[n1] = q[0];
        qim[n1] = q[1];
    }
    cpx<R> v[N1];
    if (op == FOP_NONE) {
#pragma unroll
        for (int n1 = 0; n1 < N1; ++n1) v[n1] = {(R)qre[n1], (R)qim[n1]};
    } else {
        const double kx = (op == FOP_DX) ? wavx[2 * mc] : 0.0;
#pragma unroll
        for (int n1 = 0; n1 < N1; ++n1) {
            const double k = (op == FOP_DX) ? kx : wavy[N2 * n1 + n2];
            const double re = (double)qre[n1], im = (double)qim[n1];
            v[n1] = {(R)(-k * im), (R)(k * re)};
        }
    }
    f_dft<R, 1, N1>(v);
    f_twiddle<R, 1, N1>(v, n2, tw);
    cpx<R>* Tc = T + c * TS;
#pragma unroll
    for (int k1 = 0; k1 < N1; ++k1) Tc[k1 * (N2 + 1) + n2] = v[k1];
    __syncthreads();
    if (!valid) return;
#pragma unroll
    for (int q = 0; q < kNQ<N1, N2>; ++q) {
        const int k1 = n2 + N2 * q;
        if (!f_has_col<N1, N2>(k1)) continue;
        cpx<R> u[N2];
#pragma unroll
        for (int j = 0; j < N2; ++j) u[j] = Tc[k1 * (N2 + 1) + j];
        f_dft<R, 1, N2>(u);
#pragma unroll
        for (int k2 = 0; k2 < N2; ++k2) st_c<R>(dst, (long)(k1 + N1 * k2) * ph + m, u[k2]);
    }
}

// Inverse y pass of a velocity spectrum and its x and y derivatives from one load:
// out.p[3 f] = F^-1_y(u), out.p[3 f + 1] = i kx F^-1_y(u) (kx is constant along a
// y column, so the x derivative is applied at the store), out.p[3 f + 2] =
// F^-1_y(i ky u) (ky is applied at the load).  Outputs are rows of stride ph.
template <class R, class TI, class TO, int N1, int N2, int C>
__global__ void __launch_bounds__(C * N2) k_yinv3_fast(FieldList<TI> in, FieldList<TO> out, int nplanes, int lh,
                                                       int ph, const cpx<R>* __restrict__ tw,
                                                       const double* __restrict__ wavx,
                                                       const double* __restrict__ wavy,
                                                       const double* __restrict__ ftab) {
    constexpr int TS = N1 * (N2 + 1) + 1;
    __shared__ cpx<R> T[C * TS];
    const int tid = threadIdx.x;
    const int c = tid % C, n2 = tid / C;
    const int ntile = (lh + C - 1) / C;
    const int tile = blockIdx.x % ntile;
    const long plane = blockIdx.x / ntile;
    const int f = (int)(plane / nplanes);
    const long pk = plane - (long)f * nplanes;
    const TI* src = in.p[f] + pk * (long)(N1 * N2) * (2 * lh);
    const long ooff = pk * (long)(N1 * N2) * (2 * ph);
    TO* du = out.p[3 * f] + ooff;
    TO* dx = out.p[3 * f + 1] + ooff;
    TO* dy = out.p[3 * f + 2] + ooff;
    const int m = tile * C + c;
    const bool valid = m < lh;
    const int mc = valid ? m : lh - 1;  // columns past the end read the last one, store nothing
    const double kx = wavx[2 * mc];
    double re[N1], im[N1];
#pragma unroll
    for (int n1 = 0; n1 < N1; ++n1) {
        const TI* q = src + 2 * ((long)(N2 * n1 + n2) * lh + mc);
        re[n1] = (double)q[0];
        im[n1] = (double)q[1];
    }
    if (ftab) {
        // the spectral filter as a real factor per mode: the reference's
        // magnitude/phase rebuild (specfilter_mode) equals it up to the rounding
        // of re/|u|, i.e. ~eps |re|^2/|im| on modes with |im| << |re|
        double fac[N1];
#pragma unroll
        for (int n1 = 0; n1 < N1; ++n1) fac[n1] = ftab[(N2 * n1 + n2) * lh + mc];
        __builtin_amdgcn_sched_barrier(0);  // keep the loads together, ahead of their uses
#pragma unroll
        for (int n1 = 0; n1 < N1; ++n1) {
            re[n1] *= fac[n1];
            im[n1] *= fac[n1];
        }
    }
    cpx<R>* Tc = T + c * TS;
#pragma unroll
    for (int pass = 0; pass < 2; ++pass) {
        cpx<R> v[N1];
#pragma unroll
        for (int n1 = 0; n1 < N1; ++n1) {
            if (pass == 0) {
                v[n1] = {(R)re[n1], (R)im[n1]};
            } else {
                const double k = wavy[N2 * n1 + n2];
                v[n1] = {(R)(-k * im[n1]), (R)(k * re[n1])};
            }
        }
        f_dft<R, 1, N1>(v);
        f_twiddle<R, 1, N1>(v, n2, tw);
        if (pass == 1) __syncthreads();  // the first pass has read its tile
#pragma unroll
        for (int k1 = 0; k1 < N1; ++k1) Tc[k1 * (N2 + 1) + n2] = v[k1];
        __syncthreads();
        if (valid) {
#pragma unroll
            for (int q = 0; q < kNQ<N1, N2>; ++q) {
                const int k1 = n2 + N2 * q;
                if (!f_has_col<N1, N2>(k1)) continue;
                cpx<R> u[N2];
#pragma unroll
                for (int j = 0; j < N2; ++j) u[j] = Tc[k1 * (N2 + 1) + j];
                f_dft<R, 1, N2>(u);
#pragma unroll
                for (int k2 = 0; k2 < N2; ++k2) {
                    const long o = (long)(k1 + N1 * k2) * ph + m;
                    if (pass == 0) {
                        st_c<R>(du, o, u[k2]);
                        st_c<R>(dx, o, cpx<R>{(R)(-kx) * u[k2].im, (R)kx * u[k2].re});
                    } else {
                        st_c<R>(dy, o, u[k2]);
                    }
                }
            }
        }
    }
}

// Forward y pass fused with the velocity right-hand side (one block: C kx-columns
// of one plane, one component l).  The three pieces are transformed in turn
// through the same LDS tile; N accumulates in FP64 in the order of the separate
// passes (nlt, then - i kx h_x, then - i ky h_y, each piece rounded to R after
// scaling as the separate forward pass stores it): the results of fast_yfwd followed by the
// right-hand-side kernel up to the last rounding of products that join a following sum.
// HBM-bound: 30 FP64 field passes (6.07 GB by the counters, 1.24 ms at 512x193x256: 4.9 TB/s)
// where the two passes take 46; the FP64 step there with the dynamic model 8.32 -> 7.74 ms,
// the 240x114x120 sigma step 939 -> 885 us.
template <class TN>
__device__ __forceinline__ void ld_h(const void* p, long q, double& re, double& im) {
    const TN* t = reinterpret_cast<const TN*>(p) + 2 * q;
    re = (double)t[0];
    im = (double)t[1];
}
template <class TN>
__device__ __forceinline__ void st_h(void* p, long q, double re, double im) {
    TN* t = reinterpret_cast<TN*>(p) + 2 * q;
    t[0] = (TN)re;
    t[1] = (TN)im;
}

template <class R, class TH, int N1, int N2, int C>
__global__ void __launch_bounds__(C * N2) k_yfwd_rhs(FieldList<R> pc, int nplanes, int lh,
                                                     const cpx<R>* __restrict__ tw, R scale, YRhsArgs a) {
    constexpr int L = N1 * N2;
    constexpr int TS = N1 * (N2 + 1) + 1;
    constexpr int NQ = kNQ<N1, N2>;
    __shared__ cpx<R> T[C * TS];
    __shared__ cpx<R> Tw[L];
    const int tid = threadIdx.x;
    for (int t = tid; t < L; t += C * N2) Tw[t] = tw[t];
    const int c = tid % C, n2 = tid / C;
    const int ntile = (lh + C - 1) / C;
    const int tile = blockIdx.x % ntile;
    const long rest = blockIdx.x / ntile;
    const int pk = (int)(rest % nplanes);
    const int l = (int)(rest / nplanes);
    const int m = tile * C + c;
    const bool valid = m < lh;
    const int mc = valid ? m : lh - 1;  // columns past the end read the last one, store nothing
    const double wx = a.wavx[2 * mc];
    double nr[NQ][N2], ni[NQ][N2];
    cpx<R>* Tc = T + c * TS;
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        // one piece at a time: the next piece's loads are not hoisted over this
        // piece's second stage (three live tiles would halve the occupancy)
        __builtin_amdgcn_sched_barrier(0);
        const R* src = pc.p[3 * l + q] + (long)pk * L * (2 * lh);
        cpx<R> v[N1];
#pragma unroll
        for (int n1 = 0; n1 < N1; ++n1) v[n1] = ld_c<R>(src, (long)(N2 * n1 + n2) * lh + mc);
        f_dft<R, -1, N1>(v);
        __syncthreads();  // the twiddle table is in place; the previous piece has read its tile
        f_twiddle_lds<R, -1, N1>(v, n2, Tw);
#pragma unroll
        for (int k1 = 0; k1 < N1; ++k1) Tc[k1 * (N2 + 1) + n2] = v[k1];
        __syncthreads();
#pragma unroll
        for (int qq = 0; qq < NQ; ++qq) {
            const int k1 = n2 + N2 * qq;
            if (!f_has_col<N1, N2>(k1)) continue;
            cpx<R> u[N2];
#pragma unroll
            for (int j = 0; j < N2; ++j) u[j] = Tc[k1 * (N2 + 1) + j];
            f_dft<R, -1, N2>(u);
#pragma unroll
            for (int k2 = 0; k2 < N2; ++k2) {
                const double vr = (double)(R)(u[k2].re * scale), vi = (double)(R)(u[k2].im * scale);
                if (q == 0) {
                    nr[qq][k2] = vr;
                    ni[qq][k2] = vi;
                } else if (q == 1) {
                    nr[qq][k2] = nr[qq][k2] - (-wx * vi);
                    ni[qq][k2] = ni[qq][k2] - (wx * vr);
                } else {
                    const double wy = a.wavy[k1 + N1 * k2];
                    nr[qq][k2] = nr[qq][k2] - (-wy * vi);
                    ni[qq][k2] = ni[qq][k2] - (wy * vr);
                }
            }
        }
    }
    if (!valid) return;
    const double ub = (l == 0 && m == 0) ? a.ubarpp[pk] : 0.0;
#pragma unroll
    for (int qq = 0; qq < NQ; ++qq) {
        const int k1 = n2 + N2 * qq;
        if (!f_has_col<N1, N2>(k1)) continue;
        constexpr int NB = N2 % 4 == 0 ? 4 : N2 % 3 == 0 ? 3 : 5;  // outputs per batch
        static_assert(N2 % NB == 0, "batches of the stage-2 outputs");
#pragma unroll
        for (int b0 = 0; b0 < N2; b0 += NB) {
            // the history of NB outputs is loaded before their stores (and not
            // earlier: the barrier bounds the live registers)
            __builtin_amdgcn_sched_barrier(0);
            double h1r[NB], h1i[NB], h2r[NB], h2i[NB], u0r[NB], u0i[NB], u1r[NB], u1i[NB], u2r[NB], u2i[NB];
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                const int ky = k1 + N1 * (b0 + b);
                const long qd = ((long)pk * L + ky) * lh + m;
                ld_h<TH>(a.nl[l], qd, h1r[b], h1i[b]);
                ld_h<TH>(a.nlm[l], qd, h2r[b], h2i[b]);
                ld_h<double>(a.u[l], qd, u0r[b], u0i[b]);
                ld_h<double>(a.un[l], qd, u1r[b], u1i[b]);
                ld_h<double>(a.unm[l], qd, u2r[b], u2i[b]);
            }
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                const int k2 = b0 + b;
                const int ky = k1 + N1 * k2;
                const long qd = ((long)pk * L + ky) * lh + m;
                double xr = nr[qq][k2], xi = ni[qq][k2];
                if (sizeof(TH) < sizeof(double)) {
                    xr = (double)(TH)xr;
                    xi = (double)(TH)xi;
                }
                st_h<TH>(a.nout[l], qd, xr, xi);
                const double cr = a.ab0 * xr + a.ab1 * h1r[b] + a.ab2 * h2r[b];
                const double ci = a.ab0 * xi + a.ab1 * h1i[b] + a.ab2 * h2i[b];
                double rr = -a.dtnui * (a.dt * cr + a.bdf0 * u0r[b] + a.bdf1 * u1r[b] + a.bdf2 * u2r[b]);
                const double ri = -a.dtnui * (a.dt * ci + a.bdf0 * u0i[b] + a.bdf1 * u1i[b] + a.bdf2 * u2i[b]);
                if (ky == 0) rr = rr - ub;
                st_h<double>(a.rhs[l], qd, rr, ri);
            }
        }
    }
}


// The blended ceiling on one spectral plane, out += F[m(x) F^-1 in], in one launch: m
// depends on x only, so the y transforms cancel.  Along x the rows ky and -ky of a real
// field's half spectrum, F(kx, -ky) = conj F(-kx, ky), are two real lines,
// P = (F(ky) + F(-ky)) / 2 and Q = (F(ky) - F(-ky)) / 2i: c2r, the weight (with the
// transform pair's 1/nx in it) and r2c as in the x passes above, then P + iQ and P - iQ
// are added to the two rows (ky = 0 and the Nyquist row pair with themselves, Q = 0).
// Latency-bound (two planes): 17 us at 256 x 128 where the 2-D transforms, the weight and
// the sum took six launches and 30 us.
struct XBlendArgs {
    const double* in[2];
    double* out[2];
    const double* m;
    double scale;
    int ny;
};
template <class R, int N1, int N2>
__global__ void __launch_bounds__(kXLines<N2> * N2) k_xblend(XBlendArgs a, const cpx<R>* __restrict__ tw,
                                                            const cpx<R>* __restrict__ twr) {
    constexpr int L = N1 * N2;
    constexpr int LPB = kXLines<N2>;
    constexpr int NQ = kNQ<N1, N2>;
    constexpr int TS = N1 * (N2 + 1);
    static_assert(LPB % 2 == 0, "the two lines of a pair share a block");
    __shared__ cpx<R> T[LPB * TS];
    const int tid = threadIdx.x;
    const int l = tid / N2, n2 = tid % N2;
    const int nlines = a.ny + 2;
    const int line = blockIdx.x * LPB + l;
    const bool valid = line < nlines;
    const int pr = min(line, nlines - 1) / 2;  // ky = pr and its partner
    const bool isq = line & 1;
    const int j0 = pr, j1 = (pr == 0) ? 0 : a.ny - pr;
    const double* f = a.in[blockIdx.y];
    const double* r0 = f + (long)j0 * (2 * L);
    const double* r1 = f + (long)j1 * (2 * L);
    cpx<R>* Tl = T + l * TS;
    {
        cpx<R> x[N1], y[N1];
#pragma unroll
        for (int j = 0; j < N1; ++j) {
            x[j] = ld_c<R>(r0, n2 + N2 * j);
            y[j] = ld_c<R>(r1, n2 + N2 * j);
        }
#pragma unroll
        for (int j = 0; j < N1; ++j) {
            const cpx<R> s = cadd(x[j], y[j]), d = csub(x[j], y[j]);
            Tl[n2 + N2 * j] = isq ? cpx<R>{(R)0.5 * d.im, (R)-0.5 * d.re} : cpx<R>{(R)0.5 * s.re, (R)0.5 * s.im};
        }
    }
    __syncthreads();
    cpx<R> v[N1];
#pragma unroll
    for (int n1 = 0; n1 < N1; ++n1) {
        const int n = N2 * n1 + n2;
        cpx<R> xk = Tl[n];
        cpx<R> xc;
        if (n == 0) {
            xk.im = 0;
            xc = {0, 0};
        } else {
            xc = cconj(Tl[L - n]);
        }
        const cpx<R> s = cadd(xk, xc);
        const cpx<R> d = csub(xk, xc);
        const cpx<R> wd = cmul(cconj(twr[n]), d);
        v[n1] = {s.re - wd.im, s.im + wd.re};
    }
    // the two stages of a transform of v through the line's tile, its outputs in u
    cpx<R> u[NQ][N2];
    auto stages = [&](auto sign) {
        constexpr int S = decltype(sign)::value;
        f_dft<R, S, N1>(v);
        f_twiddle<R, S, N1>(v, n2, tw);
        __syncthreads();
#pragma unroll
        for (int k1 = 0; k1 < N1; ++k1) Tl[k1 * (N2 + 1) + n2] = v[k1];
        __syncthreads();
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            const int k1 = n2 + N2 * q;
            if (f_has_col<N1, N2>(k1)) {
#pragma unroll
                for (int j = 0; j < N2; ++j) u[q][j] = Tl[k1 * (N2 + 1) + j];
                f_dft<R, S, N2>(u[q]);
            }
        }
        __syncthreads();
    };
    stages(std::integral_constant<int, 1>{});
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        const int k1 = n2 + N2 * q;
        if (!f_has_col<N1, N2>(k1)) continue;
#pragma unroll
        for (int k2 = 0; k2 < N2; ++k2) {
            const int k = k1 + N1 * k2;
            Tl[k] = {u[q][k2].re * (R)(a.scale * a.m[2 * k]), u[q][k2].im * (R)(a.scale * a.m[2 * k + 1])};
        }
    }
    __syncthreads();
#pragma unroll
    for (int n1 = 0; n1 < N1; ++n1) v[n1] = Tl[N2 * n1 + n2];
    stages(std::integral_constant<int, -1>{});
#pragma unroll
    for (int q = 0; q < NQ; ++q)
        if (f_has_col<N1, N2>(n2 + N2 * q)) {
#pragma unroll
            for (int k2 = 0; k2 < N2; ++k2) Tl[(n2 + N2 * q) + N1 * k2] = u[q][k2];
        }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < N1; ++j) {
        const int k = n2 + N2 * j;
        const cpx<R> zk = Tl[k];
        const cpx<R> zc = cconj(Tl[k == 0 ? 0 : L - k]);
        const cpx<R> s = {(R)0.5 * (zk.re + zc.re), (R)0.5 * (zk.im + zc.im)};
        const cpx<R> d = {(R)0.5 * (zk.re - zc.re), (R)0.5 * (zk.im - zc.im)};
        const cpx<R> wd = cmul(twr[k], d);
        v[j] = {s.re + wd.im, s.im - wd.re};
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < N1; ++j) Tl[n2 + N2 * j] = v[j];
    __syncthreads();
    if (!valid || (isq && j0 == j1)) return;
    const cpx<R>* Tp = T + (l ^ 1) * TS;  // the pair's other line
    double* row = a.out[blockIdx.y] + (long)(isq ? j1 : j0) * (2 * L);
#pragma unroll
    for (int j = 0; j < N1; ++j) {
        const int k = n2 + N2 * j;
        const cpx<R> p = isq ? Tp[k] : v[j], q = isq ? v[j] : Tp[k];
        const cpx<R> o = ld_c<R>(row, k);
        // P + iQ or P - iQ
        const cpx<R> x = isq ? cpx<R>{p.re + q.im, p.im - q.re} : cpx<R>{p.re - q.im, p.im + q.re};
        st_c<R>(row, k, cadd(o, x));
    }
}

// -------------------------------------------------------------- launchers
template <class R, int N1, int N2>
int launch_xblend(const XBlendArgs& a, const cpx<R>* tw, const cpx<R>* twr, hipStream_t s) {
    constexpr int LPB = kXLines<N2>;
    hipLaunchKernelGGL((k_xblend<R, N1, N2>), dim3((unsigned)((a.ny + 2 + LPB - 1) / LPB), 2), dim3(LPB * N2), 0, s, a,
                       tw, twr);
    LSB_HIP(hipGetLastError());
    return LSB_OK;
}

template <class R, class TI, class TO, int N1, int N2>
int launch_xfwd(const FieldList<TI>& in, const FieldList<TO>& out, int nrows, int nf, int istride, int ostride,
                const cpx<R>* tw, const cpx<R>* twr, hipStream_t s) {
    constexpr int LPB = kXLines<N2>;
    hipLaunchKernelGGL((k_xfwd_fast<R, TI, TO, N1, N2>), dim3((unsigned)((nrows + LPB - 1) / LPB), (unsigned)nf),
                       dim3(LPB * N2), 0, s, in, out, nrows, istride, ostride, tw, twr);
    LSB_HIP(hipGetLastError());
    return LSB_OK;
}

template <class R, class TI, class TO, int N1, int N2>
int launch_xinv(const FieldList<TI>& in, const FieldList<TO>& out, int nrows, int nf, int istride, int nxpp,
                const cpx<R>* tw, const cpx<R>* twr, hipStream_t s) {
    constexpr int LPB = kXLines<N2>;
    // the staged store: rows of exactly 2 L + 2 reals, fields 16-byte aligned
    bool aligned = nxpp == 2 * N1 * N2 + 2 && sizeof(TO) <= sizeof(R);
    const char* off = std::getenv("LSB_NO_XSTAGE");  // the direct row stores, for tests
    if (off && off[0] && std::strcmp(off, "0") != 0) aligned = false;
    for (int f = 0; f < nf && aligned; ++f) aligned = ((uintptr_t)out.p[f] & 15) == 0;
    const dim3 grid((unsigned)((nrows + LPB - 1) / LPB), (unsigned)nf);
    if (aligned)
        hipLaunchKernelGGL((k_xinv_fast<R, TI, TO, N1, N2, true>), grid, dim3(LPB * N2), 0, s, in, out, nrows, istride,
                           nxpp, tw, twr);
    else
        hipLaunchKernelGGL((k_xinv_fast<R, TI, TO, N1, N2>), grid, dim3(LPB * N2), 0, s, in, out, nrows, istride, nxpp,
                           tw, twr);
    LSB_HIP(hipGetLastError());
    return LSB_OK;
}

template <class R, class TI, class TO, int N1, int N2, int C>
int launch_yfwd(const FieldList<TI>& in, const FieldList<TO>& out, int nplanes, int nf, int lh, const cpx<R>* tw,
                R scale, hipStream_t s) {
    const long nblk = (long)((lh + C - 1) / C) * nplanes * nf;
    hipLaunchKernelGGL((k_yfwd_fast<R, TI, TO, N1, N2, C>), dim3((unsigned)nblk), dim3(C * N2), 0, s, in, out, nplanes,
                       lh, tw, scale);
    LSB_HIP(hipGetLastError());
    return LSB_OK;
}

template <class R, class TI, class TO, int N1, int N2, int C>
int launch_yinv(const FieldList<TI>& in, const FieldList<TO>& out, int nplanes, int nf, int lh, int ph,
                const cpx<R>* tw, const FftOps& ops, const double* wavx, const double* wavy, hipStream_t s) {
    const long nblk = (long)((lh + C - 1) / C) * nplanes * nf;
    hipLaunchKernelGGL((k_yinv_fast<R, TI, TO, N1, N2, C>), dim3((unsigned)nblk), dim3(C * N2), 0, s, in, out, nplanes,
                       lh, ph, tw, ops, wavx, wavy);
    LSB_HIP(hipGetLastError());
    return LSB_OK;
}

template <class R, class TI, class TO, int N1, int N2, int C>
int launch_yinv3(const FieldList<TI>& in, const FieldList<TO>& out, int nplanes, int nsrc, int lh, int ph,
                 const cpx<R>* tw, const double* wavx, const double* wavy, const double* ftab, hipStream_t s) {
    const long nblk = (long)((lh + C - 1) / C) * nplanes * nsrc;
    hipLaunchKernelGGL((k_yinv3_fast<R, TI, TO, N1, N2, C>), dim3((unsigned)nblk), dim3(C * N2), 0, s, in, out,
                       nplanes, lh, ph, tw, wavx, wavy, ftab);
    LSB_HIP(hipGetLastError());
    return LSB_OK;
}

template <class R, class TH, int N1, int N2, int C>
int launch_yrhs(const FieldList<R>& pieces, int nplanes, int lh, const cpx<R>* tw, R scale, const YRhsArgs& a,
                hipStream_t s) {
    const long nblk = (long)((lh + C - 1) / C) * nplanes * 3;
    hipLaunchKernelGGL((k_yfwd_rhs<R, TH, N1, N2, C>), dim3((unsigned)nblk), dim3(C * N2), 0, s, pieces, nplanes, lh,
                       tw, scale, a);
    LSB_HIP(hipGetLastError());
    return LSB_OK;
}

// The lengths (L, N1, N2).  Powers of two: the autotuner chooses the columns of a y tile.
#define LSB_FAST_CASES(X) \
    X(16, 4, 4)           \
    X(32, 8, 4)           \
    X(64, 8, 8)           \
    X(128, 16, 8)         \
    X(256, 16, 16)

// Lengths with a factor 3 or 5 from 24 to 240 whose balanced factors are at most 20 (125,
// 243 and 250, and everything above 256, take the LDS path); ny is even, so the odd ones
// are x lengths only.  y tiles of 16 columns.  Bound by HBM like the powers of two, where
// the LDS Stockham path is bound by its LDS passes and index divisions: 2-D pair of two
// 192 x 65 x 60 FP64 fields 58.8 -> 26.4 us; the 240 x 114 x 120 FP64 sigma step, which
// these lengths also give the fused gradient transform, 2182 -> 985 us.
constexpr int kMixedCols = 16;
#define LSB_MIXED_CASES(X)                                                                                         \
    X(24, 4, 6) X(30, 5, 6) X(36, 6, 6) X(40, 5, 8) X(48, 6, 8) X(50, 5, 10) X(54, 6, 9) X(60, 6, 10) X(72, 8, 9)  \
    X(80, 8, 10) X(90, 9, 10) X(96, 8, 12) X(100, 10, 10) X(108, 9, 12) X(120, 10, 12) X(144, 12, 12)              \
    X(150, 10, 15) X(160, 10, 16) X(162, 9, 18) X(180, 12, 15) X(192, 12, 16) X(200, 10, 20) X(216, 12, 18)        \
    X(240, 15, 16)
#define LSB_MIXED_ODD_CASES(X) \
    X(25, 5, 5) X(27, 3, 9) X(45, 5, 9) X(75, 5, 15) X(81, 9, 9) X(135, 9, 15) X(225, 15, 15)

// instantiations of the mixed lengths, one translation unit per precision and axis
#define LSB_MIXED_X(E, R, N1, N2)                                                                                \
    E template int launch_xfwd<R, R, R, N1, N2>(const FieldList<R>&, const FieldList<R>&, int, int, int, int,    \
                                                const cpx<R>*, const cpx<R>*, hipStream_t);                      \
    E template int launch_xinv<R, R, R, N1, N2>(const FieldList<R>&, const FieldList<R>&, int, int, int, int,    \
                                                const cpx<R>*, const cpx<R>*, hipStream_t);
#define LSB_MIXED_XBLEND(E, N1, N2) \
    E template int launch_xblend<double, N1, N2>(const XBlendArgs&, const cpx<double>*, const cpx<double>*, hipStream_t);
#define LSB_MIXED_YINV3(E, R, N1, N2)                                                                            \
    E template int launch_yinv3<R, double, R, N1, N2, kMixedCols>(const FieldList<double>&, const FieldList<R>&, \
                                                                  int, int, int, int, const cpx<R>*,             \
                                                                  const double*, const double*, const double*,   \
                                                                  hipStream_t);
#define LSB_MIXED_YFWD(E, R, N1, N2)                                                                         \
    E template int launch_yfwd<R, R, R, N1, N2, kMixedCols>(const FieldList<R>&, const FieldList<R>&, int, int, \
                                                            int, const cpx<R>*, R, hipStream_t);
#define LSB_MIXED_YINV(E, R, N1, N2)                                                                          \
    E template int launch_yinv<R, R, R, N1, N2, kMixedCols>(const FieldList<R>&, const FieldList<R>&, int, int,  \
                                                            int, int, const cpx<R>*, const FftOps&,           \
                                                            const double*, const double*, hipStream_t);
#define LSB_MIXED_YRHS(E, R, N1, N2)                                                                         \
    E template int launch_yrhs<R, R, N1, N2, kMixedCols>(const FieldList<R>&, int, int, const cpx<R>*, R,       \
                                                         const YRhsArgs&, hipStream_t);

}  // namespace lsb
