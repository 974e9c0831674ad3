// Dispatch of the register-resident horizontal FFT passes (kernels in fft_fast_kernels.h):
// L in {16, 32, 64, 128, 256} and the lengths with a factor 3 or 5 of LSB_MIXED_CASES.

#include "fft_fast_kernels.h"

namespace lsb {

#define X(LL, A, B)                         \
    LSB_MIXED_X(extern, double, A, B)       \
    LSB_MIXED_X(extern, float, A, B)        \
    LSB_MIXED_YINV3(extern, double, A, B)   \
    LSB_MIXED_YINV3(extern, float, A, B)    \
    LSB_MIXED_YFWD(extern, double, A, B)    \
    LSB_MIXED_YFWD(extern, float, A, B)     \
    LSB_MIXED_YINV(extern, double, A, B)    \
    LSB_MIXED_YRHS(extern, double, A, B)    \
    LSB_MIXED_YRHS(extern, float, A, B)
LSB_MIXED_CASES(X)
#undef X
#define X(LL, A, B)                   \
    LSB_MIXED_X(extern, double, A, B) \
    LSB_MIXED_X(extern, float, A, B)
LSB_MIXED_ODD_CASES(X)
#undef X
#define X(LL, A, B) LSB_MIXED_XBLEND(extern, A, B)
LSB_MIXED_CASES(X)
LSB_MIXED_ODD_CASES(X)
#undef X

bool pow2_fft_len(int L) { return L == 16 || L == 32 || L == 64 || L == 128 || L == 256; }

bool fast_fft_len(int L) {
    switch (L) {
#define X(LL, A, B) case LL:
        LSB_FAST_CASES(X)
        LSB_MIXED_CASES(X)
        LSB_MIXED_ODD_CASES(X)
#undef X
        return true;
        default: return false;
    }
}

template <class R>
int fast_xfwd(const FieldList<R>& in, const FieldList<R>& out, int nrows, int nf, int lh, int istride, int ostride,
              const cpx<R>* tw, const cpx<R>* twr, hipStream_t s) {
    if (nrows <= 0 || nf <= 0) return LSB_OK;
    switch (lh) {
#define X(LL, A, B) \
    case LL: return launch_xfwd<R, R, R, A, B>(in, out, nrows, nf, istride, ostride, tw, twr, s);
        LSB_FAST_CASES(X)
        LSB_MIXED_CASES(X)
        LSB_MIXED_ODD_CASES(X)
#undef X
        default: return LSB_E_ARG;
    }
}

template <class R>
int fast_xinv(const FieldList<R>& in, const FieldList<R>& out, int nrows, int nf, int lh, int istride, int nxpp,
              const cpx<R>* tw, const cpx<R>* twr, hipStream_t s) {
    if (nrows <= 0 || nf <= 0) return LSB_OK;
    switch (lh) {
#define X(LL, A, B) \
    case LL: return launch_xinv<R, R, R, A, B>(in, out, nrows, nf, istride, nxpp, tw, twr, s);
        LSB_FAST_CASES(X)
        LSB_MIXED_CASES(X)
        LSB_MIXED_ODD_CASES(X)
#undef X
        default: return LSB_E_ARG;
    }
}

int fast_xblend(const double* const* in, double* const* out, int ny, int lh, const double* m, const cpx<double>* tw,
                const cpx<double>* twr, hipStream_t s) {
    const XBlendArgs a{{in[0], in[1]}, {out[0], out[1]}, m, 1.0 / (2.0 * lh), ny};
    switch (lh) {
#define X(LL, A, B) \
    case LL: return launch_xblend<double, A, B>(a, tw, twr, s);
        LSB_FAST_CASES(X)
        LSB_MIXED_CASES(X)
        LSB_MIXED_ODD_CASES(X)
#undef X
        default: return LSB_E_ARG;
    }
}

// kx columns per y-pass tile: 128-byte row segments of the arithmetic type
template <class R>
constexpr int ytile_cols() {
    return 128 / (int)sizeof(cpx<R>);
}

// kx columns per tile of a y pass at the power-of-two lengths: 8, 16 or (FP32
// arithmetic) 32, from the context's tuning table; anything else gives the built-in
// default.  Each column is transformed by the same lanes in the same order whatever the
// tile width, so every choice gives the same bits.
template <class R>
static int ycols(int cols, int dflt) {
    if (cols == 8 || cols == 16 || (cols == 32 && sizeof(R) == 4)) return cols;
    return dflt;
}
// one power-of-two length of a y pass with the chosen columns nc
#define LSB_YCASE(LL, CALL8, CALL16, CALL32)                        \
    case LL:                                                        \
        switch (nc) {                                               \
            case 8: return CALL8;                                   \
            case 32:                                                \
                if constexpr (sizeof(R) == 4) return CALL32;        \
                return LSB_E_ARG;                                   \
            default: return CALL16;                                 \
        }

// The forward y pass defaults to 16 kx-columns per tile in both precisions: 256-byte row
// segments in FP64 (measured 0.57 -> 0.62 of the HBM rate against 8-column tiles on the
// 512 x 193 x 256 step, results unchanged), 128-byte ones in FP32.
template <class R>
int fast_yfwd(const FieldList<R>& in, const FieldList<R>& out, int nplanes, int nf, int lh, int ny, const cpx<R>* tw,
              R scale, hipStream_t s, int cols) {
    if (nplanes <= 0 || nf <= 0) return LSB_OK;
    const int nc = ycols<R>(cols, 16);
    switch (ny) {
#define CALL(A, B, C) launch_yfwd<R, R, R, A, B, C>(in, out, nplanes, nf, lh, tw, scale, s)
#define X(LL, A, B) LSB_YCASE(LL, (CALL(A, B, 8)), (CALL(A, B, 16)), (CALL(A, B, 32)))
        LSB_FAST_CASES(X)
#undef X
#define X(LL, A, B) \
    case LL: return CALL(A, B, kMixedCols);
        LSB_MIXED_CASES(X)
#undef X
#undef CALL
        default: return LSB_E_ARG;
    }
}

int fast_yinv(const FieldList<double>& in, const FieldList<double>& out, int nplanes, int nf, int lh, int ny, int ph,
              const cpx<double>* tw, const FftOps& ops, const double* wavx, const double* wavy, hipStream_t s) {
    if (nplanes <= 0 || nf <= 0) return LSB_OK;
    switch (ny) {
#define X(LL, A, B)                                                                                              \
    case LL:                                                                                                     \
        return launch_yinv<double, double, double, A, B, ytile_cols<double>()>(in, out, nplanes, nf, lh, ph, tw, \
                                                                               ops, wavx, wavy, s);
        LSB_FAST_CASES(X)
#undef X
#define X(LL, A, B) \
    case LL:        \
        return launch_yinv<double, double, double, A, B, kMixedCols>(in, out, nplanes, nf, lh, ph, tw, ops, wavx, wavy, s);
        LSB_MIXED_CASES(X)
#undef X
        default: return LSB_E_ARG;
    }
}

template <class R>
int fast_yinv3(const FieldList<double>& in, const FieldList<R>& out, int nplanes, int nsrc, int lh, int ny, int ph,
               const cpx<R>* tw, const double* wavx, const double* wavy, const double* ftab, hipStream_t s, int cols) {
    if (nplanes <= 0 || nsrc <= 0) return LSB_OK;
    const int nc = ycols<R>(cols, ytile_cols<R>());
    switch (ny) {
#define CALL(A, B, C) launch_yinv3<R, double, R, A, B, C>(in, out, nplanes, nsrc, lh, ph, tw, wavx, wavy, ftab, s)
#define X(LL, A, B) LSB_YCASE(LL, (CALL(A, B, 8)), (CALL(A, B, 16)), (CALL(A, B, 32)))
        LSB_FAST_CASES(X)
#undef X
#define X(LL, A, B) \
    case LL: return CALL(A, B, kMixedCols);
        LSB_MIXED_CASES(X)
#undef X
#undef CALL
        default: return LSB_E_ARG;
    }
}

template <class R>
int fast_yfwd_rhs(const FieldList<R>& pieces, int nplanes, int lh, int ny, const cpx<R>* tw, R scale,
                  const YRhsArgs& a, hipStream_t s, int cols) {
    if (nplanes <= 0) return LSB_OK;
    const int nc = ycols<R>(cols, 16);
    switch (ny) {
#define CALL(A, B, C) launch_yrhs<R, R, A, B, C>(pieces, nplanes, lh, tw, scale, a, s)
#define X(LL, A, B) LSB_YCASE(LL, (CALL(A, B, 8)), (CALL(A, B, 16)), (CALL(A, B, 32)))
        LSB_FAST_CASES(X)
#undef X
#define X(LL, A, B) \
    case LL: return CALL(A, B, kMixedCols);
        LSB_MIXED_CASES(X)
#undef X
#undef CALL
        default: return LSB_E_ARG;
    }
}

#define LSB_INST_FAST(R)                                                                                         \
    template int fast_xfwd<R>(const FieldList<R>&, const FieldList<R>&, int, int, int, int, int, const cpx<R>*,  \
                              const cpx<R>*, hipStream_t);                                                       \
    template int fast_xinv<R>(const FieldList<R>&, const FieldList<R>&, int, int, int, int, int, const cpx<R>*,  \
                              const cpx<R>*, hipStream_t);                                                       \
    template int fast_yfwd<R>(const FieldList<R>&, const FieldList<R>&, int, int, int, int, const cpx<R>*, R,    \
                              hipStream_t, int);                                                                 \
    template int fast_yinv3<R>(const FieldList<double>&, const FieldList<R>&, int, int, int, int, int,           \
                               const cpx<R>*, const double*, const double*, const double*, hipStream_t, int);   \
    template int fast_yfwd_rhs<R>(const FieldList<R>&, int, int, int, const cpx<R>*, R, const YRhsArgs&,         \
                                  hipStream_t, int);
LSB_INST_FAST(double)
LSB_INST_FAST(float)

}  // namespace lsb
