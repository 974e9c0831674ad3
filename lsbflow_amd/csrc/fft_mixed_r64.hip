// The register-resident FFT passes of the lengths with a factor 3 or 5: FP64, y, fused with the right-hand side passes.
#include "fft_fast_kernels.h"

namespace lsb {
#define X(LL, A, B) LSB_MIXED_YRHS(, double, A, B)
LSB_MIXED_CASES(X)
#undef X
}  // namespace lsb
