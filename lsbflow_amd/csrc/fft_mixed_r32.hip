// The register-resident FFT passes of the lengths with a factor 3 or 5: FP32, y, fused with the right-hand side passes.
#include "fft_fast_kernels.h"

namespace lsb {
#define X(LL, A, B) LSB_MIXED_YRHS(, float, A, B)
LSB_MIXED_CASES(X)
#undef X
}  // namespace lsb
