// The register-resident FFT passes of the lengths with a factor 3 or 5: FP32, y passes.
#include "fft_fast_kernels.h"

namespace lsb {
#define X(LL, A, B) LSB_MIXED_YINV3(, float, A, B) LSB_MIXED_YFWD(, float, A, B)
LSB_MIXED_CASES(X)
#undef X
}  // namespace lsb
