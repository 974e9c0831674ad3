// The register-resident FFT passes of the lengths with a factor 3 or 5: FP64, y passes.
#include "fft_fast_kernels.h"

namespace lsb {
#define X(LL, A, B) LSB_MIXED_YINV3(, double, A, B) LSB_MIXED_YFWD(, double, A, B) LSB_MIXED_YINV(, double, A, B)
LSB_MIXED_CASES(X)
#undef X
}  // namespace lsb
