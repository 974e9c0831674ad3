// The blended ceiling's x lines at the lengths with a factor 3 or 5 (FP64).
#include "fft_fast_kernels.h"

namespace lsb {
#define X(LL, A, B) LSB_MIXED_XBLEND(, A, B)
LSB_MIXED_CASES(X)
LSB_MIXED_ODD_CASES(X)
#undef X
}  // namespace lsb
