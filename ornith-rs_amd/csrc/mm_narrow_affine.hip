// The few-row GEMM (mm_narrow.h) over 4-bit (group 32) and 8-bit (group 64) affine weights.
#include "mm_narrow_host.h"

namespace nmm {
constexpr int affine_waves(int, int rows) { return rows == 16 ? 4 : rows == 32 ? 3 : 2; }
NMM_KERNELS(affine, true, kA4, -1, affine_waves, 8u)
}
