// The few-row GEMM (mm_narrow.h) over 4-bit (group 32) and 8-bit (group 64) affine weights.
#include "mm_narrow_host.h"

namespace nmm {
NMM_KERNELS(affine, true, 3, 3, 8u)
}
