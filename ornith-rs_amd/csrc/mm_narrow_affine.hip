// The few-row GEMM (mm_narrow.h) over 4-bit (group 32) and 8-bit (group 64) affine weights.
#include "mm_narrow_host.h"

namespace nmm {
constexpr int affine_waves(int, int rows) { return rows == 16 ? 4 : rows == 32 ? 3 : 2; }
// columns owned by wavefronts, 64-row tiles of a plain product
template <int KIND>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(KIND == kA4 ? 4 : 2))) void affine_tall_kernel(Args a) {
  body<true, 2, kTall, 64, 4, KIND>(a);
}
NMM_KERNELS(affine, true, kA4, -1, affine_waves, 8u, affine_tall_kernel<kA4>, affine_tall_kernel<-1>)
}
