// The 16x16x32 bf16 GEMM kernel's instantiations for B in VNNI panels.
#include "hmx_gemm_mi16_launch.hpp"

namespace hmx {

bool launch_mi16_vnni(const GemmArgs& g, Mi16Tile t, dim3 grid, hipStream_t s) {
  return g.c_dtype == HMX_DTYPE_BF16 ? mi16_packed<L_VNNI_PANELS, true>(g, t, grid, s)
                                     : mi16_packed<L_VNNI_PANELS, false>(g, t, grid, s);
}

}  // namespace hmx
