// The 16x16x32 bf16 GEMM kernel's instantiations for B [N, K].
#include "hmx_gemm_mi16_launch.hpp"

namespace hmx {

bool launch_mi16_nt(const GemmArgs& g, Mi16Tile t, dim3 grid, hipStream_t s) {
  return g.c_dtype == HMX_DTYPE_BF16 ? mi16_plain<L_KCONTIG, true>(g, t, grid, s)
                                     : mi16_plain<L_KCONTIG, false>(g, t, grid, s);
}

bool launch_mi16_rounds_nt(const GemmArgs& head, const GemmArgs& rest, unsigned head_blocks, unsigned rest_blocks,
                           hipStream_t s) {
  return head.c_dtype == HMX_DTYPE_BF16 ? mi16_rounds<L_KCONTIG, true>(head, rest, head_blocks, rest_blocks, s)
                                        : mi16_rounds<L_KCONTIG, false>(head, rest, head_blocks, rest_blocks, s);
}

}  // namespace hmx
