// The 16x16x32 bf16 GEMM kernel's instantiations for packed B (VNNI panels,
// K-major panels, 32 x 32 blocks), and the choice among the units.
#include "hmx_gemm_mi16_launch.hpp"

#include <cstdlib>

namespace hmx {

// The 16x16x32 MFMA kernel unless the environment sets HMX_GEMM_MFMA=32 (the
// 32x32x16 kernel, for comparison); it does not stagger K walks.
bool gemm_mi16_ok(const GemmArgs& g) {
  static const bool on = [] {
    const char* e = getenv("HMX_GEMM_MFMA");
    return !(e && e[0] == '3');
  }();
  return on && !g.k_stagger;
}

bool launch_mi16(const GemmArgs& g, int lb, Mi16Tile t, dim3 grid, hipStream_t s) {
  if (!gemm_mi16_ok(g)) return false;
  const bool bf16 = g.c_dtype == HMX_DTYPE_BF16;
  switch (lb) {
    case L_KCONTIG: return launch_mi16_nt(g, t, grid, s);
    case L_RCONTIG: return launch_mi16_nn(g, t, grid, s);
    case L_VNNI_PANELS: return bf16 ? mi16_whole<L_VNNI_PANELS, true>(g, grid, s) : mi16_whole<L_VNNI_PANELS, false>(g, grid, s);
    case L_PANELS: return bf16 ? mi16_whole<L_PANELS, true>(g, grid, s) : mi16_whole<L_PANELS, false>(g, grid, s);
    case L_BLOCKED: return bf16 ? mi16_whole<L_BLOCKED, true>(g, grid, s) : mi16_whole<L_BLOCKED, false>(g, grid, s);
  }
  return false;
}

bool launch_mi16_rounds(const GemmArgs& head, const GemmArgs& rest, int lb, unsigned head_blocks,
                        unsigned rest_blocks, hipStream_t s) {
  if (!gemm_mi16_ok(head) || !gemm_mi16_ok(rest)) return false;
  return lb == L_KCONTIG ? launch_mi16_rounds_nt(head, rest, head_blocks, rest_blocks, s)
                         : launch_mi16_rounds_nn(head, rest, head_blocks, rest_blocks, s);
}

}  // namespace hmx
