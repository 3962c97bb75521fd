// Launches of the 16x16x32 bf16 GEMM kernel (body in hmx_gemm_mi16.hpp), one
// translation unit per B layout (hmx_gemm_mi16_nt.hip, _nn.hip, _packed.hip) so
// that the instantiations compile in parallel.
#pragma once

#include <algorithm>

#include "hmx_gemm_mi16.hpp"

namespace hmx {
namespace {

template <int LB, int ACT, bool BF16, bool RAGGED = false, int BM = 256, int BN = 256, int NW = 8, int S = 2>
__global__ __launch_bounds__(NW * 64, 1) void gemm_bf16_mi16_kernel(GemmArgs g) {
  gemm_bf16_mi16_body<LB, ACT, BF16, RAGGED, BM, BN, NW, S>(g);
}

// A product of several rounds of 256 x 256 tiles and a tail of 256 x 128
// tiles in one launch: workgroup b < head_blocks runs head's tile b, the
// others rest's tile b - head_blocks (head_blocks a multiple of the XCD
// count, so the XCD-aware tile order holds for both). Both are multi-round,
// so C is streamed.
template <int LB, int ACT, bool BF16>
__global__ __launch_bounds__(512, 1) void gemm_bf16_mi16_rounds_kernel(GemmArgs head, GemmArgs rest,
                                                                        int head_blocks) {
  constexpr int kHead = mi16_lds_bytes<ACT, 256, 256, 8, 2>(), kTail = mi16_lds_bytes<ACT, 256, 128, 8, 2>();
  __shared__ __attribute__((aligned(1024))) uint8_t lds[kHead > kTail ? kHead : kTail];
  const int b = (int)blockIdx.x;
  if (b < head_blocks)
    gemm_bf16_mi16_body<LB, ACT, BF16, false, 256, 256, 8, 2>(head, lds, b, false);
  else
    gemm_bf16_mi16_body<LB, ACT, BF16, false, 256, 128, 8, 2>(rest, lds, b - head_blocks, false);
}

// g on tile t with its named register epilogue, or with any other one compiled
// in at run time; false (nothing launched) if that could not be.
template <int LB, bool BF16, bool RAGGED, int BM, int BN, int NW, int S>
bool mi16_tile(const GemmArgs& g, dim3 grid, hipStream_t s) {
  switch (g.act) {
    case HMX_EPI_IDENTITY:
      launch(gemm_bf16_mi16_kernel<LB, ACT_ID, BF16, RAGGED, BM, BN, NW, S>, grid, NW * 64, s, g);
      return true;
    case HMX_EPI_RELU:
      launch(gemm_bf16_mi16_kernel<LB, ACT_RELU, BF16, RAGGED, BM, BN, NW, S>, grid, NW * 64, s, g);
      return true;
    case HMX_EPI_SILU:
      launch(gemm_bf16_mi16_kernel<LB, ACT_SILU, BF16, RAGGED, BM, BN, NW, S>, grid, NW * 64, s, g);
      return true;
    default:
      return launch_mi16_jit(g, LB, BF16, RAGGED, BM, BN, NW, S, grid, s) == HMX_OK;
  }
}

// Whole 256 x 256 tiles: an epilogue that could not be compiled runs staged.
template <int LB, bool BF16>
bool mi16_whole(const GemmArgs& g, dim3 grid, hipStream_t s) {
  if (mi16_tile<LB, BF16, false, 256, 256, 8, 2>(g, grid, s)) return true;
  if (g.act == HMX_EPI_PROGRAM) launch(gemm_bf16_mi16_kernel<LB, ACT_PROG, BF16>, grid, 512, s, g);
  else launch(gemm_bf16_mi16_kernel<LB, ACT_ANY, BF16>, grid, 512, s, g);
  return true;
}

template <int LB, bool BF16>
bool mi16_plain(const GemmArgs& g, Mi16Tile t, dim3 grid, hipStream_t s) {
  if (t.bm == 256 && t.bn == 256)
    return t.ragged ? mi16_tile<LB, BF16, true, 256, 256, 8, 2>(g, grid, s) : mi16_whole<LB, BF16>(g, grid, s);
  if (t.bm == 256) return mi16_tile<LB, BF16, false, 256, 128, 8, 2>(g, grid, s);
  if (t.stages == 4)
    return t.ragged ? mi16_tile<LB, BF16, true, 128, 128, 4, 4>(g, grid, s)
                    : mi16_tile<LB, BF16, false, 128, 128, 4, 4>(g, grid, s);
  return t.ragged ? mi16_tile<LB, BF16, true, 128, 128, 4, 2>(g, grid, s)
                  : mi16_tile<LB, BF16, false, 128, 128, 4, 2>(g, grid, s);
}

// Packed B: whole 256 x 256 tiles, or (ragged) M of any size.
template <int LB, bool BF16>
bool mi16_packed(const GemmArgs& g, Mi16Tile t, dim3 grid, hipStream_t s) {
  if (t.bm == 256) return t.ragged ? mi16_tile<LB, BF16, true, 256, 256, 8, 2>(g, grid, s) : mi16_whole<LB, BF16>(g, grid, s);
  return t.stages == 4 ? mi16_tile<LB, BF16, true, 128, 128, 4, 4>(g, grid, s)
                       : mi16_tile<LB, BF16, true, 128, 128, 4, 2>(g, grid, s);
}

template <int LB, bool BF16>
bool mi16_rounds(const GemmArgs& head, const GemmArgs& rest, unsigned head_blocks, unsigned rest_blocks,
                 hipStream_t s) {
  const dim3 grid(head_blocks + rest_blocks);
  const int hb = (int)head_blocks;
  switch (head.act) {
    case HMX_EPI_IDENTITY: launch(gemm_bf16_mi16_rounds_kernel<LB, ACT_ID, BF16>, grid, 512, s, head, rest, hb); return true;
    case HMX_EPI_RELU: launch(gemm_bf16_mi16_rounds_kernel<LB, ACT_RELU, BF16>, grid, 512, s, head, rest, hb); return true;
    case HMX_EPI_SILU: launch(gemm_bf16_mi16_rounds_kernel<LB, ACT_SILU, BF16>, grid, 512, s, head, rest, hb); return true;
    default: return launch_mi16_rounds_jit(head, rest, LB, BF16, head_blocks, rest_blocks, s) == HMX_OK;
  }
}

}  // namespace
}  // namespace hmx
