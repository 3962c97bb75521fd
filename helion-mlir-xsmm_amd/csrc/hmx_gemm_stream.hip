// bf16 products of at most 32 rows of row-major A against a packed B (decode
// through a weight packed once): bound by reading B once. The tile kernels run
// them as 128- or 256-row tiles, most of them padding: 16 x 11008 x 4096 on VNNI
// panels took 153 us on guarded 256 x 256 tiles; this kernel takes 17.6 us (5.2
// TB/s; on 32 x 32 blocks 112 -> 24 us). With more rows A's loads, which every
// workgroup repeats, weigh as much as B's (64 rows 29 us, 100 rows 40), and 128 x
// 128 tiles of the direct-to-LDS kernel take over.
//
// A workgroup owns all rows and 64 columns; its eight waves split K and each
// streams its range of B from memory straight into MFMA operands (v_mfma_f32_16x16x32_bf16,
// B first), no LDS and no barrier on the way. Lane l (c = l % 16, g = l / 16) of a
// 32-deep step takes columns 4 c .. 4 c + 3 and K values 8 g .. 8 g + 7:
//  * VNNI panels (and blocked VNNI, panels of 32): four 16-byte loads, K pairs
//    4 g + i of the four columns; word j of the four is the operand of
//    fragment j as it stands.
//  * K-major panels and 32 x 32 blocks: eight 8-byte loads, one K row of the
//    four columns each, paired along K with v_perm_b32.
// Either way 16 lanes read 128 or 256 contiguous bytes, and fragment j holds
// columns 4 i + j, so a lane's accumulators of the four fragments are 16
// adjacent columns of one row of C. A's rows come from L2, 16 bytes a lane.
// D steps of loads are in flight per wave. The waves' sums meet in LDS in a
// fixed order: w + (w + 4), then those of waves 0 + 2 and 1 + 3, then the two.
#include "hmx_gemm_common.hpp"

namespace hmx {
namespace {

constexpr int kStreamWaves = 8, kStreamCols = 64;

template <int MB, bool VN, int D>
__global__ __launch_bounds__(kStreamWaves * 64, 1) void gemm_bf16_stream_kernel(GemmArgs g) {
  typedef float f32x4_t __attribute__((ext_vector_type(4)));
  constexpr int ROWS = 16 * MB, PITCH = kStreamCols + 4;  // f32 per LDS row
  __shared__ __attribute__((aligned(16))) float red[4 * ROWS * PITCH];
  const int lane = threadIdx.x & 63, c = lane & 15, grp = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t n0 = (int64_t)blockIdx.x * kStreamCols;
  // The lane's four columns (past B's last ones: those, never stored).
  const int64_t col = min(n0 + 4 * c, g.b.rows - 4);
  const int64_t P = g.b.panel;
  const uint32_t b_lane = (uint32_t)((col / P) * g.b.kpad * P + (col % P) * (VN ? 2 : 1) + 8 * grp * P);
  const uint16_t* b = (const uint16_t*)g.b.p;
  const uint16_t* a = (const uint16_t*)g.a.p;
  uint32_t a_lane[MB];
#pragma unroll
  for (int i = 0; i < MB; ++i) a_lane[i] = (uint32_t)(min<int64_t>(16 * i + c, g.m - 1) * g.a.ld + 8 * grp);

  const int steps = (int)(g.k / 32);
  const int t0 = wave * steps / kStreamWaves, t1 = (wave + 1) * steps / kStreamWaves;

  struct Step {
    uint4 b4[VN ? 4 : 1];
    uint2 b2[VN ? 1 : 8];
    uint4 a[MB];
  } buf[D];
  auto fetch = [&](Step& s, int t) {
    const uint16_t* bt = b + (int64_t)t * 32 * P;
    if constexpr (VN) {
#pragma unroll
      for (int i = 0; i < 4; ++i) s.b4[i] = load16(bt + b_lane + i * 2 * (uint32_t)P);
    } else {
      typedef uint32_t u32x2_any_t __attribute__((ext_vector_type(2), aligned(2)));
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const u32x2_any_t v = *reinterpret_cast<const u32x2_any_t*>(bt + b_lane + i * (uint32_t)P);
        s.b2[i] = make_uint2(v[0], v[1]);
      }
    }
    const uint16_t* at = a + t * 32;
#pragma unroll
    for (int i = 0; i < MB; ++i) s.a[i] = load16(at + a_lane[i]);
  };
  f32x4_t acc[MB][4];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  auto multiply = [&](const Step& s) {
    bf16x8_t f[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      uint4 v;
      if constexpr (VN) {
        v = make_uint4(dw(s.b4[0], j), dw(s.b4[1], j), dw(s.b4[2], j), dw(s.b4[3], j));
      } else {
        uint32_t q[4];
#pragma unroll
        for (int p = 0; p < 4; ++p) {
          const uint32_t lo = j < 2 ? s.b2[2 * p].x : s.b2[2 * p].y, hi = j < 2 ? s.b2[2 * p + 1].x : s.b2[2 * p + 1].y;
          q[p] = (j & 1) ? hi_pair(lo, hi) : lo_pair(lo, hi);
        }
        v = make_uint4(q[0], q[1], q[2], q[3]);
      }
      f[j] = __builtin_bit_cast(bf16x8_t, v);
    }
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f[j], __builtin_bit_cast(bf16x8_t, s.a[i]), acc[i][j], 0, 0, 0);
  };
  if (t0 < t1) {
#pragma unroll
    for (int d = 0; d < D; ++d) fetch(buf[d], min(t0 + d, t1 - 1));
    // Past the end the last step is fetched again, in bounds, and not used.
    for (int t = t0; t < t1; t += D) {
#pragma unroll
      for (int d = 0; d < D; ++d) {
        if (t + d < t1) multiply(buf[d]);
        fetch(buf[d], min(t + d + D, t1 - 1));
      }
    }
  }

  // Lane l holds row c of each block of 16, columns 16 grp + 4 e + j.
  auto put = [&](float* r) {
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        *(f32x4_t*)(r + (16 * i + c) * PITCH + 16 * grp + 4 * e) =
            f32x4_t{acc[i][0][e], acc[i][1][e], acc[i][2][e], acc[i][3][e]};
  };
  auto add = [&](const float* r) {
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const f32x4_t v = *(const f32x4_t*)(r + (16 * i + c) * PITCH + 16 * grp + 4 * e);
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j][e] += v[j];
      }
  };
  if (wave >= 4) put(red + (wave - 4) * ROWS * PITCH);
  __syncthreads();
  if (wave < 4) add(red + wave * ROWS * PITCH);
  __syncthreads();
  if (wave == 2 || wave == 3) put(red + (wave - 2) * ROWS * PITCH);
  __syncthreads();
  if (wave < 2) {
    add(red + wave * ROWS * PITCH);
    put(red + wave * ROWS * PITCH);
  }
  __syncthreads();
  // Every thread finishes runs of eight columns: bias, scale, shift, the
  // activation, one rounding.
  for (int u = threadIdx.x; u < ROWS * (kStreamCols / 8); u += kStreamWaves * 64) {
    const int r = u / (kStreamCols / 8), c8 = (u % (kStreamCols / 8)) * 8;
    const int64_t at = n0 + c8;
    if (r >= g.m || at >= g.n) continue;
    const float* s0 = red + r * PITCH + c8;
    float v[8];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      float cb[4], cs[4], ch[4];
      column_vectors4(g, at + 4 * h, g.n, cb, cs, ch);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float sum = s0[4 * h + e] + s0[ROWS * PITCH + 4 * h + e];
        v[4 * h + e] = apply_activation(g.act, (sum + cb[e]) * cs[e] + ch[e], g.act_arg);
      }
    }
    if (g.c_dtype == HMX_DTYPE_BF16) {
      uint16_t* p = (uint16_t*)g.c + (int64_t)r * g.ldc + at;
      if (at + 8 <= g.n) {
        store16_stream(p, Elem<uint16_t>::pack(v));
      } else {
        for (int e = 0; e < 8 && at + e < g.n; ++e) p[e] = (uint16_t)f32_to_bf16_bits(v[e]);
      }
    } else {
      float* p = (float*)g.c + (int64_t)r * g.ldc + at;
      if (at + 8 <= g.n) {
        store16_stream(p, Elem<float>::pack(v));
        store16_stream(p + 4, Elem<float>::pack(v + 4));
      } else {
        for (int e = 0; e < 8 && at + e < g.n; ++e) p[e] = v[e];
      }
    }
  }
}

template <bool VN>
void launch_stream(const GemmArgs& g, hipStream_t s) {
  const dim3 grid((unsigned)ceil_div(g.n, kStreamCols));
  constexpr int T = kStreamWaves * 64;
  if (g.m <= 16) launch(gemm_bf16_stream_kernel<1, VN, 4>, grid, T, s, g);
  else launch(gemm_bf16_stream_kernel<2, VN, 4>, grid, T, s, g);
}

}  // namespace

void launch_gemm_bf16_stream(const GemmArgs& g, int lb, hipStream_t s) {
  GemmArgs v = g;
  if (lb == L_BLOCKED || lb == L_BLOCKED_VNNI) v.b.panel = 32;
  if (lb == L_VNNI_PANELS || lb == L_BLOCKED_VNNI) launch_stream<true>(v, s);
  else launch_stream<false>(v, s);
}

}  // namespace hmx
