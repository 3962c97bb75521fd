// Small f32 products (v_mfma_f32_32x32x2_f32), bound by latency: a workgroup owns
// a 32 x 32 tile of C and its eight waves split K, each loading its operands from
// memory straight into MFMA fragments, so one launch with no workspace does
// what 64 x 64 tiles split over the grid did in two (the partials and their
// reduction). 512^3 11.9 -> 8.5 us.
//
// A 32-deep step: lane l (r = l % 32, h = l / 32) takes row (column) r and K
// values 16 h .. 16 h + 15 of it -- 64 contiguous bytes of a K-contiguous operand,
// or one value of each of 16 K rows, 128 bytes across the lanes -- and MFMA i (of
// 16) multiplies the i-th values of both. The last step of a K that is no
// multiple of 32 is loaded value by value, zeros past K. The waves' sums meet in
// LDS and are added in wave order, always the same. RMS error against f64 at
// 512^3 4.7e-6 -> 2.7e-6 (inputs N(0, 1)), at 8 x 4096 x 4096 (16 splits before)
// 1.92e-5 -> 1.89e-5.
#include "hmx_gemm_common.hpp"

namespace hmx {
namespace {

constexpr int kSmallWaves = 8;

// The 16 values of row `row` (clamped) from K k0 on.
template <int L>
__device__ __forceinline__ void load_frag(const float* p, int64_t ld, int64_t row, int64_t k0, int64_t k,
                                          float (&v)[16]) {
  if (k0 + 16 <= k) {
    if constexpr (L == L_KCONTIG) {
      const float* q = p + row * ld + k0;
#pragma unroll
      for (int i = 0; i < 4; ++i) Elem<float>::unpack(load16(q + 4 * i), &v[4 * i]);
    } else {
      const float* q = p + k0 * ld + row;
#pragma unroll
      for (int i = 0; i < 16; ++i) v[i] = q[i * ld];
    }
  } else {
#pragma unroll
    for (int i = 0; i < 16; ++i)
      v[i] = k0 + i < k ? (L == L_KCONTIG ? p[row * ld + k0 + i] : p[(k0 + i) * ld + row]) : 0.f;
  }
}

template <int LA, int LB>
__global__ __launch_bounds__(kSmallWaves * 64) void gemm_f32_small_kernel(GemmArgs g) {
  __shared__ float red[kSmallWaves * 16 * 64];
  int tm, tn;
  tile_coords(g.tiles_m, g.tiles_n, g.xcds, tm, tn);
  const int64_t m0 = (int64_t)tm * 32, n0 = (int64_t)tn * 32, batch = blockIdx.z;
  const int lane = threadIdx.x & 63, r = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const float* a = (const float*)g.a.p + batch * g.stride_a;
  const float* b = (const float*)g.b.p + batch * g.stride_b;
  const int64_t row = min(m0 + r, g.m - 1), col = min(n0 + r, g.n - 1);
  const int steps = (int)((g.k + 31) / 32);
  const int t0 = wave * steps / kSmallWaves, t1 = (wave + 1) * steps / kSmallWaves;
  // Even and odd K values apart: shorter sums, and no MFMA waits for the one
  // before it.
  f32x16_t acc[2];
#pragma unroll
  for (int e = 0; e < 16; ++e) acc[0][e] = acc[1][e] = 0.f;
  // Two steps of loads in flight.
  float av[2][16], bv[2][16];
  auto fetch = [&](int s, int t) {
    const int64_t k0 = (int64_t)min(t, t1 - 1) * 32 + 16 * h;
    load_frag<LA>(a, g.a.ld, row, k0, g.k, av[s]);
    load_frag<LB>(b, g.b.ld, col, k0, g.k, bv[s]);
  };
  auto multiply = [&](int s) {
#pragma unroll
    for (int i = 0; i < 16; ++i)
      acc[i & 1] = __builtin_amdgcn_mfma_f32_32x32x2f32(av[s][i], bv[s][i], acc[i & 1], 0, 0, 0);
  };
  if (t0 < t1) {
    fetch(0, t0);
    fetch(1, t0 + 1);
    for (int t = t0; t < t1; t += 2) {
      multiply(0);
      fetch(0, t + 2);
      if (t + 1 < t1) multiply(1);
      fetch(1, t + 3);
    }
  }
#pragma unroll
  for (int e = 0; e < 16; ++e) red[(wave * 16 + e) * 64 + lane] = acc[0][e] + acc[1][e];
  __syncthreads();
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int e = wave * 2 + q;
    const int64_t rr = m0 + 8 * (e >> 2) + 4 * h + (e & 3), cc = n0 + r;
    float s = red[e * 64 + lane];
#pragma unroll
    for (int w = 1; w < kSmallWaves; ++w) s += red[(w * 16 + e) * 64 + lane];
    if (rr >= g.m || cc >= g.n) continue;
    float bias, scale, shift;
    column_vectors(g, cc, true, bias, scale, shift);
    const float v = apply_activation(g.act, (s + bias) * scale + shift, g.act_arg);
    const int64_t off = batch * g.stride_c + rr * g.ldc + cc;
    if (g.c_dtype == HMX_DTYPE_BF16) ((uint16_t*)g.c)[off] = (uint16_t)f32_to_bf16_bits(v);
    else ((float*)g.c)[off] = v;
  }
}

}  // namespace

void launch_gemm_f32_small(const GemmArgs& g, int la, int lb, int64_t batch, hipStream_t s) {
  GemmArgs v = g;
  v.tiles_m = (int)ceil_div(g.m, 32);
  v.tiles_n = (int)ceil_div(g.n, 32);
  const dim3 grid((unsigned)(v.tiles_m * v.tiles_n), 1, (unsigned)batch);
  constexpr int T = kSmallWaves * 64;
  if (la == L_KCONTIG) {
    if (lb == L_KCONTIG) launch(gemm_f32_small_kernel<L_KCONTIG, L_KCONTIG>, grid, T, s, v);
    else launch(gemm_f32_small_kernel<L_KCONTIG, L_RCONTIG>, grid, T, s, v);
  } else {
    if (lb == L_KCONTIG) launch(gemm_f32_small_kernel<L_RCONTIG, L_KCONTIG>, grid, T, s, v);
    else launch(gemm_f32_small_kernel<L_RCONTIG, L_RCONTIG>, grid, T, s, v);
  }
}

}  // namespace hmx
