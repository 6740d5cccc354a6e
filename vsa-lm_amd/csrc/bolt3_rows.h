// Linear layers on up to 16 rows (one-token decode steps): out[m][n] = epilogue(sum_k x[m][k] W[n][k])
// for row-major bf16 weights W[N][K] (nn.Linear layout).
//
// The product is bound by streaming W once, so what counts is how many bytes of W are in flight and
// that nothing follows the stream.  A workgroup owns 16 weight rows (for the gated form 16 gate and
// 16 up rows) over the whole of K: its eight wavefronts take an eighth of the K steps each
// (v_mfma_f32_16x16x32_bf16, W rows as the A operand, x rows as the B columns), all operands loaded
// straight into registers RD steps ahead, and their fp32 partial products are added in LDS, in
// wavefront order.  The sum is then whole, so the bias, SwiGLU or residual and the one rounding
// happen here and no partial products travel through memory.  x is read from L2 by every
// workgroup, 1 KB for every KB of W; at 17 rows and more that traffic is the larger one (64 rows:
// 36 us for the input projection below, against 11.1 for rowproj_kernel, which shares x in LDS).
//
// Qwen3-4B layer, one row: packed input projection (31.7 MB) 10.3 us (9.1 by rowproj_kernel, but the
// attention then adds its partial products: 14.6 against 19.1 us), o_proj and down (21 and 49.8 MB)
// 13.3 us on average with the residual added, against 12.9 with two more kernels of 4.2 us each; gate,
// up and SwiGLU (99.6 MB) 27.5 us against 35.2 for two library products and two elementwise kernels
// of 4.4.
#pragma once
#include "bolt3_common.h"

namespace b3 {

enum : int { ROWS_PLAIN = 0, ROWS_SWIGLU = 1, ROWS_RESIDUAL = 2 };

struct RowsArgs {
  const uint16_t* x; int64_t x_rs;     // [M][K] rows
  const uint16_t* w;                   // [N][K]
  const uint16_t* w2;                  // ROWS_SWIGLU: the up projection [N][K] (w is the gate)
  const uint16_t* bias;                // [N] or null
  const uint16_t* res; int64_t res_rs; // ROWS_RESIDUAL: [M][N] added to the rounded product
  uint16_t* out; int64_t out_rs;
  int M, N, K;
};

constexpr int RW = 8;   // wavefronts per workgroup

constexpr int ROWS_MAX = 16;   // rows of x

// MODE selects the epilogue; RD: K steps loaded ahead
template <int MODE, int RD>
__global__ void __launch_bounds__(64 * RW, 6) rows_kernel(RowsArgs p) {
  constexpr int WT = MODE == ROWS_SWIGLU ? 2 : 1;
  __shared__ __attribute__((aligned(16))) float part[RW][WT][16][16];   // [wave][tile][m][n]
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, kg = lane >> 4;
  const int n0 = blockIdx.x * 16;
  const int steps = p.K >> 5, s0 = steps * wv / RW, n = steps * (wv + 1) / RW - s0;
  const uint16_t* wr[WT];
  wr[0] = p.w + (long long)(n0 + r) * p.K + 32 * s0 + 8 * kg;
  if constexpr (WT == 2) wr[1] = p.w2 + (long long)(n0 + r) * p.K + 32 * s0 + 8 * kg;
  // rows past M repeat the last one; their columns are never stored
  const uint16_t* xr = p.x + (long long)min(r, p.M - 1) * p.x_rs + 32 * s0 + 8 * kg;
  u16x8 wa[RD][WT], xa[RD];
  auto load = [&](int d, int s) {
    const int o = 32 * min(s, n - 1);   // steps past the range re-read its last one and are not multiplied
#pragma unroll
    for (int t = 0; t < WT; ++t) wa[d][t] = *reinterpret_cast<const u16x8*>(wr[t] + o);
    xa[d] = *reinterpret_cast<const u16x8*>(xr + o);
  };
  f32x4 acc[WT];
#pragma unroll
  for (int i = 0; i < WT; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  if (n > 0) {
#pragma unroll
    for (int d = 0; d < RD; ++d) load(d, d);
    for (int s = 0; s < n; s += RD) {
#pragma unroll
      for (int d = 0; d < RD; ++d) {
        if (s + d < n)
#pragma unroll
          for (int i = 0; i < WT; ++i) mma16_bf16(acc[i], wa[d][i], xa[d]);
        if (s + RD < n) load(d, s + RD + d);
      }
    }
  }
  // D: column m = r, rows n = 4 kg + i
#pragma unroll
  for (int i = 0; i < WT; ++i) *reinterpret_cast<f32x4*>(&part[wv][i][r][4 * kg]) = acc[i];
  __syncthreads();
  // four columns of one row per thread
  const int m = tid >> 2, c = 4 * (tid & 3), col = n0 + c;
  if (m < p.M) {
    f32x4 v[WT];
#pragma unroll
    for (int i = 0; i < WT; ++i) {
      v[i] = *reinterpret_cast<const f32x4*>(&part[0][i][m][c]);
#pragma unroll
      for (int w = 1; w < RW; ++w) {
        const f32x4 q = *reinterpret_cast<const f32x4*>(&part[w][i][m][c]);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[i][e] += q[e];
      }
    }
    u16x4 o;
    u16x4 rs = {0, 0, 0, 0};
    if constexpr (MODE == ROWS_RESIDUAL) rs = *reinterpret_cast<const u16x4*>(p.res + (long long)m * p.res_rs + col);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float y = round_bf(p.bias ? v[0][e] + bf2f(p.bias[col + e]) : v[0][e]);
      if constexpr (MODE == ROWS_SWIGLU) {   // each of silu's result, the up value and the product rounded
        const float g = round_bf(y / (1.0f + expf(-y)));
        o[e] = f2bf(mul_rn(g, round_bf(v[WT - 1][e])));
      } else if constexpr (MODE == ROWS_RESIDUAL) {
        o[e] = f2bf(add_rn(y, bf2f(rs[e])));
      } else {
        o[e] = f2bf(y);
      }
    }
    *reinterpret_cast<u16x4*>(p.out + (long long)m * p.out_rs + col) = o;
  }
}

// M <= ROWS_MAX, K % 32 == 0, N % 16 == 0, 16-byte aligned rows of x and W, 8-byte aligned rows of out
// and res.  K steps loaded ahead: 8 fit the registers of six wavefronts per SIMD with one W tile, 5
// with two; and 5 where a wavefront has ten steps or fewer (K <= 2560), since the second round of 8
// would be mostly loads that are not multiplied.
template <int MODE>
static int launch_rows(const RowsArgs& p, hipStream_t st) {
  const dim3 grid(p.N / 16), block(64 * RW);
  if (MODE == ROWS_SWIGLU || p.K <= 10 * 32 * RW) hipLaunchKernelGGL((rows_kernel<MODE, 5>), grid, block, 0, st, p);
  else hipLaunchKernelGGL((rows_kernel<MODE, MODE == ROWS_SWIGLU ? 5 : 8>), grid, block, 0, st, p);
  return (int)hipGetLastError();
}

}  // namespace b3
