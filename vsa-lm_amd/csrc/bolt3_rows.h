// Linear layers on up to 16 rows (one-token decode steps): out[m][n] = epilogue(sum_k x[m][k] W[n][k])
// for row-major bf16 weights W[N][K] (nn.Linear layout).
//
// The product is bound by streaming W once, so what counts is how many bytes of W are in flight and
// that nothing follows the stream.  A workgroup owns 16 weight rows (for the gated form 16 gate and
// 16 up rows) over the whole of K: its wavefronts take a range of the K steps each
// (v_mfma_f32_16x16x32_bf16, W rows as the A operand, x rows as the B columns), all operands loaded
// straight into registers RD steps ahead, and their fp32 partial products are added in LDS, in
// wavefront order.  The sum is then whole, so the bias, SwiGLU or residual and the one rounding
// happen here and no partial products travel through memory.  x is read from L2 by every
// workgroup, 1 KB for every KB of W, which grows with the rows (see ROWS_PROJ).
//
// The decode layer's projections have a form for more rows (rowproj_kernel), and a row's step must
// not depend on the batch it is in: later slot decisions follow every rounding of the layers below.
// The plain and the residual form therefore take that kernel's ranges, 512 columns of K each, in its
// order.  An eighth of K per wavefront instead (10 steps at K = 2560 against 16 in five wavefronts)
// read W a little faster (10.3 against 11.2 us for the 31.7 MB below) but gave other bits.
//
// Qwen3-4B layer, one row, in a captured step: packed input projection (31.7 MB) 11.2 us and o_proj
// (21 MB) with the residual 9.0 us; down (49.8 MB) with the residual 18.0 us against 17.6 for the
// library's product and 4.6 for the sum; gate, up and SwiGLU (99.6 MB) 27.0 us against 34.5 for two
// library products and 4.9 for SwiGLU.
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
// Rows up to which the decode layer's two projections take this kernel: it and rowproj_kernel give the
// same bits, so speed alone draws the line.  Replay of a captured step of four Qwen3-4B-shape layers, us,
// this / rowproj_kernel: 1 row 440 / 448, 2 rows 445 / 450, 4 rows 447 / 451, 7 rows 462 / 462, 8 rows
// 458 / 458, 12 rows 472 / 462, 16 rows 481 / 468.
constexpr int ROWS_PROJ = 4;

// K steps of a wavefront (32 columns each): an eighth of K, but 512 columns at least where the product
// has a form for more rows (rowproj_kernel's chunks, added in the same order: the same bits)
template <int MODE>
__host__ __device__ inline int rows_steps(int K) {
  const int eighth = (K / 32 + RW - 1) / RW;
  return MODE == ROWS_SWIGLU || eighth > 16 ? eighth : 16;
}

// MODE selects the epilogue; RD: K steps loaded ahead
template <int MODE, int RD>
__global__ void __launch_bounds__(64 * RW, 6) rows_kernel(RowsArgs p) {
  constexpr int WT = MODE == ROWS_SWIGLU ? 2 : 1;
  __shared__ __attribute__((aligned(16))) float part[RW][WT][16][16];   // [wave][tile][m][n]
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, kg = lane >> 4;
  const int n0 = blockIdx.x * 16;
  const int steps = p.K >> 5, per = rows_steps<MODE>(p.K), s0 = min(per * wv, steps), n = min(per, steps - s0);
  const int nw = (steps + per - 1) / per;       // wavefronts that hold a partial product
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
      for (int w = 1; w < RW; ++w)
        if (w < nw) {
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
// and res.  K steps loaded ahead: 8 fit the registers of six wavefronts per SIMD with one W tile (two
// rounds for a range of 512 columns; all 16 at once, at three wavefronts per SIMD, took the replays at
// ROWS_PROJ about 3 us longer), 5 with two.
template <int MODE>
static int launch_rows(const RowsArgs& p, hipStream_t st) {
  const int per = rows_steps<MODE>(p.K);
  const dim3 grid(p.N / 16), block(64 * ((p.K / 32 + per - 1) / per));
  hipLaunchKernelGGL((rows_kernel<MODE, MODE == ROWS_SWIGLU ? 5 : 8>), grid, block, 0, st, p);
  return (int)hipGetLastError();
}

}  // namespace b3
