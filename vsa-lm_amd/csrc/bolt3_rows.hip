// The MLP around the library's products: C entry of the few-row linear layers (bolt3_rows.h) of a
// one-token decode step, and the SwiGLU of more rows.
#include "bolt3_rows.h"
#include "bolt3_amd.h"

extern "C" int bolt3_rows_linear(const b3_rows_linear_args* a, void* stream) {
  if (!a || a->M < 0 || a->N <= 0 || a->K <= 0 || !a->x || !a->w || !a->out) return B3_ERR_ARG;
  if (a->mode < 0 || a->mode > 2 || (a->mode == B3_ROWS_SWIGLU && !a->w2) || (a->mode == B3_ROWS_RESIDUAL && !a->res))
    return B3_ERR_ARG;
  if (a->N % 16 || a->K % 32 || a->M > b3::ROWS_MAX) return B3_ERR_UNSUPPORTED;
  const auto odd = [](const void* p, uintptr_t n) { return reinterpret_cast<uintptr_t>(p) % n != 0; };
  if (a->x_row_stride < a->K || a->x_row_stride % 8 || a->out_row_stride < a->N || a->out_row_stride % 4 ||
      odd(a->x, 16) || odd(a->w, 16) || odd(a->w2, 16) || odd(a->out, 8) ||
      (a->mode == B3_ROWS_RESIDUAL && (a->res_row_stride < a->N || a->res_row_stride % 4 || odd(a->res, 8))))
    return B3_ERR_ARG;
  if (a->M == 0) return B3_OK;
  using u16 = const uint16_t*;
  const b3::RowsArgs p{static_cast<u16>(a->x), a->x_row_stride, static_cast<u16>(a->w), static_cast<u16>(a->w2),
                       static_cast<u16>(a->bias), static_cast<u16>(a->res), a->res_row_stride,
                       static_cast<uint16_t*>(a->out), a->out_row_stride, a->M, a->N, a->K};
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  if (a->mode == B3_ROWS_SWIGLU) return b3::launch_rows<b3::ROWS_SWIGLU>(p, st);
  if (a->mode == B3_ROWS_RESIDUAL) return b3::launch_rows<b3::ROWS_RESIDUAL>(p, st);
  return b3::launch_rows<b3::ROWS_PLAIN>(p, st);
}

namespace b3 {
// out = round(round(silu(gate)) * up), elementwise: the SwiGLU between the library's products of a
// prompt or a large batch.  Bound by its three passes over memory: 37 us for 4000 x 9728 (233 MB)
// against 68 us for torch's two kernels, which write and read silu(gate) between.
__global__ void __launch_bounds__(256) swiglu_kernel(const uint16_t* g, const uint16_t* u, uint16_t* out, long long n8) {
  for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < n8; i += (long long)gridDim.x * 256) {
    const u16x8 a = *reinterpret_cast<const u16x8*>(g + 8 * i), b = *reinterpret_cast<const u16x8*>(u + 8 * i);
    u16x8 o;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float x = bf2f(a[e]);
      o[e] = f2bf(mul_rn(round_bf(x / (1.0f + expf(-x))), bf2f(b[e])));
    }
    *reinterpret_cast<u16x8*>(out + 8 * i) = o;
  }
}
}  // namespace b3

extern "C" int bolt3_swiglu(const b3_swiglu_args* a, void* stream) {
  if (!a || a->n < 0 || (a->n > 0 && (!a->gate || !a->up || !a->out))) return B3_ERR_ARG;
  const auto odd = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 != 0; };
  if (a->n % 8 || odd(a->gate) || odd(a->up) || odd(a->out)) return B3_ERR_ARG;
  if (a->n == 0) return B3_OK;
  const long long n8 = a->n / 8, wg = (n8 + 255) / 256;
  hipLaunchKernelGGL(b3::swiglu_kernel, dim3((unsigned)(wg < (1 << 20) ? wg : (1 << 20))), dim3(256), 0,
                     reinterpret_cast<hipStream_t>(stream), static_cast<const uint16_t*>(a->gate),
                     static_cast<const uint16_t*>(a->up), static_cast<uint16_t*>(a->out), n8);
  return (int)hipGetLastError();
}
