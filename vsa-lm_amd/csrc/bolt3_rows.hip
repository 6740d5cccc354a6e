// C entry of the few-row linear layers (bolt3_rows.h): the MLP of a one-token decode step.
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
