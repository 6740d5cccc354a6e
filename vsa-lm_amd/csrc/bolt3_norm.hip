// RMSNorm of the hybrid stack around the Bolt-3 layers (block norms, final norm, q/k norms of
// the softmax-anchor layers): y = (x * rsqrt(mean(x^2) + eps)) * w, fp32 statistic, each product
// rounded in fp32, the result cast to the storage dtype once (vsa_lm/surgery.py:48-52).  One
// wavefront per row, 8 elements per 16-byte load; four rows per 256-thread workgroup.
#include "bolt3_common.h"
#include "bolt3_amd.h"

namespace b3 {

template <typename T, typename W>
__global__ void __launch_bounds__(256) rms_norm_kernel(b3_rms_norm_args a) {
  const int lane = threadIdx.x & 63;
  const long long row = (long long)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= a.rows) return;   // whole wavefronts; no barrier below
  const T* x = reinterpret_cast<const T*>(a.x) + row * a.x_row_stride;
  T* y = reinterpret_cast<T*>(a.y) + row * a.y_row_stride;
  const W* w = reinterpret_cast<const W*>(a.w);
  const int n8 = a.dim / 8;
  float ss = 0.f;
  for (int i = lane; i < n8; i += 64) {
    Vec8<T> v;
    v.load(x + 8 * i);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float f = v.get(e);
      ss += f * f;
    }
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) ss += __shfl_xor(ss, o, 64);
  const float r = 1.0f / sqrtf(div_rn(ss, (float)a.dim) + a.eps);
  for (int i = lane; i < n8; i += 64) {
    Vec8<T> v;
    v.load(x + 8 * i);
    Vec8<T> o;
#pragma unroll
    for (int e = 0; e < 8; ++e) o.set(e, mul_rn(mul_rn(v.get(e), r), St<W>::ld(w + 8 * i + e)));
    o.store(y + 8 * i);
  }
}

// Few rows: one workgroup per row, the row read once into registers by four wavefronts (NV pieces
// of 8 elements per thread).  The sum of squares keeps the order of the kernel above, so that both
// give the same bits: the row passes through LDS and every wavefront adds all of it, lane l the
// pieces l, l + 64, ...  One row of 2560 in bf16, latency bound: 4.1 us a launch in a captured
// decode step against 5.9 for the kernel above, where one wavefront reads the row twice.
constexpr int RN_NT = 256, RN_NV = 4;

template <typename T, typename W>
__global__ void __launch_bounds__(RN_NT) rms_norm_row_kernel(b3_rms_norm_args a) {
  __shared__ __attribute__((aligned(16))) T row[8 * RN_NT * RN_NV];
  const int tid = threadIdx.x, lane = tid & 63, n8 = a.dim / 8;
  const T* x = reinterpret_cast<const T*>(a.x) + (long long)blockIdx.x * a.x_row_stride;
  T* y = reinterpret_cast<T*>(a.y) + (long long)blockIdx.x * a.y_row_stride;
  Vec8<T> v[RN_NV];
  Vec8<W> w[RN_NV];
#pragma unroll
  for (int q = 0; q < RN_NV; ++q)
    if (tid + RN_NT * q < n8) {
      v[q].load(x + 8 * (tid + RN_NT * q));
      w[q].load(reinterpret_cast<const W*>(a.w) + 8 * (tid + RN_NT * q));
    }
#pragma unroll
  for (int q = 0; q < RN_NV; ++q)
    if (tid + RN_NT * q < n8) v[q].store(row + 8 * (tid + RN_NT * q));
  __syncthreads();
  float ss = 0.f;
  for (int i = lane; i < n8; i += 64) {
    Vec8<T> u;
    u.load(row + 8 * i);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float f = u.get(e);
      ss += f * f;
    }
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) ss += __shfl_xor(ss, o, 64);
  const float r = 1.0f / sqrtf(div_rn(ss, (float)a.dim) + a.eps);
#pragma unroll
  for (int q = 0; q < RN_NV; ++q)
    if (tid + RN_NT * q < n8) {
#pragma unroll
      for (int e = 0; e < 8; ++e) v[q].set(e, mul_rn(mul_rn(v[q].get(e), r), w[q].get(e)));
      v[q].store(y + 8 * (tid + RN_NT * q));
    }
}

// One workgroup per row up to a row per compute unit, where every row's latency shows, if the row fits
// the registers, is long enough for four wavefronts and its weight may be read in 16-byte pieces.
constexpr int RN_MAX_ROWS = 256;

template <typename T, typename W>
static void launch_rms_w(const b3_rms_norm_args& a, hipStream_t st) {
  if (a.rows <= RN_MAX_ROWS && a.dim > 8 * 64 && a.dim <= 8 * RN_NT * RN_NV && reinterpret_cast<uintptr_t>(a.w) % 16 == 0)
    hipLaunchKernelGGL((rms_norm_row_kernel<T, W>), dim3((unsigned)a.rows), dim3(RN_NT), 0, st, a);
  else
    hipLaunchKernelGGL((rms_norm_kernel<T, W>), dim3((unsigned)((a.rows + 3) / 4)), dim3(256), 0, st, a);
}

template <typename T>
static int launch_rms(const b3_rms_norm_args& a, hipStream_t st) {
  if (a.w_dtype == B3_F32) launch_rms_w<T, float>(a, st);
  else launch_rms_w<T, uint16_t>(a, st);
  return (int)hipGetLastError();
}

}  // namespace b3

extern "C" int bolt3_rms_norm(const b3_rms_norm_args* a, void* stream) {
  if (!a || a->rows < 0 || a->dim <= 0 || a->dim % 8 || !a->x || !a->w || !a->y) return B3_ERR_ARG;
  if ((a->dtype != B3_F32 && a->dtype != B3_BF16) || (a->w_dtype != B3_F32 && a->w_dtype != B3_BF16))
    return B3_ERR_UNSUPPORTED;
  const int64_t es = a->dtype == B3_BF16 ? 2 : 4;
  if (a->x_row_stride < a->dim || a->y_row_stride < a->dim || (a->x_row_stride * es) % 16 ||
      (a->y_row_stride * es) % 16 || reinterpret_cast<uintptr_t>(a->x) % 16 || reinterpret_cast<uintptr_t>(a->y) % 16)
    return B3_ERR_ARG;
  if (a->rows == 0) return 0;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  return a->dtype == B3_BF16 ? b3::launch_rms<uint16_t>(*a, st) : b3::launch_rms<float>(*a, st);
}
