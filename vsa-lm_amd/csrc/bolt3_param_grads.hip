// Gradients of a Bolt3Attn layer's small parameters from the partial sums that the backward's
// kernels leave: res_norm and q/k norm weights, projection biases, kappa and log_gamma, in one
// launch.  Replaces the reductions autograd makes of vsa_lm/config/bolt3.py:56-57, :59-66, :238-241
// and :253-256.
//
// Two kinds of workgroup, each owning its outputs whole, so that nothing is added across
// workgroups and every sum has one order: PG_C columns of a partial-sum array (PG_RG rows at a
// time, PG_UN loads per thread in flight), and one per kv head for kappa and log_gamma.  Bound by
// the latency of those loads: 49 us at the Qwen3-4B shape with 4 x 4096 tokens (164 us with 32
// columns per workgroup), 18 us at the SmolLM shape with 4 x 1100.  It takes the place of about 25
// elementwise and reduction launches, which bound the second (forward and backward 1.59 -> 1.23
// ms); in the first their column sums of the projection gradient ran beside its two products,
// slowing them, and for 55 us after them.  Where q, k and v have biases (all 6192 columns of the
// first shape instead of 40) forward and backward take 5.26-5.28 ms against 5.32-5.45 with those sums.
#include "bolt3_common.h"
#include "bolt3_amd.h"

namespace b3 {
namespace pgrad {

constexpr int PG_NT = 1024, PG_UN = 16, PG_S = 128;   // threads, loads in flight, slots
constexpr int PG_C = 8;                // columns of a workgroup: few, so that the long columns take few rounds
constexpr int PG_RG = PG_NT / PG_C;    // rows that it reads at a time

__device__ __forceinline__ float ldf(const float* p) { return *p; }
__device__ __forceinline__ float ldf(const uint16_t* p) { return bf2f(*p); }

// sum over the rows of column c (0 where not live), in the PG_C threads of row group 0
template <typename T>
__device__ __forceinline__ float column_sum(const T* src, long long rows, long long stride, int c, bool live,
                                            float (*red)[PG_C + 1]) {
  const int rg = threadIdx.x / PG_C;
  float s = 0.f;
  if (live)
    for (long long r = rg; r < rows; r += (long long)PG_RG * PG_UN) {
      float x[PG_UN];
#pragma unroll
      for (int u = 0; u < PG_UN; ++u) {
        const long long q = r + (long long)PG_RG * u;
        x[u] = q < rows ? ldf(src + q * stride + c) : 0.f;
      }
#pragma unroll
      for (int u = 0; u < PG_UN; ++u) s += x[u];
    }
  // the row groups of a wavefront, then the wavefronts in order
#pragma unroll
  for (int o = PG_C; o < 64; o <<= 1) s += __shfl_xor(s, o, 64);
  if ((threadIdx.x & 63) < PG_C) red[threadIdx.x >> 6][threadIdx.x & 63] = s;
  __syncthreads();
  s = 0.f;
  if (rg == 0)
    for (int i = 0; i < PG_NT / 64; ++i) s += red[i][threadIdx.x];
  return s;
}

__device__ __forceinline__ float block_sum(float v, float* red) {
  v = wave_sum(v);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  v = 0.f;
  for (int i = 0; i < PG_NT / 64; ++i) v += red[i];
  __syncthreads();
  return v;
}

template <typename T>
__global__ void __launch_bounds__(PG_NT) param_grads_kernel(b3_param_grads_args a) {
  __shared__ float red[PG_NT / 64][PG_C + 1];
  const int tid = threadIdx.x, col = tid % PG_C, HD = a.HD;
  const long long BH = (long long)a.B * a.HKV;
  int w = blockIdx.x;
  // ---- column sums: res_norm, q_norm, k_norm, biases
  const int tn = HD / PG_C, tb = (a.n_bias + PG_C - 1) / PG_C;
  const float* src[3] = {a.d_res_w, a.d_qn_w, a.d_kn_w};
  float* dst[3] = {a.g_res_w, a.g_qn_w, a.g_kn_w};
  const long long rows[3] = {BH * a.n_chunks, a.n_blocks, a.n_blocks};
  for (int k = 0; k < 3; ++k) {
    if (!src[k]) continue;
    if (w < tn) {
      const float s = column_sum(src[k], rows[k], HD, PG_C * w + col, true, red);
      if (tid < PG_C) dst[k][PG_C * w + col] = s;
      return;
    }
    w -= tn;
  }
  if (w < tb) {
    const int c = PG_C * w + col;
    const float s = column_sum(static_cast<const T*>(a.dz), (long long)a.B * a.T, a.dz_row_stride, a.bias_col + c,
                               c < a.n_bias, red);
    if (tid < PG_C && c < a.n_bias) a.g_bias[c] = s;
    return;
  }
  w -= tb;
  // ---- kv head w: kappa (the slot bias is kappa log(max(mass, 1))) and gamma
  // 128 threads per (step, batch row), a slot each: the row's G heads x query tiles are contiguous
  const int hkv = w, slot = tid & (PG_S - 1);
  float kap = 0.f, gam = 0.f;
  const int nr = a.H / a.HKV * a.n_qtiles;
  for (long long sb = tid / PG_S; sb < (long long)a.n_steps * a.B; sb += PG_NT / PG_S) {
    const float* d = a.d_bias + (sb * a.HKV + hkv) * nr * PG_S + slot;
    const float lm = logf(fmaxf(a.snap_mass[(sb * a.HKV + hkv) * PG_S + slot], 1.0f));
    float s = 0.f;
#pragma unroll 16
    for (int r = 0; r < nr; ++r) s += d[r * PG_S];
    kap += s * lm;
  }
  for (int i = tid; i < a.B * a.n_chunks; i += PG_NT)
    gam += a.d_gamma[(long long)(i / a.n_chunks * a.HKV + hkv) * a.n_chunks + i % a.n_chunks];
  const int nm = HD / 32;
  for (int i = tid; i < a.n_steps * a.B * nm; i += PG_NT)
    gam += a.d_gamma_chain[((long long)(i / nm) * a.HKV + hkv) * nm + i % nm];
  kap = block_sum(kap, &red[0][0]);
  gam = block_sum(gam, &red[0][0]);
  if (tid == 0) {
    a.g_kappa[hkv] = kap;
    // gamma = clamp(0.999 sigmoid(log_gamma), 1e-3, 0.999); clamp passes its bounds inclusive
    const float x = a.log_gamma[hkv], sg = 1.0f / (1.0f + expf(-x)), g0 = 0.999f * sg;
    a.g_log_gamma[hkv] = g0 >= 1e-3f && g0 <= 0.999f ? gam * 0.999f * sg / (1.0f + expf(x)) : 0.f;
  }
}

}  // namespace pgrad
}  // namespace b3

extern "C" int bolt3_param_grads(const b3_param_grads_args* a, void* stream) {
  if (!a) return B3_ERR_ARG;
  if (a->dtype != B3_F32 && a->dtype != B3_BF16) return B3_ERR_UNSUPPORTED;
  if (a->HD != 64 && a->HD != 128) return B3_ERR_UNSUPPORTED;
  if (a->B <= 0 || a->T <= 0 || a->H <= 0 || a->HKV <= 0 || a->H % a->HKV || a->S <= 0 || a->n_chunks <= 0 ||
      a->n_qtiles <= 0 || a->n_steps < 0 || a->n_blocks < 0 || a->n_bias < 0 || a->bias_col < 0)
    return B3_ERR_ARG;
  if (!a->d_res_w || !a->d_gamma || !a->log_gamma || !a->g_res_w || !a->g_kappa || !a->g_log_gamma) return B3_ERR_ARG;
  if (a->n_steps > 0 && a->S != b3::pgrad::PG_S) return B3_ERR_UNSUPPORTED;
  if (a->n_steps > 0 && (!a->d_bias || !a->snap_mass || !a->d_gamma_chain)) return B3_ERR_ARG;
  if ((a->d_qn_w && !a->g_qn_w) || (a->d_kn_w && !a->g_kn_w)) return B3_ERR_ARG;
  if (a->n_bias > 0 && (!a->dz || !a->g_bias || a->dz_row_stride < (int64_t)a->bias_col + a->n_bias)) return B3_ERR_ARG;
  const int tn = a->HD / b3::pgrad::PG_C;
  const dim3 grid(tn * (1 + (a->d_qn_w != nullptr) + (a->d_kn_w != nullptr)) + (a->n_bias + b3::pgrad::PG_C - 1) / b3::pgrad::PG_C + a->HKV);
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  using namespace b3::pgrad;
  if (a->dtype == B3_BF16) hipLaunchKernelGGL((param_grads_kernel<uint16_t>), grid, dim3(PG_NT), 0, st, *a);
  else hipLaunchKernelGGL((param_grads_kernel<float>), grid, dim3(PG_NT), 0, st, *a);
  return (int)hipGetLastError();
}
