// Strided copies of several pieces in one launch: loading a decoder state (ring halves, sinks, slots)
// from tensors on the same device (vsa_lm/config/bolt3.py:450-457 leaves these in its kv_caches).
//
// A piece is rows of contiguous bytes.  Each piece has its own row of workgroups (blockIdx.y), which
// step over it in units of 16 bytes, or of 4 or 1 where an address, a stride or a length asks for it;
// a unit per thread at a time (with four in flight the pieces' bounds took longer than the loads: 16 us).
// What it saves is launches: a prefill's layer loads 17 pieces, 4.4 us each as copies of their own
// (75 us, with 2 x 256 tokens of 8 kv heads) and 4.6 us together.
#include "bolt3_common.h"
#include "bolt3_amd.h"

namespace b3 {
namespace copy {

struct Piece {
  const char* src;
  char* dst;
  long long src_stride, dst_stride;   // bytes between rows
  unsigned units, per_row, size;      // units in all and in a row, bytes of a unit
};
struct Pieces {
  Piece p[B3_COPY_MAX];
};

constexpr int NT = 256;

template <typename V>
__device__ __forceinline__ void copy_units(const Piece c) {
  const char* src = c.src;
  char* dst = c.dst;
  for (unsigned long long i = blockIdx.x * NT + threadIdx.x; i < c.units; i += gridDim.x * NT) {
    const unsigned r = (unsigned)i / c.per_row;
    const long long o = (long long)((unsigned)i - r * c.per_row) * sizeof(V);
    *reinterpret_cast<V*>(dst + r * c.dst_stride + o) = *reinterpret_cast<const V*>(src + r * c.src_stride + o);
  }
}

__global__ void __launch_bounds__(NT) copy_pieces_kernel(const Pieces a) {
  const Piece& c = a.p[blockIdx.y];
  if (c.size == 16)
    copy_units<uint4>(c);
  else if (c.size == 4)
    copy_units<uint32_t>(c);
  else
    copy_units<uint8_t>(c);
}

}  // namespace copy
}  // namespace b3

extern "C" int bolt3_copy_pieces(const b3_copy_pieces_args* a, void* stream) {
  using namespace b3::copy;
  if (!a || a->n < 0 || a->n > B3_COPY_MAX) return B3_ERR_ARG;
  Pieces k{};
  int n = 0;
  unsigned wg = 1;
  for (int i = 0; i < a->n; ++i) {
    const b3_copy_piece& q = a->piece[i];
    if (q.rows < 0 || q.row_bytes < 0) return B3_ERR_ARG;
    if (q.rows == 0 || q.row_bytes == 0) continue;
    if (!q.src || !q.dst || q.src_stride < 0 || q.dst_stride < 0 || (q.rows > 1 && q.dst_stride < q.row_bytes))
      return B3_ERR_ARG;
    const uint64_t all = reinterpret_cast<uintptr_t>(q.src) | reinterpret_cast<uintptr_t>(q.dst) | (uint64_t)q.row_bytes |
                         (q.rows > 1 ? (uint64_t)q.src_stride | (uint64_t)q.dst_stride : 0);
    const unsigned size = all % 16 == 0 ? 16 : all % 4 == 0 ? 4 : 1;
    const long long per_row = q.row_bytes / size;
    if (per_row > 0x7fffffffLL / q.rows) return B3_ERR_UNSUPPORTED;
    const unsigned units = (unsigned)(per_row * q.rows);
    k.p[n++] = Piece{static_cast<const char*>(q.src), static_cast<char*>(q.dst), q.src_stride, q.dst_stride,
                     units, (unsigned)per_row, size};
    const unsigned need = (units - 1) / NT + 1;
    wg = need > wg ? need : wg;
  }
  if (n == 0) return B3_OK;
  hipLaunchKernelGGL(copy_pieces_kernel, dim3(wg < 256 ? wg : 256, n), dim3(NT), 0,
                     reinterpret_cast<hipStream_t>(stream), k);
  return (int)hipGetLastError();
}
