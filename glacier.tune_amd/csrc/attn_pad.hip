// attn_pad.hip -- head sizes the attention kernels are not built for.
//
// GpuLoraEngine.SupportsAttention (GpuLoraEngine.cs:111-112) takes any head
// size; the kernels are instantiated for 32, 64, 96, 128 and 256.  A call
// with another head size d runs them on copies of its rows padded to the
// next of those sizes, dp, laid out so that the rotation pairs
// (i, i + d/2) of RoPEKernel.cs:74-84 stay pairs of the padded row: the first
// half's d/2 elements go to columns 0 .. d/2 - 1, the second half's to
// dp/2 .. dp/2 + d/2 - 1, an odd d's last (unrotated) element to column d/2,
// and every other column is zero.  The engine's RoPE table for such a call
// holds the angles of d in its first d/2 columns and the identity rotation
// (cos 1, sin 0) after them, so padded columns stay zero (or keep the odd
// element) through every rotation, contribute nothing to a score or a row
// term, and come out of dQ/dK/dV as zeros; the softmax scale is that of d.
#include "attn_common.hpp"
#include "attn_launch.hpp"

namespace glacier {
namespace {

// The source column of padded column j (-1: a zero column).
__device__ inline int pad_source(int j, int d, int dp) {
  const int h = d / 2, hp = dp / 2;
  if (j < hp) {
    if (j < h) return j;
    return ((d & 1) && j == h) ? 2 * h : -1;
  }
  const int i = j - hp;
  return i < h ? h + i : -1;
}

// The padded column of source column s.
__device__ inline int pad_target(int s, int d, int dp) {
  const int h = d / 2, hp = dp / 2;
  if (s < h) return s;
  if (s < 2 * h) return hp + (s - h);
  return h;  // an odd d's last element
}

// Every tensor of one direction of a call in one launch (blockIdx.y: the
// tensor), V consecutive elements of a row per thread: whole 16-byte pieces
// where half a row is a whole number of them and the arrays are aligned (then a
// piece lies in one half, and is copied or zeroed as one), else one element.
// A workgroup takes 256 / (pieces per row) rows, so no index is divided by
// more than a row's pieces.  Bound by the launch: a step at head size 80, 16
// heads, 600 tokens made 14 launches of 3.9 us, one per tensor and element by
// element; these are 4 of about 4.
template <typename T, int V, bool PAD>
__global__ __launch_bounds__(256) void pad_rows_kernel(const PadCall a, int d, int dp) {
  const PadJob& job = a.j[blockIdx.y];
  const int width = PAD ? dp : d, pieces = width / V, per_block = 256 / pieces;
  const int sub = (int)threadIdx.x / pieces, j = V * ((int)threadIdx.x - sub * pieces);
  const long r = (long)blockIdx.x * per_block + sub;
  if (sub >= per_block || r >= job.rows) return;
  const T* src = static_cast<const T*>(job.src) + r * (PAD ? d : dp);
  T* dst = static_cast<T*>(job.dst) + r * width + j;
  const int from = PAD ? pad_source(j, d, dp) : pad_target(j, d, dp);
  if constexpr (V == 1) {
    *dst = from >= 0 ? src[from] : static_cast<T>(0.0f);
  } else {
    i32x4 x{0, 0, 0, 0};
    if (from >= 0) x = *reinterpret_cast<const i32x4*>(src + from);
    *reinterpret_cast<i32x4*>(dst) = x;
  }
}

template <typename T, bool PAD>
hipError_t launch_pad(const PadCall& a, int d, int dp, hipStream_t st) {
  constexpr int W = 16 / sizeof(T);
  bool wide = (d / 2) % W == 0 && d % 2 == 0;
  long rows = 0;
  for (int i = 0; i < a.n; ++i) {
    rows = rows > a.j[i].rows ? rows : a.j[i].rows;
    wide = wide && (reinterpret_cast<uintptr_t>(a.j[i].src) & 15) == 0 &&
           (reinterpret_cast<uintptr_t>(a.j[i].dst) & 15) == 0;
  }
  if (rows == 0) return hipSuccess;
  const int per_block = 256 / ((PAD ? dp : d) / (wide ? W : 1));
  const dim3 grid(static_cast<unsigned>((rows + per_block - 1) / per_block), a.n);
  if (wide)
    hipLaunchKernelGGL((pad_rows_kernel<T, W, PAD>), grid, dim3(256), 0, st, a, d, dp);
  else
    hipLaunchKernelGGL((pad_rows_kernel<T, 1, PAD>), grid, dim3(256), 0, st, a, d, dp);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_pad_rows(bool io_bf16, const PadCall& a, int d, int dp, hipStream_t st) {
  return io_bf16 ? launch_pad<bf16, true>(a, d, dp, st) : launch_pad<float, true>(a, d, dp, st);
}

hipError_t launch_unpad_rows(bool io_bf16, const PadCall& a, int d, int dp, hipStream_t st) {
  return io_bf16 ? launch_pad<bf16, false>(a, d, dp, st) : launch_pad<float, false>(a, d, dp, st);
}

}  // namespace glacier
