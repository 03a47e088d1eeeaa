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

// Every tensor of one direction of a call in one launch, in pieces of V
// consecutive elements: the most, up to 16 bytes, that half a row is a whole
// number of and the arrays are aligned to (a piece then lies in one half of its
// row, and is copied or zeroed as one).  A workgroup takes per_block whole rows, up
// to 256 N pieces, N of each thread in flight at once.
template <typename T, int V, int N, bool PAD>
__global__ __launch_bounds__(256) void pad_rows_kernel(const PadCall a, int d, int dp, int per_block,
                                                      unsigned inv) {
  typedef T Piece __attribute__((ext_vector_type(V)));
  // short calls (N 1): a tensor per row of a grid that its longest one fills;
  // long ones: each tensor its own workgroups, one after another
  int z = (int)blockIdx.y;
  if constexpr (N > 1)
    while (z + 1 < a.n && (int)blockIdx.x >= a.j[z + 1].first) ++z;
  const PadJob& job = a.j[z];
  const int width = PAD ? dp : d, pieces = width / V;
  const long r0 = (long)((int)blockIdx.x - (N > 1 ? job.first : 0)) * per_block;
  if (N == 1 && r0 >= job.rows) return;
  const int rows = static_cast<int>(min((long)per_block, job.rows - r0));
  const T* src = static_cast<const T*>(job.src) + r0 * (PAD ? d : dp);
  T* dst = static_cast<T*>(job.dst) + r0 * width;
  Piece x[N];
  int to[N];
#pragma unroll
  for (int n = 0; n < N; ++n) {
    const int i = (int)threadIdx.x + 256 * n;
    // i / pieces: inv is 2^20 / pieces rounded up, i below 2^10, pieces at most 2^8
    const int r = static_cast<int>(((unsigned)i * inv) >> 20), j = V * (i - r * pieces);
    const int from = PAD ? pad_source(j, d, dp) : pad_target(j, d, dp);
    to[n] = r < rows ? r * width + j : -1;
    x[n] = *reinterpret_cast<const Piece*>(src + min(r, rows - 1) * (PAD ? d : dp) + max(from, 0));
    if (from < 0) x[n] = Piece(static_cast<T>(0.0f));
  }
#pragma unroll
  for (int n = 0; n < N; ++n)
    if (to[n] >= 0) *reinterpret_cast<Piece*>(dst + to[n]) = x[n];
}

template <typename T, bool PAD>
hipError_t launch_pad(PadCall a, int d, int dp, hipStream_t st) {
  int v = 16 / sizeof(T);
  auto whole = [&](int n) {
    if (d % 2 != 0 || (d / 2) % n != 0) return n == 1;
    for (int i = 0; i < a.n; ++i)
      if (reinterpret_cast<uintptr_t>(a.j[i].src) % (n * sizeof(T)) != 0 ||
          reinterpret_cast<uintptr_t>(a.j[i].dst) % (n * sizeof(T)) != 0)
        return n == 1;
    return true;
  };
  while (!whole(v)) v /= 2;
  const int pieces = (PAD ? dp : d) / v;
  const unsigned inv = ((1u << 20) + pieces - 1) / pieces;
  int per_block = 4 * 256 / pieces;
  long blocks = 0, most = 0;
  for (int i = 0; i < a.n; ++i) {
    a.j[i].first = static_cast<int>(blocks);
    blocks += (a.j[i].rows + per_block - 1) / per_block;
    most = std::max(most, a.j[i].rows);
  }
  if (blocks == 0) return hipSuccess;
  // Bound by the launch on short calls, by the pieces on long ones.  Forward that
  // saves, then backward, bf16: 1500 tokens, 40/8 heads of 200: 168 + 534 us, where
  // one element a thread took 265 + 694 and a launch per tensor 223 + 647.  Four
  // pieces a thread once they give every CU two workgroups, one before (64
  // tokens, 14/2 heads of 80: 14.5 + 16.8 us, 15.4 + 17.6 with four).
  const bool four = blocks >= 512;
  if (!four) {
    per_block = 256 / pieces;
    blocks = (most + per_block - 1) / per_block;
  }
  auto pick = [&](auto nc) {
    constexpr int N = decltype(nc)::value;
    if constexpr (sizeof(T) == 2)
      if (v == 8) return pad_rows_kernel<T, 8, N, PAD>;
    return v == 4 ? pad_rows_kernel<T, 4, N, PAD> : v == 2 ? pad_rows_kernel<T, 2, N, PAD> : pad_rows_kernel<T, 1, N, PAD>;
  };
  auto fn = four ? pick(std::integral_constant<int, 4>{}) : pick(std::integral_constant<int, 1>{});
  hipLaunchKernelGGL(fn, dim3(static_cast<unsigned>(blocks), four ? 1 : a.n), dim3(256), 0, st, a, d, dp, per_block, inv);
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
