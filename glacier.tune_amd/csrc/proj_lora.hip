// proj_lora.hip -- the projection step either side of attention, on the
// device: a frozen base projection plus a trainable LoRA adapter, for the q,
// k and v projections of one normalised input (GpuLoraEngine.ForwardQKV,
// GpuLoraEngine.Forward.cs:205-245, whose LoRA delta the reference adds on
// the host, AddLoraDeltaHost :366-399), and the reverse
// (LoraAdapter.Backward, LoraAdapter.cs:190-247).
//
// Per projection p, with X [T][in], W_p [out][in], A_p [in][r], B_p [r][out]:
//   forward   Y_p  = X W_p^T + bias_p + s_p (X A_p) B_p
//   backward  dX   = sum_p dY_p W_p + s_p (dY_p B_p^T) A_p^T
//             dA_p += s_p X^T (dY_p B_p^T),  dB_p += s_p (X A_p)^T dY_p
//
// bf16 tensors (every width a multiple of 8, 16-byte aligned): three launches
// forward, four backward.
//   lowrank_split   L = X A_p and dL = dY_p B_p^T, and the split terms
//                   (split3.hpp) of s L and of the adapters
//   lowrank_cols    backward: grad_A += s X^T dL, grad_B += s L^T dY (reduction
//                   over the tokens): 64-column slabs, tokens split over 8 waves
//   proj_gemm       (proj_gemm.hip) Y_p = X W_p^T + bias_p + (s L_p) B_p for
//                   every projection, or dX = sum_p dY_p W_p + (s dL_p) A_p^T
// Other calls (fp32 tensors, widths that are multiples of 4 only):
//   proj_gemm_f32   the base products, fp32 results, one launch per projection
//   lowrank_rows    L and dL: 16-row slabs, the reduction split over workgroups
//                   and over their 8 waves, fp32 MFMAs
//   lowrank_reduce  adds the workgroups' split sums in split order
//   lowrank_cols    as above
//   lowrank_out     Y_p = io(Yf_p + bias_p + (s L_p) B_p) and dX = io(dXf +
//                   sum_p (s dL_p) A_p^T): 16 x 256 tiles, the rank-r
//                   product on MFMAs, fused with the dtype conversion
// The adapters, the low-rank activations and the gradients stay fp32, as in
// the reference (LoraAdapter.cs:23-24); bf16 tensors round only the base
// operands and the outputs.  Every reduction has a fixed order, so every
// result is bitwise repeatable.
#include "attn_common.hpp"
#include "lds_mfma.hpp"
#include "proj_launch.hpp"
#include "split3.hpp"

namespace glacier {
namespace {

constexpr int kLrWaves = 8;  // waves of a rows/cols workgroup, splitting the reduction
constexpr int kLrThreads = 64 * kLrWaves;
constexpr int kOutThreads = 256;  // lowrank_out: 4 waves of 16 x 64
constexpr int kMaxJobs = 2 * kMaxProj;

__device__ inline void load4(const float* p, float (&x)[4]) {
  const float4 a = *reinterpret_cast<const float4*>(p);
  x[0] = a.x; x[1] = a.y; x[2] = a.z; x[3] = a.w;
}

// 4 consecutive elements as loaded, converted (or zeroed) only when used:
// every load of a step is issued at an in-bounds (clamped) address before any
// value is used, and out-of-range values of ONE operand of each product are
// zeroed afterwards; the other operand's clamped values then meet zeros, or
// reach only outputs that are not stored.  (A load under a condition makes
// the wave wait for each load in turn; so would a select on both operands,
// which the compiler turns back into conditional loads.)
template <typename IO>
struct Raw4;
template <>
struct Raw4<float> {
  using T = float4;
};
template <>
struct Raw4<bf16> {
  using T = bf16x4;
};
template <typename IO>
__device__ inline typename Raw4<IO>::T ld_raw4(const IO* p) {
  return *reinterpret_cast<const typename Raw4<IO>::T*>(p);
}
__device__ inline void sel4(float4 r, bool ok, float (&x)[4]) {
  x[0] = ok ? r.x : 0.0f;
  x[1] = ok ? r.y : 0.0f;
  x[2] = ok ? r.z : 0.0f;
  x[3] = ok ? r.w : 0.0f;
}
__device__ inline void sel4(bf16x4 r, bool ok, float (&x)[4]) {
#pragma unroll
  for (int e = 0; e < 4; ++e) x[e] = ok ? (float)r[e] : 0.0f;
}

__device__ inline f32x4 mma_f32(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// The [lo, hi) share of part p of n of a range [0, len), cut at multiples of g.
__device__ inline void share(int len, int n, int p, int g, int& lo, int& hi) {
  const int per = (len + n * g - 1) / (n * g) * g;
  lo = min(len, p * per);
  hi = min(len, lo + per);
}

// One product Out [T][r] = U [T][K] V of lowrank_rows: V = A [K][r] (vt 0)
// or B^T with B [r][K] (vt 1); U in the call's dtype.
struct RowsJob {
  const void* u;
  const float* v;
  int K;
  int vt;
};
struct RowsJobs {
  RowsJob j[kMaxJobs];
};

// The k range [kb, ke) of one wave of lowrank_rows_kernel, added into acc.
// In a step of 16 lane (i = lane % 16, q = lane / 16) loads U[row i][k0 + 4q
// .. +4] and, for MFMA e of the step, supplies U[i][k0 + 4q + e] and V(k0 +
// 4q + e, 16 jt + i): each MFMA's reduction index q maps to one k for both
// operands.  U is zeroed for k past the slice and for rows >= T.
template <typename IO, int NT, bool VT>
__device__ inline void rows_accumulate(const IO* __restrict__ urow, bool row_ok,
                                       const float* __restrict__ v, int K, int rank, int kb, int ke,
                                       f32x4 (&acc)[NT]) {
  constexpr int CH = NT <= 2 ? 8 : 4;  // steps whose loads are issued together
  const int lane = threadIdx.x & 63, i = lane & 15, q = lane >> 4;
  for (int k0 = kb; k0 < ke; k0 += 16 * CH) {
    typename Raw4<IO>::T xr[CH];
    float w[CH][NT][4];
#pragma unroll
    for (int s = 0; s < CH; ++s) {
      if (k0 + 16 * s >= ke) break;  // the wave's slice ends (uniform)
      const int kc = min(k0 + 16 * s + 4 * q, K - 4);  // K % 4 == 0
      xr[s] = ld_raw4(urow + kc);
#pragma unroll
      for (int jt = 0; jt < NT; ++jt) {
        const int jc = min(16 * jt + i, rank - 1);
        if constexpr (VT) {
          const float4 r = *reinterpret_cast<const float4*>(v + (long)jc * K + kc);
          w[s][jt][0] = r.x; w[s][jt][1] = r.y; w[s][jt][2] = r.z; w[s][jt][3] = r.w;
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) w[s][jt][e] = v[(long)(kc + e) * rank + jc];
        }
      }
    }
#pragma unroll
    for (int s = 0; s < CH; ++s) {
      if (k0 + 16 * s >= ke) break;
      const bool k_ok = k0 + 16 * s + 4 * q < ke;  // a 4-chunk is all in or all out
      float x[4];
      sel4(xr[s], k_ok && row_ok, x);
#pragma unroll
      for (int jt = 0; jt < NT; ++jt)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[jt] = mma_f32(x[e], w[s][jt][e], acc[jt]);
    }
  }
}

// Workgroup (x, y, z): rows 16x.. of job z, split y of its K; wave w reduces
// a contiguous slice of that split (rows_accumulate).  The workgroup's sums
// (waves added in order through LDS) go to part[z][y][x][16][16 NT].
template <typename IO, int NT>
__global__ __launch_bounds__(kLrThreads) void lowrank_rows_kernel(RowsJobs jobs, int rows, int rank,
                                                                  float* __restrict__ part) {
  constexpr int kOut = 16 * NT * 16;  // outputs of the workgroup
  __shared__ float red[kLrWaves * kOut];
  const RowsJob& job = jobs.j[blockIdx.z];
  const int K = job.K;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int i = lane & 15, q = lane >> 4;
  const int t0 = blockIdx.x * 16;
  const bool row_ok = t0 + i < rows;
  const IO* urow = static_cast<const IO*>(job.u) + (long)(row_ok ? t0 + i : 0) * K;
  int k_lo, k_hi, kb, ke;
  share(K, gridDim.y, blockIdx.y, 16, k_lo, k_hi);
  share(k_hi - k_lo, kLrWaves, wave, 16, kb, ke);
  f32x4 acc[NT];
#pragma unroll
  for (int jt = 0; jt < NT; ++jt) acc[jt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  if (job.vt)
    rows_accumulate<IO, NT, true>(urow, row_ok, job.v, K, rank, k_lo + kb, k_lo + ke, acc);
  else
    rows_accumulate<IO, NT, false>(urow, row_ok, job.v, K, rank, k_lo + kb, k_lo + ke, acc);
  // D of tile jt: lane (i, q), register c holds row 4q + c, column 16 jt + i.
#pragma unroll
  for (int jt = 0; jt < NT; ++jt)
#pragma unroll
    for (int c = 0; c < 4; ++c) red[wave * kOut + (4 * q + c) * (16 * NT) + 16 * jt + i] = acc[jt][c];
  __syncthreads();
  float* mine = part + (((long)blockIdx.z * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x) * kOut;
  for (int idx = threadIdx.x; idx < kOut; idx += kLrThreads) {
    float sum = 0.0f;
#pragma unroll
    for (int wv = 0; wv < kLrWaves; ++wv) sum += red[wv * kOut + idx];
    mine[idx] = sum;
  }
}

// dense[z][t][j] = sum over the splits s (ascending) of part[z][s][t / 16]
// [t % 16][j], for every job z of a lowrank_rows launch.
__global__ __launch_bounds__(256) void lowrank_reduce_kernel(const float* __restrict__ part,
                                                             float* __restrict__ dense, int n_jobs,
                                                             int splits, int slabs, int width,
                                                             int T, int rank) {
  const long idx = (long)blockIdx.x * 256 + threadIdx.x;
  const long per_job = (long)T * rank;
  if (idx >= n_jobs * per_job) return;
  const int z = (int)(idx / per_job), t = (int)(idx % per_job / rank), j = (int)(idx % rank);
  const long slab_floats = 16L * width;
  const float* p = part + ((long)z * splits * slabs + t / 16) * slab_floats + (t % 16) * width + j;
  float sum = 0.0f;
  for (int s = 0; s < splits; ++s) sum += p[(long)s * slabs * slab_floats];
  dense[idx] = sum;
}

// ---- bf16 tensors: the low-rank products and their split terms ----------
// L [T][r] = U [T][K] V for each job (V as in RowsJob), with U in bf16: V goes
// onto the bf16 MFMAs in its three terms (split3.hpp), so every product is
// exact and the sums are fp32, at 3/8 of the fp32 MFMA's time.  The results
// go out as L in fp32 (lowrank_cols) and, where the job has `terms`, as the
// split terms of s L, the B operand of the GEMM's low-rank segment; the last
// kTermBlocks workgroups write the adapters' own terms, its A operand.  A row
// of terms holds six stretches of r: the products of the same stretch of the
// two operands are h h, h m, m h, m m, h l, l h.
// Bound by the vector-memory unit (V is read a column at a time, 64-byte
// pieces): 11-15 us at 512 x 3584 -> 3584/512/512 and 23-39 us at 4096 x 4096
// -> 4096/1024/1024, rank 16, where the fp32 form with its separate reduction
// took 14 and 38 us without forming the terms.
struct SplitJob {
  const void* u;  // [T][K] (bf16)
  const float* v;
  float* l;       // [T][r]
  void* terms;    // [T][P] (bf16) or null
  float s;        // the terms are those of s L
  int K;
  int vt;
};
// terms [n][P] of V [r][n] (across 0), or terms [P][n] of V [n][r] (across 1)
struct TermJob {
  const float* v;
  void* terms;
  int n;
};
struct SplitCall {
  SplitJob j[kMaxJobs];
  TermJob v[kMaxProj];
  int n, nv, across;
  int slabs;   // row slabs of a job
  int* odd;    // [kTermBlocks], then [n][slabs]: a non-finite value among what that workgroup wrote
};

__device__ inline bool not_finite(float x) { return (__float_as_uint(x) & 0x7f800000u) == 0x7f800000u; }

// The six entries of a terms row for x: side 0 the adapters', side 1 (s L).
template <typename Put>
__device__ inline void put_terms(float x, int side, Put&& put) {
  const bf16 h = (bf16)x;
  const float r1 = x - (float)h;
  const bf16 m = (bf16)r1, l = (bf16)(r1 - (float)m);
  put(0, h);
  put(1, side ? m : h);
  put(2, side ? h : m);
  put(3, m);
  put(4, side ? l : h);
  put(5, side ? h : l);
}

// x has a split: its terms are finite (false also for a finite x that rounds
// to infinity).
[[maybe_unused]] __device__ inline bool has_split(float x) { return !not_finite((float)(bf16)x); }

constexpr int kTermBlocks = 64;
// Waves of a lowrank_split workgroup
constexpr int split_waves(int nt, int rb) { return rb == 1 && nt % 2 == 1 ? 16 : 8; }

#if defined(__HIP_DEVICE_COMPILE__)
// The k range [kb, ke) of one wave of lowrank_split_kernel, added into acc.
// Steps of 32: lane (i, q) holds U[row i][k0 + 8q .. +7] and V[k0 + 8q ..
// +7][16 jt + i].  K % 8 == 0, so a lane's 8 are all in or all out; out of
// range V is zeroed, U clamped (and finite, or the step goes the fp32 way,
// where U is zeroed as well).
template <int NT, int RB, bool VT>
__device__ inline void split_accumulate(const bf16* const (&u)[RB], const float* __restrict__ v0, int K,
                                        int rank, int kb, int ke, f32x4 (&acc)[RB][NT]) {
  const int lane = threadIdx.x & 63, i = lane & 15, q = lane >> 4;
  constexpr int CH = NT * RB <= 2 ? 4 : NT * RB <= 8 ? 2 : 1;  // steps whose loads are issued together
  for (int k0 = kb; k0 < ke; k0 += 32 * CH) {
    bf16x8 ur[CH][RB];
    float vr[CH][NT][8];
#pragma unroll
    for (int s = 0; s < CH; ++s) {
      const int kc = min(k0 + 32 * s + 8 * q, K - 8);
#pragma unroll
      for (int b = 0; b < RB; ++b) ur[s][b] = *reinterpret_cast<const bf16x8*>(u[b] + kc);
#pragma unroll
      for (int jt = 0; jt < NT; ++jt) {
        const int jc = min(16 * jt + i, rank - 1);
        if constexpr (VT) {
          load8(v0 + (long)jc * K + kc, vr[s][jt]);
        } else {
#pragma unroll
          for (int e = 0; e < 8; ++e) vr[s][jt][e] = v0[(long)(kc + e) * rank + jc];
        }
      }
    }
#pragma unroll
    for (int s = 0; s < CH; ++s) {
      if (k0 + 32 * s >= ke) break;
      const bool k_ok = k0 + 32 * s + 8 * q < ke;
      float chk = 0.0f;  // NaN once an element of U is not finite
#pragma unroll
      for (int b = 0; b < RB; ++b)
#pragma unroll
        for (int e = 0; e < 8; ++e) chk += 0.0f * (float)ur[s][b][e];
#pragma unroll
      for (int jt = 0; jt < NT; ++jt) {
#pragma unroll
        for (int e = 0; e < 8; ++e) vr[s][jt][e] = k_ok ? vr[s][jt][e] : 0.0f;
        Split3 v;
        const bool bad = v.set(vr[s][jt]) || chk != chk;
        if (__any(bad)) {
#pragma unroll
          for (int b = 0; b < RB; ++b)
#pragma unroll
            for (int e = 0; e < 8; ++e)
              acc[b][jt] = mma_f32(k_ok ? (float)ur[s][b][e] : 0.0f, vr[s][jt][e], acc[b][jt]);
        } else {
#pragma unroll
          for (int b = 0; b < RB; ++b) {
            acc[b][jt] = Mfma<bf16>::mma(ur[s][b], v.l, acc[b][jt]);
            acc[b][jt] = Mfma<bf16>::mma(ur[s][b], v.m, acc[b][jt]);
            acc[b][jt] = Mfma<bf16>::mma(ur[s][b], v.h, acc[b][jt]);
          }
        }
      }
    }
  }
}
#endif

template <int NT, int RB>
__global__ __launch_bounds__(64 * split_waves(NT, RB)) void lowrank_split_kernel(const SplitCall a, int T,
                                                                             int rank) {
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr int W = split_waves(NT, RB);  // waves, splitting K
  constexpr int kRow = 16 * NT + 1;
  __shared__ float red[W * 16 * RB * kRow];
  const int P = term_pitch(rank);
  bool odd = false;
  const int rows_blocks = a.n * a.slabs;
  if ((int)blockIdx.x >= rows_blocks) {
    // the adapters' terms: four ranks of one feature a thread, its loads
    // together (tied, so that none sinks under the bounds tests below),
    // features consecutive over the threads
    const int chunks = (rank + 3) / 4;
    int total = 0;
    for (int p = 0; p < a.nv; ++p) total += a.v[p].n * chunks;
    for (int g = ((int)blockIdx.x - rows_blocks) * (64 * W) + (int)threadIdx.x; g < total;
         g += kTermBlocks * 64 * W) {
      int p = 0, idx = g;
      while (idx >= a.v[p].n * chunks) idx -= a.v[p++].n * chunks;
      const float* v = a.v[p].v;
      bf16* out = static_cast<bf16*>(a.v[p].terms);
      const int n = a.v[p].n, f = idx % n, j0 = 4 * (idx / n);
      float x[4];
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        const int j = min(j0 + m, rank - 1);
        x[m] = v[a.across ? (long)f * rank + j : (long)j * n + f];
      }
#pragma unroll
      for (int m = 0; m < 4; ++m) tie_v(x[m]);
      if (!a.across && rank % 4 == 0) {  // four entries of a row in one store
        bf16x4 t4[6];
#pragma unroll
        for (int m = 0; m < 4; ++m) {
          odd |= !has_split(x[m]);
          put_terms(x[m], 0, [&](int e, bf16 t) { t4[e][m] = t; });
        }
#pragma unroll
        for (int e = 0; e < 6; ++e) *reinterpret_cast<bf16x4*>(out + (long)f * P + e * rank + j0) = t4[e];
      } else {
#pragma unroll
        for (int m = 0; m < 4; ++m) {
          if (j0 + m >= rank) break;
          odd |= !has_split(x[m]);
          put_terms(x[m], 0, [&](int e, bf16 t) {
            const int q = e * rank + j0 + m;
            out[a.across ? (long)q * n + f : (long)f * P + q] = t;
          });
        }
      }
      if (j0 == 0)
        for (int q = 6 * rank; q < P; ++q) out[a.across ? (long)q * n + f : (long)f * P + q] = (bf16)0.0f;
    }
    odd = __syncthreads_or(odd);
    if (threadIdx.x == 0) a.odd[(int)blockIdx.x - rows_blocks] = odd;
    return;
  }
  const int z = (int)blockIdx.x / a.slabs, slab = (int)blockIdx.x % a.slabs;
  const SplitJob& job = a.j[z];
  const int K = job.K;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int i = lane & 15, q = lane >> 4;
  const int t0 = slab * 16 * RB;
  const bf16* u[RB];
#pragma unroll
  for (int b = 0; b < RB; ++b)
    u[b] = static_cast<const bf16*>(job.u) + (long)min(t0 + 16 * b + i, T - 1) * K;
  int kb, ke;
  share(K, W, wave, 32, kb, ke);
  f32x4 acc[RB][NT];
#pragma unroll
  for (int b = 0; b < RB; ++b)
#pragma unroll
    for (int jt = 0; jt < NT; ++jt) acc[b][jt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  if (job.vt)
    split_accumulate<NT, RB, true>(u, job.v, K, rank, kb, ke, acc);
  else
    split_accumulate<NT, RB, false>(u, job.v, K, rank, kb, ke, acc);
  // D of (b, jt): lane (i, q), register c holds row 16 b + 4q + c, column 16 jt + i
#pragma unroll
  for (int b = 0; b < RB; ++b)
#pragma unroll
    for (int jt = 0; jt < NT; ++jt)
#pragma unroll
      for (int c = 0; c < 4; ++c)
        red[(wave * 16 * RB + 16 * b + 4 * q + c) * kRow + 16 * jt + i] = acc[b][jt][c];
  __syncthreads();
  for (int idx = threadIdx.x; idx < 16 * RB * 16 * NT; idx += 64 * W) {
    const int r = idx / (16 * NT), j = idx % (16 * NT), t = t0 + r;
    if (t >= T || j >= rank) continue;
    float sum = 0.0f;
#pragma unroll
    for (int w = 0; w < W; ++w) sum += red[(w * 16 * RB + r) * kRow + j];
    job.l[(long)t * rank + j] = sum;
    if (job.terms == nullptr) continue;
    bf16* row = static_cast<bf16*>(job.terms) + (long)t * P;
    const float x = job.s * sum;
    odd |= !has_split(x);
    put_terms(x, 1, [&](int e, bf16 v) { row[e * rank + j] = v; });
    if (j == 0)
      for (int e = 6 * rank; e < P; ++e) row[e] = (bf16)0.0f;
  }
  odd = __syncthreads_or(odd);
  if (threadIdx.x == 0) a.odd[kTermBlocks + (int)blockIdx.x] = odd;
#endif
}

// One product Out (+)= alpha U^T W of lowrank_cols: U [T][cols] in the call's
// dtype, W [T][r] fp32; Out [cols][r] or, transposed, [r][cols];
// workgroups first .. first + ceil(cols / 64) - 1.
struct ColsJob {
  const void* u;
  const float* w;
  float* out;
  int cols;
  float alpha;
  int transposed;
  int first;
};
struct ColsJobs {
  ColsJob j[kMaxJobs];
  int n;
};

// Workgroup: 64 columns of one job; wave w reduces a contiguous slice of the
// tokens in steps of 4.  Lane (i, q) loads U[t0 + q][c0 + 4i .. +4]: element
// e feeds tile e, whose row i is column c0 + 4i + e, with W[t0 + q][16 jt +
// i] as the other operand.  The waves' sums are added in order through LDS.
template <typename IO, int NT>
__global__ __launch_bounds__(kLrThreads) void lowrank_cols_kernel(ColsJobs jobs, int T, int rank) {
  constexpr int CH = 8;
  constexpr int kPad = 17;  // LDS row stride: the 4 lane groups fall in different banks
  __shared__ float red[kLrWaves * 64 * kPad];
  int z = 0;
  while (z + 1 < jobs.n && (int)blockIdx.x >= jobs.j[z + 1].first) ++z;
  const ColsJob& job = jobs.j[z];
  const IO* u = static_cast<const IO*>(job.u);
  const float* w = job.w;
  const int cols = job.cols;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int i = lane & 15, q = lane >> 4;
  const int c0 = ((int)blockIdx.x - job.first) * 64;
  const bool col_ok = c0 + 4 * i < cols;  // cols % 4 == 0
  int tb, te;
  share(T, kLrWaves, wave, 4, tb, te);
  f32x4 acc[4][NT];
#pragma unroll
  for (int e = 0; e < 4; ++e)
#pragma unroll
    for (int jt = 0; jt < NT; ++jt) acc[e][jt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  const IO* ucol = u + min(c0 + 4 * i, cols - 4);
  for (int t0 = tb; t0 < te; t0 += 4 * CH) {
    typename Raw4<IO>::T xr[CH];
    float wv[CH][NT];
#pragma unroll
    for (int s = 0; s < CH; ++s) {
      if (t0 + 4 * s >= te) break;  // the wave's slice ends (uniform)
      const int tc = min(t0 + 4 * s + q, T - 1);
      xr[s] = ld_raw4(ucol + (long)tc * cols);
#pragma unroll
      for (int jt = 0; jt < NT; ++jt) wv[s][jt] = w[(long)tc * rank + min(16 * jt + i, rank - 1)];
    }
#pragma unroll
    for (int s = 0; s < CH; ++s) {
      if (t0 + 4 * s >= te) break;
      const bool t_ok = t0 + 4 * s + q < te;
      float x[4];
      sel4(xr[s], t_ok && col_ok, x);
#pragma unroll
      for (int jt = 0; jt < NT; ++jt)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[e][jt] = mma_f32(x[e], wv[s][jt], acc[e][jt]);
    }
  }
  // D of tile (e, jt): lane (i, q), register c holds column c0 + 4 (4q + c) +
  // e, rank 16 jt + i.  One rank tile at a time through LDS.
#pragma unroll
  for (int jt = 0; jt < NT; ++jt) {
    if (jt > 0) __syncthreads();
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int c = 0; c < 4; ++c) red[(wave * 64 + 4 * (4 * q + c) + e) * kPad + i] = acc[e][jt][c];
    __syncthreads();
    for (int idx = threadIdx.x; idx < 64 * 16; idx += kLrThreads) {
      // transposed output: consecutive threads take consecutive columns
      const int cl = job.transposed ? idx % 64 : idx / 16, jl = job.transposed ? idx / 64 : idx % 16;
      float sum = 0.0f;
#pragma unroll
      for (int wv2 = 0; wv2 < kLrWaves; ++wv2) sum += red[(wv2 * 64 + cl) * kPad + jl];
      const int c = c0 + cl, j = 16 * jt + jl;
      if (c < cols && j < rank) {
        float* o = job.transposed ? job.out + (long)j * cols + c : job.out + (long)c * rank + j;
        *o += job.alpha * sum;
      }
    }
  }
}

// One output of lowrank_out: out [T][n] = io(base [T][n] + bias [n] + sum
// over the terms of (s L [T][r]) V), V = B [r][n] (forward) or A^T with A
// [n][r] (dX); workgroups first .. first + ceil(T / 16) ceil(n / 256) - 1.
struct OutJob {
  const float* base;
  const float* bias;  // or null
  void* out;
  int n;
  int n_terms;
  int first;
  const float* l[kMaxProj];
  const float* v[kMaxProj];
  float s[kMaxProj];
};
struct OutJobs {
  OutJob j[kMaxProj];
  int n;
};

// Workgroup: 16 tokens x 256 columns of one output, wave w the columns 64w..
// of those.  Lane (i, q) owns columns col = n0 + 4i .. +4: tile e's column i
// is n0 + 4i + e, so that register c of the 4 tiles holds out[t0 + 4q +
// c][col .. col + 4].  In MFMA step m of a group of 16 ranks m0.., the
// reduction index q is rank m0 + 4q + m: a lane's 4 ranks are consecutive,
// one 16-byte load of L, and of A (dX) or of each row of B (forward), when
// r % 4 == 0 (VEC).
template <typename IO, bool AT, bool VEC>
__global__ __launch_bounds__(kOutThreads) void lowrank_out_kernel(OutJobs jobs, int T, int rank) {
  int z = 0;
  while (z + 1 < jobs.n && (int)blockIdx.x >= jobs.j[z + 1].first) ++z;
  const OutJob& job = jobs.j[z];
  const int n = job.n;
  const int b = (int)blockIdx.x - job.first, ncb = (n + 255) / 256;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int i = lane & 15, q = lane >> 4;
  const int t0 = (b / ncb) * 16, col = (b % ncb) * 256 + 64 * wave + 4 * i;
  const bool col_ok = col < n;  // n % 4 == 0
  const int colc = min(col, n - 4);
  f32x4 base[4];
#pragma unroll
  for (int c = 0; c < 4; ++c)
    base[c] = *reinterpret_cast<const f32x4*>(job.base + (long)min(t0 + 4 * q + c, T - 1) * n + colc);
  f32x4 acc[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) acc[e] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  const bool row_ok = t0 + i < T;
  for (int term = 0; term < job.n_terms; ++term) {
    const float* L = job.l[term] + (long)min(t0 + i, T - 1) * rank;
    const float* V = job.v[term];
    const float s = job.s[term];
    for (int m0 = 0; m0 < rank; m0 += 16) {
      const int jb = m0 + 4 * q;  // this lane's ranks jb .. jb + 3
      float a[4], bv[4][4];       // a[m] = L[t][jb + m], bv[m][e] = V(jb + m, col + e)
      if constexpr (VEC) {  // r % 4 == 0
        const int jc = min(jb, rank - 4);
        load4(L + jc, a);
        if constexpr (AT) {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            float r4[4];
            load4(V + (long)(colc + e) * rank + jc, r4);
#pragma unroll
            for (int m = 0; m < 4; ++m) bv[m][e] = r4[m];
          }
        } else {
#pragma unroll
          for (int m = 0; m < 4; ++m) load4(V + (long)(jc + m) * n + colc, bv[m]);
        }
      } else {
#pragma unroll
        for (int m = 0; m < 4; ++m) {
          const int j = min(jb + m, rank - 1);
          a[m] = L[j];
#pragma unroll
          for (int e = 0; e < 4; ++e) bv[m][e] = AT ? V[(long)(colc + e) * rank + j] : V[(long)j * n + colc + e];
        }
      }
#pragma unroll
      for (int m = 0; m < 4; ++m) a[m] = jb + m < rank && row_ok ? s * a[m] : 0.0f;
#pragma unroll
      for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[e] = mma_f32(a[m], bv[m][e], acc[e]);
    }
  }
  if (!col_ok) return;
  f32x4 bias = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  if (job.bias != nullptr) {
#pragma unroll
    for (int e = 0; e < 4; ++e) bias[e] = job.bias[col + e];
  }
  IO* out = static_cast<IO*>(job.out);
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const int t = t0 + 4 * q + c;
    if (t >= T) continue;
    f32x4 y;
#pragma unroll
    for (int e = 0; e < 4; ++e) y[e] = base[c][e] + bias[e] + acc[e][c];
    store4(out + (long)t * n + col, y);
  }
}

unsigned blocks(long n, int per) { return static_cast<unsigned>((n + per - 1) / per); }

// The low-rank products X A_p / dY_p B_p^T of a call: which are needed, and
// where their results go (slot z of ProjLaunch::lowrank, [T][r] each).
struct RowsPlan {
  RowsJobs jobs{};
  int n = 0, kmax = 0;
  int slot_l[kMaxProj], slot_dl[kMaxProj];  // -1: not computed
};

RowsPlan rows_plan(const ProjLaunch& a, bool backward) {
  RowsPlan plan;
  for (int p = 0; p < a.n_proj; ++p) {
    const ProjSpec& s = a.p[p];
    plan.slot_l[p] = plan.slot_dl[p] = -1;
    if (s.a == nullptr) continue;
    if (backward) {
      plan.slot_dl[p] = plan.n;
      plan.jobs.j[plan.n++] = RowsJob{s.dy, s.b, s.out, 1};
      plan.kmax = std::max(plan.kmax, s.out);
    }
    if (!backward || s.grad_b != nullptr) {
      plan.slot_l[p] = plan.n;
      plan.jobs.j[plan.n++] = RowsJob{a.x, s.a, a.in, 0};
      plan.kmax = std::max(plan.kmax, a.in);
    }
  }
  return plan;
}

// Workgroups splitting each reduction of lowrank_rows: about 512 workgroups
// in all, at least 128 reduction elements per split.
int rows_splits(const ProjLaunch& a, const RowsPlan& plan) {
  const int slabs = (a.T + 15) / 16, per = std::max(1, slabs * plan.n);
  return std::max(1, std::min({(512 + per - 1) / per, plan.kmax / 128, 16}));
}

template <typename IO>
hipError_t run_rows(const ProjLaunch& a, const RowsPlan& plan, hipStream_t st) {
  if (plan.n == 0) return hipSuccess;
  const int slabs = (a.T + 15) / 16, splits = rows_splits(a, plan), nt = (a.rank + 15) / 16;
  const dim3 grid(slabs, splits, plan.n), block(kLrThreads);
  switch (nt) {
#define GL_ROWS(NT) \
  hipLaunchKernelGGL((lowrank_rows_kernel<IO, NT>), grid, block, 0, st, plan.jobs, a.T, a.rank, a.part)
    case 1: GL_ROWS(1); break;
    case 2: GL_ROWS(2); break;
    case 3: GL_ROWS(3); break;
    case 4: GL_ROWS(4); break;
#undef GL_ROWS
    default: return hipErrorInvalidValue;
  }
  GL_CHECK(hipGetLastError());
  const long n = (long)plan.n * a.T * a.rank;
  hipLaunchKernelGGL(lowrank_reduce_kernel, dim3(blocks(n, 256)), dim3(256), 0, st, a.part,
                     a.lowrank, plan.n, splits, slabs, 16 * nt, a.T, a.rank);
  return hipGetLastError();
}

template <typename IO, bool AT>
hipError_t run_out(const ProjLaunch& a, OutJobs& jobs, hipStream_t st) {
  int total = 0;
  for (int z = 0; z < jobs.n; ++z) {
    jobs.j[z].first = total;
    total += ((a.T + 15) / 16) * ((jobs.j[z].n + 255) / 256);
  }
  if (a.rank % 4 == 0)
    hipLaunchKernelGGL((lowrank_out_kernel<IO, AT, true>), dim3(total), dim3(kOutThreads), 0, st,
                       jobs, a.T, a.rank);
  else
    hipLaunchKernelGGL((lowrank_out_kernel<IO, AT, false>), dim3(total), dim3(kOutThreads), 0, st,
                       jobs, a.T, a.rank);
  return hipGetLastError();
}

float* slot(const ProjLaunch& a, int z) { return a.lowrank + (long)z * a.T * a.rank; }

// Row blocks (of 16) per lowrank_split workgroup: V is read once per
// workgroup, U once per job, so taller slabs save V's reads while the
// launch still fills the CUs.
int split_row_blocks(int T, int jobs, int nt) {
  if (nt <= 2 && (T + 63) / 64 * jobs >= 128) return 4;
  if ((T + 31) / 32 * jobs >= 128) return 2;
  return 1;
}

// Calls whose tensors the fused GEMM (proj_gemm.hip) takes: bf16, whole
// 16-byte pieces in every row, 16-byte aligned tensors.  The others (fp32
// tensors, widths that are multiples of 4 only) form the base products in
// fp32 and add the rest in lowrank_out.
bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }
bool fused(const ProjLaunch& a, bool backward) {
  if (!a.io_bf16 || a.in % 8 != 0 || !aligned16(a.x) || (backward && !aligned16(a.dx))) return false;
  for (int p = 0; p < a.n_proj; ++p)
    if (a.p[p].out % 8 != 0 || !aligned16(a.p[p].w) || !aligned16(backward ? a.p[p].dy : a.p[p].y)) return false;
  return true;
}

hipError_t run_cols_any(const ProjLaunch& a, const RowsPlan& plan, hipStream_t st);

// The fused form: the low-rank products and the split terms, then (backward)
// the adapters' gradients, then one GEMM launch for everything else.
hipError_t fused_impl(const ProjLaunch& a, bool backward, hipStream_t st) {
  const RowsPlan plan = rows_plan(a, backward);
  const int P = term_pitch(a.rank), nt = (a.rank + 15) / 16;
  GemmCall g{};
  g.dx = a.dx;
  g.T = a.T;
  g.K = a.in;
  g.rank = a.rank;
  g.n = a.n_proj;
  bf16* vt = static_cast<bf16*>(a.terms);  // the adapters' terms, one after another
  bf16* lt = vt;                           // then those of s L, [T][P] each
  for (int p = 0; p < a.n_proj; ++p)
    if (a.p[p].a != nullptr) lt += (long)P * (backward ? a.in : a.p[p].out);
  SplitCall c{};
  c.across = backward;
  c.odd = a.odd;
  for (int p = 0; p < a.n_proj; ++p) {
    const ProjSpec& s = a.p[p];
    g.j[p] = GemmJob{s.y, s.bias, nullptr, nullptr, s.scaling, s.out, 0};
    g.seg[p] = GemmSeg{s.w, backward ? s.dy : a.x, backward ? s.out : a.in};
    const int slot_l = backward ? plan.slot_dl[p] : plan.slot_l[p];
    if (slot_l < 0) continue;
    g.j[p].l = slot(a, slot_l);
    g.j[p].v = backward ? s.a : s.b;
    g.seg[kMaxProj + p] = GemmSeg{vt, lt, P};
    const int n = backward ? a.in : s.out;
    c.v[c.nv++] = TermJob{g.j[p].v, vt, n};
    const RowsJob& r = plan.jobs.j[slot_l];
    c.j[slot_l] = SplitJob{r.u, r.v, slot(a, slot_l), lt, s.scaling, r.K, r.vt};
    vt += (long)P * n;
    lt += (long)a.T * P;
  }
  if (backward)
    for (int p = 0; p < a.n_proj; ++p)
      if (const int z = plan.slot_l[p]; z >= 0) {
        const RowsJob& r = plan.jobs.j[z];
        c.j[z] = SplitJob{r.u, r.v, slot(a, z), nullptr, 0.0f, r.K, r.vt};
      }
  c.n = plan.n;
  if (plan.n > 0) {
    const int rb = split_row_blocks(a.T, plan.n, nt);
    c.slabs = (a.T + 16 * rb - 1) / (16 * rb);
    const dim3 grid(c.n * c.slabs + kTermBlocks), block(64 * split_waves(nt, rb));
    switch (8 * rb + nt) {
#define GL_SPLIT(RB, NT)                                                                                \
  case 8 * RB + NT:                                                                                     \
    hipLaunchKernelGGL((lowrank_split_kernel<NT, RB>), grid, block, 0, st, c, a.T, a.rank); \
    break;
      GL_SPLIT(1, 1) GL_SPLIT(1, 2) GL_SPLIT(1, 3) GL_SPLIT(1, 4)
      GL_SPLIT(2, 1) GL_SPLIT(2, 2) GL_SPLIT(2, 3) GL_SPLIT(2, 4)
      GL_SPLIT(4, 1) GL_SPLIT(4, 2)
#undef GL_SPLIT
      default: return hipErrorInvalidValue;
    }
    GL_CHECK(hipGetLastError());
    g.odd = a.odd;
    g.n_odd = kTermBlocks + c.n * c.slabs;
  }
  if (backward) GL_CHECK(run_cols_any(a, plan, st));
  return launch_gemm(g, backward, st);
}

template <typename IO>
hipError_t forward_impl(const ProjLaunch& a, hipStream_t st) {
  long off = 0;
  OutJobs out{};
  out.n = a.n_proj;
  for (int p = 0; p < a.n_proj; ++p) {
    const ProjSpec& s = a.p[p];
    out.j[p] = OutJob{a.yf + off, s.bias, s.y, s.out, 0, 0, {}, {}, {}};
    // Yf_p = X W_p^T
    GL_CHECK(launch_generic_fwd(WideFwd{a.x, s.w, a.yf + off, a.T, a.in, s.out}, a.io_bf16, st));
    off += (long)a.T * s.out;
  }
  const RowsPlan plan = rows_plan(a, false);
  GL_CHECK(run_rows<IO>(a, plan, st));  // L_p = X A_p
  for (int p = 0; p < a.n_proj; ++p) {
    if (plan.slot_l[p] < 0) continue;
    OutJob& o = out.j[p];
    o.n_terms = 1;
    o.l[0] = slot(a, plan.slot_l[p]);
    o.v[0] = a.p[p].b;
    o.s[0] = a.p[p].scaling;
  }
  return run_out<IO, false>(a, out, st);  // Y_p = io(Yf_p + bias_p + (s L_p) B_p)
}

// grad_A_p += s X^T dL_p;  grad_B_p += s L_p^T dY_p
template <typename IO>
hipError_t run_cols(const ProjLaunch& a, const RowsPlan& plan, hipStream_t st) {
  ColsJobs cj{};
  int total = 0;
  for (int p = 0; p < a.n_proj; ++p) {
    const ProjSpec& s = a.p[p];
    if (s.a == nullptr) continue;
    if (s.grad_a != nullptr) {
      cj.j[cj.n++] = ColsJob{a.x, slot(a, plan.slot_dl[p]), s.grad_a, a.in, s.scaling, 0, total};
      total += (a.in + 63) / 64;
    }
    if (s.grad_b != nullptr) {
      cj.j[cj.n++] = ColsJob{s.dy, slot(a, plan.slot_l[p]), s.grad_b, s.out, s.scaling, 1, total};
      total += (s.out + 63) / 64;
    }
  }
  if (cj.n > 0) {
    switch ((a.rank + 15) / 16) {
#define GL_COLS(NT) \
  hipLaunchKernelGGL((lowrank_cols_kernel<IO, NT>), dim3(total), dim3(kLrThreads), 0, st, cj, a.T, a.rank)
      case 1: GL_COLS(1); break;
      case 2: GL_COLS(2); break;
      case 3: GL_COLS(3); break;
      case 4: GL_COLS(4); break;
#undef GL_COLS
      default: return hipErrorInvalidValue;
    }
    GL_CHECK(hipGetLastError());
  }
  return hipSuccess;
}

hipError_t run_cols_any(const ProjLaunch& a, const RowsPlan& plan, hipStream_t st) {
  return a.io_bf16 ? run_cols<bf16>(a, plan, st) : run_cols<float>(a, plan, st);
}

template <typename IO>
hipError_t backward_impl(const ProjLaunch& a, hipStream_t st) {
  // dXf = sum_p dY_p W_p in one launch
  WideBwd gb{};
  gb.c = a.dxf;
  gb.T = a.T;
  gb.K = a.in;
  for (int p = 0; p < a.n_proj; ++p) gb.j[gb.n++] = WideJob{a.p[p].w, a.p[p].dy, a.p[p].out};
  GL_CHECK(launch_generic_bwd(gb, a.io_bf16, st));
  // dL_p = dY_p B_p^T, and L_p = X A_p where grad_B_p is wanted
  const RowsPlan plan = rows_plan(a, true);
  GL_CHECK(run_rows<IO>(a, plan, st));
  GL_CHECK(run_cols<IO>(a, plan, st));
  // dX = io(dXf + sum_p (s dL_p) A_p^T)
  OutJobs out{};
  out.n = 1;
  OutJob& o = out.j[0];
  o = OutJob{a.dxf, nullptr, a.dx, a.in, 0, 0, {}, {}, {}};
  for (int p = 0; p < a.n_proj; ++p) {
    if (plan.slot_dl[p] < 0) continue;
    o.l[o.n_terms] = slot(a, plan.slot_dl[p]);
    o.v[o.n_terms] = a.p[p].a;
    o.s[o.n_terms] = a.p[p].scaling;
    ++o.n_terms;
  }
  return run_out<IO, true>(a, out, st);
}

}  // namespace

ProjScratchNeed proj_scratch_need(const ProjLaunch& a, bool backward) {
  ProjScratchNeed need{};
  const bool f = fused(a, backward);
  if (!f && backward) need.dxf = (long)a.T * a.in;
  if (!f && !backward)
    for (int p = 0; p < a.n_proj; ++p) need.yf += (long)a.T * a.p[p].out;
  const RowsPlan plan = rows_plan(a, backward);
  if (plan.n > 0) {
    need.lowrank = (long)plan.n * a.T * a.rank;
    if (f) {
      need.odd = kTermBlocks + (long)plan.n * ((a.T + 15) / 16);
      for (int p = 0; p < a.n_proj; ++p)
        if (a.p[p].a != nullptr)
          need.terms += (long)term_pitch(a.rank) * (a.T + (backward ? a.in : a.p[p].out));
    } else {
      const long slabs = (a.T + 15) / 16, nt = (a.rank + 15) / 16;
      need.part = (long)plan.n * rows_splits(a, plan) * slabs * 256 * nt;
    }
  }
  return need;
}

hipError_t launch_proj_forward(const ProjLaunch& a, hipStream_t st) {
  if (fused(a, false)) return fused_impl(a, false, st);
  return a.io_bf16 ? forward_impl<bf16>(a, st) : forward_impl<float>(a, st);
}

hipError_t launch_proj_backward(const ProjLaunch& a, hipStream_t st) {
  if (fused(a, true)) return fused_impl(a, true, st);
  return a.io_bf16 ? backward_impl<bf16>(a, st) : backward_impl<float>(a, st);
}

}  // namespace glacier
