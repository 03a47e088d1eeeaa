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
// Two launches forward, three backward:
//   lowrank_split   L = X A_p and dL = dY_p B_p^T; for bf16 tensors in whole
//                   16-byte pieces also the split terms (split3.hpp) of s L and of
//                   the adapters
//   lowrank_cols    backward: grad_A += s X^T dL, grad_B += s L^T dY (reduction
//                   over the tokens): 64-column slabs, tokens split over 8 waves
//   proj_gemm       (proj_gemm.hip) Y_p = X W_p^T + bias_p + (s L_p) B_p for
//                   every projection, or dX = sum_p dY_p W_p + (s dL_p) A_p^T:
//                   by DMA for such bf16 tensors, else (fp32 tensors, widths that
//                   are multiples of 4 only, unaligned weights) with every
//                   operand split as it is loaded
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
constexpr int kMaxJobs = 2 * kMaxProj;

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
[[maybe_unused]] __device__ inline float raw_at(float4 r, int e) { return e == 0 ? r.x : e == 1 ? r.y : e == 2 ? r.z : r.w; }
[[maybe_unused]] __device__ inline bf16 raw_at(bf16x4 r, int e) { return r[e]; }
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

// One product L [T][r] = U [T][K] V: V = A [K][r] (vt 0) or B^T with B
// [r][K] (vt 1); U in the call's dtype.
struct RowsJob {
  const void* u;
  const float* v;
  int K;
  int vt;
};
struct RowsJobs {
  RowsJob j[kMaxJobs];
};

// ---- the low-rank products and their split terms ------------------------
// L [T][r] = U [T][K] V for each job (V as in RowsJob) on bf16 MFMAs, V (and U,
// for fp32 tensors) in three terms (split3.hpp): the sums are fp32, at 3/16 of
// the fp32 MFMA's time (6/16 for fp32 tensors).  The results
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
  const void* u;  // [T][K]
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
  int groups;  // rank groups of a slab
  int* odd;    // [kTermBlocks], then [groups][n][slabs]: a value without split
               // terms among what that workgroup wrote; null: no terms are written
};

// The six entries of a terms row for x: side 0 the adapters', side 1 (s L).
// True if x has no split (split3.hpp): the entries are then meaningless.
template <typename Put>
__device__ inline bool put_terms(float x, int side, Put&& put) {
  const bf16 h = (bf16)x;
  const float r1 = x - (float)h;
  const bf16 m = (bf16)r1;
  const float r2 = r1 - (float)m;
  const bf16 l = (bf16)r2;
  put(0, h);
  put(1, side ? m : h);
  put(2, side ? h : m);
  put(3, m);
  put(4, side ? l : h);
  put(5, side ? h : l);
  const unsigned left = __float_as_uint(r2);
  return (left & 0xffffu) != 0 || (left & 0x7f800000u) == 0x7f800000u;
}

// Workgroups for the adapters' terms: 32 took up to 21% longer a call (16 tokens,
// 3584 -> 3584/512/512 at rank 64), 128 from 3% less to 5% more.
constexpr int kTermBlocks = 64;
// Waves of a lowrank_split workgroup.  16 where a workgroup has one tile: its
// registers let all run at once, and with 8 a forward of 3584 inputs took 2-5%
// longer (a backward of 896 inputs 6% less).
constexpr int split_waves(int nt, int rb) { return rb == 1 && nt == 1 ? 16 : 8; }

#if defined(__HIP_DEVICE_COMPILE__)
// The k range [kb, ke) of one wave of lowrank_split_kernel, added into acc and,
// the products of lower terms, into small (so that acc rounds once a step).
// Steps of 32: lane (i, q) holds U[row i][k0 + 8q .. +7] and V[k0 + 8q ..
// +7][j0 + 16 jt + i].  Lengths are multiples of 4 (of 8 with WIDE), so each half
// of a lane's 8 is all in or all out; out of range V is zeroed, U clamped
// (and, where a step goes the fp32 way, zeroed as well).
template <typename IO, bool WIDE, int NT, int RB, bool VT>
__device__ inline void split_accumulate(const IO* const (&u)[RB], const float* __restrict__ v0, int K,
                                        int rank, int j0, int kb, int ke, f32x4 (&acc)[RB][NT],
                                        f32x4 (&small)[RB][NT]) {
  const int lane = threadIdx.x & 63, i = lane & 15, q = lane >> 4;
  constexpr bool kF32 = sizeof(IO) == 4;
  constexpr int W = NT * RB * (kF32 ? 2 : 1);
  // steps whose loads are issued together (fp32 at one tile: four would spill
  // beside the 16 waves)
  constexpr int CH = W <= 2 && !kF32 ? 4 : W <= 8 ? 2 : 1;
  for (int k0 = kb; k0 < ke; k0 += 32 * CH) {
    typename Raw4<IO>::T ur[CH][RB][2];
    float vr[CH][NT][8];
#pragma unroll
    for (int s = 0; s < CH; ++s) {
      const int k = k0 + 32 * s + 8 * q;
      const int kc[2] = {WIDE ? min(k, K - 8) : min(k, K - 4), WIDE ? min(k, K - 8) + 4 : min(k + 4, K - 4)};
#pragma unroll
      for (int b = 0; b < RB; ++b)
#pragma unroll
        for (int h = 0; h < 2; ++h) ur[s][b][h] = ld_raw4(u[b] + kc[h]);
#pragma unroll
      for (int jt = 0; jt < NT; ++jt) {
        const int jc = min(j0 + 16 * jt + i, rank - 1);
#pragma unroll
        for (int e = 0; e < 8; e += VT ? 4 : 1) {
          const int kk = kc[e / 4] + e % 4;
          if constexpr (VT) {
            const float4 r = *reinterpret_cast<const float4*>(v0 + (long)jc * K + kk);
            vr[s][jt][e] = r.x, vr[s][jt][e + 1] = r.y, vr[s][jt][e + 2] = r.z, vr[s][jt][e + 3] = r.w;
          } else {
            vr[s][jt][e] = v0[(long)kk * rank + jc];
          }
        }
      }
    }
#pragma unroll
    for (int s = 0; s < CH; ++s) {
      if (k0 + 32 * s >= ke) break;
      const int k = k0 + 32 * s + 8 * q;
      const bool ok[2] = {k < ke, k + 4 < ke};
      float x[RB][8];
      Split3 us[kF32 ? RB : 1];
      bf16x8 ub[RB];
      bool odd_u = false;
#pragma unroll
      for (int b = 0; b < RB; ++b) {
        SplitMarks mark;  // bf16: NaN once an element is not finite
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          x[b][e] = (float)raw_at(ur[s][b][e / 4], e % 4);
          if constexpr (!kF32) {
            ub[b][e] = (bf16)x[b][e];
            mark.sum += 0.0f * x[b][e];
          }
        }
        if constexpr (kF32) us[b].set(x[b], mark);
        odd_u |= mark.bad();
      }
#pragma unroll
      for (int jt = 0; jt < NT; ++jt) {
#pragma unroll
        for (int e = 0; e < 8; ++e) vr[s][jt][e] = ok[e / 4] ? vr[s][jt][e] : 0.0f;
        Split3 v;
        SplitMarks mark;
        v.set(vr[s][jt], mark);
        if (__any(mark.bad() || odd_u)) {
#pragma unroll
          for (int b = 0; b < RB; ++b)
#pragma unroll
            for (int e = 0; e < 8; ++e)
              acc[b][jt] = mma_f32(ok[e / 4] ? x[b][e] : 0.0f, vr[s][jt][e], acc[b][jt]);
        } else {
#pragma unroll
          for (int b = 0; b < RB; ++b) {
            if constexpr (kF32) {
              small[b][jt] = Mfma<bf16>::mma(us[b].l, v.h, small[b][jt]);
              small[b][jt] = Mfma<bf16>::mma(us[b].h, v.l, small[b][jt]);
              small[b][jt] = Mfma<bf16>::mma(us[b].m, v.m, small[b][jt]);
              small[b][jt] = Mfma<bf16>::mma(us[b].m, v.h, small[b][jt]);
              small[b][jt] = Mfma<bf16>::mma(us[b].h, v.m, small[b][jt]);
              acc[b][jt] = Mfma<bf16>::mma(us[b].h, v.h, acc[b][jt]);
            } else {
              small[b][jt] = Mfma<bf16>::mma(ub[b], v.l, small[b][jt]);
              small[b][jt] = Mfma<bf16>::mma(ub[b], v.m, small[b][jt]);
              acc[b][jt] = Mfma<bf16>::mma(ub[b], v.h, acc[b][jt]);
            }
          }
        }
      }
    }
  }
}
#endif

template <typename IO, bool WIDE, int NT, int RB>
__global__ __launch_bounds__(64 * split_waves(NT, RB)) void lowrank_split_kernel(const SplitCall a, int T,
                                                                             int rank) {
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr int W = split_waves(NT, RB);  // waves, splitting K
  constexpr int kRow = 16 * NT + 1;
  __shared__ float red[W * 16 * RB * kRow];
  const int P = term_pitch(rank);
  bool odd = false;
  const int rows_blocks = a.groups * a.n * a.slabs;
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
        for (int m = 0; m < 4; ++m) odd |= put_terms(x[m], 0, [&](int e, bf16 t) { t4[e][m] = t; });
#pragma unroll
        for (int e = 0; e < 6; ++e) *reinterpret_cast<bf16x4*>(out + (long)f * P + e * rank + j0) = t4[e];
      } else {
#pragma unroll
        for (int m = 0; m < 4; ++m) {
          if (j0 + m >= rank) break;
          odd |= put_terms(x[m], 0, [&](int e, bf16 t) {
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
  const int slab = (int)blockIdx.x % a.slabs, z = (int)blockIdx.x / a.slabs % a.n;
  const int j0 = 16 * NT * ((int)blockIdx.x / (a.slabs * a.n));  // the workgroup's ranks from j0
  const SplitJob& job = a.j[z];
  const int K = job.K;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int i = lane & 15, q = lane >> 4;
  const int t0 = slab * 16 * RB;
  const IO* u[RB];
#pragma unroll
  for (int b = 0; b < RB; ++b)
    u[b] = static_cast<const IO*>(job.u) + (long)min(t0 + 16 * b + i, T - 1) * K;
  int kb, ke;
  share(K, W, wave, 32, kb, ke);
  f32x4 acc[RB][NT], small[RB][NT];
#pragma unroll
  for (int b = 0; b < RB; ++b)
#pragma unroll
    for (int jt = 0; jt < NT; ++jt) acc[b][jt] = small[b][jt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  if (job.vt)
    split_accumulate<IO, WIDE, NT, RB, true>(u, job.v, K, rank, j0, kb, ke, acc, small);
  else
    split_accumulate<IO, WIDE, NT, RB, false>(u, job.v, K, rank, j0, kb, ke, acc, small);
  // D of (b, jt): lane (i, q), register c holds row 16 b + 4q + c, column j0 + 16 jt + i
#pragma unroll
  for (int b = 0; b < RB; ++b)
#pragma unroll
    for (int jt = 0; jt < NT; ++jt)
#pragma unroll
      for (int c = 0; c < 4; ++c)
        red[(wave * 16 * RB + 16 * b + 4 * q + c) * kRow + 16 * jt + i] = acc[b][jt][c] + small[b][jt][c];
  __syncthreads();
  for (int idx = threadIdx.x; idx < 16 * RB * 16 * NT; idx += 64 * W) {
    const int r = idx / (16 * NT), jl = idx % (16 * NT), j = j0 + jl, t = t0 + r;
    if (t >= T || j >= rank) continue;
    float sum = 0.0f;
#pragma unroll
    for (int w = 0; w < W; ++w) sum += red[(w * 16 * RB + r) * kRow + jl];
    job.l[(long)t * rank + j] = sum;
    if (job.terms == nullptr) continue;
    bf16* row = static_cast<bf16*>(job.terms) + (long)t * P;
    odd |= put_terms(job.s * sum, 1, [&](int e, bf16 v) { row[e * rank + j] = v; });
    if (j == 0)
      for (int e = 6 * rank; e < P; ++e) row[e] = (bf16)0.0f;
  }
  if (a.odd == nullptr) return;
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

// The low-rank products X A_p / dY_p B_p^T of a call: which are needed, and
// where their results go (slot z of ProjLaunch::lowrank, [T][r] each).
struct RowsPlan {
  RowsJobs jobs{};
  int n = 0;
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
    }
    if (!backward || s.grad_b != nullptr) {
      plan.slot_l[p] = plan.n;
      plan.jobs.j[plan.n++] = RowsJob{a.x, s.a, a.in, 0};
    }
  }
  return plan;
}

float* slot(const ProjLaunch& a, int z) { return a.lowrank + (long)z * a.T * a.rank; }

// Row blocks (of 16) per lowrank_split workgroup: V is read once per
// workgroup, U once per job, so taller slabs save V's reads while the
// launch still fills half of the CUs.  Two blocks only from 256 slabs on took up to
// 1.55 times as long a call where they start at 128 (2100 tokens), never at rank
// 64 1.05-1.16 times; without four blocks bf16 forwards at rank 16 and 32 took
// 1.03-1.15 times from 3000 tokens on.
template <typename IO, bool WIDE>
int split_row_blocks(int T, int jobs, int nt) {
  if (sizeof(IO) == 2 && WIDE && nt <= 2 && (T + 63) / 64 * jobs >= 128) return 4;
  if ((T + 31) / 32 * jobs >= 128) return 2;
  return 1;
}

// Rank tiles (of 16) per workgroup of a launch of `slabs` single-block slabs: as
// few as leave one workgroup a CU.  A workgroup reads its V columns whole, so a
// tile of its own costs only U again, and splits K over 16 waves.  Calls at rank
// 64, all four tiles in one workgroup before: 16 x 3584 -> 3584 bf16 47.3 + 56.5 ->
// 30.4 + 39.6 us, 512 tokens 54.7 + 77.3 -> 39.0 + 62.8.  Two or four workgroups a
// CU allowed: up to 1.21 and 1.30 times as long.
int rank_tiles(int slabs, int tiles) {
  for (int nt : {1, 2})
    if (slabs * ((tiles + nt - 1) / nt) <= 256) return nt;
  return 4;
}

// Every row of bf16 x and dY in whole 16-byte pieces.
bool eights(const ProjLaunch& a) {
  bool ok = a.in % 8 == 0;
  for (int p = 0; p < a.n_proj; ++p) ok = ok && a.p[p].out % 8 == 0;
  return ok;
}
bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }
// Calls whose tensors the DMA of proj_gemm takes as they are: bf16, whole
// 16-byte pieces in every row, 16-byte aligned tensors.
bool whole_pieces(const ProjLaunch& a, bool backward) {
  if (!a.io_bf16 || !eights(a) || !aligned16(a.x) || (backward && !aligned16(a.dx))) return false;
  for (int p = 0; p < a.n_proj; ++p)
    if (!aligned16(a.p[p].w) || !aligned16(backward ? a.p[p].dy : a.p[p].y)) return false;
  return true;
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

template <typename IO, bool WIDE>
hipError_t launch_lowrank(const ProjLaunch& a, SplitCall& c, hipStream_t st) {
  const int tiles = (a.rank + 15) / 16, rb = split_row_blocks<IO, WIDE>(a.T, c.n, tiles);
  c.slabs = (a.T + 16 * rb - 1) / (16 * rb);
  const int nt = rb == 1 ? rank_tiles(c.slabs * c.n, tiles) : tiles;
  c.groups = (tiles + nt - 1) / nt;
  const dim3 grid(c.groups * c.n * c.slabs + (c.nv > 0 ? kTermBlocks : 0)), block(64 * split_waves(nt, rb));
  switch (8 * rb + nt) {
#define GL_SPLIT(RB, NT)                                                                             \
  case 8 * RB + NT:                                                                                  \
    hipLaunchKernelGGL((lowrank_split_kernel<IO, WIDE, NT, RB>), grid, block, 0, st, c, a.T, a.rank); \
    break;
    GL_SPLIT(1, 1) GL_SPLIT(1, 2) GL_SPLIT(1, 4)
    GL_SPLIT(2, 1) GL_SPLIT(2, 2) GL_SPLIT(2, 3) GL_SPLIT(2, 4)
    default:
      if constexpr (sizeof(IO) == 2 && WIDE) {
        switch (8 * rb + nt) {
          GL_SPLIT(4, 1) GL_SPLIT(4, 2)
          default: return hipErrorInvalidValue;
        }
        break;
      }
      return hipErrorInvalidValue;
#undef GL_SPLIT
  }
  return hipGetLastError();
}

// Whether output p of the call (forward: y_p; backward: dX, p 0) shares memory
// with what its GEMM launch reads while it writes: x or every dY, and the W.
bool in_place(const ProjLaunch& a, bool backward, int p) {
  const size_t esz = a.io_bf16 ? 2 : 4;
  const uintptr_t out = reinterpret_cast<uintptr_t>(backward ? a.dx : a.p[p].y);
  const size_t out_bytes = (size_t)a.T * (backward ? a.in : a.p[p].out) * esz;
  auto shares = [&](const void* q, size_t n) {
    const uintptr_t at = reinterpret_cast<uintptr_t>(q);
    return at < out + out_bytes && out < at + n * esz;
  };
  bool any = !backward && shares(a.x, (size_t)a.T * a.in);
  for (int i = 0; i < a.n_proj; ++i)
    any = any || shares(a.p[i].w, (size_t)a.p[i].out * a.in) ||
          (backward && shares(a.p[i].dy, (size_t)a.T * a.p[i].out));
  return any;
}
// Bytes of output p in ProjLaunch::shadow: none unless in_place.
size_t shadow_bytes(const ProjLaunch& a, bool backward, int p) {
  if (!in_place(a, backward, p)) return 0;
  const size_t n = (size_t)a.T * (backward ? a.in : a.p[p].out) * (a.io_bf16 ? 2 : 4);
  return (n + 15) / 16 * 16;
}

// A call: the low-rank products (and split terms), then (backward) the
// adapters' gradients, then one GEMM launch for everything else.
hipError_t run_call(const ProjLaunch& a, bool backward, hipStream_t st) {
  const bool whole = whole_pieces(a, backward);
  const RowsPlan plan = rows_plan(a, backward);
  const int P = term_pitch(a.rank);
  GemmCall g{};
  // the outputs, or where the launch writes them instead
  const int n_out = backward ? 1 : a.n_proj;
  void* to[kMaxProj];
  size_t shadowed[kMaxProj], at = 0;
  for (int p = 0; p < n_out; ++p) {
    shadowed[p] = shadow_bytes(a, backward, p);
    to[p] = shadowed[p] > 0 ? static_cast<char*>(a.shadow) + at : backward ? a.dx : a.p[p].y;
    at += shadowed[p];
  }
  g.dx = backward ? to[0] : nullptr;
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
  c.odd = whole ? a.odd : nullptr;
  for (int p = 0; p < a.n_proj; ++p) {
    const ProjSpec& s = a.p[p];
    g.j[p] = GemmJob{backward ? nullptr : to[p], s.bias, nullptr, nullptr, s.scaling, s.out, 0};
    g.seg[p] = GemmSeg{s.w, backward ? s.dy : a.x, backward ? s.out : a.in};
    const int slot_l = backward ? plan.slot_dl[p] : plan.slot_l[p];
    if (slot_l < 0) continue;
    g.j[p].l = slot(a, slot_l);
    g.j[p].v = backward ? s.a : s.b;
    g.seg[kMaxProj + p] = GemmSeg{vt, lt, P};
    const int n = backward ? a.in : s.out;
    c.v[c.nv++] = TermJob{g.j[p].v, vt, n};
    const RowsJob& r = plan.jobs.j[slot_l];
    c.j[slot_l] = SplitJob{r.u, r.v, slot(a, slot_l), whole ? lt : nullptr, s.scaling, r.K, r.vt};
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
    if (!whole) c.nv = 0;
    if (!a.io_bf16)
      GL_CHECK((launch_lowrank<float, false>(a, c, st)));
    else if (eights(a))
      GL_CHECK((launch_lowrank<bf16, true>(a, c, st)));
    else
      GL_CHECK((launch_lowrank<bf16, false>(a, c, st)));
    g.odd = c.odd;
    g.n_odd = whole ? kTermBlocks + c.groups * c.n * c.slabs : 0;
  }
  if (backward) GL_CHECK(run_cols_any(a, plan, st));
  GL_CHECK(whole ? launch_gemm(g, backward, st) : launch_gemm_split(g, backward, a.io_bf16, st));
  for (int p = 0; p < n_out; ++p)
    if (shadowed[p] > 0)
      GL_CHECK(hipMemcpyAsync(backward ? a.dx : a.p[p].y, to[p],
                              (size_t)a.T * (backward ? a.in : a.p[p].out) * (a.io_bf16 ? 2 : 4),
                              hipMemcpyDeviceToDevice, st));
  return hipSuccess;
}

}  // namespace

ProjScratchNeed proj_scratch_need(const ProjLaunch& a, bool backward) {
  ProjScratchNeed need{};
  for (int p = 0; p < (backward ? 1 : a.n_proj); ++p) need.shadow += shadow_bytes(a, backward, p);
  const RowsPlan plan = rows_plan(a, backward);
  if (plan.n == 0) return need;
  need.lowrank = (long)plan.n * a.T * a.rank;
  if (!whole_pieces(a, backward)) return need;
  need.odd = kTermBlocks + (long)plan.n * ((a.T + 15) / 16) * ((a.rank + 15) / 16);
  for (int p = 0; p < a.n_proj; ++p)
    if (a.p[p].a != nullptr)
      need.terms += (long)term_pitch(a.rank) * (a.T + (backward ? a.in : a.p[p].out));
  return need;
}

hipError_t launch_proj_forward(const ProjLaunch& a, hipStream_t st) { return run_call(a, false, st); }

hipError_t launch_proj_backward(const ProjLaunch& a, hipStream_t st) { return run_call(a, true, st); }

}  // namespace glacier
