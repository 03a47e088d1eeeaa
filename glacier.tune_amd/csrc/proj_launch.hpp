// proj_launch.hpp -- host-side interface of proj_lora.hip (the projection
// with LoRA adapters) for engine.cpp.
#pragma once

#include <hip/hip_runtime.h>

namespace glacier {

constexpr int kMaxRank = 64;  // largest LoRA rank taken
constexpr int kMaxProj = 4;   // projections of one input per call

// One projection p of the input: W [out][in] (io dtype), bias [out] fp32 or
// null, A [in][r] and B [r][out] fp32 (A null: no adapter), y [T][out]
// (forward), dy [T][out] (backward), grad_a [in][r] and grad_b [r][out]
// accumulated (+=) when not null.
struct ProjSpec {
  const void* w;
  const float* bias;
  const float* a;
  const float* b;
  float scaling;
  int out;
  void* y;
  const void* dy;
  float* grad_a;
  float* grad_b;
};

struct ProjLaunch {
  int T, in, rank;
  bool io_bf16;
  int n_proj;
  ProjSpec p[kMaxProj];
  const void* x;  // [T][in]
  void* dx;       // [T][in] (backward; overwritten)
  // scratch, sized by proj_scratch_need
  float* lowrank;  // [slot][T][r] X A_p and dY_p B_p^T
  void* terms;     // fused calls: the split terms (bf16) of the adapters, then of s L
  int* odd;        // fused calls: marks of values without a split (SplitCall)
  void* shadow;    // outputs in the memory of x, dY or a W: written here, then copied
};

// ---- bf16 tensors: base products, low-rank delta, bias and conversion in ----
// one launch per direction (proj_gemm.hip)
struct GemmSeg {  // a stretch of the reduction: k elements
  const void* a;  // forward [n][k], backward [k][K] (bf16)
  const void* b;  // [T][k] (bf16)
  int k;          // a multiple of 8
};
struct GemmJob {
  void* y;            // forward: Y_p [T][n] (bf16)
  const float* bias;  // forward: [n] or null
  const float* l;     // L_p (forward) or dL_p (backward) [T][r]; null: no adapter
  const float* v;     // B_p [r][n] (forward) or A_p [K][r] (backward)
  float s;            // the adapter's scaling
  int n;              // outputs of the projection
  int first;          // forward: its first feature tile (set by launch_gemm)
};
struct GemmCall {
  void* dx;         // backward: dX [T][K] (bf16)
  const int* odd;   // [n_odd] marks: the low-rank operands hold values without a split
  int n_odd;
  int T, K, rank, n;
  int ftiles;       // set by launch_gemm
  GemmJob j[kMaxProj];
  GemmSeg seg[2 * kMaxProj];  // p: W_p with X (forward) or dY_p; kMaxProj + p: the adapter's split terms
};
// Elements of a row of split terms: six stretches of r, in whole 16-byte pieces.
__host__ __device__ constexpr int term_pitch(int rank) { return (6 * rank + 7) / 8 * 8; }
hipError_t launch_gemm(GemmCall a, bool backward, hipStream_t st);

// Every other call (fp32 tensors; bf16 ones of other widths or alignments),
// the operands split as they are loaded; the adapter's terms are not used.
hipError_t launch_gemm_split(const GemmCall& a, bool backward, bool io_bf16, hipStream_t st);

// Elements of each ProjLaunch scratch buffer for a forward or backward call.
struct ProjScratchNeed {
  long lowrank;  // floats
  long terms;    // bf16
  long odd;      // ints
  long shadow;   // bytes
};
ProjScratchNeed proj_scratch_need(const ProjLaunch& a, bool backward);

// Enqueue on st.
hipError_t launch_proj_forward(const ProjLaunch& a, hipStream_t st);
hipError_t launch_proj_backward(const ProjLaunch& a, hipStream_t st);

}  // namespace glacier
