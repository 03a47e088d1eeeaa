// proj_gemm.hip -- the projections' base products on the matrix cores, with
// the LoRA delta, the bias and the output conversion in the same pass.
//
// GpuLoraEngine.ForwardQKV (GpuLoraEngine.Forward.cs:205-245) and
// LoraAdapter.Backward (LoraAdapter.cs:190-247) compute the same products.
#include "attn_common.hpp"
#include "lds_mfma.hpp"
#include "proj_launch.hpp"
#include "split3.hpp"

namespace glacier {
namespace {

// The hardware deals workgroup ids to the 8 XCDs round-robin (id % 8), each
// XCD with its own L2.  Renumbering so that consecutive logical indices run
// on one XCD keeps the workgroups that share operand tiles (tile_of) on one
// L2: each XCD then fetches only its own share of the weights, instead of
// every XCD fetching all of them.
[[maybe_unused]] __device__ inline int xcd_logical(int id, int total) {
  constexpr int kXcds = 8;
  const int q = total / kXcds, r = total % kXcds, x = id % kXcds;
  return x * q + min(x, r) + id / kXcds;
}

// ---------------------------------------------------------------------------
// bf16 tensors.  One launch per direction takes every projection of the call:
//   forward  (NT) Y_p[t][f] = sum_k X[t][k] W_p[f][k] + bias_p[f] + s_p (L_p B_p)[t][f]
//   backward (NN) dX[t][c]  = sum_p sum_f dY_p[t][f] W_p[f][c] + s_p (dL_p A_p^T)[t][c]
// with L_p = X A_p and dL_p = dY_p B_p^T in fp32 from lowrank_split.
//
// A workgroup of 8 waves computes a FT-feature x TT-token tile of the
// transposed product C^T on v_mfma_f32_32x32x16_bf16: WF x WT waves of FB x
// TB blocks of 32 x 32, times WK groups that share the k-steps of a stage
// (their sums are added in group order through LDS at the end).  Stages of KT
// reduction elements go global -> LDS by DMA (buffer_load ... lds, 16 bytes a
// lane) into a ring of RING slots.  LDS rows are KT elements of a feature or
// token (backward A: 64 features of one reduction row, FT / 64 such
// sub-tiles), unpadded, their 16-byte pieces XOR-swizzled (lds_sw): fragment
// reads and transposing reads (ds_read_b64_tr_b16) are free of bank conflicts.
// Rows past T or past a projection's outputs, and the pieces past the
// reduction's end, are outside the DMA's buffer range and arrive as zeros.
//
// The low-rank product is a further stretch of the same reduction: both fp32
// operands are split in three bf16 terms (split3.hpp), laid out six times r
// wide by lowrank_split so that one bf16 product sums the six term products.
// A call that holds a value without a split there (its marks, `odd`) takes fp32
// MFMAs for it instead.  The bias starts the accumulators, and the bf16
// conversion happens as the tile leaves through LDS in whole row pieces.  So
// no fp32 product goes to memory and back.
// MFMA layout (lane l, c = l % 32, h = l / 32): A[row c][k = 8h .. 8h + 7],
// B[k = 8h ..][col c]; accumulator element e holds column c, row
// 8 (e / 4) + 4h + e % 4.
//
// What bounds it: large calls, the matrix cores at the clock the chip holds
// under them (1.45-1.5 GHz with every CU on MFMAs of random data): 4096 x 4096
// x 4096 forward 137 us (1.0 PFLOP/s), the products alone 117 us; 220 us before
// (and 24 us of lowrank_out).  Small calls, the DMA: a 1 KB instruction takes
// 16 clocks of the CU's vector-memory unit from L2 (24 with 64-byte rows, 24-28
// when the chip's CUs share the fabric), and a stage's DMA is issued in a burst
// behind its barrier.  512 x 3584 -> 3584/512/512: forward 33 us, backward 35
// us, against 21.6 + 11.7 + 6.3 and 24.9 + 15.0 + 8.4 us in three launches.
// ---------------------------------------------------------------------------
constexpr int kGThreads = 512;  // 8 waves
[[maybe_unused]] constexpr int kOob = 0x7ffffff0;  // a buffer offset past every range: reads as zero

#if defined(__HIP_DEVICE_COMPILE__)
__device__ inline f32x16 mma32(const bf16x8& a, const bf16x8& b, const f32x16& c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// Byte offset, inside a tile of rows of KT elements, of this lane's fragment
// read of k-step 0 for rows row0 + lane % 32 (row0 a multiple of 16); k-step
// s reads at that offset ^ 32 s, the 32 rows after at + 64 KT.
template <int KT>
__device__ inline unsigned frag_off(int lane, int row0) {
  const int r = row0 + (lane & 31), h = lane >> 5;
  return static_cast<unsigned>(r * 2 * KT + 16 * (h ^ lds_sw<KT>(r)));
}
// Byte offset, inside a sub-tile of 64 reduction rows x 64 features, of this
// lane's transposing read j (0, 1) of k-step 0 for features col0 + 16 (G & 1)
// + 4 (i & 3) (quarter-wave G, lane i in it): rows 8 h + 4 j + i / 4; k-step
// s reads 16 s rows further (+2048 s).
__device__ inline unsigned tr_off128(int lane, int col0, int j) {
  const int G = lane >> 4, i = lane & 15, h = lane >> 5;
  const int r = 8 * h + 4 * j + (i >> 2);
  const int col = col0 + 16 * (G & 1) + 4 * (i & 3);
  return static_cast<unsigned>(r * 128 + 16 * ((col >> 3) ^ lds_sw<64>(r)) + 2 * (col & 7));
}
#endif

// Tile id -> (feature tile, token tile): bands of 4 feature tiles, feature
// fastest inside a band, so that the 32 workgroups an XCD runs at once cover
// a block of about 4 x 8 tiles and share both operands through its L2.
[[maybe_unused]] __device__ inline void tile_of(int id, int ftiles, int ttiles, int& f, int& t) {
  const int band = id / (4 * ttiles), in = id - band * 4 * ttiles;
  const int width = min(4, ftiles - 4 * band);
  t = in / width;
  f = 4 * band + in - t * width;
}

template <int FB, int TB, int WK>
constexpr int block_owner(int fb, int tb) {
  if constexpr (WK == 1)
    return 0;
  else if constexpr (FB % 2 == 0)
    return fb / (FB / 2);
  else if constexpr (TB % 2 == 0)
    return tb / (TB / 2);
  else
    return 0;
}

#if defined(__HIP_DEVICE_COMPILE__)
// WK == 2: each group hands the other the blocks that one finishes, and adds
// its own to what it receives.  All of the workgroup is past its last use of
// lds; barriers on both sides.
template <int FB, int TB, int WK>
__device__ inline void merge_groups(f32x16 (&acc)[FB][TB], unsigned char* lds, int place, int wk, int lane) {
  if constexpr (WK == 2) {
    f32x4* ex = reinterpret_cast<f32x4*>(lds) + place * (FB * TB * 256);
#pragma unroll
    for (int fb = 0; fb < FB; ++fb)
#pragma unroll
      for (int tb = 0; tb < TB; ++tb)
        if (block_owner<FB, TB, WK>(fb, tb) != wk)
#pragma unroll
          for (int q = 0; q < 4; ++q)
            ex[(fb * TB + tb) * 256 + q * 64 + lane] =
                f32x4{acc[fb][tb][4 * q], acc[fb][tb][4 * q + 1], acc[fb][tb][4 * q + 2], acc[fb][tb][4 * q + 3]};
    __syncthreads();
#pragma unroll
    for (int fb = 0; fb < FB; ++fb)
#pragma unroll
      for (int tb = 0; tb < TB; ++tb)
        if (block_owner<FB, TB, WK>(fb, tb) == wk)
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const f32x4 o = ex[(fb * TB + tb) * 256 + q * 64 + lane];
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[fb][tb][4 * q + e] += o[e];
          }
    __syncthreads();
  }
}
#endif

template <bool NN, int KT, int FB, int TB, int WF, int WT, int WK, int G, int RING>
__global__ __launch_bounds__(kGThreads) void proj_gemm_kernel(const GemmCall a) {
#if defined(__HIP_DEVICE_COMPILE__)
  static_assert(WF * WT * WK == 8 && (WK == 1 || WK == 2), "8 waves");
  constexpr int FT = WF * FB * 32, TT = WT * TB * 32;
  constexpr int RI = 1024 / (2 * KT);  // operand rows per DMA instruction
  constexpr int NA = FT / (8 * RI), NB = TT / (8 * RI), ND = NA + NB;  // per wave and stage
  constexpr int kA = FT * KT * 2, kStage = (FT + TT) * KT * 2;
  static_assert(FT % (8 * RI) == 0 && TT % (8 * RI) == 0 && RING >= 2 && RING * kStage <= 160 * 1024, "tile");
  constexpr int KS = KT / 16 / WK;  // k-steps of a stage per wave
  constexpr int U = KS / G;         // units of a stage: G k-steps each
  static_assert(KS % G == 0 && (U == 1 || U % 2 == 0), "fragment buffers alternate");
  __shared__ __align__(1024) unsigned char lds[RING * kStage];
  const int ttiles = (a.T + TT - 1) / TT;
  const int id = xcd_logical((int)blockIdx.x, (int)gridDim.x);
  int ft, tt;
  tile_of(id, a.ftiles, ttiles, ft, tt);
  int z = 0;  // forward: the tile's projection
  if constexpr (!NN)
    while (z + 1 < a.n && ft >= a.j[z + 1].first) ++z;
  const int f0 = NN ? FT * ft : FT * (ft - a.j[z].first), t0 = TT * tt;
  const int nf = NN ? a.K : a.j[z].n;  // features of the output
  const int lane = threadIdx.x & 63, w = wave_id();
  const int wf = w % WF, wt = w / WF % WT, wk = w / (WF * WT);
  // a value without a split among the low-rank operands: see below
  bool slow = false;
  for (int i = lane; i < a.n_odd; i += 64) slow |= a.odd[i] != 0;
  slow = __any(slow);

  // DMA: instruction i of this wave covers RI rows of an operand (backward A:
  // 8 reduction rows of a sub-tile); a lane writes one 16-byte slot of a row
  // and fetches the piece that belongs there.
  constexpr int PR = KT / 8;  // pieces per row
  const int row = RI * w + lane / PR;
  const int piece = (lane % PR) ^ lds_sw<KT>(row);
  int va[NA], vb[NB];
  __amdgpu_buffer_rsrc_t ra, rb;
  if constexpr (NN) {
#pragma unroll
    for (int i = 0; i < NA; ++i) {
      const int n = w + 8 * i, r = 8 * (n % (KT / 8)) + (lane >> 3);
      const int c = 64 * (n / (KT / 8)) + 8 * ((lane & 7) ^ lds_sw<64>(r));
      va[i] = f0 + c < a.K ? r * a.K * 2 + 2 * c : kOob;
    }
  }
  // the segments of the reduction: forward X W^T then L_p B_p, backward
  // every dY_p W_p then every dL_p A_p^T (seg[kMaxProj + p], in split terms)
  const int T = a.T, K = a.K, n_seg = a.n;
  int nst = 0, sg = NN ? -1 : z - kMaxProj, kend = 0, kbase = 0, kcur = 0;
  for (int y = NN ? 0 : z; y < (NN ? n_seg : z + 1); ++y)
    nst += (a.seg[y].k + KT - 1) / KT + (slow ? 0 : (a.seg[kMaxProj + y].k + KT - 1) / KT);
  // advance(st) (in order: 0, 1, ...) points the DMA at stage st; dma<i>(slot)
  // issues its instruction i into ring slot `slot`
  const bf16* wrow = nullptr;  // backward: A's rows from the segment's first, column f0
  int k0 = 0;
  bool past = false;  // this lane's piece lies past the segment's end
  auto advance = [&](int st) {
    while (st >= kend) {  // the next segment
      sg = NN ? (sg + 1 == n_seg ? kMaxProj : sg + 1) : sg + kMaxProj;
      kbase = kend;
      kcur = a.seg[sg].k;
      kend += (kcur + KT - 1) / KT;
      const int rowb = kcur * 2;
      rb = wave_rsrc(static_cast<const bf16*>(a.seg[sg].b) + (long)t0 * kcur, min(TT, T - t0) * rowb);
#pragma unroll
      for (int i = 0; i < NB; ++i) vb[i] = (8 * RI * i + row) * rowb + 16 * piece;
      if constexpr (NN) {
        wrow = static_cast<const bf16*>(a.seg[sg].a) + f0;
      } else {
        ra = wave_rsrc(static_cast<const bf16*>(a.seg[sg].a) + (long)f0 * kcur, min(FT, nf - f0) * rowb);
#pragma unroll
        for (int i = 0; i < NA; ++i) va[i] = (8 * RI * i + row) * rowb + 16 * piece;
      }
    }
    k0 = (st - kbase) * KT;
    if constexpr (NN)
      ra = wave_rsrc(wrow + (long)k0 * K, (min(KT, kcur - k0) - 1) * K * 2 + (K - f0) * 2);
    past = k0 + KT > kcur && k0 + 8 * piece >= kcur;
  };
  auto dma = [&](auto ic, int slot) {
    constexpr int I = decltype(ic)::value;
    unsigned char* base = lds + slot * kStage + 1024 * w;
    if constexpr (I < NA)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (GLACIER_LDS void*)(base + 8192 * I), 16,
                                               NN ? va[I] : past ? kOob : va[I], NN ? 0 : 2 * k0, 0, 0);
    else
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, (GLACIER_LDS void*)(base + kA + 8192 * (I - NA)), 16,
                                               past ? kOob : vb[I - NA], 2 * k0, 0, 0);
  };
#pragma unroll
  for (int i = 0; i < RING; ++i)
    if (i < nst) {
      advance(i);
      static_for<ND>([&](auto ic) { dma(ic, i); });
    }

  // the accumulators start at the bias (in one group's)
  f32x16 acc[FB][TB];
  const int fw = f0 + 32 * FB * wf, tw = t0 + 32 * TB * wt;
  const float* bias = NN || wk != 0 ? nullptr : a.j[z].bias;
#pragma unroll
  for (int fb = 0; fb < FB; ++fb)
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const int f = fw + 32 * fb + 8 * (e / 4) + 4 * (lane >> 5) + e % 4;
      const float b = bias == nullptr ? 0.0f : bias[min(f, nf - 1)];
#pragma unroll
      for (int tb = 0; tb < TB; ++tb) acc[fb][tb][e] = b;
    }
  if (slow && wk == 0) {
    // the low-rank products of a call with values that have no split terms:
    // sum over the terms of (s L [T][r]) V, V = B [r][n]
    // (forward) or A^T with A [K][r], on fp32 MFMAs
    for (int p = NN ? 0 : z; p < (NN ? a.n : z + 1); ++p) {
      const GemmJob& job = a.j[p];
      if (job.l == nullptr) continue;
#pragma clang loop unroll(disable)
      for (int k0 = 0; k0 < a.rank; k0 += 2) {
        const int kk = min(k0 + (lane >> 5), a.rank - 1);
        const bool k_ok = k0 + (lane >> 5) < a.rank;
        float lv[TB], vv[FB];
#pragma unroll
        for (int tb = 0; tb < TB; ++tb) {
          const float v = job.l[(long)min(tw + 32 * tb + (lane & 31), a.T - 1) * a.rank + kk];
          lv[tb] = k_ok ? job.s * v : 0.0f;
        }
#pragma unroll
        for (int fb = 0; fb < FB; ++fb) {
          const int f = min(fw + 32 * fb + (lane & 31), nf - 1);
          const float v = NN ? job.v[(long)f * a.rank + kk] : job.v[(long)kk * nf + f];
          vv[fb] = k_ok ? v : 0.0f;
        }
#pragma unroll
        for (int fb = 0; fb < FB; ++fb)
#pragma unroll
          for (int tb = 0; tb < TB; ++tb)
            acc[fb][tb] = __builtin_amdgcn_mfma_f32_32x32x2f32(vv[fb], lv[tb], acc[fb][tb], 0, 0, 0);
      }
    }
  }

  // read addresses of k-step s of slot 0: A (NT: fragments, blocks 32 rows
  // apart; NN: transposing reads j of each block), B fragments
  const unsigned sbase = static_cast<unsigned>(reinterpret_cast<uintptr_t>((GLACIER_LDS void*)lds));
  unsigned oa[NN ? 2 * FB : KS], ob[KS];
  {
    const unsigned b = frag_off<KT>(lane, 32 * TB * wt);
#pragma unroll
    for (int s = 0; s < KS; ++s) ob[s] = sbase + kA + (b ^ (32u * (KS * wk + s)));
    if constexpr (NN) {
#pragma unroll
      for (int fb = 0; fb < FB; ++fb) {
        const int col = 32 * (FB * wf + fb);
#pragma unroll
        for (int j = 0; j < 2; ++j)
          oa[2 * fb + j] = sbase + 128u * KT * (col / 64) + tr_off128(lane, col % 64, j) + 2048u * KS * wk;
      }
    } else {
      const unsigned o = frag_off<KT>(lane, 32 * FB * wf);
#pragma unroll
      for (int s = 0; s < KS; ++s) oa[s] = sbase + (o ^ (32u * (KS * wk + s)));
    }
  }
  // fragments in two buffers of one unit (G k-steps) each
  constexpr int NRK = (NN ? 2 * FB : FB) + TB, NRD = G * NRK, NM = G * FB * TB;
  bf16x8 fa[2][G][FB], fbk[2][G][TB];
  bf16x4 ta[2][G][FB][2];
  // read i of unit N of a stage into buffer P: the A blocks' first, then B's
  auto rd = [&](auto pc, auto nc, auto ic, unsigned so) {
    constexpr int P = decltype(pc)::value, I = decltype(ic)::value % NRK, g = decltype(ic)::value / NRK;
    constexpr int S = decltype(nc)::value * G + g;
    if constexpr (I >= NRK - TB)
      fbk[P][g][I - (NRK - TB)] = rd128<64 * KT * (I - (NRK - TB))>(ob[S] + so);
    else if constexpr (NN)
      ta[P][g][I / 2][I & 1] = rdtr<2048 * S>(oa[I] + so);
    else
      fa[P][g][I] = rd128<64 * KT * I>(oa[S] + so);
  };
  // the reads into buffer P have arrived
  auto arrive = [&](auto pc) {
    constexpr int P = decltype(pc)::value;
    lgkm<0>();
    static_for<G>([&](auto gc) {
      constexpr int g = decltype(gc)::value;
      static_for<FB>([&](auto fc) {
        constexpr int F = decltype(fc)::value;
        if constexpr (NN) {
          tie_v(ta[P][g][F][0]);
          tie_v(ta[P][g][F][1]);
          fa[P][g][F] = join8(ta[P][g][F][0], ta[P][g][F][1]);
        } else {
          tie_v(fa[P][g][F]);
        }
      });
      static_for<TB>([&](auto tc) { tie_v(fbk[P][g][decltype(tc)::value]); });
    });
  };
  // Between the MFMAs of a unit go the fragment reads of the next one, one
  // at a time (eight waves' reads in a row fill the LDS queue and hold up the
  // products behind them).  The one barrier of a stage stands before its last
  // unit, whose fragments have then arrived: past it every wave is done with
  // the stage's slot, so the DMA of the stage RING ahead goes into it, and the
  // next stage has landed (each wave waited for its own DMA of it), so the
  // next unit's fragments are read behind the last products as usual.
  // Every read is waited for in the stage that issues it: the loop carries
  // only values that have arrived.
  vm_wait_v((min(nst, RING) - 1) * ND);
  wg_barrier();
  static_for<NRD>([&](auto ic) { rd(std::integral_constant<int, 0>{}, std::integral_constant<int, 0>{}, ic, 0u); });
  arrive(std::integral_constant<int, 0>{});
  int slot = 0;
  auto stage = [&](int st, auto p0c) {
    const int next = slot + 1 == RING ? 0 : slot + 1;
    const unsigned so = static_cast<unsigned>(slot * kStage), sn = static_cast<unsigned>(next * kStage);
    const bool more = st + RING < nst;
    static_for<U>([&](auto uc) {
      constexpr int UN = decltype(uc)::value, P = (decltype(p0c)::value + UN) & 1, N = (UN + 1) % U;
      constexpr bool kLast = UN == U - 1;
      constexpr int NI = NM > NRD ? NM : NRD;
      if constexpr (kLast) {
        if (more)
          vmw<(RING - 2) * ND>();
        else
          vm_wait_v(max(nst - 2 - st, 0) * ND);
        wg_barrier();
        if (more) advance(st + RING);
      }
      __builtin_amdgcn_sched_barrier(0);
      static_for<(kLast && ND > NI ? ND : NI)>([&](auto ic) {
        constexpr int I = decltype(ic)::value;
        if constexpr (I < NM) {
          constexpr int g = I / (FB * TB), fb = I % (FB * TB) / TB, tb = I % TB;
          acc[fb][tb] = mma32(fa[P][g][fb], fbk[P][g][tb], acc[fb][tb]);
        }
        if constexpr (I < NRD)  // past the last stage: a slot's old rows, unused
          rd(std::integral_constant<int, P ^ 1>{}, std::integral_constant<int, N>{}, ic, kLast ? sn : so);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (kLast && I < ND) {
          if (more) dma(ic, slot);
          __builtin_amdgcn_sched_barrier(0);
        }
      });
      arrive(std::integral_constant<int, P ^ 1>{});
    });
    slot = next;
  };
  for (int st = 0; st < nst; ++st) {
    stage(st, std::integral_constant<int, 0>{});
    if constexpr (U == 1)  // the buffers change roles
      if (++st < nst) stage(st, std::integral_constant<int, 1>{});
  }

  __syncthreads();
  merge_groups<FB, TB, WK>(acc, lds, w % (WF * WT), wk, lane);
  // bf16, and out through LDS: 32 tokens x 32 FB features per wave at a
  // time, rows of kOutRow bytes (padded), then 16-byte row pieces
  constexpr int kOutRow = 64 * FB + 16;
  unsigned char* mine = lds + w * 32 * kOutRow;
  static_assert(8 * 32 * kOutRow <= RING * kStage, "output staging fits the ring");
  const int h = lane >> 5;
  bf16* out = static_cast<bf16*>(NN ? a.dx : a.j[z].y);
#pragma unroll
  for (int tb = 0; tb < TB; ++tb) {
#pragma unroll
    for (int fb = 0; fb < FB; ++fb) {
      if (block_owner<FB, TB, WK>(fb, tb) != wk) continue;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int fl = 32 * fb + 8 * q + 4 * h;
        bf16x4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = (bf16)acc[fb][tb][4 * q + e];
        *reinterpret_cast<bf16x4*>(mine + (lane & 31) * kOutRow + 2 * fl) = v;
      }
    }
    __builtin_amdgcn_wave_barrier();
    constexpr int PC = 4 * FB;  // 16-byte pieces per row
#pragma unroll
    for (int i = 0; i < 32 * PC / 64; ++i) {
      const int idx = 64 * i + lane, r = idx / PC, pc = idx % PC;
      const int t = tw + 32 * tb + r, f = fw + 8 * pc;
      if (block_owner<FB, TB, WK>(pc / 4, tb) == wk && t < a.T && f < nf)
        *reinterpret_cast<i32x4*>(out + (long)t * nf + f) = *reinterpret_cast<const i32x4*>(mine + r * kOutRow + 16 * pc);
    }
    __builtin_amdgcn_wave_barrier();
  }
#endif
}

// ---------------------------------------------------------------------------
// Every other call (fp32 tensors, and bf16 tensors of other widths or
// alignments): the same sums, operands through registers.  Each fp32 element is
// split in three bf16 terms (split3.hpp) on its way from global memory to LDS, and
// a product of fragments is six v_mfma_f32_32x32x16_bf16; bf16 elements are one
// term, and one product.  The low-rank product is again a stretch of the
// reduction, the adapters' ranks one after another, its operands split as they
// are (fp32, B and A read down their columns); it goes first, while the base
// products' first stages are on their way.
//
// 8 waves: WF x WT waves of FB x TB blocks of 32 x 32, times WK groups that
// share a stage's two k-steps.  Stages of 32 reduction elements go global ->
// registers (PF stages ahead) -> three LDS planes of bf16 rows (layout as above:
// 64-byte rows, backward A 64-feature sub-tiles; one plane for one term), two
// buffers, one barrier a stage.  Loads are unconditional at clamped addresses;
// elements past the reduction are zeroed in A (in one term in both), rows past
// an edge reach no stored result.  A tile that meets an element without a split
// is done over on fp32 MFMAs, straight from global memory.
//
// What bounds it: fp32 at one small tile per CU the chain of a stage (split, LDS,
// six dependent products: 0.75 us); once the chip is full the six products
// (6/16 of the fp32 MFMA's time) and the split's 11 vector instructions for each
// 2 elements beside them.  201 x 896 -> 896/128/128: forward 24 us in one
// launch (three of 35, and two low-rank passes, before), backward 31 us (46
// and two).  bf16, the chain of a stage (0.25 us): 512 x 3584 -> 3584/512/12, whole
// calls, 61 + 81 us (177 + 219 split in three terms, 198 + 72 with q on a DMA
// GEMM of its own); a 3584 x 3584 W off 16 bytes, 63 + 82 (177 + 230; 58 + 71).
// 16-byte loads take 5-10% less than two of 8 bytes; planes of 96 reduction
// elements in place of the terms took as long (a third of the barriers, but
// 40 more VGPRs: one 64 x 64 workgroup a CU).
// ---------------------------------------------------------------------------
// Ends a run of products where control flow joins: 16 wait states, so that the
// copies of accumulators that the compiler may place there read what the last
// MFMA wrote.  (It leaves too few of its own before copies in a loop's header:
// built without this, the bf16 backward 64 x 64 instance copied one 5 wait states
// behind a product that takes 12, and lost its sums.  The loops without it have no
// such copies as built; tests/test_mfma_waits.py looks.)
template <int FB, int TB>
__device__ inline void settle(f32x16 (&acc)[FB][TB]) {
#pragma unroll
  for (int fb = 0; fb < FB; ++fb)
#pragma unroll
    for (int tb = 0; tb < TB; ++tb) tie_v(acc[fb][tb]);
  asm volatile("s_nop 15" : "+v"(acc[FB - 1][TB - 1]));
}

template <typename E>
__device__ inline void load4_any(const E* p, float (&x)[8], int at) {
  typedef E E4 __attribute__((ext_vector_type(4)));
  E4 v;
  __builtin_memcpy(&v, p, sizeof(v));
#pragma unroll
  for (int e = 0; e < 4; ++e) x[at + e] = (float)v[e];
}
// A thread's 8 elements of a stage on their way to LDS, as loaded: the first
// `valid` count, the rest are zeros.
struct Piece {
  float x[8];
  int valid;
};
struct Piece16 {  // of bf16 tensors
  bf16x8 x;
  int valid;
  bool late;  // the 8 loaded begin 4 before the piece
};

template <typename IO, bool NN, bool kTiny, int FB, int TB, int WF, int WT, int WK, int PF>
__global__ __launch_bounds__(kGThreads) void proj_gemm_split_kernel(const GemmCall a) {
#if defined(__HIP_DEVICE_COMPILE__)
  static_assert(WF * WT * WK == 8 && (WK == 1 || WK == 2), "8 waves");
  constexpr int FT = WF * FB * 32, TT = WT * TB * 32, KT = 32, KS = 2 / WK;
  constexpr int NA = FT * 4 / kGThreads, NB = TT * 4 / kGThreads;  // 8-element pieces per thread
  constexpr int PA = FT * 4, PB = TT * 4;                          // pieces in all
  constexpr int kPlaneA = FT * 64, kPlaneB = TT * 64, kBuf = 3 * (kPlaneA + kPlaneB);
  static_assert((PA % kGThreads == 0 && PB % kGThreads == 0) || (NA == 0 && NB == 0 && PA + PB == kGThreads),
                "pieces per thread");
  constexpr bool kOne = sizeof(IO) == 2;  // base operands: bf16 already, one term
  constexpr bool kShared = NA == 0;  // half of the threads bring A, half B
  constexpr int LA = kShared ? 1 : NA, LB = kShared ? 0 : NB;
  __shared__ __align__(1024) unsigned char lds[2 * kBuf];
  const int T = a.T, K = a.K, rank = a.rank;
  const int ttiles = (T + TT - 1) / TT;
  const int id = xcd_logical((int)blockIdx.x, (int)gridDim.x);
  int ft, tt;
  tile_of(id, a.ftiles, ttiles, ft, tt);
  int z = 0;
  if constexpr (!NN)
    while (z + 1 < a.n && ft >= a.j[z + 1].first) ++z;
  const int f0 = NN ? FT * ft : FT * (ft - a.j[z].first), t0 = TT * tt;
  const int nf = NN ? K : a.j[z].n;
  const int tid = threadIdx.x, lane = tid & 63, w = wave_id();
  const int wf = w % WF, wt = w / WF % WT, wk = w / (WF * WT);

  // the base products: forward X W^T, backward every dY_p W_p
  const int seg0 = NN ? 0 : z, seg1 = NN ? a.n : z + 1;
  int nst = 0, terms = 0;
  for (int y = seg0; y < seg1; ++y) {
    nst += (a.seg[y].k + KT - 1) / KT;
    terms += a.j[y].l != nullptr;
  }
  // the terms in order: with element kk of the low-rank stretch in term kk / rank
  const int n_low = terms * rank, low_st = (n_low + KT - 1) / KT;
  auto job_of = [&](int term) {  // the term's projection
    int y = seg0;
    for (;; ++y)
      if (a.j[y].l != nullptr && term-- == 0) break;
    return y;
  };

  // Piece idx of a stage of the base products, reduction elements k0 .. of
  // segment `cur`: A (forward: row f, 8 reduction elements; backward:
  // reduction row, 8 features) and B (row t, 8 reduction elements).
  int sg = seg0 - 1, kend = 0, kbase = 0, kcur = 0;
  const IO *ca = nullptr, *cb = nullptr;
  using Base = std::conditional_t<kOne, Piece16, Piece>;
  // elements k .. k + 7 of a row of len (a multiple of 4), in bounds
  auto eight = [&](const IO* row, int k, int len, Base& p) {
    if constexpr (kOne && kTiny) {
      p.late = false;
      __builtin_memcpy(&p.x, row + min(k, len - 4), 8);
      __builtin_memcpy(reinterpret_cast<char*>(&p.x) + 8, row + min(k + 4, len - 4), 8);
    } else if constexpr (kOne) {
      // one load, 4 early where the row ends inside it
      const int at = min(k, len - 8);
      p.late = k > at;
      __builtin_memcpy(&p.x, row + at, 16);
    } else {
      load4_any(row + min(k, len - 4), p.x, 0);
      load4_any(row + min(k + 4, len - 4), p.x, 4);
    }
  };
  auto load_a = [&](int idx, int k0, Base& p) {
    if constexpr (NN) {
      const int k = k0 + (idx >> 3) % 32, f = f0 + 64 * (idx >> 8) + 8 * (idx & 7);
      p.valid = k < kcur ? 8 : 0;
      eight(ca + (long)min(k, kcur - 1) * K, f, K, p);
    } else {
      const int f = min(f0 + (idx >> 2), nf - 1), k = k0 + 8 * (idx & 3);
      p.valid = kcur - k;
      eight(ca + (long)f * kcur, k, kcur, p);
    }
  };
  auto load_b = [&](int idx, int k0, Base& p) {
    const int t = min(t0 + (idx >> 2), T - 1), k = k0 + 8 * (idx & 3);
    p.valid = kOne ? kcur - k : 8;  // one term: nothing marks a non-finite value that A's zeros meet
    eight(cb + (long)t * kcur, k, kcur, p);
  };
  // the same of the low-rank stretch, its elements kk0 ..
  auto low_a = [&](int idx, int kk0, Piece& p) {
    const int kk = NN ? kk0 + (idx >> 3) % 32 : kk0 + 8 * (idx & 3);
    const int f = NN ? f0 + 64 * (idx >> 8) + 8 * (idx & 7) : min(f0 + (idx >> 2), nf - 1);
    p.valid = NN ? (kk < n_low ? 8 : 0) : n_low - kk;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int q = min(NN ? kk : kk + e, n_low - 1), term = q / rank, j = q - term * rank;
      const float* v = a.j[job_of(term)].v;
      p.x[e] = NN ? v[(long)min(f + e, K - 1) * rank + j] : v[(long)j * nf + f];
    }
  };
  auto low_b = [&](int idx, int kk0, Piece& p) {
    const int t = min(t0 + (idx >> 2), T - 1), kk = kk0 + 8 * (idx & 3);
    p.valid = 8;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int q = min(kk + e, n_low - 1), term = q / rank, j = q - term * rank;
      const GemmJob& job = a.j[job_of(term)];
      p.x[e] = job.s * job.l[(long)t * rank + j];
    }
  };
  struct Pieces {
    Piece a[LA], b[LB > 0 ? LB : 1];
  };
  struct BasePieces {
    Base a[LA], b[LB > 0 ? LB : 1];
  };
  auto load = [&](int st, BasePieces& p) {
    while (st >= kend && sg + 1 < seg1) {
      ++sg;
      kbase = kend;
      kcur = a.seg[sg].k;
      kend += (kcur + KT - 1) / KT;
      ca = static_cast<const IO*>(a.seg[sg].a);
      cb = static_cast<const IO*>(a.seg[sg].b);
    }
    const int k0 = (st - kbase) * KT;
    if constexpr (kShared) {
      if (w < PA / 64)
        load_a(tid, k0, p.a[0]);
      else
        load_b(tid - PA, k0, p.a[0]);
    } else {
#pragma unroll
      for (int i = 0; i < LA; ++i) load_a(tid + kGThreads * i, k0, p.a[i]);
#pragma unroll
      for (int i = 0; i < LB; ++i) load_b(tid + kGThreads * i, k0, p.b[i]);
    }
  };
  auto load_low = [&](int st, Pieces& p) {
    if constexpr (kShared) {
      if (w < PA / 64)
        low_a(tid, st * KT, p.a[0]);
      else
        low_b(tid - PA, st * KT, p.a[0]);
    } else {
#pragma unroll
      for (int i = 0; i < LA; ++i) low_a(tid + kGThreads * i, st * KT, p.a[i]);
#pragma unroll
      for (int i = 0; i < LB; ++i) low_b(tid + kGThreads * i, st * KT, p.b[i]);
    }
  };
  SplitMarks mark;
  // piece idx of operand `b` (0: A, 1: B) into the planes of a buffer
  auto put = [&](unsigned char* base, int idx, bool b, auto& q) {
    int off;
    if (NN && !b) {
      const int r = (idx >> 3) % 32;
      off = 4096 * (idx >> 8) + 128 * r + 16 * ((idx & 7) ^ lds_sw<64>(r));
    } else {
      const int r = idx >> 2;
      off = 64 * r + 16 * ((idx & 3) ^ lds_sw<32>(r));
    }
    unsigned char* p = base + (b ? 3 * kPlaneA : 0) + off;
    if constexpr (std::is_same_v<std::decay_t<decltype(q)>, Piece16>) {
      tie_v(q.x);  // the load stays unconditional
      const bf16x4 zero{}, lo{q.x[0], q.x[1], q.x[2], q.x[3]}, hi{q.x[4], q.x[5], q.x[6], q.x[7]};
      *reinterpret_cast<bf16x8*>(p) = join8(q.valid <= 0 ? zero : q.late ? hi : lo, q.valid <= 4 ? zero : hi);
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        tie_v(q.x[e]);
        q.x[e] = e < q.valid ? q.x[e] : 0.0f;
      }
      Split3 s;
      s.set(q.x, mark);
      const int plane = b ? kPlaneB : kPlaneA;
      *reinterpret_cast<bf16x8*>(p) = s.h;
      *reinterpret_cast<bf16x8*>(p + plane) = s.m;
      *reinterpret_cast<bf16x8*>(p + 2 * plane) = s.l;
    }
  };
  auto put_all = [&](unsigned char* base, auto& p) {
    if constexpr (kShared) {
      put(base, w < PA / 64 ? tid : tid - PA, w >= PA / 64, p.a[0]);
    } else {
#pragma unroll
      for (int i = 0; i < LA; ++i) put(base, tid + kGThreads * i, false, p.a[i]);
#pragma unroll
      for (int i = 0; i < LB; ++i) put(base, tid + kGThreads * i, true, p.b[i]);
    }
  };

  const int fw = f0 + 32 * FB * wf, tw = t0 + 32 * TB * wt;
  const float* bias = NN || wk != 0 ? nullptr : a.j[z].bias;
  // fp32 tensors: the five small products of a step sum apart from the large
  // one, whose sum then rounds once a step; bf16 results round far above that
  constexpr bool kApart = sizeof(IO) == 4;
  f32x16 acc[FB][TB], small[FB][TB];
#pragma unroll
  for (int fb = 0; fb < FB; ++fb)
#pragma unroll
    for (int tb = 0; tb < TB; ++tb)
#pragma unroll
      for (int e = 0; e < 16; ++e) small[fb][tb][e] = 0.0f;
  auto clear = [&] {
#pragma unroll
    for (int fb = 0; fb < FB; ++fb)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int f = fw + 32 * fb + 8 * (e / 4) + 4 * (lane >> 5) + e % 4;
        const float b = bias == nullptr ? 0.0f : bias[min(f, nf - 1)];
#pragma unroll
        for (int tb = 0; tb < TB; ++tb) acc[fb][tb][e] = b;
      }
  };
  clear();

  // LDS offsets of the fragments of k-step s of this wave
  unsigned oa[NN ? 2 * FB : KS], ob[KS];
  {
    const unsigned b = frag_off<32>(lane, 32 * TB * wt);
#pragma unroll
    for (int s = 0; s < KS; ++s) ob[s] = 3 * kPlaneA + (b ^ (32u * (KS * wk + s)));
    if constexpr (NN) {
#pragma unroll
      for (int fb = 0; fb < FB; ++fb) {
        const int col = 32 * (FB * wf + fb);
#pragma unroll
        for (int j = 0; j < 2; ++j)
          oa[2 * fb + j] = 4096u * (col / 64) + tr_off128(lane, col % 64, j) + 2048u * KS * wk;
      }
    } else {
      const unsigned o = frag_off<32>(lane, 32 * FB * wf);
#pragma unroll
      for (int s = 0; s < KS; ++s) oa[s] = o ^ (32u * (KS * wk + s));
    }
  }
  bf16x8 fa[KS][FB][3], fbk[KS][TB][3];
  // k-step s of a stage in one term or three
  auto fragments = [&](const unsigned char* base, int s, auto terms) {
#pragma unroll
    for (int p = 0; p < decltype(terms)::value; ++p) {
#pragma unroll
      for (int fb = 0; fb < FB; ++fb) {
        if constexpr (NN) {
          auto tr = [&](int j) {
            return __builtin_amdgcn_ds_read_tr16_b64_v4bf16((bf16x4 GLACIER_LDS*)const_cast<unsigned char*>(
                base + oa[2 * fb + j] + kPlaneA * p + 2048 * s));
          };
          fa[s][fb][p] = join8(tr(0), tr(1));
        } else {
          fa[s][fb][p] = *reinterpret_cast<const bf16x8*>(base + oa[s] + kPlaneA * p + 2048 * fb);
        }
      }
#pragma unroll
      for (int tb = 0; tb < TB; ++tb)
        fbk[s][tb][p] = *reinterpret_cast<const bf16x8*>(base + ob[s] + kPlaneB * p + 2048 * tb);
    }
  };
  auto products = [&](int s, auto terms) {
    // the small products first
    constexpr int kPa[6] = {2, 0, 1, 1, 0, 0}, kPb[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
    for (int q = decltype(terms)::value == 1 ? 5 : 0; q < 6; ++q)
#pragma unroll
      for (int fb = 0; fb < FB; ++fb)
#pragma unroll
        for (int tb = 0; tb < TB; ++tb) {
          f32x16& sum = kApart && q < 5 ? small[fb][tb] : acc[fb][tb];
          sum = mma32(fa[s][fb][kPa[q]], fbk[s][tb][kPb[q]], sum);
        }
  };
  // Stage n in buffer n % 2: its fragments are read, the next stage's pieces
  // split and written to the other buffer (every wave is past its reads of it)
  // behind those reads, then come the products, then the barrier that makes
  // the next stage's rows visible.
  int n = 0;
  auto turn = [&](auto terms, auto&& next) {
    const unsigned char* base = lds + (n & 1) * kBuf;
    fragments(base, 0, terms);
    ++n;
    next(lds + (n & 1) * kBuf);
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      if (s > 0) fragments(base, s, terms);
      products(s, terms);
    }
    lgkm<0>();
    wg_barrier();
  };
  constexpr std::integral_constant<int, 3> kThree{};
  constexpr std::integral_constant<int, kOne ? 1 : 3> kBase{};
  BasePieces ring[PF];
  {
    Pieces low;
    if (low_st > 0) load_low(0, low);
    static_for<PF>([&](auto jc) { load(decltype(jc)::value, ring[decltype(jc)::value]); });
    if (low_st > 0) {
      put_all(lds, low);
      if (low_st > 1) load_low(1, low);
      lgkm<0>();
      wg_barrier();
      for (int st = 1; st < low_st; ++st)
        turn(kThree, [&](unsigned char* base) {
          put_all(base, low);
          if (st + 1 < low_st) load_low(st + 1, low);
        });
      turn(kThree, [&](unsigned char* base) { put_all(base, ring[0]); });
    } else {
      put_all(lds, ring[0]);
      lgkm<0>();
      wg_barrier();
    }
    load(PF, ring[0]);
  }
  settle(acc);
  if constexpr (kApart) settle(small);
  for (int st0 = 0; st0 < nst; st0 += PF) {
    static_for<PF>([&](auto jc) {
      // stages past the end hold zeros (no valid element), and add nothing
      constexpr int J = (decltype(jc)::value + 1) % PF;
      turn(kBase, [&](unsigned char* base) {
        put_all(base, ring[J]);
        load(st0 + decltype(jc)::value + 1 + PF, ring[J]);
      });
    });
    settle(acc);
    if constexpr (kApart) settle(small);
  }
  if constexpr (kApart) {
#pragma unroll
    for (int fb = 0; fb < FB; ++fb)
#pragma unroll
      for (int tb = 0; tb < TB; ++tb) acc[fb][tb] += small[fb][tb];
  }
  if (__syncthreads_or(mark.bad())) {
    // the same sums on fp32 MFMAs: lane l supplies A[row l % 32][k + l / 32]
    // and B's column likewise; group 0 sums everything
    clear();
    if (wk == 0) {
      for (int i = 2 * seg0; i < 2 * seg1; ++i) {
        const int y = i / 2;
        const bool low = i & 1;
        const GemmJob& job = a.j[y];
        const int len = !low ? a.seg[y].k : job.l == nullptr ? 0 : rank;
#pragma clang loop unroll(disable)
        for (int k0 = 0; k0 < len; k0 += 2) {
          const int k = min(k0 + (lane >> 5), len - 1);
          const bool ok = k0 + (lane >> 5) < len;
          float va[FB], vb[TB];
#pragma unroll
          for (int fb = 0; fb < FB; ++fb) {
            const int f = min(fw + 32 * fb + (lane & 31), nf - 1);
            const float v = low ? (NN ? job.v[(long)f * rank + k] : job.v[(long)k * nf + f])
                                : (float)static_cast<const IO*>(a.seg[y].a)[NN ? (long)k * K + f : (long)f * len + k];
            va[fb] = ok ? v : 0.0f;
          }
#pragma unroll
          for (int tb = 0; tb < TB; ++tb) {
            const long at = (long)min(tw + 32 * tb + (lane & 31), T - 1) * len + k;
            const float v = low ? job.s * job.l[at] : (float)static_cast<const IO*>(a.seg[y].b)[at];
            vb[tb] = ok ? v : 0.0f;
          }
#pragma unroll
          for (int fb = 0; fb < FB; ++fb)
#pragma unroll
            for (int tb = 0; tb < TB; ++tb)
              acc[fb][tb] = __builtin_amdgcn_mfma_f32_32x32x2f32(va[fb], vb[tb], acc[fb][tb], 0, 0, 0);
        }
      }
    }
  }
  merge_groups<FB, TB, WK>(acc, lds, w % (WF * WT), wk, lane);
  IO* out = static_cast<IO*>(NN ? a.dx : a.j[z].y);
#pragma unroll
  for (int tb = 0; tb < TB; ++tb) {
    const int t = tw + 32 * tb + (lane & 31);
    if (t >= T) continue;
#pragma unroll
    for (int fb = 0; fb < FB; ++fb) {
      if (block_owner<FB, TB, WK>(fb, tb) != wk) continue;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int f = fw + 32 * fb + 8 * q + 4 * (lane >> 5);
        if (f < nf)  // nf % 4 == 0
          store4(out + (long)t * nf + f,
                 f32x4{acc[fb][tb][4 * q], acc[fb][tb][4 * q + 1], acc[fb][tb][4 * q + 2], acc[fb][tb][4 * q + 3]});
      }
    }
  }
#endif
}

// Tile shapes (features x tokens), the times a stage of theirs was measured
// to take, and their instances.  us per launch, forward / backward (rank 16):
//   T, in -> outs                    256x256  128x128/2  128x128  128x64  64x64
//   4096, 4096 -> 4096               137/138  162/174    182/193  219/237 278/295
//   4096, 4096 -> 4096/1024/1024     225/202  228/244    259/272  314/339 406/418
//   1290, 3584 -> 3584/512/512       82/108   59/69      67/88    76/94   97/103
//   512, 3584 -> 3584/512/512        76/105   44/58      33/45    42/36   44/44
//   201, 896 -> 896/128/128          24/31    11/15      12/16    9.5/12  7.9/9.9
//   37, 3584 -> 3584/512/512         72/100   40/51      28/40    20/31   16/21
struct GemmShape {
  int slots;            // workgroups resident at once
  float alone, loaded;  // us per 64 reduction elements: few workgroups, every slot taken
  int kt;
  int ft, tt;
  void (*nt)(GemmCall);
  void (*nn)(GemmCall);
};
#define GL_GEMM(SLOTS, ALONE, LOADED, KT, FB, TB, WF, WT, WK, G, RING)                                                       \
  GemmShape { SLOTS, ALONE, LOADED, KT, 32 * FB * WF, 32 * TB * WT, proj_gemm_kernel<false, KT, FB, TB, WF, WT, WK, G, RING>,  \
              proj_gemm_kernel<true, KT, FB, TB, WF, WT, WK, G, RING> }
const GemmShape kShapes[] = {
    GL_GEMM(256, 1.20f, 2.00f, 64, 4, 2, 2, 4, 1, 1, 2),   // 256 x 256
    GL_GEMM(512, 0.68f, 1.20f, 64, 2, 2, 2, 2, 2, 1, 2),   // 128 x 128, two per CU
    GL_GEMM(256, 0.50f, 0.66f, 64, 2, 2, 2, 2, 2, 2, 4),   // 128 x 128
    GL_GEMM(256, 0.34f, 0.43f, 128, 2, 1, 2, 2, 2, 2, 3),  // 128 x 64
    GL_GEMM(256, 0.23f, 0.27f, 128, 1, 1, 2, 2, 2, 4, 5),  // 64 x 64
};
#undef GL_GEMM

int tiles_of(const GemmCall& a, bool nn, const GemmShape& s) {
  int ftiles = 0;
  if (nn)
    ftiles = (a.K + s.ft - 1) / s.ft;
  else
    for (int z = 0; z < a.n; ++z) ftiles += (a.j[z].n + s.ft - 1) / s.ft;
  return ftiles * ((a.T + s.tt - 1) / s.tt);
}

// The shape with the least estimated time: rounds of the CUs times the time
// of a stage, which grows with the share of the chip at work (the clock falls
// under load).  One pair of times serves both directions: the order of the
// shapes is what they have to tell, and the table's rows bear it out in both.
int gemm_shape(const GemmCall& a, bool nn) {
  int best = 0;
  float best_t = 0.0f;
  for (int i = 0; i < (int)(sizeof(kShapes) / sizeof(kShapes[0])); ++i) {
    const GemmShape& s = kShapes[i];
    const int tiles = tiles_of(a, nn, s), full = tiles / s.slots, rest = tiles % s.slots;
    const float t = full * s.loaded + (rest > 0 ? s.alone + (s.loaded - s.alone) * rest / s.slots : 0.0f);
    if (i == 0 || t < best_t) best = i, best_t = t;
  }
  return best;
}

hipError_t launch_gemm_shape(GemmCall a, bool nn, int shape, hipStream_t st) {
  const GemmShape& s = kShapes[shape];
  a.ftiles = 0;
  if (nn) {
    a.ftiles = (a.K + s.ft - 1) / s.ft;
  } else {
    for (int z = 0; z < a.n; ++z) {
      a.j[z].first = a.ftiles;
      a.ftiles += (a.j[z].n + s.ft - 1) / s.ft;
    }
  }
  const int ttiles = (a.T + s.tt - 1) / s.tt;
  if (ttiles == 0 || a.ftiles == 0) return hipSuccess;
  hipLaunchKernelGGL(nn ? s.nn : s.nt, dim3(a.ftiles * ttiles), dim3(kGThreads), 0, st, a);
  return hipGetLastError();
}

template <typename IO, bool NN>
hipError_t launch_split(GemmCall a, hipStream_t st) {
  // 128 x 128 tiles (one workgroup a CU) once they are more than the 64 x 64 ones
  // that fit the chip at once: half of its CUs, as fp32 tensors have one of those
  // on a CU of twice the time, bf16 tensors two.  Time at 128 x 128 over time at
  // 64 x 64, forward and backward: fp32 32-64 tiles 1.50-1.76, 72-112 0.92-1.02,
  // 128 0.95, 144-192 0.71, over that 0.72-0.87 (264: 1.06); bf16 up to 116 tiles
  // 1.05-1.42, 128 1.08-1.14, 132-256 0.82-0.84 (1.07 at 132 with 1000 inputs),
  // over that 0.69-1.05.
  constexpr int kBigTiles = sizeof(IO) == 2 ? 129 : 128;
  auto tiles = [&](int ft) {
    a.ftiles = 0;
    for (int z = 0; z < (NN ? 1 : a.n); ++z) {
      a.j[z].first = a.ftiles;
      a.ftiles += ((NN ? a.K : a.j[z].n) + ft - 1) / ft;
    }
    return a.ftiles * ((a.T + ft - 1) / ft);
  };
  // bf16 rows of 4 elements: no 8 to load at once
  bool tiny = a.K < 8;
  for (int z = 0; z < a.n; ++z) tiny = tiny || a.j[z].n < 8;
  tiny = tiny && sizeof(IO) == 2;
  int n = tiles(128);
  const bool big = n >= kBigTiles && !tiny;
  if (!big) n = tiles(64);
  if (n == 0) return hipSuccess;
  auto fn = big ? proj_gemm_split_kernel<IO, NN, false, 2, 1, 2, 4, 1, 2>
                : proj_gemm_split_kernel<IO, NN, false, 1, 1, 2, 2, 2, 4>;
  if constexpr (sizeof(IO) == 2)
    if (tiny) fn = proj_gemm_split_kernel<IO, NN, true, 1, 1, 2, 2, 2, 4>;
  hipLaunchKernelGGL(fn, dim3(n), dim3(kGThreads), 0, st, a);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_gemm(GemmCall a, bool nn, hipStream_t st) {
  return launch_gemm_shape(a, nn, gemm_shape(a, nn), st);
}

hipError_t launch_gemm_split(const GemmCall& a, bool nn, bool io_bf16, hipStream_t st) {
  if (io_bf16) return nn ? launch_split<bf16, true>(a, st) : launch_split<bf16, false>(a, st);
  return nn ? launch_split<float, true>(a, st) : launch_split<float, false>(a, st);
}

}  // namespace glacier
