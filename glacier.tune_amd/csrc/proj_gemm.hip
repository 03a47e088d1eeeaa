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
__device__ inline int xcd_logical(int id, int total) {
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
// A call that holds a non-finite value there (its marks, `odd`) takes fp32
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
  // a non-finite value among the low-rank operands: see below
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
    // the low-rank products of a call with non-finite values, which have no
    // split terms: sum over the terms of (s L [T][r]) V, V = B [r][n]
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

  // Epilogue.  WK == 2: each group hands the other the blocks that one
  // finishes, and adds its own to what it receives (group 0's first).
  __syncthreads();
  if constexpr (WK == 2) {
    f32x4* ex = reinterpret_cast<f32x4*>(lds) + (w % (WF * WT)) * (FB * TB * 256);
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
  // bias, bf16, and out through LDS: 32 tokens x 32 FB features per wave at a
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
// Every other projection (fp32 tensors, the fp32-operand mode, or bf16
// tensors of a shape neither kernel above takes): both directions on
// v_mfma_f32_16x16x4f32, any shape, operands converted to fp32 on load.  A workgroup computes a 64-feature x
// 64-token tile of C^T, 4 waves of 32 x 32 (2 x 2 blocks of 16 x 16).
// Stages of 32 reduction elements go global -> registers -> LDS (two
// buffers, one barrier per stage, the next stage's loads in flight during
// the products); elements past any edge load as zero.
//   forward  (NT) C^T[f][t] = sum_k W[f][k] X[t][k]   (A tile [f][k])
//   backward (NN) C^T[c][t] = sum_z sum_f W_z[f][c] dY_z[t][f]   (A tile [f][c])
// MFMA layout (lane l, c = l % 16, g = l / 16): A[row c][k = g],
// B[k = g][col c]; accumulator i holds column c, row 4 g + i: four
// consecutive features of one token.
// ---------------------------------------------------------------------------
constexpr int kFT = 64;       // features and tokens per tile
constexpr int kFK = 32;       // reduction elements per stage
constexpr int kFS = kFK + 4;  // row stride of [row][k] tiles (floats): conflict-free
constexpr int kFC = kFT + 16; // row stride of the backward's [k][feature] tile
constexpr int kFThreads = 256;

// Four elements k .. k + 3 of a row (len elements valid) as fp32, zero past
// the end; vec: the row allows one aligned vector load.
template <typename IO>
__device__ inline f32x4 load4_f32(const IO* row, int k, int len, bool vec) {
  if (vec && k + 3 < len) {
    if constexpr (sizeof(IO) == 4) {
      return *reinterpret_cast<const f32x4*>(row + k);
    } else {
      const bf16x4 h = *reinterpret_cast<const bf16x4*>(row + k);
      return f32x4{(float)h[0], (float)h[1], (float)h[2], (float)h[3]};
    }
  }
  f32x4 v;
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = k + i < len ? (float)row[k + i] : 0.0f;
  return v;
}

template <typename IO, bool NN>
__global__ __launch_bounds__(kFThreads) void proj_gemm_f32_kernel(const WideFwd fa, const WideBwd ba) {
  __shared__ __align__(16) float la[2][NN ? kFK * kFC : kFT * kFS];
  __shared__ __align__(16) float lb[2][kFT * kFS];
  const int T = NN ? ba.T : fa.T;
  const int nout = NN ? ba.K : fa.n;  // C^T rows: features
  const int ttiles = (T + kFT - 1) / kFT;
  const int id = xcd_logical((int)blockIdx.x, (int)gridDim.x);
  const int t0 = kFT * (id % ttiles), f0 = kFT * (id / ttiles);
  const int tid = threadIdx.x, lane = tid & 63, w = wave_id();
  const int wf = w & 1, wt = w >> 1, c = lane & 15, g = lane >> 4;
  // stages: forward over K; backward over every job's outputs in turn
  int nst = 0;
  if constexpr (NN) {
    for (int z = 0; z < ba.n; ++z) nst += (ba.j[z].n + kFK - 1) / kFK;
  } else {
    nst = (fa.K + kFK - 1) / kFK;
  }
  f32x4 ra[2], rb[2];
  auto load = [&](int st) {
    const IO* wsrc;
    const IO* bsrc;
    int k0, klen, bstride;
    if constexpr (NN) {
      int z = 0, base = 0;
      while (z + 1 < ba.n && st >= base + (ba.j[z].n + kFK - 1) / kFK) base += (ba.j[z++].n + kFK - 1) / kFK;
      k0 = kFK * (st - base);
      klen = ba.j[z].n;
      wsrc = static_cast<const IO*>(ba.j[z].w);
      bsrc = static_cast<const IO*>(ba.j[z].dy);
      bstride = klen;
    } else {
      k0 = kFK * st;
      klen = fa.K;
      wsrc = static_cast<const IO*>(fa.w);
      bsrc = static_cast<const IO*>(fa.x);
      bstride = fa.K;
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int idx = tid + kFThreads * i;
      if constexpr (NN) {
        // A: W_z rows k0 + idx / 16 (of klen), columns f0 + 4 (idx % 16)
        const int kr = k0 + (idx >> 4), cc = f0 + 4 * (idx & 15);
        ra[i] = kr < klen ? load4_f32(wsrc + (long)kr * ba.K, cc, nout, (ba.K & 3) == 0) : f32x4{0, 0, 0, 0};
      } else {
        // A: W rows f0 + idx / 8, columns k0 + 4 (idx % 8)
        const int fr = f0 + (idx >> 3), kc = k0 + 4 * (idx & 7);
        ra[i] = fr < nout ? load4_f32(wsrc + (long)fr * fa.K, kc, klen, (fa.K & 3) == 0) : f32x4{0, 0, 0, 0};
      }
      // B: rows t0 + idx / 8 (tokens), columns k0 + 4 (idx % 8)
      const int tr = t0 + (idx >> 3), kc = k0 + 4 * (idx & 7);
      rb[i] = tr < T ? load4_f32(bsrc + (long)tr * bstride, kc, klen, (bstride & 3) == 0) : f32x4{0, 0, 0, 0};
    }
  };
  auto store = [&](int buf) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int idx = tid + kFThreads * i;
      if constexpr (NN)
        *reinterpret_cast<f32x4*>(&la[buf][(idx >> 4) * kFC + 4 * (idx & 15)]) = ra[i];
      else
#pragma unroll
        for (int e = 0; e < 4; ++e) la[buf][(idx >> 3) * kFS + 4 * (idx & 7) + e] = ra[i][e];
#pragma unroll
      for (int e = 0; e < 4; ++e) lb[buf][(idx >> 3) * kFS + 4 * (idx & 7) + e] = rb[i][e];
    }
  };
  f32x4 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  if (nst > 0) {
    load(0);
    store(0);
  }
  __syncthreads();
  for (int st = 0; st < nst; ++st) {
    const int buf = st & 1;
    if (st + 1 < nst) load(st + 1);
#pragma unroll
    for (int kk = 0; kk < kFK / 4; ++kk) {
      float av[2], bv[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int fr = 32 * wf + 16 * i + c, tr = 32 * wt + 16 * i + c, k = 4 * kk + g;
        av[i] = NN ? la[buf][k * kFC + fr] : la[buf][fr * kFS + k];
        bv[i] = lb[buf][tr * kFS + k];
      }
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[i], bv[j], acc[i][j], 0, 0, 0);
    }
    if (st + 1 < nst) store(buf ^ 1);
    __syncthreads();
  }
  // C [T][nout]: token t0 + 32 wt + 16 j + c, features f0 + 32 wf + 16 i + 4 g ..
  float* cdst = NN ? ba.c : fa.c;
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int t = t0 + 32 * wt + 16 * j + c;
    if (t >= T) continue;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int f = f0 + 32 * wf + 16 * i + 4 * g;
      float* d = cdst + (long)t * nout + f;
      if (f + 3 < nout && (nout & 3) == 0) {
        *reinterpret_cast<f32x4*>(d) = acc[i][j];
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (f + e < nout) d[e] = acc[i][j][e];
      }
    }
  }
}

}  // namespace

namespace {

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
// under load).
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

}  // namespace

hipError_t launch_gemm(GemmCall a, bool nn, hipStream_t st) {
  return launch_gemm_shape(a, nn, gemm_shape(a, nn), st);
}

hipError_t launch_generic_fwd(const WideFwd& a, bool io_bf16, hipStream_t st) {
  const int ttiles = (a.T + kFT - 1) / kFT, ftiles = (a.n + kFT - 1) / kFT;
  if (ttiles == 0 || ftiles == 0) return hipSuccess;
  auto fn = io_bf16 ? proj_gemm_f32_kernel<bf16, false> : proj_gemm_f32_kernel<float, false>;
  hipLaunchKernelGGL(fn, dim3(ttiles * ftiles), dim3(kFThreads), 0, st, a, WideBwd{});
  return hipGetLastError();
}

hipError_t launch_generic_bwd(const WideBwd& a, bool io_bf16, hipStream_t st) {
  const int ttiles = (a.T + kFT - 1) / kFT, ftiles = (a.K + kFT - 1) / kFT;
  if (ttiles == 0 || ftiles == 0 || a.n == 0) return hipSuccess;
  auto fn = io_bf16 ? proj_gemm_f32_kernel<bf16, true> : proj_gemm_f32_kernel<float, true>;
  hipLaunchKernelGGL(fn, dim3(ttiles * ftiles), dim3(kFThreads), 0, st, WideFwd{}, a);
  return hipGetLastError();
}

}  // namespace glacier
