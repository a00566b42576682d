// K6: split-activation GEMM for prompt-sized row counts (prefill) on bf16 MFMA (gfx950), with
// the RMSNorm of its input in the prologue and the SwiGLU gate or the residual add in the
// epilogue, so a prefill layer needs no fp32 gate / up round trip and no add+RMSNorm pass.
//
//   acc[m, n] (fp32) = sum_k (a_hi[m, k] + a_lo[m, k]) * w[n, k],   k < K
//
// w: bf16 [N, K] in the MFMA tile layout (MDL_LAYOUT_TILES, the decode copies of the weights).
// a (AMODE): A_ROWS  split [M, 2K] row-major (hi in [0, K), lo in [K, 2K)), row stride lda;
//            A_TILES the same matrix in the tile layout;
//            A_NORM  split(x * gamma) of the fp32 residual stream x [M, K] in the fp32 tile
//                    layout, formed after the LDS read; the block sees whole rows, so it sums
//                    x^2 and has rstd.
// AP (activation parts) 1 drops the lo term: A_ROWS / A_TILES then hold hi alone ([M, K]),
// A_NORM uses bf16(x * gamma); half the MFMAs and, for the split forms, a third fewer loads.
// epilogue (EPI): E_STORE     out = acc (fp32 row-major; with A_NORM also rstd[m]);
//                 E_SWIGLU    h = split(silu(rstd g + b_g) * (rstd u + b_u)) from the gate / up
//                             accumulator pairs (weights with 16-row gate / up blocks
//                             interleaved), h [M, 2F] in the tile layout (h_parts 1: hi alone,
//                             [M, F], for a consumer with AP 1);
//                 E_RESIDUAL  x[m, n] += acc (+ bias[n]) in place, x [M, N] in the fp32 tile
//                             layout;
//                 E_QKV       K2 on the qkv accumulators (A_NORM): rstd, 3D RoPE of q and k, the
//                             softmax scale on q; q bf16 [M, d], K / V bf16 into their cache
//                             slots, and fp32 acc only for the lead rows (the first `lead` tokens
//                             of each row, which the exact lead-attention pass reads).
//
// Block: a tile of activation rows x weight rows (see Shape), e.g. 128 x 256 on 4 waves, each
// owning 32 MFMA tiles (128 fp32 accumulators per lane): 64 rows x 128 weight rows in a 2 x 2 wave
// grid for the split forms, 32 rows x 256 weight rows (4 x 1) for A_NORM.  K advances through a
// ring of LDS stages; a k-step of 32 of this tile is 32 KB: 16 weight fragments and 16 activation
// fragments of 1 KB in MFMA lane order (bf16 {hi, lo} of 8 row blocks; for A_NORM the fp32 x of
// 8 row blocks in the fp32 tile layout, split after the read), so every fragment read is one
// conflict-free 16-byte LDS read per lane.  Global data goes straight to LDS
// (global_load_lds_dwordx4, 16 bytes per lane, one kilobyte per wave instruction), issued RING - 1
// stages ahead; nothing is staged in registers, and a stage ends with one barrier after an exact
// vmcnt wait for the next stage's loads.
//
// What bounds it.  A CU takes in one such copy every 25-32 cycles, and a wave issues in order: the
// copies of a stage handed out in one go, each with a chain of address arithmetic before it, held
// back the MFMAs behind them until all were accepted, and a block took the sum of its copy time
// and its MFMA time (down projection at 731 rows of d = 768, F = 2048, 64 x 64 tiles, us: 25 whole,
// 12 without the MFMAs, 9 without the copies).  So each copy has a scalar pointer that it moves
// on by itself, and the shapes that run one or two tiles per CU spread a stage's copies over its
// MFMAs (17 in that test, 13 with four k-steps a stage).
// At prompt sizes the chip's power is the limit: 282,695 rows' down projection keeps its MFMAs
// busy 78% of the cycles, at 1.4 GHz.  There two blocks of 128 x 256 per CU, their copies ahead of
// the MFMAs at an even pace, take the least time: one block's LDS reads and epilogues run under
// the other's MFMAs.  Against one block of 256 x 256 on 8 waves (the same fragment reads per MFMA,
// a quarter fewer copies), us per launch (qkv / out / gate-up / down): 2,059 / 712 / 3,351 / 1,507
// -> 1,974 / 666 / 3,240 / 1,375 at 282,695 rows, 157 / 50 / 227 / 103 -> 132 / 43 / 195 / 86 at
// 16,669.
//
// Blocks are persistent (each walking its tiles), and the load ring runs on across tile
// boundaries, so a tile's epilogue overlaps the next tile's first loads.  Every weight
// fragment feeds two MFMAs (hi and lo rows), as in K5.  Blocks are numbered so that an XCD (block
// i runs on XCD i mod 8) takes a contiguous run of tiles, row tile major: the N tiles of one row
// tile share its activation rows in one L2.  Summation order is fixed (k-steps in order, hi
// before lo), so results are reproducible, and it is the same in every shape: a row's results do
// not depend on how many rows run beside it.  The forms for fp32 weights take K5's order (eight
// runs of k-steps, each summed from zero, added in order), because a few rows run on K5.
#include <algorithm>

#include <type_traits>

#include "common.h"
#include "lds_dma.h"
#include "mfma.h"
#include "rope.h"

namespace mdl {

namespace {

// A block shape: a BM x BN output tile on WMW x WNW waves, K through a ring of RING LDS stages of
// KS k-steps (of 32) each (K a multiple of 32 KS); the blocks that fit a CU's LDS and registers
// together are OCC.  SPREAD: the copies of a stage go out between the MFMAs of a step, otherwise
// ahead of them.  GK: the largest K of the norm forms (gamma lives in LDS).
template <int BM_, int BN_, int WMW_, int WNW_, int KS_, int RING_, int OCC_, bool SPREAD_,
          int GK_ = 2048>
struct Shape {
  static constexpr int BM = BM_, BN = BN_, WMW = WMW_, WNW = WNW_, KS = KS_, RING = RING_;
  static constexpr int OCC = OCC_, NW = WMW_ * WNW_, GK = GK_;
  static constexpr bool SPREAD = SPREAD_;
};
constexpr int kMaxNormK = 2048;   // the norm forms' largest K

enum AMode { A_ROWS = 0, A_TILES = 1, A_NORM = 2 };
enum Epi { E_STORE = 0, E_SWIGLU = 1, E_RESIDUAL = 2, E_QKV = 3 };

struct Args {
  const uint16_t* a;   // A_ROWS / A_TILES
  int64_t lda;
  const float* x;      // A_NORM: [M, K] in the fp32 tile layout
  const float* gamma;
  float eps;
  const uint16_t* w;   // tiled [N, K]
  const uint16_t* wl;  // WL forms: low bf16 part of an fp32 weight, tiled like w
  float* out;          // E_STORE
  int64_t ldo;
  float* rstd_out;     // E_STORE with A_NORM (may be NULL)
  const float* bias_a; // E_SWIGLU gate bias / E_RESIDUAL bias (may be NULL)
  const float* bias_b; // E_SWIGLU up bias (may be NULL)
  uint16_t* h;         // E_SWIGLU: tiled [M, h_parts d_ff] (hi, then lo when h_parts is 2)
  int d_ff, h_parts;
  float* x_res;        // E_RESIDUAL: [M, N] in the fp32 tile layout
  // E_QKV: row m is token slot tok_slot[m] of batch row tok_row[m] (packed), or slot m % seq of
  // row m / seq; out (may be NULL) receives the lead rows' fp32 acc
  const int64_t* pos;
  const float* rope_tab;
  RopeArgs ra;
  float q_scale;
  void* q_out;   // bf16, or fp32 with fp32 weights (WL), like the caches
  void* kc;
  void* vc;
  const int32_t* tok_row;
  const int32_t* tok_slot;
  const int32_t* kv_start;
  int slots, seq, batch, lead;
  int M, N, K, tiles_n, tiles, per_xcd;
};

// Wait until at most N of this wave's global memory operations are in flight, then a block
// barrier that also waits for this wave's LDS traffic; the memory clobbers keep the compiler from
// moving LDS accesses across either.  N counts the copies issued for later stages; any other
// load or store the wave issued after this stage's copies (epilogue traffic of the previous
// tile) only makes the wait stricter.
template <int N>
__device__ __forceinline__ void stage_barrier() {
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_waitcnt lgkmcnt(0)\n\ts_barrier" :: "n"(N) : "memory");
}

// The epilogue's own loads are used here, on every path: a load whose value only a branch uses is
// still in flight for the compiler where that branch is not taken, and it then waits for it at the
// first reuse of its registers, in the middle of the next tile's k-loop and on every pass through
// it, where vmcnt(0) also waits for the copies of the stages ahead.
__device__ __forceinline__ void landed(float v) { asm volatile("" ::"v"(v)); }
__device__ __forceinline__ void landed(const float4& v) {
  asm volatile("" ::"v"(v.x), "v"(v.y), "v"(v.z), "v"(v.w));
}

template <int AMODE, int EPI, int AP, bool WL, class S>
__global__ __launch_bounds__(64 * S::NW, S::NW * S::OCC / 4) void prefill_gemm_kernel(
    const Args p) {
  static_assert(AP == 1 || AP == 2, "activation parts: hi, or hi and lo");
  static_assert(!WL || AP == 2, "the low weight part goes with split activations");
  constexpr int kBM = S::BM, kBN = S::BN, kWaves = S::NW, kThreads = 64 * S::NW;
  constexpr int KS = S::KS, kRing = S::RING;
  // fragments of 1 KB in one k-step of a stage: {hi, lo} (A_NORM: the two kilobytes of fp32) of
  // each row block, then the weight row blocks, then (WL) their low parts
  constexpr int kAFrags = (kBM / 16) * 2, kWFrags = kBN / 16 * (WL ? 2 : 1);
  constexpr int kStep = (kAFrags + kWFrags) * 1024, kStage = KS * kStep;
  // copies per wave and stage; the split forms with the hi part alone make half the activation's
  constexpr bool kHiOnly = AMODE != A_NORM && AP == 1;
  constexpr int kACopies = KS * kAFrags / (kHiOnly ? 2 : 1) / kWaves;
  constexpr int kWCopies = KS * kWFrags / kWaves;
  constexpr int kLoads = kACopies + kWCopies;
  static_assert(kACopies * kWaves * (kHiOnly ? 2 : 1) == KS * kAFrags &&
                kWCopies * kWaves == KS * kWFrags, "every wave makes the same copies");
  constexpr int kGammaBytes = AMODE == A_NORM ? S::GK * 4 : 0;
  __shared__ __align__(16) uint8_t lds[kRing * kStage + kGammaBytes];
  __shared__ float rstd_s[kBM];
  // Persistent blocks: XCD x = blockIdx % 8 owns logical tiles [x per_xcd, (x + 1) per_xcd), row
  // tile major; its bpx blocks take every bpx-th of them, so the XCD's CUs work on consecutive
  // tiles at any time.
  const int bpx = gridDim.x >> 3;
  const int t_lo = (blockIdx.x & 7) * p.per_xcd;
  const int t_hi = min(t_lo + p.per_xcd, p.tiles);
  const int first = t_lo + (blockIdx.x >> 3);
  if (first >= t_hi) return;   // whole block, before any barrier
  const int M = p.M, N = p.N, K = p.K, nk = K >> 5;
  const int ns = nk / KS;                                  // stages per tile
  const int total = (t_hi - first + bpx - 1) / bpx * ns;   // stages over this block's tiles
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // wave grid WMW x WNW over the tile: wave (wm, wn) owns FM row blocks and FN weight fragments.
  // The A_NORM forms split x * gamma in registers after the LDS read, so there every row block
  // belongs to one wave (WNW 1) and is converted once; the split forms of the large shape use
  // 2 x 2 (8 activation and 8 weight fragment reads per wave and k-step).
  constexpr int WMW = S::WMW, WNW = S::WNW;
  constexpr int FM = kBM / 16 / WMW, FN = kBN / 16 / WNW;
  const int wm = wave % WMW, wn = wave / WMW;
  const int c = lane & 15, g = lane >> 4;
  const int last_nb = (N + 15) / 16 - 1, last_mb = (M + 15) / 16 - 1;
  const uint32_t lds0 = lds_addr(lds);

  // The copies of a stage: the waves take its fragments in turn.  Weight fragment f is row block
  // n0 / 16 + f (WL: f / 2, part f % 2, hi / lo); activation fragment f is row block f / 2, part
  // f % 2 (hi / lo; for A_NORM the first or second kilobyte of the fp32 16 x 32 block, lane l's
  // columns 0..3 or 4..7); with the hi part alone (AP 1, split forms) only the even f exist.
  // Fragment f lands in slot f of its k-step either way.  Every copy is one contiguous kilobyte
  // per wave, except row-major A.  Row blocks past M or N load valid memory (clamped to the last;
  // tile-layout buffers hold its padding rows); their results are never used.
  //
  // `seek` finds each copy's first address in a tile, a scalar pointer, and `copy` makes it and
  // moves the pointer on: six scalar instructions.  Found anew each time the address is a chain of
  // a dozen (two clamps, 64-bit multiplies) in front of every copy.
  const uint8_t* wsrc[kWCopies];
  const uint8_t* asrc[AMODE == A_ROWS ? 1 : kACopies];
  const uint32_t lane16 = 16 * lane;
  constexpr int kPer = kHiOnly ? kAFrags / 2 : kAFrags;   // activation fragments of a k-step
  constexpr int kXStep = AMODE == A_NORM ? 2048 : 1024;   // bytes of an activation block's k-step
  int am0 = 0, as = 0;                                    // A_ROWS: the cursor itself
  auto seek = [&](int m0, int n0) {
#pragma unroll
    for (int j = 0; j < kWCopies; ++j) {
      const int f = kWaves * j + wave, ks = f / kWFrags, fw = f - ks * kWFrags;
      const int nb = min(n0 / 16 + (WL ? fw >> 1 : fw), last_nb);
      const uint16_t* src = WL && (fw & 1) ? p.wl : p.w;
      wsrc[j] = reinterpret_cast<const uint8_t*>(src) + (static_cast<int64_t>(nb) * nk + ks) * 1024;
    }
    if constexpr (AMODE == A_ROWS) {
      am0 = m0;
      as = 0;
    } else {
#pragma unroll
      for (int j = 0; j < kACopies; ++j) {
        const int fa = kWaves * j + wave, ks = fa / kPer;
        const int f = (kHiOnly ? 2 : 1) * (fa - ks * kPer), rb = f >> 1, part = f & 1;
        const int64_t blk = min(m0 / 16 + rb, last_mb);
        if constexpr (AMODE == A_NORM)
          asrc[j] = reinterpret_cast<const uint8_t*>(p.x) + (blk * nk + ks) * 2048 + part * 1024;
        else
          asrc[j] = reinterpret_cast<const uint8_t*>(p.a) +
                    (blk * AP * nk + part * nk + ks) * 1024;
      }
    }
  };
  auto copy = [&](int q, uint32_t base) {   // copy q < kLoads of the stage at LDS address base
    if (q < kWCopies) {
      const int f = kWaves * q + wave, ks = f / kWFrags, fw = f - ks * kWFrags;
      dma16_free(wsrc[q], lane16,
                 __builtin_amdgcn_readfirstlane(base + ks * kStep + (kAFrags + fw) * 1024));
      wsrc[q] += KS * 1024;
    } else {
      const int j = q - kWCopies;
      const int fa = kWaves * j + wave, ks = fa / kPer;
      const int f = (kHiOnly ? 2 : 1) * (fa - ks * kPer), rb = f >> 1, part = f & 1;
      const uint32_t dst = __builtin_amdgcn_readfirstlane(base + ks * kStep + f * 1024);
      if constexpr (AMODE == A_ROWS) {
        const int row = min(am0 + 16 * rb + c, M - 1);
        dma16(p.a + static_cast<int64_t>(row) * p.lda + part * K + 32 * (KS * as + ks) + 8 * g,
              dst);
      } else {
        dma16_free(asrc[j], lane16, dst);
        asrc[j] += KS * kXStep;
      }
    }
  };

  const float* gam_s = reinterpret_cast<const float*>(lds + kRing * kStage);
  if constexpr (AMODE == A_NORM) {
    float* gw = reinterpret_cast<float*>(lds + kRing * kStage);
    for (int i = tid; i < K; i += kThreads) gw[i] = p.gamma[i];
    __syncthreads();   // before any stage load is in flight (it waits for every load)
  }

  f32x4_t acc[FN][FM];
  float ss[FM];   // A_NORM: this lane's part of sum(x^2) of row 16 (FM wm + j) + c
  // WL: the sums of the runs of k-steps before this one (acc and ss are of the present run)
  f32x4_t tot[WL ? FN : 1][WL ? FM : 1];
  float ss_tot[WL ? FM : 1];
  auto clear = [&]() {
#pragma unroll
    for (int i = 0; i < FN; ++i)
#pragma unroll
      for (int j = 0; j < FM; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < FM; ++j) ss[j] = 0.f;
  };
  auto over_groups = [&](float v) {   // a row's four lane groups, in a fixed order
    v += __shfl_xor(v, 16, kWave);
    return v + __shfl_xor(v, 32, kWave);
  };
  // WL: run w of a tile's k-steps is [nk w / 8, nk (w + 1) / 8), what wave w of a K5 block takes;
  // each is summed from zero and the sums are added in order, as that block's reduction does.
  // `run_end` is where the present one ends (the tile's first k-step moves past empty ones).
  int run = 0, run_end = 0;
  auto next_run = [&](int s) {   // s: the next k-step
    do {
      ++run;
      run_end = (nk * run) >> 3;
    } while (run_end <= s && run < 8);
  };
  auto reset = [&]() {
    clear();
    if constexpr (WL) {
#pragma unroll
      for (int i = 0; i < FN; ++i)
#pragma unroll
        for (int j = 0; j < FM; ++j) tot[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < FM; ++j) ss_tot[j] = 0.f;
      run = 0;
      next_run(0);
    }
  };
  auto fold = [&](int s) {   // after k-step s
    if constexpr (WL) {
      if (s + 1 != run_end) return;
#pragma unroll
      for (int i = 0; i < FN; ++i)
#pragma unroll
        for (int j = 0; j < FM; ++j) tot[i][j] += acc[i][j];
      if constexpr (AMODE == A_NORM) {
#pragma unroll
        for (int j = 0; j < FM; ++j) ss_tot[j] += over_groups(ss[j]);
      }
      clear();
      next_run(s + 1);
    }
  };
  auto result = [&](int i, int j) -> const f32x4_t& {
    if constexpr (WL) return tot[i][j];
    else return acc[i][j];
  };

  // k-step s from LDS, with the copies q0 .. q1 - 1 of the stage at `dst` spread over its MFMAs:
  // the CU takes in a copy every 25-30 cycles, and a wave that has to wait for that issues
  // nothing else meanwhile
  constexpr int kParts = AP + (WL ? 1 : 0);
  auto compute = [&](int s, const uint8_t* base, uint32_t dst, int q0, int q1) {
    constexpr int kGroup = AMODE == A_NORM ? (FN < 4 ? FN : 4) : 1;
    constexpr int kGroups = FN / kGroup * kParts;
    int grp = 0;
    auto copies = [&]() {   // after the MFMAs of group grp
#pragma unroll
      for (int q = q0 + (q1 - q0) * grp / kGroups; q < q0 + (q1 - q0) * (grp + 1) / kGroups; ++q)
        copy(q, dst);
      if (S::SPREAD) __builtin_amdgcn_sched_barrier(0x106);   // VALU, SALU, LDS reads may cross
      ++grp;
    };
    bf16x8_t ah[FM], al[FM];
    if constexpr (AMODE == A_NORM) {
      // x of row 16 (FM wm + j) + c, columns 8 g .. 8 g + 7: the split of x * gamma, as the
      // norm kernels write it (t rounded, then split)
      const float4 g0 = *reinterpret_cast<const float4*>(gam_s + 32 * s + 8 * g);
      const float4 g1 = *reinterpret_cast<const float4*>(gam_s + 32 * s + 8 * g + 4);
      const float ge[8] = {g0.x, g0.y, g0.z, g0.w, g1.x, g1.y, g1.z, g1.w};
#pragma unroll
      for (int j = 0; j < FM; ++j) {
        const float4 x0 =
            *reinterpret_cast<const float4*>(base + (2 * (FM * wm + j)) * 1024 + 16 * lane);
        const float4 x1 =
            *reinterpret_cast<const float4*>(base + (2 * (FM * wm + j) + 1) * 1024 + 16 * lane);
        const float xe[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
        float t[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          t[e] = xe[e] * ge[e];
          ss[j] = fmaf(xe[e], xe[e], ss[j]);
        }
        if constexpr (AP == 2) {
          uint4 hi, lo;
          split8(t, hi, lo);
          ah[j] = as_bf16x8(hi);
          al[j] = as_bf16x8(lo);
        } else {
          ah[j] = as_bf16x8(pack8(t));
        }
      }
    } else {
#pragma unroll
      for (int j = 0; j < FM; ++j) {
        ah[j] =
            *reinterpret_cast<const bf16x8_t*>(base + (2 * (FM * wm + j)) * 1024 + 16 * lane);
        if constexpr (AP == 2)
          al[j] = *reinterpret_cast<const bf16x8_t*>(base + (2 * (FM * wm + j) + 1) * 1024 +
                                                     16 * lane);
      }
    }
    // The hi products before the lo products, so that consecutive MFMAs write different
    // accumulators (each accumulator still adds hi before lo).  The split forms (8 weight
    // fragments) hold all their weight fragments and run two passes; the norm forms (16, whose
    // registers that would exhaust) take four fragments at a time: hi for the four fragments
    // and both row blocks, then lo, so an accumulator's lo product issues eight MFMAs after its
    // hi product (measured at config 2 against one fragment at a time: qkv 7%, gate/up 6%
    // faster; two at a time sits between; eight is within 1% of four and takes the E_QKV form
    // to the 256-register limit).
    constexpr int kWPer = WL ? 2 : 1;   // fragments per weight row block
    if constexpr (AMODE == A_NORM) {
      static_assert(FN % kGroup == 0, "the norm forms group their weight fragments");
#pragma unroll
      for (int i = 0; i < FN; i += kGroup) {
        bf16x8_t wf[kGroup];
#pragma unroll
        for (int u = 0; u < kGroup; ++u)
          wf[u] = *reinterpret_cast<const bf16x8_t*>(
              base + (kAFrags + kWPer * (FN * wn + i + u)) * 1024 + 16 * lane);
        bf16x8_t wlf[WL ? kGroup : 1];
        if constexpr (WL) {
#pragma unroll
          for (int u = 0; u < kGroup; ++u)
            wlf[u] = *reinterpret_cast<const bf16x8_t*>(
                base + (kAFrags + 2 * (FN * wn + i + u) + 1) * 1024 + 16 * lane);
        }
#pragma unroll
        for (int u = 0; u < kGroup; ++u)
#pragma unroll
          for (int j = 0; j < FM; ++j)
            acc[i + u][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[u], ah[j], acc[i + u][j],
                                                                    0, 0, 0);
        copies();
        if constexpr (AP == 2) {
#pragma unroll
          for (int u = 0; u < kGroup; ++u)
#pragma unroll
            for (int j = 0; j < FM; ++j)
              acc[i + u][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[u], al[j],
                                                                      acc[i + u][j], 0, 0, 0);
          copies();
        }
        if constexpr (WL) {
#pragma unroll
          for (int u = 0; u < kGroup; ++u)
#pragma unroll
            for (int j = 0; j < FM; ++j)
              acc[i + u][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wlf[u], ah[j],
                                                                      acc[i + u][j], 0, 0, 0);
          copies();
        }
      }
    } else {
      bf16x8_t wf[FN];
#pragma unroll
      for (int i = 0; i < FN; ++i)
        wf[i] = *reinterpret_cast<const bf16x8_t*>(
            base + (kAFrags + kWPer * (FN * wn + i)) * 1024 + 16 * lane);
      bf16x8_t wlf[WL ? FN : 1];
      if constexpr (WL) {
#pragma unroll
        for (int i = 0; i < FN; ++i)
          wlf[i] = *reinterpret_cast<const bf16x8_t*>(
              base + (kAFrags + 2 * (FN * wn + i) + 1) * 1024 + 16 * lane);
      }
#pragma unroll
      for (int i = 0; i < FN; ++i) {
#pragma unroll
        for (int j = 0; j < FM; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[i], ah[j], acc[i][j], 0, 0, 0);
        copies();
      }
      if constexpr (AP == 2) {
#pragma unroll
        for (int i = 0; i < FN; ++i) {
#pragma unroll
          for (int j = 0; j < FM; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[i], al[j], acc[i][j], 0, 0, 0);
          copies();
        }
      }
      if constexpr (WL) {
#pragma unroll
        for (int i = 0; i < FN; ++i) {
#pragma unroll
          for (int j = 0; j < FM; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wlf[i], ah[j], acc[i][j], 0, 0,
                                                                0);
          copies();
        }
      }
    }
  };

  // the finished tile at (m0, n0): lane (c, g) of accumulator tile (i, j) holds
  // acc[row 16 (FM wm + j) + c][weight rows 16 (FN wn + i) + 4 g ..]
  auto epilogue = [&](int m0, int n0) {
    if constexpr (AMODE == A_NORM) {
      // the four lane groups of a row in a fixed order (one wave per row block); the barrier waits
      // for LDS only, so the next tile's loads stay in flight (rstd_s was last read in the
      // previous tile's epilogue, ns >= 1 stage barriers ago)
#pragma unroll
      for (int j = 0; j < FM; ++j) {
        float v;
        if constexpr (WL) v = ss_tot[j];
        else v = over_groups(ss[j]);
        if (g == 0) rstd_s[16 * (FM * wm + j) + c] = rsqrtf(v / static_cast<float>(K) + p.eps);
      }
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    }
    if constexpr (AMODE == A_NORM && (EPI == E_STORE || EPI == E_QKV)) {
      static_assert(kBM <= kThreads, "one thread per row of the tile");
      if (p.rstd_out && n0 == 0 && tid < kBM && m0 + tid < M) p.rstd_out[m0 + tid] = rstd_s[tid];
    }
    if constexpr (EPI == E_QKV) {
      static_assert(AMODE == A_NORM, "E_QKV follows the norm prologue");
      // the arithmetic of K2 (rope_cache.hip); n0 and d are multiples of 64, so lane (c, g) of
      // the tile's weight fragment f holds dims 16 (f % 4) + 4 g .. + 3 of its head: RoPE pairs
      // 8 (f % 4) + 2 g and + 1
      constexpr int kQ = FN < 4 ? FN : 4;   // distinct f % 4 of this wave
      static_assert(4 % kQ == 0 && FN % kQ == 0, "the wave's fragments cycle through their dims");
      const int d = N / 3;
      const int64_t head_stride = static_cast<int64_t>(p.slots) * kHeadDim;
#pragma unroll
      for (int j = 0; j < FM; ++j) {
        const int r = 16 * (FM * wm + j) + c;
        const int m = m0 + r;
        if (m >= M) continue;
        int64_t b;
        int slot;
        if (p.tok_slot) {
          b = p.tok_row[m];
          slot = p.tok_slot[m];
        } else {
          b = m / p.seq;
          slot = static_cast<int>(m - b * p.seq);
        }
        const bool in_cache = slot >= 0 && slot < p.slots && b >= 0 && b < p.batch;
        // clamped below at 0 as the lead-attention pass (K4c) clamps it, so the rows written
        // here are exactly the rows it reads
        const int ks = (p.kv_start && b >= 0 && b < p.batch) ? max(p.kv_start[b], 0) : 0;
        const bool lead_row = !WL && p.out != nullptr && slot >= ks && slot - ks < p.lead;
        const float rs = rstd_s[r];
        const int64_t* pos3 = p.pos + static_cast<int64_t>(m) * 3;
        float cs[2 * kQ], sn[2 * kQ];
#pragma unroll
        for (int t = 0; t < 2 * kQ; ++t)
          rope_cos_sin(8 * ((FN * wn + (t >> 1)) & 3) + 2 * g + (t & 1), pos3, p.rope_tab, p.ra,
                       cs[t], sn[t]);
#pragma unroll
        for (int t = 0; t < 2 * kQ; ++t) {
          landed(cs[t]);
          landed(sn[t]);
        }
        const int64_t cache_row = (b * (d / kHeadDim) * static_cast<int64_t>(p.slots) + slot) *
                                  kHeadDim;
#pragma unroll
        for (int i = 0; i < FN; ++i) {
          const int n = n0 + 16 * (FN * wn + i) + 4 * g;
          if (n >= N) continue;
          const f32x4_t v = result(i, j);
          if (lead_row)
            *reinterpret_cast<float4*>(p.out + static_cast<int64_t>(m) * p.ldo + n) =
                make_float4(v[0], v[1], v[2], v[3]);
          const int part = n / d, e = n - part * d;
          const int head = e / kHeadDim, dim = e - head * kHeadDim;
          const int q4 = i % kQ;
          const float a0 = v[0] * rs, a1 = v[1] * rs, a2 = v[2] * rs, a3 = v[3] * rs;
          using TO = std::conditional_t<WL, float, uint16_t>;
          const int64_t at = cache_row + head * head_stride + dim;
          if (part == 2) {
            if (in_cache) st_ch4<false>(static_cast<TO*>(p.vc) + at, a0, a1, a2, a3);
            continue;
          }
          float y0, y1, y2, y3;
          rope_rot(a0, a1, cs[2 * q4], sn[2 * q4], y0, y1);
          rope_rot(a2, a3, cs[2 * q4 + 1], sn[2 * q4 + 1], y2, y3);
          if (part == 0)
            st_ch4<false>(static_cast<TO*>(p.q_out) + static_cast<int64_t>(m) * d + e,
                          y0 * p.q_scale, y1 * p.q_scale, y2 * p.q_scale, y3 * p.q_scale);
          else if (in_cache)
            st_ch4<false>(static_cast<TO*>(p.kc) + at, y0, y1, y2, y3);
        }
      }
    } else if constexpr (EPI == E_SWIGLU) {
      // Gate fragment 2 pb, up fragment 2 pb + 1: channels 16 (n0 / 32 + FN / 2 * wn + pb) + 4 g.
      // The bias loads of kG pairs are issued together, and those of the next kG pairs before
      // this group's stores: the compiler's wait for a load also waits for every older memory
      // operation (the stores before it, the next tile's copies), so loads issued one pair at a
      // time after the previous pair's stores took a full round trip per pair.
      const int F = p.d_ff;
      constexpr int NP = FN / 2, kG = NP % 4 == 0 ? 2 : 1;
      static_assert(FN % 2 == 0 && (NP == 1 || NP % (2 * kG) == 0), "bias groups");
      auto chan = [&](int pb) { return 16 * (n0 / 32 + FN / 2 * wn + pb) + 4 * g; };
      auto load_bias = [&](int pb0, float4 (&bg)[kG], float4 (&bu)[kG]) {
#pragma unroll
        for (int q = 0; q < kG; ++q) {
          const int ch = min(chan(pb0 + q), F - 4);   // in bounds; unused past F
          bg[q] = p.bias_a ? *reinterpret_cast<const float4*>(p.bias_a + ch)
                           : make_float4(0.f, 0.f, 0.f, 0.f);
          bu[q] = p.bias_b ? *reinterpret_cast<const float4*>(p.bias_b + ch)
                           : make_float4(0.f, 0.f, 0.f, 0.f);
        }
      };
      auto store_h = [&](int pb0, const float4 (&bg)[kG], const float4 (&bu)[kG]) {
#pragma unroll
        for (int q = 0; q < kG; ++q) {
          landed(bg[q]);
          landed(bu[q]);
          const int pb = pb0 + q, ch = chan(pb);
          if (2 * ch >= N) continue;
#pragma unroll
          for (int j = 0; j < FM; ++j) {
            const int r = 16 * (FM * wm + j) + c;
            const int m = m0 + r;
            if (m >= M) continue;
            const float rs = AMODE == A_NORM ? rstd_s[r] : 1.f;
            const f32x4_t gs = result(2 * pb, j), us = result(2 * pb + 1, j);
            // the arithmetic of K3 (swiglu.hip)
            const float o[4] = {silu_mul(fmaf(rs, gs[0], bg[q].x), fmaf(rs, us[0], bu[q].x)),
                                silu_mul(fmaf(rs, gs[1], bg[q].y), fmaf(rs, us[1], bu[q].y)),
                                silu_mul(fmaf(rs, gs[2], bg[q].z), fmaf(rs, us[2], bu[q].z)),
                                silu_mul(fmaf(rs, gs[3], bg[q].w), fmaf(rs, us[3], bu[q].w))};
            uint2 hi, lo;
            split4(o, hi, lo);
            *reinterpret_cast<uint2*>(p.h + tile_off(m, ch, p.h_parts * F)) = hi;
            if (p.h_parts == 2) *reinterpret_cast<uint2*>(p.h + tile_off(m, F + ch, 2 * F)) = lo;
          }
        }
      };
      float4 ga[kG], ua[kG], gb[kG], ub[kG];
      load_bias(0, ga, ua);
#pragma unroll
      for (int pb0 = 0; pb0 < NP; pb0 += 2 * kG) {
        if (pb0 + kG < NP) load_bias(pb0 + kG, gb, ub);
        store_h(pb0, ga, ua);
        if (pb0 + 2 * kG < NP) load_bias(pb0 + 2 * kG, ga, ua);
        if (pb0 + kG < NP) store_h(pb0 + kG, gb, ub);
      }
    } else {
      // The residual's loads of kG weight fragments are issued together, and those of the next
      // kG before this group's stores (see E_SWIGLU: one load and its wait per fragment, after
      // the previous fragment's store, took a full round trip each).
      constexpr int kG = FN % 4 == 0 ? 2 : 1;
      static_assert(FN == 1 || FN % (2 * kG) == 0, "residual groups");
      auto col = [&](int i) { return n0 + 16 * (FN * wn + i) + 4 * g; };
      auto row = [&](int j) { return m0 + 16 * (FM * wm + j) + c; };
      auto load_x = [&](int i0, float4 (&xv)[kG][FM], float4 (&bv)[kG]) {
        if constexpr (EPI == E_RESIDUAL) {
#pragma unroll
          for (int u = 0; u < kG; ++u) {
            const int n = min(col(i0 + u), N - 4);   // in bounds; unused past N or M
            bv[u] = p.bias_a ? *reinterpret_cast<const float4*>(p.bias_a + n)
                             : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
            for (int j = 0; j < FM; ++j)
              xv[u][j] = *reinterpret_cast<const float4*>(
                  p.x_res + tile_off32(min(row(j), M - 1), n, N));
          }
        }
      };
      auto store_x = [&](int i0, const float4 (&xv)[kG][FM], const float4 (&bv)[kG]) {
#pragma unroll
        for (int u = 0; u < kG; ++u) {
          if constexpr (EPI == E_RESIDUAL) {
            landed(bv[u]);
#pragma unroll
            for (int j = 0; j < FM; ++j) landed(xv[u][j]);
          }
          const int n = col(i0 + u);
          if (n >= N) continue;
#pragma unroll
          for (int j = 0; j < FM; ++j) {
            const int m = row(j);
            if (m >= M) continue;
            const f32x4_t v = result(i0 + u, j);
            if constexpr (EPI == E_RESIDUAL) {
              // x + delta, then + bias: the order of the add+RMSNorm kernel it replaces
              float4 x = xv[u][j];
              x.x += v[0]; x.y += v[1]; x.z += v[2]; x.w += v[3];
              if (p.bias_a) {
                x.x += bv[u].x; x.y += bv[u].y; x.z += bv[u].z; x.w += bv[u].w;
              }
              *reinterpret_cast<float4*>(p.x_res + tile_off32(m, n, N)) = x;
            } else {
              *reinterpret_cast<float4*>(p.out + static_cast<int64_t>(m) * p.ldo + n) =
                  make_float4(v[0], v[1], v[2], v[3]);
            }
          }
        }
      };
      float4 xa[kG][FM], ba[kG], xb[kG][FM], bb[kG];
      load_x(0, xa, ba);
#pragma unroll
      for (int i0 = 0; i0 < FN; i0 += 2 * kG) {
        if (i0 + kG < FN) load_x(i0 + kG, xb, bb);
        store_x(i0, xa, ba);
        if (i0 + 2 * kG < FN) load_x(i0 + 2 * kG, xa, ba);
        if (i0 + kG < FN) store_x(i0 + kG, xb, bb);
      }
    }
  };

  // Step u (over all stages of this block's tiles, tile after tile) computes ring stage
  // u % kRing while the next kRing - 1 stages load -- across a tile boundary too, so the next
  // tile's first stages are in flight during this tile's epilogue.  The stage that step u's
  // copies overwrite, (u + kAhead) % kRing, was last read in step u - 1, before that step's
  // barrier.  Every wave runs the same steps (all counters are block-uniform), so every barrier
  // is reached by all.
  auto tile_origin = [&](int t, int& m0, int& n0) {
    const int mt = t / p.tiles_n;
    m0 = mt * kBM;
    n0 = (t - mt * p.tiles_n) * kBN;
  };
  constexpr int kAhead = kRing - 1;   // stages in flight beyond the one being computed
  int it = first, is = 0, im0, in0;   // issue cursor: tile, stage of the tile
  tile_origin(it, im0, in0);
  seek(im0, in0);
  auto advance_issue = [&]() {
    ++as;
    if (++is == ns) {
      is = 0;
      it += bpx;
      tile_origin(it, im0, in0);
      seek(im0, in0);
    }
  };
#pragma unroll
  for (int r = 0; r < kAhead; ++r) {
#pragma unroll
    for (int q = 0; q < kLoads; ++q) copy(q, lds0 + r * kStage);
    advance_issue();
  }
  stage_barrier<(kAhead - 1) * kLoads>();
  int ct = first, cs = 0, cm0, cn0;   // compute cursor
  tile_origin(ct, cm0, cn0);
  reset();
  int b = 0;
  for (int u = 0; u < total; ++u) {
    // past the block's last stage the copies go on (clamped addresses, stages no one reads), so
    // that every step makes the same copies and waits for the same number
    const uint32_t dst = lds0 + (b == 0 ? kRing - 1 : b - 1) * kStage;   // (u + kAhead) % kRing
    if constexpr (!S::SPREAD) {
#pragma unroll
      for (int q = 0; q < kLoads; ++q) {
        copy(q, dst);
        // one copy every 80 cycles (14 wait states and six scalar instructions of 4 cycles):
        // 310 us for the down projection of 65,536 rows; 336-352 at 24-64 cycles, 324 at 104
        asm volatile("s_nop 13");
      }
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      constexpr int n = S::SPREAD ? kLoads : 0;
      compute(KS * cs + ks, lds + b * kStage + ks * kStep, dst, n * ks / KS, n * (ks + 1) / KS);
      fold(KS * cs + ks);
    }
    advance_issue();
    stage_barrier<(kAhead - 1) * kLoads>();
    b = b == kRing - 1 ? 0 : b + 1;
    if (++cs == ns) {
      epilogue(cm0, cn0);
      reset();
      cs = 0;
      ct += bpx;
      tile_origin(ct, cm0, cn0);
    }
  }
  stage_barrier<0>();   // the last copies land while the LDS is still this block's
}

// CUs of the current device (hipDeviceAttributeMultiprocessorCount), cached per device
int device_cus() {
  static int cached[64] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  if (cached[dev] == 0) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        n <= 0)
      n = 256;
    cached[dev] = n;
  }
  return cached[dev];
}

template <int AMODE, int EPI, int AP, bool WL, class S>
int launch_shape(Args p, hipStream_t st) {
  const int64_t tm = (static_cast<int64_t>(p.M) + S::BM - 1) / S::BM;
  const int64_t tn = (static_cast<int64_t>(p.N) + S::BN - 1) / S::BN;
  const int64_t tiles = tm * tn;
  if (tiles > 0x7fffffff - 8) return MDL_ERR_SHAPE;
  const int64_t per_xcd = (tiles + 7) / 8;
  // the blocks that fit the chip at a time; blocks per XCD capped by its tiles
  const int64_t bpx = std::min<int64_t>(S::OCC * ((device_cus() + 7) / 8), per_xcd);
  p.tiles_n = static_cast<int>(tn);
  p.tiles = static_cast<int>(tiles);
  p.per_xcd = static_cast<int>(per_xcd);
  prefill_gemm_kernel<AMODE, EPI, AP, WL, S>
      <<<dim3(static_cast<unsigned>(8 * bpx)), 64 * S::NW, 0, st>>>(p);
  return launch_status();
}

// The block shapes, smallest tile first: the more blocks a product gives, the more it pays to hand
// each a tile that reads less per MFMA.  Every norm form keeps a row block in one wave; gamma's
// room bounds the K of all but the last (GK).
struct NormShapes {
  using S0 = Shape<64, 64, 4, 1, 2, 3, 2, true, 1920>;
  using S1 = Shape<128, 128, 4, 1, 1, 3, 2, true, 1920>;
  using S2 = Shape<128, 256, 8, 1, 1, 4, 1, true, 1920>;
  using S3 = Shape<128, 256, 4, 1, 1, 2, 2, true>;
  using S4 = Shape<128, 256, 4, 1, 1, 2, 2, false>;
};
struct SplitShapes {
  using S0 = Shape<64, 64, 4, 2, 2, 3, 2, true>;
  using S1 = Shape<128, 128, 4, 2, 2, 3, 1, true>;
  using S2 = Shape<128, 256, 4, 2, 1, 4, 1, true>;
  using S3 = Shape<128, 256, 2, 2, 1, 2, 2, false>;
  using S4 = S3;
};
// fp32 weights: twice the weight fragments, so half the weight rows a tile
struct NormShapesF32 {
  using S0 = Shape<64, 64, 4, 1, 2, 2, 2, true, 1920>;
  using S1 = Shape<64, 128, 4, 1, 1, 3, 2, true, 1920>;
  using S2 = Shape<128, 128, 4, 1, 1, 2, 2, true>;   // every K
  using S3 = S2;
  using S4 = S2;
};
struct SplitShapesF32 {
  using S0 = Shape<64, 64, 4, 2, 2, 2, 2, true>;
  using S1 = Shape<128, 64, 2, 2, 1, 3, 2, true>;
  using S2 = Shape<128, 128, 2, 2, 1, 2, 2, false>;
  using S3 = S2;
  using S4 = S2;
};

// What a k-step takes (us) on tiles of a shape: `single` with at most one per CU, else `base` +
// `round` for every filling of the chip (CUs x OCC blocks), for up to `limit` of these.  Fitted to
// launches of d = 768, F = 2048 and d = 1280, F = 3392 at 64 to 282,695 rows.
struct StepCost {
  int bm, bn, ks, gk, occ;
  float single, base, round;
  int limit;
};
constexpr int kAnyRounds = 0x7fffffff;

template <class S>
constexpr StepCost step_cost(float single, float base, float round, int limit = kAnyRounds) {
  return {S::BM, S::BN, S::KS, S::GK, S::OCC, single, base, round, limit};
}

// The index of the cheapest shape for an [m, k] x [n, k]^T product; the last one takes every size
template <int COUNT>
int cheapest(const StepCost (&costs)[COUNT], bool norm, int m, int n, int k) {
  int best = COUNT - 1;
  float best_cost = 1e30f;
  for (int i = 0; i < COUNT; ++i) {
    const StepCost& c = costs[i];
    if (k % (32 * c.ks) || (norm && k > c.gk)) continue;
    const int64_t tiles = ((static_cast<int64_t>(m) + c.bm - 1) / c.bm) *
                          ((static_cast<int64_t>(n) + c.bn - 1) / c.bn);
    const int64_t slots = static_cast<int64_t>(device_cus()) * c.occ;
    const int64_t rounds = (tiles + slots - 1) / slots;
    if (rounds > c.limit) continue;
    const float cost =
        tiles <= device_cus() ? c.single : c.base + c.round * static_cast<float>(rounds);
    if (cost < best_cost) {
      best = i;
      best_cost = cost;
    }
  }
  return best;
}

// Measured at d = 768, F = 2048, us per launch (qkv / out / gate-up / down), one block of 256 x 256
// per CU (what every size ran on before these shapes) -> the shape taken here:
//   256 rows    50 / 37 / 43 / 87      12 / 6 / 12 / 11     S0
//   731 rows    53 / 38 / 45 / 88      17 / 7 / 21 / 13     S0 / S0 / S1 / S0
//   2,300 rows  55 / 38 / 48 / 88      30 / 10 / 40 / 22    S2 / S0 / S3 / S0
//   4,096 rows  57 / 41 / 54 / 90      50 / 16 / 51 / 31    S3 / S1 / S3 / S1
//   8,192 rows  106 / 42 / 99 / 92     77 / 28 / 92 / 55    S2 / S2 / S3 / S2
//   16,669      157 / 50 / 227 / 103   126 / 45 / 185 / 90  S3
// Past five rounds the power limit sets in, and the paced copies of the norm forms' S4 win: 701
// against 729 us for the gate / up projection of 65,536 rows.
int pick_shape(bool norm, int m, int n, int k) {
  static constexpr StepCost kNorm[] = {
      step_cost<NormShapes::S0>(0.5f, 0.35f, 0.375f), step_cost<NormShapes::S1>(0.97f, 0.25f, 1.12f),
      step_cost<NormShapes::S2>(1.25f, 0.22f, 1.03f),
      step_cost<NormShapes::S3>(1.6f, 0.15f, 1.7f, 5), step_cost<NormShapes::S4>(1.7f, 0.5f, 1.7f)};
  static constexpr StepCost kSplit[] = {
      step_cost<SplitShapes::S0>(0.26f, 0.1f, 0.3f), step_cost<SplitShapes::S1>(0.5f, 0.05f, 0.52f),
      step_cost<SplitShapes::S2>(0.9f, 0.1f, 0.9f), step_cost<SplitShapes::S3>(1.2f, 0.1f, 1.45f)};
  return norm ? cheapest(kNorm, true, m, n, k) : cheapest(kSplit, false, m, n, k);
}

// The same for fp32 weights, us on K5 / here (qkv and K2, out, gate-up, down; d = 768, F = 2048):
//   1,536 rows   45 / 18 / 57 / 39        31 / 13 / 40 / 27
//   2,304 rows   68 / 23 / 87 / 45        45 / 14 / 74 / 31
//   11,242 rows  260 / 98 / 388 / 211     171 / 53 / 297 / 128
// The fold of the runs of k-steps (`fold`) is in these: in one run over all k-steps 28 / 12 / 35 /
// 25, 41 / 13 / 80 / 30 and 160 / 52 / 280 / 126.
int pick_shape_f32(bool norm, int m, int n, int k) {
  static constexpr StepCost kNorm[] = {step_cost<NormShapesF32::S0>(0.47f, 0.2f, 0.52f),
                                       step_cost<NormShapesF32::S1>(0.72f, 0.3f, 0.65f),
                                       step_cost<NormShapesF32::S2>(1.1f, 0.2f, 1.25f)};
  static constexpr StepCost kSplit[] = {step_cost<SplitShapesF32::S0>(0.35f, 0.1f, 0.37f),
                                        step_cost<SplitShapesF32::S1>(0.5f, 0.1f, 0.63f),
                                        step_cost<SplitShapesF32::S2>(1.05f, 0.05f, 1.27f)};
  return norm ? cheapest(kNorm, true, m, n, k) : cheapest(kSplit, false, m, n, k);
}

template <int AMODE, int EPI, bool WL, class T>
int launch_of(int shape, const Args& p, hipStream_t st) {
  switch (shape) {
    case 0: return launch_shape<AMODE, EPI, 2, WL, typename T::S0>(p, st);
    case 1: return launch_shape<AMODE, EPI, 2, WL, typename T::S1>(p, st);
    case 2: return launch_shape<AMODE, EPI, 2, WL, typename T::S2>(p, st);
    case 3: return launch_shape<AMODE, EPI, 2, WL, typename T::S3>(p, st);
    default: return launch_shape<AMODE, EPI, 2, WL, typename T::S4>(p, st);
  }
}

template <int EPI>
int launch_norm(const Args& p, hipStream_t st) {
  return launch_of<A_NORM, EPI, false, NormShapes>(pick_shape(true, p.M, p.N, p.K), p, st);
}

template <int EPI>
int launch_f32w(const Args& p, hipStream_t st) {
  if constexpr (EPI == E_RESIDUAL)
    return launch_of<A_TILES, EPI, true, SplitShapesF32>(pick_shape_f32(false, p.M, p.N, p.K), p,
                                                         st);
  else
    return launch_of<A_NORM, EPI, true, NormShapesF32>(pick_shape_f32(true, p.M, p.N, p.K), p, st);
}

// fp32 weights: up to this many rows the projections run on K5, whose waves split K and need no
// ring to fill, with the same bits; qkv up to the last, since past it K5 and K2 are slower than the
// one launch.  Out, gate / up and down, us on K5 / on K6: d = 768 at 384 rows 37 / 53, 768 53 / 60,
// 896 60 / 63, 1,536 114 / 80; d = 1,280 at 768 rows 104 / 116, 896 150 / 120.  At d = 256 a k-step's
// share of the fold is larger: gate / up at 1,024 rows 10.1 / 10.6, 1,536 14.1 / 13.1; out and down at
// 1,536 9.9 / 13.9, 2,304 14.0 / 14.6.  qkv: d = 768 at 384 rows 17.3 / 19.0, 512 24.5 / 22.4;
// d = 1,280 at 256 24.9 / 28.9, 384 35.0 / 32.2.
constexpr int kK5Rows = 768, kK5RowsNarrow = 1024, kK5RowsNarrowResidual = 2048;
constexpr int kK5RowsQkv = MDL_F32W_QKV_ROWS;   // 448
constexpr int kNarrow = 512;                    // channels

bool on_k5_norm(int m, int k) { return m <= (k < kNarrow ? kK5RowsNarrow : kK5Rows); }
bool on_k5_residual(int m, int n) { return m <= (n < kNarrow ? kK5RowsNarrowResidual : kK5Rows); }

// the split forms by A layout and parts: row-major activations, and the forms with the hi part
// alone, are not on the prompt path and run on the large shape
template <int EPI>
int launch_split(const Args& p, int a_layout, int a_parts, hipStream_t st) {
  using Large = SplitShapes::S4;
  if (a_layout == MDL_LAYOUT_ROWS)
    return a_parts == 1 ? launch_shape<A_ROWS, EPI, 1, false, Large>(p, st)
                        : launch_shape<A_ROWS, EPI, 2, false, Large>(p, st);
  if (a_parts == 1) return launch_shape<A_TILES, EPI, 1, false, Large>(p, st);
  return launch_of<A_TILES, EPI, false, SplitShapes>(pick_shape(false, p.M, p.N, p.K), p, st);
}

// shared argument checks: k a positive multiple of 32, n of 16, 16-byte aligned operands
int check_common(const uint16_t* w, int m, int n, int k) {
  if (!w) return MDL_ERR_NULL;
  if (m < 0 || n <= 0 || k <= 0 || k % 32 != 0 || n % 16 != 0) return MDL_ERR_SHAPE;
  if (!aligned16(w)) return MDL_ERR_ALIGN;
  return MDL_OK;
}

int check_a(const uint16_t* a, int64_t lda, int a_layout, int a_parts, int k) {
  if (!a) return MDL_ERR_NULL;
  if (a_layout != MDL_LAYOUT_ROWS && a_layout != MDL_LAYOUT_TILES) return MDL_ERR_SHAPE;
  if (a_parts != 1 && a_parts != 2) return MDL_ERR_SHAPE;
  if (a_layout == MDL_LAYOUT_ROWS && lda < a_parts * static_cast<int64_t>(k))
    return MDL_ERR_SHAPE;
  if (!aligned16(a) || (a_layout == MDL_LAYOUT_ROWS && lda % 8 != 0)) return MDL_ERR_ALIGN;
  return MDL_OK;
}

}  // namespace
}  // namespace mdl

using namespace mdl;

extern "C" int mdl_prefill_gemm_split(const uint16_t* a, int64_t lda, int a_layout, int a_parts,
                                      const uint16_t* w, float* out, int64_t ldo, int m, int n,
                                      int k, void* stream) {
  int rc = check_common(w, m, n, k);
  if (rc == MDL_OK) rc = check_a(a, lda, a_layout, a_parts, k);
  if (rc != MDL_OK) return rc;
  if (!out) return MDL_ERR_NULL;
  if (ldo < n) return MDL_ERR_SHAPE;
  if (!aligned16(out) || ldo % 4 != 0) return MDL_ERR_ALIGN;
  if (m == 0) return MDL_OK;
  Args p{};
  p.a = a; p.lda = lda; p.w = w; p.out = out; p.ldo = ldo; p.M = m; p.N = n; p.K = k;
  return launch_split<E_STORE>(p, a_layout, a_parts, static_cast<hipStream_t>(stream));
}

extern "C" int mdl_prefill_gemm_norm(const float* x, const float* gamma, float eps,
                                     const uint16_t* w, float* out, int64_t ldo, float* rstd_out,
                                     int m, int n, int k, void* stream) {
  int rc = check_common(w, m, n, k);
  if (rc != MDL_OK) return rc;
  if (!x || !gamma || !out) return MDL_ERR_NULL;
  if (ldo < n || k > kMaxNormK) return MDL_ERR_SHAPE;
  if (!aligned16(x) || !aligned16(gamma) || !aligned16(out) || ldo % 4 != 0)
    return MDL_ERR_ALIGN;
  if (m == 0) return MDL_OK;
  Args p{};
  p.x = x; p.gamma = gamma; p.eps = eps; p.w = w; p.out = out; p.ldo = ldo;
  p.rstd_out = rstd_out; p.M = m; p.N = n; p.K = k;
  return launch_norm<E_STORE>(p, static_cast<hipStream_t>(stream));
}

extern "C" int mdl_prefill_gemm_norm_swiglu(const float* x, const float* gamma, float eps,
                                            int a_parts, const uint16_t* w_gu,
                                            const float* bias_gate, const float* bias_up,
                                            uint16_t* h_out, int h_parts, int m, int d_ff, int k,
                                            void* stream) {
  if (d_ff <= 0 || d_ff % 16 != 0 || d_ff > (1 << 28)) return MDL_ERR_SHAPE;
  if ((a_parts != 1 && a_parts != 2) || (h_parts != 1 && h_parts != 2)) return MDL_ERR_SHAPE;
  int rc = check_common(w_gu, m, 2 * d_ff, k);
  if (rc != MDL_OK) return rc;
  if (!x || !gamma || !h_out) return MDL_ERR_NULL;
  if (k > kMaxNormK) return MDL_ERR_SHAPE;
  if (!aligned16(x) || !aligned16(gamma) || !aligned8(h_out) ||
      (bias_gate && !aligned16(bias_gate)) || (bias_up && !aligned16(bias_up)))
    return MDL_ERR_ALIGN;
  if (m == 0) return MDL_OK;
  Args p{};
  p.x = x; p.gamma = gamma; p.eps = eps; p.w = w_gu; p.bias_a = bias_gate; p.bias_b = bias_up;
  p.h = h_out; p.d_ff = d_ff; p.h_parts = h_parts; p.M = m; p.N = 2 * d_ff; p.K = k;
  const hipStream_t st = static_cast<hipStream_t>(stream);
  return a_parts == 1 ? launch_shape<A_NORM, E_SWIGLU, 1, false, NormShapes::S4>(p, st)
                      : launch_norm<E_SWIGLU>(p, st);
}

extern "C" int mdl_prefill_gemm_split_residual(const uint16_t* a, int64_t lda, int a_layout,
                                               int a_parts, const uint16_t* w, float* x,
                                               const float* bias, int m, int n, int k,
                                               void* stream) {
  int rc = check_common(w, m, n, k);
  if (rc == MDL_OK) rc = check_a(a, lda, a_layout, a_parts, k);
  if (rc != MDL_OK) return rc;
  if (!x) return MDL_ERR_NULL;
  if (n % 32 != 0) return MDL_ERR_SHAPE;   // x in the fp32 tile layout: whole 32-column blocks
  if (!aligned16(x) || (bias && !aligned16(bias))) return MDL_ERR_ALIGN;
  if (m == 0) return MDL_OK;
  Args p{};
  p.a = a; p.lda = lda; p.w = w; p.x_res = x; p.bias_a = bias; p.M = m; p.N = n; p.K = k;
  return launch_split<E_RESIDUAL>(p, a_layout, a_parts, static_cast<hipStream_t>(stream));
}

extern "C" int mdl_prefill_gemm_norm_qkv(
    const float* x, const float* gamma, float eps, const uint16_t* w, int m, int n_heads,
    float* rstd_out, float* qkv_lead, int64_t ldq, int lead, const int32_t* kv_start,
    const int64_t* pos, const float* rope_tab, int max_x, int max_y, int max_z, int px, int py,
    int pz, float q_scale, uint16_t* q_out, uint16_t* k_cache, uint16_t* v_cache,
    int cache_slots, int batch, int seq, const int32_t* token_row, const int32_t* token_slot,
    void* stream) {
  if (n_heads <= 0 || n_heads * kHeadDim > kMaxNormK) return MDL_ERR_SHAPE;
  const int d = n_heads * kHeadDim;
  int rc = check_common(w, m, 3 * d, d);
  if (rc != MDL_OK) return rc;
  if (!x || !gamma || !pos || !rope_tab || !q_out || !k_cache || !v_cache) return MDL_ERR_NULL;
  if ((token_row == nullptr) != (token_slot == nullptr)) return MDL_ERR_NULL;
  if (max_x <= 0 || max_y <= 0 || max_z <= 0 || px < 0 || py < 0 || pz < 0 ||
      px + py + pz != kHeadDim / 2 || batch < 0 || cache_slots <= 0 || lead < 0)
    return MDL_ERR_SHAPE;
  if (!token_slot) {   // [batch, seq] rows: token i of row b is slot i
    if (seq <= 0 || static_cast<int64_t>(batch) * seq != m) return MDL_ERR_SHAPE;
    if (seq > cache_slots) return MDL_ERR_CACHE;
  }
  if (qkv_lead && (ldq < 3 * static_cast<int64_t>(d) || ldq % 4 != 0 || !aligned16(qkv_lead)))
    return qkv_lead && ldq < 3 * static_cast<int64_t>(d) ? MDL_ERR_SHAPE : MDL_ERR_ALIGN;
  if (!aligned16(x) || !aligned16(gamma) || !aligned8(q_out) || !aligned8(k_cache) ||
      !aligned8(v_cache) || !aligned4(rope_tab))
    return MDL_ERR_ALIGN;
  if (m == 0) return MDL_OK;
  Args p{};
  p.x = x; p.gamma = gamma; p.eps = eps; p.w = w; p.out = qkv_lead; p.ldo = ldq;
  p.rstd_out = rstd_out; p.pos = pos; p.rope_tab = rope_tab;
  p.ra = RopeArgs{max_x, max_y, max_z, px, py, pz};
  p.q_scale = q_scale; p.q_out = q_out; p.kc = k_cache; p.vc = v_cache;
  p.tok_row = token_row; p.tok_slot = token_slot; p.kv_start = kv_start;
  p.slots = cache_slots; p.seq = seq; p.batch = batch; p.lead = lead;
  p.M = m; p.N = 3 * d; p.K = d;
  return launch_norm<E_QKV>(p, static_cast<hipStream_t>(stream));
}

extern "C" int mdl_prefill_gemm_shapes(int form) {
  switch (form) {
    case MDL_GEMM_NORM: return 5;
    case MDL_GEMM_SPLIT: return 4;
    case MDL_GEMM_NORM_F32W:
    case MDL_GEMM_SPLIT_F32W: return 3;
    default: return MDL_ERR_SHAPE;
  }
}

extern "C" int mdl_prefill_gemm_pick(int form, int m, int n, int k) {
  if (form < MDL_GEMM_NORM || form > MDL_GEMM_SPLIT_F32W || m <= 0 || n <= 0 || k <= 0 || k % 32)
    return MDL_ERR_SHAPE;
  const bool norm = form == MDL_GEMM_NORM || form == MDL_GEMM_NORM_F32W;
  if (norm && k > kMaxNormK) return MDL_ERR_SHAPE;
  return form < MDL_GEMM_NORM_F32W ? pick_shape(norm, m, n, k) : pick_shape_f32(norm, m, n, k);
}

extern "C" int mdl_prefill_gemm_norm_f32w(const float* x, const float* gamma, float eps,
                                          const uint16_t* w, const uint16_t* w_lo, float* out,
                                          int64_t ldo, float* rstd_out, int m, int n, int k,
                                          void* stream) {
  int rc = check_common(w, m, n, k);
  if (rc != MDL_OK) return rc;
  if (!w_lo || !x || !gamma || !out) return MDL_ERR_NULL;
  if (ldo < n || k > kMaxNormK) return MDL_ERR_SHAPE;
  if (!aligned16(w_lo) || !aligned16(x) || !aligned16(gamma) || !aligned16(out) || ldo % 4 != 0)
    return MDL_ERR_ALIGN;
  if (m == 0) return MDL_OK;
  if (on_k5_norm(m, k))
    return mdl_gemm_norm(x, gamma, eps, w, w_lo, out, ldo, rstd_out, m, n, k, 0, stream);
  Args p{};
  p.x = x; p.gamma = gamma; p.eps = eps; p.w = w; p.wl = w_lo; p.out = out; p.ldo = ldo;
  p.rstd_out = rstd_out; p.M = m; p.N = n; p.K = k;
  return launch_f32w<E_STORE>(p, static_cast<hipStream_t>(stream));
}

extern "C" int mdl_prefill_gemm_norm_qkv_f32w(
    const float* x, const float* gamma, float eps, const uint16_t* w, const uint16_t* w_lo, int m,
    int n_heads, float* qkv, int64_t ldq, float* rstd, const int64_t* pos, const float* rope_tab,
    int max_x, int max_y, int max_z, int px, int py, int pz, float q_scale, float* q_out,
    float* k_cache, float* v_cache, int cache_slots, int batch, int seq, const int32_t* token_row,
    const int32_t* token_slot, void* stream) {
  if (n_heads <= 0 || n_heads * kHeadDim > kMaxNormK) return MDL_ERR_SHAPE;
  const int d = n_heads * kHeadDim;
  int rc = check_common(w, m, 3 * d, d);
  if (rc != MDL_OK) return rc;
  if (!w_lo || !x || !gamma || !qkv || !rstd || !pos || !rope_tab || !q_out || !k_cache ||
      !v_cache)
    return MDL_ERR_NULL;
  if ((token_row == nullptr) != (token_slot == nullptr)) return MDL_ERR_NULL;
  if (max_x <= 0 || max_y <= 0 || max_z <= 0 || px < 0 || py < 0 || pz < 0 ||
      px + py + pz != kHeadDim / 2 || batch < 0 || cache_slots <= 0 || ldq < 3 * d)
    return MDL_ERR_SHAPE;
  if (!token_slot) {   // [batch, seq] rows: token i of row b is slot i
    if (seq <= 0 || static_cast<int64_t>(batch) * seq != m) return MDL_ERR_SHAPE;
    if (seq > cache_slots) return MDL_ERR_CACHE;
  }
  if (!aligned16(w_lo) || !aligned16(x) || !aligned16(gamma) || !aligned16(qkv) || ldq % 4 != 0 ||
      !aligned16(q_out) || !aligned16(k_cache) || !aligned16(v_cache) || !aligned4(rope_tab))
    return MDL_ERR_ALIGN;
  if (m == 0) return MDL_OK;
  if (m <= kK5RowsQkv) {
    rc = mdl_gemm_norm(x, gamma, eps, w, w_lo, qkv, ldq, rstd, m, 3 * d, d, 0, stream);
    if (rc != MDL_OK) return rc;
    return token_slot
               ? mdl_qkv_rope_cache_packed(qkv, ldq, rstd, pos, rope_tab, m, token_row, token_slot,
                                           batch, n_heads, kHeadDim, max_x, max_y, max_z, px, py,
                                           pz, q_scale, q_out, k_cache, v_cache, MDL_DTYPE_F32,
                                           cache_slots, stream)
               : mdl_qkv_rope_cache(qkv, ldq, rstd, pos, rope_tab, batch, seq, n_heads, kHeadDim,
                                    max_x, max_y, max_z, px, py, pz, q_scale, q_out, k_cache,
                                    v_cache, MDL_DTYPE_F32, cache_slots, 0, nullptr, stream);
  }
  Args p{};
  p.x = x; p.gamma = gamma; p.eps = eps; p.w = w; p.wl = w_lo;
  p.pos = pos; p.rope_tab = rope_tab;
  p.ra = RopeArgs{max_x, max_y, max_z, px, py, pz};
  p.q_scale = q_scale; p.q_out = q_out; p.kc = k_cache; p.vc = v_cache;
  p.tok_row = token_row; p.tok_slot = token_slot;
  p.slots = cache_slots; p.seq = seq; p.batch = batch;
  p.M = m; p.N = 3 * d; p.K = d;
  return launch_f32w<E_QKV>(p, static_cast<hipStream_t>(stream));
}

extern "C" int mdl_prefill_gemm_norm_swiglu_f32w(const float* x, const float* gamma, float eps,
                                                 const uint16_t* w_gu, const uint16_t* w_gu_lo,
                                                 const float* bias_gate, const float* bias_up,
                                                 uint16_t* h_out, int m, int d_ff, int k,
                                                 void* stream) {
  if (d_ff <= 0 || d_ff % 16 != 0 || d_ff > (1 << 28)) return MDL_ERR_SHAPE;
  int rc = check_common(w_gu, m, 2 * d_ff, k);
  if (rc != MDL_OK) return rc;
  if (!w_gu_lo || !x || !gamma || !h_out) return MDL_ERR_NULL;
  if (k > kMaxNormK) return MDL_ERR_SHAPE;
  if (!aligned16(w_gu_lo) || !aligned16(x) || !aligned16(gamma) || !aligned8(h_out) ||
      (bias_gate && !aligned16(bias_gate)) || (bias_up && !aligned16(bias_up)))
    return MDL_ERR_ALIGN;
  if (m == 0) return MDL_OK;
  if (on_k5_norm(m, k))
    return mdl_gemm_norm_swiglu(x, gamma, eps, w_gu, w_gu_lo, bias_gate, bias_up, h_out, m, d_ff,
                                k, 0, stream);
  Args p{};
  p.x = x; p.gamma = gamma; p.eps = eps; p.w = w_gu; p.wl = w_gu_lo; p.bias_a = bias_gate;
  p.bias_b = bias_up; p.h = h_out; p.d_ff = d_ff; p.h_parts = 2; p.M = m; p.N = 2 * d_ff; p.K = k;
  return launch_f32w<E_SWIGLU>(p, static_cast<hipStream_t>(stream));
}

extern "C" int mdl_prefill_gemm_split_residual_f32w(const uint16_t* a, const uint16_t* w,
                                                    const uint16_t* w_lo, float* x,
                                                    const float* bias, int m, int n, int k,
                                                    void* stream) {
  int rc = check_common(w, m, n, k);
  if (rc == MDL_OK) rc = check_a(a, 0, MDL_LAYOUT_TILES, 2, k);
  if (rc != MDL_OK) return rc;
  if (!w_lo || !x) return MDL_ERR_NULL;
  if (n % 32 != 0) return MDL_ERR_SHAPE;   // x in the fp32 tile layout: whole 32-column blocks
  if (!aligned16(w_lo) || !aligned16(x) || (bias && !aligned16(bias))) return MDL_ERR_ALIGN;
  if (m == 0) return MDL_OK;
  if (on_k5_residual(m, n)) return mdl_gemm_split_residual(a, w, w_lo, x, bias, m, n, k, 0, stream);
  Args p{};
  p.a = a; p.w = w; p.wl = w_lo; p.x_res = x; p.bias_a = bias; p.M = m; p.N = n; p.K = k;
  return launch_f32w<E_RESIDUAL>(p, static_cast<hipStream_t>(stream));
}
