// K4f -- attention over an fp32 static cache on fp32 MFMA (gfx950 v_mfma_f32_16x16x4_f32).
//
// A model whose parameters are fp32 keeps its cache in fp32 (the reference allocates the cache in
// the parameter dtype, src/inference.py:522, :544) and computes its attention in fp32
// (F.scaled_dot_product_attention at src/inference.py:409 and :452).  This kernel is that
// attention for the fp32 form of the inference path: q, K and V enter the products unrounded, the
// scores and probabilities stay fp32, and only the output is stored as the split (hi|lo bf16)
// input of the out projection, which carries it to ~2^-17.
//
// A wave computes 16 consecutive query positions of one (batch row, head) against 16 keys at a
// time.  Lane l = (c, g), c = l % 16, g = l / 16:
//
//   S^T = K . Q^T   16 keys x 16 queries, 16 MFMAs of k = 4.  MFMA kb pairs lane group g's
//                   A element K[key c][16 g + kb] with its B element q[query c][16 g + kb], so a
//                   lane holds dims 16 g .. 16 g + 15 of one key row and of one query row: four
//                   float4 each.  The accumulator of lane (c, g) holds S^T[keys 4 g .. 4 g + 3]
//                   [query c].
//   softmax         per query column c over the four lane groups (base 2: q carries the softmax
//                   scale times log2(e)), online across key tiles.
//   O^T = V^T . P^T 64 dims x 16 queries as 4 dim blocks x 4 key steps.  Key step r pairs lane
//                   group g's B element P^T[key 4 g + r][query c] -- accumulator element r of
//                   the score MFMA, no data movement -- with A element V[key 4 g + r][4 c + db] of
//                   dim block db, so a lane holds one float4 (dims 4 c .. 4 c + 3) per key step.
//                   Row i of dim block db's accumulator is dim 4 i + db, so lane (c, g) ends
//                   with dims 16 g .. 16 g + 15 of query c (element r of block db = dim
//                   16 g + 4 r + db).
//
// Modes: prefill over [batch, seq] query rows (row b * seq + i), prefill over a packed token
// list (row q_offset[b] + i - kv_start[b], queries i >= kv_start[b] only), and decode (one query
// per batch row at cache slot t).  Key j is visible to the query at position i iff
// kv_start[b] <= j < n_keys, (causal) j <= i, and (j >= mask_len or mask[b * mask_len + j] != 0);
// a query with no visible key outputs 0 (what torch's CPU SDPA returns for an all -inf row).
//
// Prefill (attn_f32_prefill_kernel): a block of QW = 4 waves takes 64 queries, and key tiles of 32
// go through a ring of two LDS stages (K and V, 8 KB each) filled by direct global -> LDS copies,
// the next tile's while this one is worked on; one barrier per tile.  The 16-byte chunks of a
// 256-byte row are XOR-swizzled with the row's low four bits, so both reads (16 rows of one chunk;
// four whole rows) touch every bank once.  What bounds it is the fp32 matrix rate (154 TFLOP/s in
// a large product on this card).  A wave that loaded its own 16 queries' keys from L2 waited for
// every tile and moved four times the bytes: 16 rows of up to 811 tokens and 12 heads
// 271 -> 178 us (92 us of MFMAs), 8 of up to 1,001 and 4 heads 126 -> 61.  A small launch is
// bound by its longest block, whose SIMDs each work through all keys of 16 queries (64 fp32 MFMAs
// of 32 cycles for 32 keys): there KG = 4 groups of QW waves take the tiles in turn, each with a
// ring of its own, and merge their states in LDS at the end (8 ragged rows of up
// to 1,001 tokens and 4 heads 61 -> 49 us).
//
// Order of the sums, causal: tile t of a row (from kv_start) belongs to chain t % 4, each chain is
// an online softmax of its own, and chains 1, 2 and 3 are merged into chain 0 in that order.  The
// four groups of waves hold one chain each; a block of one group holds all four (CH = 4, 72
// registers: 3 waves per SIMD in place of 4), so a query's result does not depend on the size of
// the launch.  That costs the large launches little (16 rows of up to 811 tokens and 12 heads 138 ->
// 142 us, 64 of 200 and 16 heads 66 -> 69, 6 of 811 and 12 heads 72 -> 67).  Without the causal limit
// there is one chain.
//
// Decode (attn_f32_decode_kernel): a work item is one split_len-slot chunk of one (row, head), a
// wave of its own without LDS or barriers; the chunks are what fills the GPU.  The query fills all
// 16 columns, and 32 slots are loaded and worked on at a time.  Lane (c, g) holds dims 16 i + 4 g
// .. + 3 (i = 0..3) of its key row and of the query here (the same order in both, so the products
// pair up), which makes each load 64 contiguous bytes of 16 rows.  With several chunks each writes
// its running state (m, l, unnormalised o) to the workspace, and attn_f32_combine_kernel merges
// them.  What bounds it is the latency of a chunk's few dependent loads, then HBM: 16 rows of 12
// heads over some 750 slots (74 MB) with the merge 26 -> 20 us, 8 rows of 4 heads 19 -> 12 (16-slot
// steps at 128-slot chunks before; a lane's mask bytes were read one by one after the products).
#include "common.h"
#include "lds_dma.h"
#include "mfma.h"

namespace mdl {

namespace {

constexpr int kQT = 16;          // queries of a wave
constexpr int kWavesF = 4;       // decode: waves per block
constexpr int kKT = 32;              // prefill: keys of a tile
constexpr int kTileF = kKT * kHeadDim * 4;   // bytes of a K or V tile

struct F32Args {
  const float* q;                // [rows, H, 64], pre-scaled (softmax scale * log2(e))
  const float* kc;               // [batch, H, slots, 64]
  const float* vc;
  const uint8_t* mask;           // [batch, mask_len] or NULL
  int mask_len;
  const int32_t* kv_start;       // [batch] or NULL (0)
  const int32_t* q_offset;       // packed prefill: [batch]
  const int32_t* seq_dev;        // decode: slot of the query (NULL: seq_pos)
  int seq_pos;
  int batch, heads, slots, seq;  // seq: prefill query / key count
  int causal;
  int q_tiles;                   // work items per (row, head): query blocks, or decode chunks
  int64_t items;                 // decode: chunks; prefill: (row, head) pairs
  uint16_t* out;                 // split bf16 [rows, 2 d]
  int out_layout;
  int split_len;                 // decode: slots per chunk
  float* ws;                     // decode with more than one chunk: kPartF floats per chunk
};

constexpr int kPartF = 2 + kHeadDim;   // m, l, o[64] of one decode chunk

typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ void load16(const float* p, float* v) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float4 t = *reinterpret_cast<const float4*>(p + 4 * i);
    v[4 * i] = t.x; v[4 * i + 1] = t.y; v[4 * i + 2] = t.z; v[4 * i + 3] = t.w;
  }
}

// o / l of query c as the split output of row qrow: lane (c, g) holds dims 16 g + 4 r + db as
// element r of block db
__device__ __forceinline__ void store_out(const F32Args& p, int64_t qrow, int h, int g, float l,
                                          const f32x4 (&o)[4]) {
  const int d = p.heads * kHeadDim;
  const float inv = l > 0.f ? 1.f / l : 0.f;
  float res[16];
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int db = 0; db < 4; ++db) res[4 * r + db] = o[db][r] * inv;
  uint4 hi0, lo0, hi1, lo1;
  split8(res, hi0, lo0);
  split8(res + 8, hi1, lo1);
  const int col = h * kHeadDim + 16 * g;
  if (p.out_layout == MDL_LAYOUT_TILES) {
    *reinterpret_cast<uint4*>(p.out + tile_off(qrow, col, 2 * d)) = hi0;
    *reinterpret_cast<uint4*>(p.out + tile_off(qrow, col + 8, 2 * d)) = hi1;
    *reinterpret_cast<uint4*>(p.out + tile_off(qrow, d + col, 2 * d)) = lo0;
    *reinterpret_cast<uint4*>(p.out + tile_off(qrow, d + col + 8, 2 * d)) = lo1;
  } else {
    uint16_t* orow = p.out + qrow * 2 * d;
    *reinterpret_cast<uint4*>(orow + col) = hi0;
    *reinterpret_cast<uint4*>(orow + col + 8) = hi1;
    *reinterpret_cast<uint4*>(orow + d + col) = lo0;
    *reinterpret_cast<uint4*>(orow + d + col + 8) = lo1;
  }
}

// Blocks: (row, head) pair i % 8 + 8 j on XCD i % 8, the latest (longest) query block of every pair
// first, so that the short ones fill the end of the launch (pair by pair, the last pair's longest
// blocks ran on alone: 213 -> 178 us).
template <int QW, int KG, int CH>
__global__ __launch_bounds__(64 * QW * KG, CH > 1 ? 3 : QW == 2 ? 2 : 4) void
attn_f32_prefill_kernel(const F32Args p) {
  static_assert(KG == 1 || CH == 1, "the key groups or the chains take the tiles in turn");
  static_assert(CH % 2 == 0 || CH == 1, "a turn of the chains ends on the ring's first stage");
  constexpr int kQB = kQT * QW;   // queries of a block
  const int slot = blockIdx.x >> 3, pairs = gridDim.x / (8 * p.q_tiles);   // pairs of an XCD
  const int qt = p.q_tiles - 1 - slot / pairs;
  const int bh = (blockIdx.x & 7) + 8 * (slot % pairs);
  if (bh >= p.items) return;   // pairs padded to a multiple of 8: whole blocks exit
  const int b = bh / p.heads, h = bh - b * p.heads;
  const int S = p.seq;
  const int kstart = p.kv_start ? min(max(p.kv_start[b], 0), S) : 0;
  // packed rows: queries from kstart on, query i at row q_offset[b] + i - kstart
  const int q0 = (p.q_offset ? kstart : 0) + kQB * qt;
  if (q0 >= S) return;         // the whole block lies past the row
  const int64_t qbase = p.q_offset ? static_cast<int64_t>(p.q_offset[b]) - kstart
                                   : static_cast<int64_t>(b) * S;
  const int tid = threadIdx.x, lane = tid & 63, c = lane & 15, g = lane >> 4;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wave = wv % QW, kg = wv / QW;   // query group, key group
  const int wq0 = q0 + kQT * wave;
  const int qi = wq0 + c;
  const int64_t qrow = qbase + min(qi, S - 1);

  __shared__ __attribute__((aligned(16))) uint8_t lds[KG][2][2][kTileF];   // [stage][K, V]
  const int64_t head = (static_cast<int64_t>(b) * p.heads + h) * p.slots * kHeadDim;
  const float* K = p.kc + head;
  const float* V = p.vc + head;
  const uint8_t* mrow = p.mask ? p.mask + static_cast<int64_t>(b) * p.mask_len : nullptr;
  // a row without a valid key attends to nothing
  const int kend = kstart >= S ? kstart : (p.causal ? min(S, q0 + kQB) : S);

  float qv[16];
  load16(p.q + (qrow * p.heads + h) * kHeadDim + 16 * g, qv);

  // Tile kt -> stage st: wave w copies key rows 16 j + 4 w .. + 3 of K and V (j = 0, 1), one
  // kilobyte each; lane l takes physical chunk l % 16 of its row, i.e. logical chunk
  // (l % 16) ^ (row % 16).  Rows past S copy the last key (their weights are 0).
  const uint32_t lds0 = lds_addr(lds) + kg * 4 * kTileF;
  auto issue = [&](int kt, int st) {
#pragma unroll
    for (int j = 0; j < 8 / QW; ++j) {
      const int row = 4 * (QW * j + wave) + (lane >> 4);
      const uint32_t off = min(row, S - 1 - kt) * (kHeadDim * 4) + 16 * (c ^ (row & 15));
      const uint32_t dst = lds0 + 2 * st * kTileF + 4 * (QW * j + wave) * 256;
      const int64_t tile = static_cast<int64_t>(kt) * kHeadDim;
      dma16_sbase(K + tile, off, __builtin_amdgcn_readfirstlane(dst));
      dma16_sbase(V + tile, off, __builtin_amdgcn_readfirstlane(dst + kTileF));
    }
  };
  // lanes 0 .. 31: this lane's key of tile kt is valid (inside the row and not masked)
  auto key_ok = [&](int kt) -> int {
    const int j = kt + (lane & 31);
    if (j >= S) return 0;
    return mrow && j < p.mask_len ? mrow[j] : 1;
  };

  float m[CH], l[CH];   // l: this lane group's part of the sum
  f32x4 o[CH][4];
#pragma unroll
  for (int ch = 0; ch < CH; ++ch) {
    m[ch] = -INFINITY;
    l[ch] = 0.f;
#pragma unroll
    for (int db = 0; db < 4; ++db) o[ch][db] = f32x4{0.f, 0.f, 0.f, 0.f};
  }

  // the tile of keys kt .. kt + 31 at Kt / Vt into the state of chain ch
  auto work = [&](int kt, uint32_t valid, const uint8_t* Kt, const uint8_t* Vt, int ch) {
    f32x4 s[2];
    float kv[2][16];
#pragma unroll
    for (int nb = 0; nb < 2; ++nb) {
      s[nb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float4 t = *reinterpret_cast<const float4*>(Kt + (16 * nb + c) * 256 +
                                                          16 * ((4 * g + i) ^ c));
        kv[nb][4 * i] = t.x; kv[nb][4 * i + 1] = t.y;
        kv[nb][4 * i + 2] = t.z; kv[nb][4 * i + 3] = t.w;
      }
    }
#pragma unroll
    for (int kb = 0; kb < 16; ++kb)
#pragma unroll
      for (int nb = 0; nb < 2; ++nb)
        s[nb] = __builtin_amdgcn_mfma_f32_16x16x4f32(kv[nb][kb], qv[kb], s[nb], 0, 0, 0);
    if (valid != ~0u || (p.causal && kt + kKT - 1 > wq0)) {
      uint32_t vis = valid;
      if (p.causal) {
        const int x = qi - kt;   // offset of the last key query qi may see
        vis &= x >= 31 ? ~0u : (x < 0 ? 0u : (2u << x) - 1u);
      }
#pragma unroll
      for (int nb = 0; nb < 2; ++nb)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (!((vis >> (16 * nb + 4 * g + r)) & 1u)) s[nb][r] = -INFINITY;
    }
    float tmax = -INFINITY;
#pragma unroll
    for (int nb = 0; nb < 2; ++nb)
#pragma unroll
      for (int r = 0; r < 4; ++r) tmax = fmaxf(tmax, s[nb][r]);
    const float m_new = fmaxf(m[ch], max_over_groups(tmax));
    const float base = m_new == -INFINITY ? 0.f : m_new;   // no visible key yet: weights 0
    const float alpha = exp2f(m[ch] - base);
    m[ch] = m_new;
    // exp2f scales its argument to keep results below 2^-126, five instructions more than the bare
    // one, which gives the same bits above: taken where a weight may lie there (2,496 blocks 142 us
    // without it, 150 with it for every weight, 144 so)
    float least = s[0][0];
#pragma unroll
    for (int nb = 0; nb < 2; ++nb)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        least = fminf(least, s[nb][r]);
        s[nb][r] -= base;
      }
    if (__any(least - base < -126.f)) {
#pragma unroll
      for (int nb = 0; nb < 2; ++nb)
#pragma unroll
        for (int r = 0; r < 4; ++r) s[nb][r] = exp2f(s[nb][r]);
    } else {
#pragma unroll
      for (int nb = 0; nb < 2; ++nb)
#pragma unroll
        for (int r = 0; r < 4; ++r) s[nb][r] = __builtin_amdgcn_exp2f(s[nb][r]);
    }
    float psum = 0.f;
#pragma unroll
    for (int nb = 0; nb < 2; ++nb)
#pragma unroll
      for (int r = 0; r < 4; ++r) psum += s[nb][r];
    l[ch] = fmaf(l[ch], alpha, psum);
#pragma unroll
    for (int db = 0; db < 4; ++db) o[ch][db] *= alpha;
#pragma unroll
    for (int nb = 0; nb < 2; ++nb) {
      // sixteen keys past the row or in this wave's future: their weights are zero, but zero times
      // a value that is not finite is NaN
      if (nb == 1 && (kt + 16 >= S || (p.causal && kt + 16 > wq0 + kQT - 1))) continue;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = 16 * nb + 4 * g + r;
        const float4 v = *reinterpret_cast<const float4*>(Vt + row * 256 + 16 * (c ^ (row & 15)));
        const float ve[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int db = 0; db < 4; ++db)
          o[ch][db] = __builtin_amdgcn_mfma_f32_16x16x4f32(ve[db], s[nb][r], o[ch][db], 0, 0, 0);
      }
    }
  };

  constexpr int kStep = kKT * KG;
  int ok_next = 0;
  if (kstart + kKT * kg < kend) {
    ok_next = key_ok(kstart + kKT * kg);
    issue(kstart + kKT * kg, 0);
  }
  // every wave of the block makes the same number of turns, so the barriers match; a group whose
  // tile would start past the end neither copies nor computes
  int st = 0;
  for (int t0 = kstart; t0 < kend; t0 += kStep * CH) {
#pragma unroll
    for (int ch = 0; ch < CH; ++ch) {
      const int kt = t0 + kStep * ch + kKT * kg;
      if (CH > 1 && kt >= kend) break;   // whole block (KG is 1)
      // tile kt has landed for every wave, and every wave is done with the other stage (the builtin
      // wait, so that the compiler counts its own loads, q and the mask bytes, as landed too)
      __builtin_amdgcn_s_waitcnt(kWaitAll);
      asm volatile("s_barrier" ::: "memory");
      const uint32_t valid = static_cast<uint32_t>(__ballot(ok_next != 0));
      const int cur = CH > 1 ? ch & 1 : st;   // the tile's stage
      st ^= 1;
      if (kt + kStep < kend) {
        ok_next = key_ok(kt + kStep);
        issue(kt + kStep, cur ^ 1);
      }
      // nothing past the end, nor a tile that lies wholly in this wave's future
      if (kt < kend && !(p.causal && kt > wq0 + kQT - 1))
        work(kt, valid, lds[kg][cur][0], lds[kg][cur][1], ch);
    }
  }
  // chain j's state (m, l, o) into chain 0's, j = 1, 2, 3 in order, whatever holds it
  auto merge = [&](float mj, float lj, auto oj) {
    const float m_new = fmaxf(m[0], mj);
    const float base = m_new == -INFINITY ? 0.f : m_new;
    const float a = exp2f(m[0] - base), aj = exp2f(mj - base);
    m[0] = m_new;
    l[0] = fmaf(lj, aj, l[0] * a);
#pragma unroll
    for (int i = 0; i < 16; ++i)
      o[0][i >> 2][i & 3] = fmaf(oj(i), aj, o[0][i >> 2][i & 3] * a);
  };
  if constexpr (CH > 1) {
#pragma unroll
    for (int j = 1; j < CH; ++j)
      merge(m[j], l[j], [&](int i) { return o[j][i >> 2][i & 3]; });
  }
  if constexpr (KG > 1) {
    // the other groups' states through the ring's memory, one float per lane at a time
    __syncthreads();   // every wave is done with its tiles
    float* part = reinterpret_cast<float*>(lds);
    if (kg > 0) {
      float* w = part + ((kg - 1) * QW + wave) * 18 * kWave + lane;
      w[0] = m[0];
      w[kWave] = l[0];
#pragma unroll
      for (int i = 0; i < 16; ++i) w[(2 + i) * kWave] = o[0][i >> 2][i & 3];
    }
    __syncthreads();
    if (kg > 0) return;
#pragma unroll
    for (int j = 0; j < KG - 1; ++j) {
      const float* w = part + (j * QW + wave) * 18 * kWave + lane;
      merge(w[0], w[kWave], [&](int i) { return w[(2 + i) * kWave]; });
    }
  }
  if (qi >= S) return;
  float sum = l[0];
  sum += __shfl_xor(sum, 16, kWave);
  sum += __shfl_xor(sum, 32, kWave);
  store_out(p, qrow, h, g, sum, o[0]);
}

__global__ __launch_bounds__(64 * kWavesF) void attn_f32_decode_kernel(const F32Args p) {
  const int64_t item = static_cast<int64_t>(blockIdx.x) * kWavesF + (threadIdx.x >> 6);
  if (item >= p.items) return;   // whole wave; the kernel has no barrier
  const int lane = threadIdx.x & 63, c = lane & 15, g = lane >> 4;
  const int64_t bh = item / p.q_tiles;
  const int chunk = p.q_tiles - 1 - static_cast<int>(item - bh * p.q_tiles);
  const int b = static_cast<int>(bh / p.heads), h = static_cast<int>(bh - b * p.heads);
  const int t = p.seq_dev ? *p.seq_dev : p.seq_pos;
  const int n_keys = min(t + 1, p.slots);
  int klo = p.kv_start ? min(max(p.kv_start[b], 0), n_keys) : 0;
  klo = min(klo + chunk * p.split_len, n_keys);
  const int khi = min(klo + p.split_len, n_keys);   // slots of this chunk: [klo, khi)

  float qv[16];   // element 4 i + e: dim 16 i + 4 g + e of the query
  const float* qp = p.q + (static_cast<int64_t>(b) * p.heads + h) * kHeadDim + 4 * g;
#pragma unroll
  for (int i = 0; i < 4; ++i)
    *reinterpret_cast<float4*>(qv + 4 * i) = *reinterpret_cast<const float4*>(qp + 16 * i);
  const int64_t head = (static_cast<int64_t>(b) * p.heads + h) * p.slots * kHeadDim;
  const float* K = p.kc + head;
  const float* V = p.vc + head;
  const uint8_t* mrow = p.mask ? p.mask + static_cast<int64_t>(b) * p.mask_len : nullptr;

  float m_run = -INFINITY, l_run = 0.f;   // l_run: this lane group's part of the sum
  f32x4 o[4];
#pragma unroll
  for (int db = 0; db < 4; ++db) o[db] = f32x4{0.f, 0.f, 0.f, 0.f};

  for (int k0 = klo; k0 < khi; k0 += 2 * kQT) {
    // the 32 slots' visibility, one lane each, read with the keys
    const int kj = k0 + (lane & 31);
    bool ok = kj < khi;
    if (mrow && kj < p.mask_len) ok = ok && mrow[kj] != 0;
    // rows past the chunk load its last slot; their weights are 0
    float4 kv[2][4], vv[2][4];   // V rows k0 + 16 nb + 4 g + r, dims 4 c .. 4 c + 3
#pragma unroll
    for (int nb = 0; nb < 2; ++nb) {
      const float* kp =
          K + static_cast<int64_t>(min(k0 + 16 * nb + c, khi - 1)) * kHeadDim + 4 * g;
#pragma unroll
      for (int i = 0; i < 4; ++i) kv[nb][i] = ld_f4<true>(kp + 16 * i);
    }
#pragma unroll
    for (int nb = 0; nb < 2; ++nb)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        vv[nb][r] = ld_f4<true>(
            V + static_cast<int64_t>(min(k0 + 16 * nb + 4 * g + r, khi - 1)) * kHeadDim + 4 * c);
    f32x4 s[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int nb = 0; nb < 2; ++nb) {
          const float4 k4 = kv[nb][i];
          const float a = e == 0 ? k4.x : e == 1 ? k4.y : e == 2 ? k4.z : k4.w;
          s[nb] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, qv[4 * i + e], s[nb], 0, 0, 0);
        }
    const uint32_t vis = static_cast<uint32_t>(__ballot(ok));
    if (vis != ~0u) {
#pragma unroll
      for (int nb = 0; nb < 2; ++nb)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (!((vis >> (16 * nb + 4 * g + r)) & 1u)) s[nb][r] = -INFINITY;
    }
    float tmax = -INFINITY;
#pragma unroll
    for (int nb = 0; nb < 2; ++nb)
#pragma unroll
      for (int r = 0; r < 4; ++r) tmax = fmaxf(tmax, s[nb][r]);
    const float m_old = m_run;
    m_run = fmaxf(m_run, max_over_groups(tmax));
    const float base = m_run == -INFINITY ? 0.f : m_run;   // no visible slot yet: weights 0
    const float alpha = exp2f(m_old - base);
    float psum = 0.f;
#pragma unroll
    for (int nb = 0; nb < 2; ++nb)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        s[nb][r] = exp2f(s[nb][r] - base);
        psum += s[nb][r];
      }
    l_run = fmaf(l_run, alpha, psum);
#pragma unroll
    for (int db = 0; db < 4; ++db) o[db] *= alpha;
    // O^T += V^T . P^T, key step r: lane group g contributes key 4 g + r
#pragma unroll
    for (int nb = 0; nb < 2; ++nb)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float ve[4] = {vv[nb][r].x, vv[nb][r].y, vv[nb][r].z, vv[nb][r].w};
#pragma unroll
        for (int db = 0; db < 4; ++db)
          o[db] = __builtin_amdgcn_mfma_f32_16x16x4f32(ve[db], s[nb][r], o[db], 0, 0, 0);
      }
  }
  l_run += __shfl_xor(l_run, 16, kWave);
  l_run += __shfl_xor(l_run, 32, kWave);

  if (c != 0) return;   // every column holds the same
  if (p.ws) {
    // this chunk's state: m and l, o unnormalised
    float* part = p.ws + item * kPartF;
    if (g == 0) {
      part[0] = m_run;
      part[1] = l_run;
    }
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int db = 0; db < 4; ++db) part[2 + 16 * g + 4 * r + db] = o[db][r];
    return;
  }
  store_out(p, b, h, g, l_run, o);
}

// The decode chunks of one (row, head) merged, lane = channel: the states rescaled to their
// largest m (base 2), o / l, stored as the split output of mdl_attn_decode_f32.
__global__ __launch_bounds__(256) void attn_f32_combine_kernel(const float* __restrict__ ws,
                                                               int n_bh, int n_heads,
                                                               int n_split,
                                                               uint16_t* __restrict__ out,
                                                               int out_layout) {
  const int bh = blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (bh >= n_bh) return;
  const float v = merge_parts<kPartF>(ws + static_cast<int64_t>(bh) * n_split * kPartF, n_split,
                                      lane);
  const int b = bh / n_heads, h = bh - b * n_heads;
  const int d = n_heads * kHeadDim, col = h * kHeadDim + lane;
  const uint16_t hi = static_cast<uint16_t>(f2bf(v));
  const uint16_t lo = static_cast<uint16_t>(f2bf(v - bf2f(hi)));
  if (out_layout == MDL_LAYOUT_TILES) {
    out[tile_off(b, col, 2 * d)] = hi;
    out[tile_off(b, d + col, 2 * d)] = lo;
  } else {
    out[static_cast<int64_t>(b) * 2 * d + col] = hi;
    out[static_cast<int64_t>(b) * 2 * d + d + col] = lo;
  }
}

constexpr int kBlocksSplit32 = 256, kBlocksSplit64 = 512;   // 64-query blocks

template <int QW, int KG, int CH>
int launch_prefill_f32(F32Args p, hipStream_t st) {
  p.q_tiles = (p.seq + kQT * QW - 1) / (kQT * QW);
  const int64_t blocks = (p.items + 7) / 8 * 8 * p.q_tiles;
  if (blocks > 0x7fffffff) return MDL_ERR_SHAPE;
  hipLaunchKernelGGL((attn_f32_prefill_kernel<QW, KG, CH>), dim3(static_cast<unsigned>(blocks)),
                     dim3(64 * QW * KG), 0, st, p);
  return launch_status();
}

int check_f32(const float* q, const float* k_cache, const float* v_cache, int batch,
              int n_heads, int head_dim, int cache_slots, const uint16_t* out, int out_layout) {
  if (!q || !k_cache || !v_cache || !out) return MDL_ERR_NULL;
  if (head_dim != kHeadDim) return MDL_ERR_HEAD_DIM;
  if (batch < 0 || n_heads <= 0 || n_heads > (1 << 16) || cache_slots <= 0 ||
      (out_layout != MDL_LAYOUT_ROWS && out_layout != MDL_LAYOUT_TILES))
    return MDL_ERR_SHAPE;
  if (!aligned16(q) || !aligned16(k_cache) || !aligned16(v_cache) || !aligned16(out))
    return MDL_ERR_ALIGN;
  return MDL_OK;
}

}  // namespace

}  // namespace mdl

using namespace mdl;

extern "C" int mdl_attn_prefill_f32(const float* q, const float* k_cache, const float* v_cache,
                                    int batch, int seq, int n_heads, int head_dim,
                                    int cache_slots, const uint8_t* key_mask,
                                    const int32_t* kv_start, const int32_t* q_offset, int causal,
                                    uint16_t* out, int out_layout, void* stream) {
  const int rc = check_f32(q, k_cache, v_cache, batch, n_heads, head_dim, cache_slots, out,
                           out_layout);
  if (rc != MDL_OK) return rc;
  if (seq <= 0) return MDL_ERR_SHAPE;
  if (seq > cache_slots) return MDL_ERR_CACHE;
  if (q_offset && !kv_start) return MDL_ERR_NULL;
  F32Args p{};
  p.q = q; p.kc = k_cache; p.vc = v_cache;
  p.mask = key_mask; p.mask_len = seq;
  p.kv_start = kv_start; p.q_offset = q_offset;
  p.batch = batch; p.heads = n_heads; p.slots = cache_slots; p.seq = seq;
  p.causal = causal != 0;
  p.items = static_cast<int64_t>(batch) * n_heads;
  p.out = out; p.out_layout = out_layout;
  if (p.items == 0) return MDL_OK;
  const hipStream_t st = static_cast<hipStream_t>(stream);
  // How the longest block's key tiles are split while 64-query blocks number one or two per CU:
  // four groups of waves take the tiles in turn, on 32 queries at up to one block per CU (so that
  // twice as many CUs work) and on 64 at up to two.  Causal, us as one group of 64 / here: 60
  // blocks 17.0 / 10.9, 144 34.7 / 20.3, 432 33.3 / 28.5, 512 60.1 / 49.4.  Past that as one group
  // (here) / as four: 528 45.1 / 43.7, 600 44.5 / 47.9, 624 56.9 / 50.0, 936 67 / 74, 2,496 142 /
  // 182.  Without the causal limit every block is as long as the longest, and one group is as good
  // or better (144: 37.5 / 39.2, 432: 47.6 / 49.7).
  const int64_t blocks = p.items * ((seq + 63) / 64);
  if (p.causal && blocks <= kBlocksSplit32) return launch_prefill_f32<2, 4, 1>(p, st);
  if (p.causal && blocks <= kBlocksSplit64) return launch_prefill_f32<4, 4, 1>(p, st);
  return p.causal ? launch_prefill_f32<4, 1, 4>(p, st) : launch_prefill_f32<4, 1, 1>(p, st);
}

extern "C" int mdl_attn_decode_f32(const float* q, const float* k_cache, const float* v_cache,
                                   int batch, int n_heads, int head_dim, int cache_slots,
                                   const uint8_t* prompt_mask, int prompt_len,
                                   const int32_t* kv_start, int seq_pos, const int32_t* seq_dev,
                                   float* workspace, int64_t workspace_bytes, int split_len,
                                   uint16_t* out, int out_layout, void* stream) {
  const int rc = check_f32(q, k_cache, v_cache, batch, n_heads, head_dim, cache_slots, out,
                           out_layout);
  if (rc != MDL_OK) return rc;
  if (prompt_len < 0 || (prompt_mask && prompt_len == 0) || split_len < kQT ||
      split_len % kQT != 0)
    return MDL_ERR_SHAPE;
  if (!seq_dev && (seq_pos < 0 || seq_pos >= cache_slots)) return MDL_ERR_CACHE;
  const int n_split = (cache_slots + split_len - 1) / split_len;
  const int64_t n_bh = static_cast<int64_t>(batch) * n_heads;
  if (n_split > 1) {
    if (!workspace) return MDL_ERR_WORKSPACE;
    if (workspace_bytes < n_bh * n_split * kPartF * static_cast<int64_t>(sizeof(float)))
      return MDL_ERR_WORKSPACE;
    if (!aligned16(workspace)) return MDL_ERR_ALIGN;
  }
  F32Args p{};
  p.q = q; p.kc = k_cache; p.vc = v_cache;
  p.mask = prompt_mask; p.mask_len = prompt_len;
  p.kv_start = kv_start;
  p.seq_dev = seq_dev; p.seq_pos = seq_pos;
  p.batch = batch; p.heads = n_heads; p.slots = cache_slots; p.seq = cache_slots;
  p.causal = 1;
  p.q_tiles = n_split;
  p.split_len = split_len;
  p.ws = n_split > 1 ? workspace : nullptr;
  p.items = n_bh * n_split;
  p.out = out; p.out_layout = out_layout;
  const hipStream_t st = static_cast<hipStream_t>(stream);
  if (p.items == 0) return MDL_OK;
  const int64_t blocks = (p.items + kWavesF - 1) / kWavesF;
  if (blocks > 0x7fffffff) return MDL_ERR_SHAPE;
  hipLaunchKernelGGL(attn_f32_decode_kernel, dim3(static_cast<unsigned>(blocks)),
                     dim3(64 * kWavesF), 0, st, p);
  const int rc2 = launch_status();
  if (rc2 != MDL_OK || n_split == 1) return rc2;
  if ((n_bh + 3) / 4 > 0x7fffffff) return MDL_ERR_SHAPE;
  hipLaunchKernelGGL(attn_f32_combine_kernel, dim3(static_cast<unsigned>((n_bh + 3) / 4)),
                     dim3(256), 0, st, workspace, static_cast<int>(n_bh), n_heads, n_split, out,
                     out_layout);
  return launch_status();
}
