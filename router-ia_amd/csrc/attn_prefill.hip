// Causal GQA full-attention prefill over the paged KV cache, for gfx950.
//
// Equal to `length` decode steps of the reference (qwen36_attention_cache.py:
// 306-317) run one token at a time, which is how the reference prefills
// (qwen36_chat_batch.py:255-258): token t of the prompt, at absolute position
// start + t, is RoPE-rotated, appended, and attends to every resident token
// 0 .. start + t; the output is softmax(q K^T * scale) V * sigmoid(gate).
//
// Two launches: the prompt's k (rotated) and v go into the pages first (the
// append kernel in sequence mode), then one workgroup per (query block of 16
// or 32 tokens, KV head[, piece of its keys]) streams the keys 0 .. last query
// of the block in blocks of 32 keys (two pages); a third launch merges the
// pieces where query blocks are split.
//   * bound by LDS operand reads and the softmax between the MFMAs: with 16
//     tokens a wave reads one operand (8 cycles of the CU's LDS) per 16-cycle
//     MFMA of its SIMD, so the MFMAs could run half the time at best (16384
//     tokens: 2.25 ms, 0.98 PFLOP/s); with 32 tokens (fp16 operands: q 64 and
//     O 128 of the 256 registers) each operand feeds two, 1.82 ms, 1.21
//     PFLOP/s on the same box, where a large fp16 matrix product of the
//     library reaches 1.5;
//   * 8 waves, one query head each (GQA group <= 8), two waves per SIMD: one
//     wave's softmax (VALU, transcendental) overlaps the other's MFMAs, and
//     every key block fetched serves the block's tokens x 8 heads;
//   * key blocks travel HBM/L2 -> LDS by direct-to-LDS loads into a 4-slot
//     ring, in pairs two blocks ahead of the one being computed, with no
//     registers in flight and one barrier per pair;
//   * scores S^T = K Q^T on 16x16x32 MFMA (16 keys x 16 tokens per tile): the
//     K tile is already in A-operand order (8 dims of one token are 16
//     contiguous bytes); the two score tiles of a block take their rows from
//     the block's tokens in an order that leaves lane group g with exactly 8
//     consecutive tokens of one page, whose V^T column is then one 16-byte
//     operand of O^T = V^T P^T (16x16x32, k = those 32 keys);
//   * with a bf16 cache the rotated q and the probabilities are carried as
//     bf16 hi + lo pairs (near-fp32 operands on MFMA); with an fp16 cache the
//     fp16 hi part alone (11 significant bits); the online softmax is kept in log2
//     units (q is pre-scaled) with a lazy rescale (only when a block max
//     exceeds the running max by 2^8); row statistics combine across lane
//     groups with permlane swaps;
//   * the gated result leaves through LDS so the output stores are coalesced;
//   * query blocks are scheduled from the last (most keys) to the first.
#include <float.h>
#include <math.h>
#include <algorithm>

#include "ria_common.h"

namespace ria {

constexpr int kTile = kPageTokens * kAttnHeadDim;  // elements per (page, KV head) tile
constexpr int kTileVec = kTile * 2 / 16;           // 16-byte vectors per tile (512)
// Ring slot layout (16-byte vectors): K page 0 at 0, K page 1 at kSlotK1 (64
// bytes further than back-to-back, so the rows of the two pages that one
// 16-lane read pass touches fall on different banks), V^T pages 0 and 1 at
// kSlotV + 512 m, each stored as [token half][dim][8 tokens].
constexpr int kSlotK1 = kTileVec + 4;
constexpr int kSlotV = kSlotK1 + kTileVec;
constexpr int kSlotVec = kSlotV + 2 * kTileVec;
constexpr int kRingSlots = 4;
constexpr int kPrefillWaves = 8;                   // one query head per wave
constexpr int kPrefillThreads = 64 * kPrefillWaves;
constexpr int kStagePitch = kAttnHeadDim + 4;      // floats per staged output row
constexpr int kPrefillLds = kPrefillWaves * 16 * kStagePitch * 4;  // output stage; the ring (128 KiB) aliases it
constexpr int kMaxPieces = 32;      // pieces of a query block's keys
constexpr int kMinPieceBlocks = 4;  // 32-key blocks of a piece: two refills of the ring
static_assert(kRingSlots * kSlotVec * 16 <= kPrefillLds, "ring must fit in the LDS block");

struct PrefillAttnArgs {
  const void* q;
  int64_t q_stride;
  const void* gate;
  int64_t gate_stride;
  const uint16_t* k_cache;
  const uint16_t* v_cache;
  int num_pages;
  int64_t pt_len;  // entries in the sequence's page-table row
  int start;   // tokens resident before the prompt
  int length;  // prompt tokens
  const float* inv_freq;
  int rope_dim;
  const float* q_norm_w;  // q_norm weight [256] f32, or null: q arrives normalised
  float scale;
  int num_q_heads;
  int num_kv_heads;
  int group;
  void* out;
  int staged;  // keys from an fp16 stage with tile (page p, KV head) at p * Hkv + kvh, not the page table
  int chunk;   // 32-key blocks per piece of a query block's keys (even); 0: no query block is split
  float* part;     // split pieces: unnormalised O, [piece][head of the group][token 16][256]
  float2* part_ml;  // .. and the columns' (max, sum), [piece][head of the group][token 16]
};

// Pieces.  The keys of a query block are split every `chunk` 32-key blocks,
// as far as a piece's first key is visible to the block's first query (so
// every column of every piece sees a key); the last piece takes the rest.  Piece s exists for the query blocks qb >= first_query_block(s).  A
// launch lists the pieces by s, each s from the last query block down, and
// both kernels find a piece's index by the same counts.
__host__ __device__ inline int first_query_block(int s, int chunk, int start, int nqb, int qt) {
  if (s == 0) return 0;
  const int64_t k0 = (int64_t)s * chunk * 32 - start;  // query tokens from here on see the piece's first key
  return k0 <= 0 ? 0 : static_cast<int>(k0 + qt - 1 < (int64_t)qt * nqb ? (k0 + qt - 1) / qt : nqb);
}
__host__ __device__ inline int query_block_pieces(int qb, int chunk, int start, int qt) {
  return chunk ? 1 + (start + qt * qb) / (32 * chunk) : 1;
}

// Key held by row r (0..15) of score tile m (0, 1) of a 32-key block, as
// (page of the block, token): lane group g = r / 4 of both tiles together
// holds tokens 8 (g % 2) .. 8 (g % 2) + 7 of page g / 2, tile m the half
// 8 (g % 2) + 4 m .. + 3.
__device__ __forceinline__ int tile_row_page(int r) { return r >> 3; }
__device__ __forceinline__ int tile_row_token(int m, int r) { return 8 * ((r >> 2) & 1) + 4 * m + (r & 3); }

// max of three scores (never NaN: finite products, or -inf where masked) in
// one instruction; fmaxf would first quiet each MFMA result for IEEE NaN rules
__device__ __forceinline__ float max3_f(float a, float b, float c) {
  float r;
  asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}

// acc + the two fp16 values of w (exact products with 1, fp32 sum)
__device__ __forceinline__ float sum_pair_f16(uint32_t w, float acc) {
  typedef _Float16 h2 __attribute__((ext_vector_type(2)));
  return __builtin_amdgcn_fdot2(__builtin_bit_cast(h2, w), h2{1, 1}, acc, false);
}

__device__ __forceinline__ float swap_max(float x, bool rows16) {
  const auto s = rows16 ? __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false)
                        : __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(s[0]), __uint_as_float(s[1]));
}

__device__ __forceinline__ float swap_sum(float x, bool rows16) {
  const auto s = rows16 ? __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false)
                        : __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(s[0]) + __uint_as_float(s[1]);
}

template <int AT, int KVT, int NC>
__global__ __launch_bounds__(kPrefillThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) void attn_prefill_kernel(
    PrefillAttnArgs a, const int32_t* __restrict__ pt) {
  using KV = Kv16<KVT>;
  // bf16 operands carry q and the probabilities as hi + lo pairs; fp16 ones
  // keep 11 significant bits in the hi part alone, which is enough here
  constexpr bool kSplit = KVT == RIA_DT_BF16;
  static_assert(NC == 1 || !kSplit, "two column tiles of hi + lo operands do not fit the registers");
  constexpr int QT = 16 * NC;             // tokens of a query block
  constexpr int KG = NC == 1 ? 8 : 1;     // 32-dim steps of K operands loaded at a time
  constexpr int VG = NC == 1 ? 16 : 4;    // dim tiles of V^T operands loaded at a time
  constexpr int NO = NC == 1 ? 17 : 16;   // O tiles of a column tile (17: the all-ones product)
  const int nqb = (a.length + QT - 1) / QT;
  int piece = 0, unit = static_cast<int>(blockIdx.x);
  if (a.chunk)
    for (int n; unit >= (n = (nqb - first_query_block(piece, a.chunk, a.start, nqb, QT)) * a.num_kv_heads); unit -= n) ++piece;
  const int qb = nqb - 1 - unit / a.num_kv_heads;  // heaviest blocks first
  const int kvh = unit % a.num_kv_heads;
  const int pieces = query_block_pieces(qb, a.chunk, a.start, QT);
  const int tid = threadIdx.x, lane = tid & 63;
  // in a scalar register: the copies' LDS destinations and bases are then scalar
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 15;   // MFMA column (token QT qb + 16 c + n) / row (key or dim)
  const int g4 = lane >> 4;  // lane group: k slice of the operands, row group of the results

  __shared__ __attribute__((aligned(16))) unsigned char smem[kPrefillLds];
  u32x4* ring = reinterpret_cast<u32x4*>(smem);
  float* stage = reinterpret_cast<float*>(smem);

  const bool head_ok = wave < a.group;
  const int head = kvh * a.group + wave;
  const int ctx_total = a.start + a.length;  // keys that exist

  // ---- q operands: column n, dims 32 kd + 8 g4 + j, RoPE'd, scaled by
  //      scale * log2(e) (scores come out in log2 units), as hi + lo pairs
  u32x4 qh[NC][8], ql[8];
  // SEP: fp16 values converted one at a time, so hipcc folds the multiply
  // that produced each (q times its scale) into the conversion
  // (v_fma_mixlo_f16, one rounding); the probabilities, which no multiply
  // produces, take the paired conversion.
  auto pack = [&](const float (&x)[8], u32x4& hi, u32x4& lo, auto sep) {
    uint32_t h4[4], l4[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if constexpr (decltype(sep)::value && KVT == RIA_DT_F16)
        h4[j] = uint32_t(f32_to_f16_bits(x[2 * j])) | (uint32_t(f32_to_f16_bits(x[2 * j + 1])) << 16);
      else
        h4[j] = KV::pack2(x[2 * j], x[2 * j + 1]);
      l4[j] = KV::pack2(x[2 * j] - KV::lo_f32(h4[j]), x[2 * j + 1] - KV::hi_f32(h4[j]));
    }
    hi = u32x4{h4[0], h4[1], h4[2], h4[3]};
    lo = u32x4{l4[0], l4[1], l4[2], l4[3]};
  };
  const float sl2 = a.scale * 1.4426950408889634f;
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const int t_row = QT * qb + 16 * c + n;
    const bool row_ok = head_ok && t_row < a.length;
    const int qpos = a.start + t_row;
    const int64_t base = (int64_t)t_row * a.q_stride + (int64_t)head * kAttnHeadDim + 8 * g4;
    auto load_q8 = [&](int kd, float (&x)[8]) {
      if (row_ok) {
        load_act8<AT>(a.q, base + 32 * kd, x);
      } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) x[j] = 0.f;
      }
    };
    float y[8][8];
#pragma unroll
    for (int kd = 0; kd < 8; ++kd) load_q8(kd, y[kd]);
    // q_norm (qwen36_attention_cache.py:302-304) before RoPE: the row's sum of
    // squares, whose four 64-dim slices sit in lanes n, n + 16, n + 32, n + 48.
    if (a.q_norm_w) {
      float ss = 0.f;
#pragma unroll
      for (int kd = 0; kd < 8; ++kd)
#pragma unroll
        for (int j = 0; j < 8; ++j) ss = add_rn(ss, mul_rn(y[kd][j], y[kd][j]));
      const float qs = rms_scale(swap_sum(swap_sum(ss, true), false), kAttnHeadDim);
#pragma unroll
      for (int kd = 0; kd < 8; ++kd) {
        const f32x4* wp = reinterpret_cast<const f32x4*>(a.q_norm_w + 32 * kd + 8 * g4);
        const f32x4 w0 = wp[0], w1 = wp[1];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          y[kd][j] = rmsnorm_elem<AT>(y[kd][j], qs, w0[j]);
          y[kd][4 + j] = rmsnorm_elem<AT>(y[kd][4 + j], qs, w1[j]);
        }
      }
    }
    // dims [0, 64) are kd 0, 1; rotate_half pairs dim 8 g4 + j with 32 + 8 g4 + j
    if (a.rope_dim == 64) {
      const float pos = static_cast<float>(qpos);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float ang = mul_rn(pos, a.inv_freq[8 * g4 + j]);
        float cs, sn;
        sincosf(ang, &sn, &cs);
        const float x1 = y[0][j], x2 = y[1][j];
        y[0][j] = add_rn(mul_rn(x1, cs), mul_rn(-x2, sn));
        y[1][j] = add_rn(mul_rn(x2, cs), mul_rn(x1, sn));
      }
    }
#pragma unroll
    for (int kd = 0; kd < 8; ++kd) {
#pragma unroll
      for (int j = 0; j < 8; ++j) y[kd][j] *= sl2;
      pack(y[kd], qh[c][kd], ql[kd], std::true_type{});
    }
  }

  const int q_last = a.start + min(QT * qb + QT - 1, a.length - 1);  // last query position of the block
  const int npages = q_last / kPageTokens + 1;                   // <= pt_len (checked on the host)
  const int blk0 = piece * a.chunk;  // this piece's key blocks: blk0 (even) .. nblk - 1
  const int nblk = piece + 1 < pieces ? blk0 + a.chunk : (npages + 1) / 2;
  const int kmax = min(q_last, ctx_total - 1);  // last key any column of the block uses
  const int q_first = a.start + QT * qb;         // first query position of the block

  // Direct-to-LDS copy of key block b (K and V tiles of pages 2b, 2b+1) into
  // ring slot b % 4: 4 loads of 16 bytes per thread; a page past the block's
  // range reads page 0 and is masked out.
  auto slot_of = [&](int b) { return ring + (b % kRingSlots) * kSlotVec; };
  auto issue = [&](int b) {
    u32x4* slot = slot_of(b);
    int ln = lane;
    asm volatile("" : "+v"(ln));  // its multiples computed here, not held over the loop
#pragma unroll
    for (int pg = 0; pg < 2; ++pg) {
      const int p = 2 * b + pg;
      int phys = p < npages ? (a.staged ? p : pt[p]) : 0;
      phys = (phys < 0 || phys >= a.num_pages) ? 0 : phys;  // unallocated entries never fault
      const int64_t tile = (int64_t)phys * a.num_kv_heads + kvh;
      // through a buffer resource per tile, in scalar registers, so the lane's
      // part of the address is a 32-bit offset
      const auto kr = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(a.k_cache + tile * kTile), 0, kTile * 2,
                                                        kBufferWord3);
      const auto vr = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(a.v_cache + tile * kTile), 0, kTile * 2,
                                                        kBufferWord3);
      const int v = wave * 64;  // this wave's 64 vectors of each tile; lane l lands at +l
      __builtin_amdgcn_raw_ptr_buffer_load_lds(kr, slot + pg * kSlotK1 + v, 16, 16 * ln, 16 * v, 0, 0);
      // V^T position (half, dim) = v + lane holds tile vector 2 dim + half
      __builtin_amdgcn_raw_ptr_buffer_load_lds(vr, slot + kSlotV + pg * kTileVec + v, 16, 32 * ln,
                                               32 * (wave & 3) * 64 + 16 * (wave >> 2), 0, 0);
    }
  };

  // O^T tiles: dims 16 dt + 4 g4 + i, column n.  The softmax's normaliser is
  // the sum of the probabilities as the MFMAs weight V with them.  One column
  // tile: o[16], the product with an all-ones V^T tile, every row that sum (no
  // VALU adds and no cross-lane sum).  Two: l_run, the lane's own keys' part
  // of it by v_dot2, summed across lanes at the end (the eight registers of
  // the all-ones tiles are not there).
  f32x4 o[NC][NO];
  float m_run[NC], l_run[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) {
#pragma unroll
    for (int dt = 0; dt < NO; ++dt) o[c][dt] = f32x4{0.f, 0.f, 0.f, 0.f};
    // below every score, and finite: a block or piece whose scores are all -inf
    // (infinite keys) then weighs 0 instead of exp2(-inf + inf)
    m_run[c] = -FLT_MAX;
    l_run[c] = 0.f;
  }
  constexpr uint32_t kOne2 = KVT == RIA_DT_F16 ? 0x3C003C00u : 0x3F803F80u;  // two 16-bit 1.0

  // K operands of this lane (row n of score tile m, dims 32 kd + 8 g4 .. + 7):
  // token tile_row_token(m, n) of page tile_row_page(n), dim group q8 = 4 kd +
  // g4 at vector ((q8 % 8) * 4 + q8 / 8) * 16, so k_vec + 256 (kd % 2) +
  // 16 (kd / 2) + 4 m.
  const int k_vec = tile_row_page(n) * kSlotK1 + tile_row_token(0, n) + 64 * g4;
  // V^T operand of this lane for dim tile dt: dim 16 dt + n, tokens
  // 8 (g4 % 2) .. + 7 of page g4 / 2 (one 16-byte vector).
  const int v_vec = kSlotV + (g4 >> 1) * kTileVec + (g4 & 1) * 256 + n;
  // key of result row i of score tile m in this lane: 32 b + 8 g4 + 4 m + i

  // Each phase first issues all of its LDS operand reads, then its MFMAs
  // (scheduling barriers keep the compiler from re-serialising them); the
  // V^T reads of a block go out before its softmax so they land meanwhile.
  //
  // ---- scores of block b: two 16-key tiles; q_hi and q_lo products in separate
  //      accumulators so no MFMA waits on the one just before it
  auto qk = [&](int b, f32x4 (&sc)[NC][2]) {
    const u32x4* slot = slot_of(b);
    u32x4 kop[8 / KG > 1 ? 2 : 1][KG][2];
    auto load_k = [&](int g, u32x4 (&dst)[KG][2]) {
#pragma unroll
      for (int i = 0; i < KG; ++i) {
        const int kd = KG * g + i;
        dst[i][0] = slot[k_vec + 256 * (kd & 1) + 16 * (kd >> 1)];
        dst[i][1] = slot[k_vec + 256 * (kd & 1) + 16 * (kd >> 1) + 4];
      }
    };
    load_k(0, kop[0]);
    __builtin_amdgcn_sched_barrier(0);  // groups land in order
    f32x4 acc[NC][2], acl[2];
#pragma unroll
    for (int m = 0; m < 2; ++m) {
      acl[m] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int c = 0; c < NC; ++c) acc[c][m] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int g = 0; g < 8 / KG; ++g) {
      if (g + 1 < 8 / KG) load_k(g + 1, kop[(g + 1) & 1]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < KG; ++i)
#pragma unroll
        for (int m = 0; m < 2; ++m) {
          const int kd = KG * g + i;
#pragma unroll
          for (int c = 0; c < NC; ++c) acc[c][m] = KV::mfma_k32(kop[g & 1][i][m], qh[c][kd], acc[c][m]);
          if (kSplit) acl[m] = KV::mfma_k32(kop[g & 1][i][m], ql[kd], acl[m]);
        }
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
      for (int c = 0; c < NC; ++c) sc[c][m] = kSplit ? acc[c][m] + acl[m] : acc[c][m];
  };

  // ---- online softmax of block b (log2 units), then O^T += V^T P^T over its 32 keys
  auto softmax_pv = [&](int b, const f32x4 (&sc)[NC][2], auto tail) {
    const u32x4* slot = slot_of(b);
    int tile0_keys = 0;  // of the lane's 8 keys, those the first column tile sees
    if constexpr (decltype(tail)::value) {
      int ln = lane;
      asm volatile("" : "+v"(ln));
      tile0_keys = q_first + 16 - (32 * b + 8 * (ln >> 4));
    }
    u32x4 vop[16 / VG > 1 ? 2 : 1][VG];
    auto load_v = [&](int g, u32x4 (&dst)[VG]) {
#pragma unroll
      for (int i = 0; i < VG; ++i) dst[i] = slot[v_vec + 16 * (VG * g + i)];
    };
    load_v(0, vop[0]);
    __builtin_amdgcn_sched_barrier(0);
    u32x4 ph[NC], pl;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      float s[8];
#pragma unroll
      for (int m = 0; m < 2; ++m)
#pragma unroll
        for (int i = 0; i < 4; ++i) s[4 * m + i] = sc[c][m][i];
      if (32 * b + 31 > q_first) {
        // blocks reaching past the block's first query need the causal mask
        int ln = lane;
        asm volatile("" : "+v"(ln));  // computed here: held over the loop, these values cost registers
        const int qlim = min(q_first + 16 * c + (ln & 15), ctx_total - 1);  // last key this column sees
        const int key0 = 32 * b + 8 * (ln >> 4);
#pragma unroll
        for (int m = 0; m < 2; ++m)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (key0 + 4 * m + i > qlim) s[4 * m + i] = -INFINITY;
      }
      // The probabilities against the running max go out at once; only a
      // block with a score more than 2^8 above it (every column's first block
      // among them) needs the column max (permlane swaps), the rescale and the
      // probabilities again.  m_run is the same in the four lanes of a column,
      // so a lane's own max decides as the column max would.
      const float mloc = max3_f(max3_f(s[0], s[1], s[2]), max3_f(s[3], s[4], s[5]), max3_f(s[6], s[7], s[7]));
      float pr[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        pr[j] = __builtin_amdgcn_exp2f(s[j] - m_run[c]);
        asm volatile("" : "+v"(pr[j]));  // computed here, beside the vote, not sunk past the branch
      }
      if (__any(mloc > m_run[c] + 8.0f)) {
        const float mx = swap_max(swap_max(mloc, true), false);
        // m_run is finite, so masked scores give exp2(-inf) = 0
        const bool grow = mx > m_run[c] + 8.0f;
        const float m_new = grow ? mx : m_run[c];
        const float alpha = __builtin_amdgcn_exp2f(m_run[c] - m_new);  // 0 on the first block, where o and l are 0
#pragma unroll
        for (int dt = 0; dt < NO; ++dt) o[c][dt] *= alpha;
        l_run[c] *= alpha;
        m_run[c] = m_new;
#pragma unroll
        for (int j = 0; j < 8; ++j) pr[j] = __builtin_amdgcn_exp2f(s[j] - m_run[c]);
      }
      pack(pr, ph[c], pl, std::false_type{});
      if constexpr (NC > 1) {
        asm volatile("" : "+v"(ph[c]));  // packed here, before the next column tile's probabilities
#pragma unroll
        for (int j = 0; j < 4; ++j) l_run[c] = sum_pair_f16(ph[c][j], l_run[c]);
      }
    }
#pragma unroll
    for (int g = 0; g < 16 / VG; ++g) {
      if (g + 1 < 16 / VG) load_v(g + 1, vop[(g + 1) & 1]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < VG; ++i)
#pragma unroll
        for (int c = 0; c < NC; ++c) {
          u32x4 w = vop[g & 1][i];
          if constexpr (decltype(tail)::value) {
            // V of the keys past the first column tile's last query, which the
            // second tile still sees, counts as zero for the first: its
            // probabilities there are 0, but 0 * inf is NaN
            if (c == 0)
#pragma unroll
              for (int j = 0; j < 4; ++j) w[j] = tile0_keys >= 2 * j + 2 ? w[j] : tile0_keys == 2 * j + 1 ? w[j] & 0xffffu : 0u;
          }
          o[c][VG * g + i] = KV::mfma_k32(w, ph[c], o[c][VG * g + i]);
        }
      if constexpr (NC == 1) {  // one group: all hi products, then all lo products (17 MFMAs between dependent ones)
        const u32x4 ones{kOne2, kOne2, kOne2, kOne2};
        o[0][16] = KV::mfma_k32(ones, ph[0], o[0][16]);
        if (kSplit) {
#pragma unroll
          for (int dt = 0; dt < 16; ++dt) o[0][dt] = KV::mfma_k32(vop[0][dt], pl, o[0][dt]);
          o[0][16] = KV::mfma_k32(ones, pl, o[0][16]);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  // Key blocks arrive in pairs, two blocks ahead.  At an even block every
  // copy this thread has in flight (the pair b, b + 1, issued two iterations
  // earlier) is waited for, then the barrier makes every thread's copies
  // landed and every wave done with blocks b - 2 and b - 1, whose slots take
  // the next pair.  An odd block's pair has already landed, so odd blocks
  // pass no barrier and the waves drift apart by up to a block (the two
  // waves of a SIMD then rarely reach the softmax at once).  The wait is for
  // all copies, not a count of them: it relies on no ordering among the
  // direct-to-LDS copies, only on each being written to LDS when the counter
  // no longer holds it; pairing gives each copy two iterations to land.
  f32x4 sc[NC][2];
  issue(blk0);
  if (blk0 + 1 < nblk) issue(blk0 + 1);
  auto step = [&](int b, auto tail) __attribute__((always_inline)) {
    if ((b & 1) == 0) {
      asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
      if (b + 2 < nblk) issue(b + 2);
      if (b + 3 < nblk) issue(b + 3);
    }
    u32x4* slot = slot_of(b);
    if (32 * b + 31 > kmax) {
      // last block: zero V of keys past the last one used, so that
      // 0-probability keys cannot bring NaN/Inf from unwritten slots
#pragma unroll
      for (int j2 = 0; j2 < 2; ++j2) {
        int vi = j2 * kPrefillThreads + tid;  // vector of the block's two V^T tiles
        asm volatile("" : "+v"(vi));                 // computed here, not held over the loop
        const int m = vi / kTileVec;                 // page of the block
        const int half = (vi % kTileVec) >> 8;       // token half: tokens 8 half .. + 7 of one dim
        const int k0 = 32 * b + 16 * m + 8 * half;
        u32x4 w = slot[kSlotV + vi];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          uint32_t x = w[j];
          if (k0 + 2 * j > kmax) x &= 0xffff0000u;
          if (k0 + 2 * j + 1 > kmax) x &= 0x0000ffffu;
          w[j] = x;
        }
        slot[kSlotV + vi] = w;
      }
      lds_barrier();
    }

    // The scores' MFMAs go ahead of the other wave's softmax on this SIMD: the
    // sooner a wave reaches its own softmax, the more of it runs beside MFMAs
    // (hi + lo operands: 197 -> 185 us for 500 tokens after 12000).
    __builtin_amdgcn_s_setprio(1);
    qk(b, sc);
    __builtin_amdgcn_s_setprio(0);
    softmax_pv(b, sc, tail);
  };
  // A second column tile sees 16 more keys than the first.  The blocks that
  // hold them (one or two, the last) run apart: masked in one loop, the
  // operands spilled (212 registers); apart, 16384 tokens 1711 -> 1720 us.
  const int tail0 = NC > 1 ? min(nblk, (q_first + 16) / 32) : nblk;
  for (int b = blk0; b < tail0; ++b) step(b, std::false_type{});
  if constexpr (NC > 1)
    for (int b = max(blk0, tail0); b < nblk; ++b) step(b, std::true_type{});

  if (NC > 1) {
#pragma unroll
    for (int c = 0; c < NC; ++c) l_run[c] = swap_sum(swap_sum(l_run[c], true), false);
  } else {
    l_run[0] = o[0][NO - 1][0];
  }
  if (pieces > 1) {  // a split query block: the combine launch merges the pieces
    if (!head_ok) return;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int64_t row = ((int64_t)blockIdx.x * a.group + wave) * QT + 16 * c + n;
      float* pp = a.part + row * kAttnHeadDim + 4 * g4;
#pragma unroll
      for (int dt = 0; dt < 16; ++dt) *reinterpret_cast<f32x4*>(pp + 16 * dt) = o[c][dt];
      if (g4 == 0) a.part_ml[row] = float2{m_run[c], l_run[c]};
    }
    return;
  }
  // ---- normalise, stage (the ring is dead once every wave has left the loop), gate, store
  lds_barrier();
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const float inv = 1.0f / l_run[c];  // every valid query sees at least itself
    float* st = stage + (wave * 16 + n) * kStagePitch;
#pragma unroll
    for (int dt = 0; dt < 16; ++dt) *reinterpret_cast<f32x4*>(st + 16 * dt + 4 * g4) = o[c][dt] * inv;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    if (!head_ok) return;
    // Gate rows in batches of 8 loads (rows past the prompt repeat its last
    // one): row by row, each row's load latency was exposed, 16 in a row.
    const int d = 4 * lane;
    const int t0 = QT * qb + 16 * c;
#pragma unroll
    for (int r0 = 0; r0 < 16; r0 += 8) {
      float g[8][4];
#pragma unroll
      for (int r = 0; r < 8; ++r)
        load_act4<AT>(a.gate, (int64_t)min(t0 + r0 + r, a.length - 1) * a.gate_stride + (int64_t)head * kAttnHeadDim + d, g[r]);
#pragma unroll
      for (int r = 0; r < 8; ++r) {
        const int t = t0 + r0 + r;
        if (t >= a.length) break;
        // one 16-byte read of the staged row (element reads would hit 4-way bank conflicts)
        const f32x4 row = *reinterpret_cast<const f32x4*>(stage + (wave * 16 + r0 + r) * kStagePitch + d);
        float y[4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
          y[i] = AT == RIA_DT_BF16 ? gate_mul_to_bf16(row[i], g[r][i]) : mul_rn(row[i], sigmoid_f(g[r][i]));
        store_act4<AT>(a.out, ((int64_t)t * a.num_q_heads + head) * kAttnHeadDim + d, y);
      }
    }
    __builtin_amdgcn_wave_barrier();  // the next tile's rows take the same region after these reads
  }
}

// Merges the pieces of every split query block: one wave per (token, query
// head), lane l dims 4 l .. + 3.  out = sum_s w_s O_s / sum_s w_s l_s * sigmoid(gate),
// w_s = 2^(m_s - max m).  Bound by the partials' bytes (16 tokens x 8 heads x
// 1 KB per piece, written and read once).
template <int AT>
__global__ __launch_bounds__(256) void attn_prefill_combine_kernel(PrefillAttnArgs a, int qt) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t r = (int64_t)blockIdx.x * 4 + wave;
  const int t = static_cast<int>(r / a.num_q_heads), head = static_cast<int>(r % a.num_q_heads);
  if (t >= a.length) return;
  const int nqb = (a.length + qt - 1) / qt, qb = t / qt;
  const int pieces = query_block_pieces(qb, a.chunk, a.start, qt);
  if (pieces == 1) return;  // its workgroup stored the result
  const int d = 4 * lane;
  float g[4], y[4];
  load_act4<AT>(a.gate, (int64_t)t * a.gate_stride + (int64_t)head * kAttnHeadDim + d, g);
  const int kvh = head / a.group;
  // row of piece s in the partials: its index in the launch, this head and token
  auto row_of = [&](int s, int64_t before) {
    return ((before + (int64_t)(nqb - 1 - qb) * a.num_kv_heads + kvh) * a.group + head % a.group) * qt + t % qt;
  };
  int64_t before = 0;
  float m = -INFINITY, l = 0.f;
  f32x4 o = {0.f, 0.f, 0.f, 0.f};
  for (int s0 = 0; s0 < pieces; s0 += 4) {  // four pieces' loads in flight
    float2 ml[4];
    f32x4 po[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int s = min(s0 + j, pieces - 1);
      const int64_t row = row_of(s, before);
      ml[j] = a.part_ml[row];
      po[j] = *reinterpret_cast<const f32x4*>(a.part + row * kAttnHeadDim + d);
      if (s0 + j + 1 < pieces) before += (int64_t)(nqb - first_query_block(s, a.chunk, a.start, nqb, qt)) * a.num_kv_heads;
    }
    float mx = m;
#pragma unroll
    for (int j = 0; j < 4; ++j) mx = fmaxf(mx, ml[j].x);
    const float keep = __builtin_amdgcn_exp2f(m - mx);
    o *= keep;
    l *= keep;
    m = mx;
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (s0 + j < pieces) {
        const float w = __builtin_amdgcn_exp2f(ml[j].x - mx);
        o += po[j] * w;
        l = fmaf(ml[j].y, w, l);
      }
  }
  const float inv = 1.0f / l;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float x = o[i] * inv;
    y[i] = AT == RIA_DT_BF16 ? gate_mul_to_bf16(x, g[i]) : mul_rn(x, sigmoid_f(g[i]));
  }
  store_act4<AT>(a.out, ((int64_t)t * a.num_q_heads + head) * kAttnHeadDim + d, y);
}

template <int AT>
static void launch_prefill(const PrefillAttnArgs& a, const int32_t* pt, int kv_dtype, int qt, dim3 grid, hipStream_t st) {
  if (kv_dtype == RIA_DT_BF16)
    hipLaunchKernelGGL((attn_prefill_kernel<AT, RIA_DT_BF16, 1>), grid, dim3(kPrefillThreads), 0, st, a, pt);
  else if (qt == 16)
    hipLaunchKernelGGL((attn_prefill_kernel<AT, RIA_DT_F16, 1>), grid, dim3(kPrefillThreads), 0, st, a, pt);
  else
    hipLaunchKernelGGL((attn_prefill_kernel<AT, RIA_DT_F16, 2>), grid, dim3(kPrefillThreads), 0, st, a, pt);
  if (a.chunk) {
    const int64_t rows = (int64_t)a.length * a.num_q_heads;
    hipLaunchKernelGGL((attn_prefill_combine_kernel<AT>), dim3(static_cast<unsigned>((rows + 3) / 4)), dim3(256), 0, st, a, qt);
  }
}

// How a prompt's query blocks are formed (16 or 32 tokens) and split
// (PrefillAttnArgs::chunk).  One workgroup per CU runs at a time, so a launch
// takes about max(longest piece, work / CUs).  Blocks of 32 tokens do twice
// the MFMAs per LDS operand read and win once every CU is busy (8000 tokens
// 604 -> 471 us), but halve the workgroups and double the longest chain (4096
// tokens: 179 us in blocks of 16, 206 in blocks of 32).  A prompt whose query
// blocks number fewer than the CUs, or whose last blocks hold most keys, is
// cut into pieces where the prologue of each piece, the partials' traffic and
// the combine launch cost less than it evens out (500 tokens after 12000: 585
// -> 190 us; 1000 tokens 49 -> 43; 300 tokens 26.2 whole, 27.2 cut).
// Costs in microseconds on MI355X, from a sweep of both choices over 17 ..
// 8000 tokens after 0 .. 12000: a 32-key block (while other CUs idle, while
// all are busy) of 16 tokens with fp16 keys 1.05, 1.15, of 32 tokens 1.36,
// 1.65, of 16 tokens with bf16 hi + lo operands 1.8; prologue and epilogue 14
// per 16 tokens; combine 6 + one per 40 pieces of 16 tokens.
// A split has to promise 3%: of 644 prompts of other lengths, positions and head
// counts those promised less (2500 tokens after 13, 0.8%: 145 us whole, 166 cut;
// 300 after 700 with 8 KV heads, 1%: 66 and 71) were the only ones it slowed down.
struct PrefillPlan {
  int qt;          // tokens of a query block
  int chunk;       // 0: unsplit
  int64_t pieces;  // workgroups of the launch
};
static PrefillPlan plan_prefill(int length, int start, int num_kv_heads, bool fp16_keys, int max_pieces) {
  const int cus = device_cus();
  const int most = ((start + length - 1) / kPageTokens + 2) / 2;  // key blocks of the last query block
  PrefillPlan best[2]{};  // whole query blocks; split
  double best_cost[2] = {-1, -1};
  for (int qt = 16; qt <= (fp16_keys ? 32 : 16); qt += 16) {
    const int nqb = (length + qt - 1) / qt;
    const double block = !fp16_keys ? 1.8 : qt == 16 ? 1.05 : 1.36;
    const double block_busy = !fp16_keys ? 1.8 : qt == 16 ? 1.15 : 1.65;
    const double fixed = 14.0 * qt / 16;
    for (int k = 1; k <= max_pieces; ++k) {
      const int chunk = k == 1 ? 0 : ((most + k - 1) / k + 1) / 2 * 2;
      if (k > 1 && chunk < kMinPieceBlocks) break;
      int64_t pieces = 0;
      for (int s = 0; s < k; ++s) pieces += (int64_t)(nqb - first_query_block(s, chunk, start, nqb, qt)) * num_kv_heads;
      if (k > 1 && pieces * qt > 32 * cus) continue;  // partials of at most 64 MB for 8 heads a group
      // key blocks in all: query block qb has about (start + qt qb) / 32 + 1 of them
      const double work =
          (double)num_kv_heads * nqb * ((start + 0.5 * qt * nqb) / 32 + 1) * block_busy + pieces * fixed;
      const double longest = (k == 1 ? most : chunk + 1) * block + fixed;
      double cost = std::max(longest, work / cus);
      if (k > 1) {  // whole query blocks run longest first and end together; pieces of several sizes do not
        if (pieces > cus) cost = std::max(cost, work / cus + longest / 4);
        cost += 6.0 + pieces * qt / 640.0;
      }
      const int split = k > 1;
      if (best_cost[split] < 0 || cost < best_cost[split]) {
        best_cost[split] = cost;
        best[split] = PrefillPlan{qt, chunk, pieces};
      }
    }
  }
  return best_cost[1] >= 0 && best_cost[1] < 0.97 * best_cost[0] ? best[1] : best[0];
}

static int64_t partial_bytes(const PrefillPlan& p, int group) {
  return p.chunk ? p.pieces * group * p.qt * (int64_t)(kAttnHeadDim * sizeof(float) + sizeof(float2)) : 0;
}

}  // namespace ria

using namespace ria;



namespace ria {
int kv_append_seq_impl(int length, int num_kv_heads, const void* k, int k_dtype, int64_t k_row_stride,
                       const void* v, int v_dtype, int64_t v_row_stride, void* k_cache, void* v_cache, int kv_dtype,
                       int num_pages, const int32_t* page_table_row, int64_t page_capacity, int32_t start_pos,
                       const float* inv_freq, int rope_dim, const float* k_norm_weight, uint16_t* stage_k,
                       uint16_t* stage_v, void* stream);

static int64_t stage_half_bytes(int length, int num_kv_heads) {
  return (int64_t)((length + kPageTokens - 1) / kPageTokens) * num_kv_heads * kTile * 2;
}

static int prefill_impl(int length, int num_q_heads, int num_kv_heads, const void* q, int64_t q_row_stride,
                        const void* k, int64_t k_row_stride, const void* v, int64_t v_row_stride, const void* gate,
                        int64_t gate_row_stride, int act_dtype, void* k_cache, void* v_cache, int kv_dtype,
                        int num_pages, const int32_t* page_table_row, int64_t page_capacity, int32_t start_pos,
                        const float* inv_freq, int rope_dim, const float* q_norm_weight, const float* k_norm_weight,
                        float scale, void* stage, int64_t stage_bytes, void* workspace, int64_t workspace_bytes,
                        void* out, int phase, void* stream) {
  if (phase < RIA_PREFILL_APPEND || phase > RIA_PREFILL_BOTH)
    return set_error(RIA_ERR_INVALID, "ria_attn_prefill: phase must be 1 (append), 2 (attention) or 3 (both)");
  if (length < 0 || start_pos < 0) return set_error(RIA_ERR_INVALID, "ria_attn_prefill: negative length or start");
  if (num_kv_heads <= 0 || num_q_heads <= 0 || num_q_heads % num_kv_heads)
    return set_error(RIA_ERR_INVALID, "ria_attn_prefill: num_q_heads must be a multiple of num_kv_heads");
  const int group = num_q_heads / num_kv_heads;
  if (group > 8) return set_error(RIA_ERR_INVALID, "ria_attn_prefill: at most 8 query heads per KV head");
  if (act_dtype != RIA_DT_BF16 && act_dtype != RIA_DT_F16 && act_dtype != RIA_DT_F32)
    return set_error(RIA_ERR_INVALID, "ria_attn_prefill: unknown dtype code");
  if (kv_dtype != RIA_DT_BF16 && kv_dtype != RIA_DT_F16)
    return set_error(RIA_ERR_INVALID, "ria_attn_prefill: the KV cache must be bf16 or fp16");
  if (!q || !k || !v || !gate || !k_cache || !v_cache || !page_table_row || !out)
    return set_error(RIA_ERR_INVALID, "ria_attn_prefill: null pointer");
  if (rope_dim != 0 && rope_dim != 64) return set_error(RIA_ERR_INVALID, "ria_attn_prefill: rope_dim must be 0 or 64");
  if (rope_dim && !inv_freq) return set_error(RIA_ERR_INVALID, "ria_attn_prefill: inv_freq is null");
  if (reinterpret_cast<uintptr_t>(q_norm_weight) % 16)
    return set_error(RIA_ERR_INVALID, "ria_attn_prefill: q_norm_weight must be 16-byte aligned");
  if ((int64_t)start_pos + length > page_capacity * kPageTokens)
    return set_error(RIA_ERR_INVALID, "ria_attn_prefill: %d + %d tokens exceed the row's %lld pages", start_pos,
                     length, (long long)page_capacity);
  if (q_row_stride < (int64_t)num_q_heads * kAttnHeadDim || gate_row_stride < (int64_t)num_q_heads * kAttnHeadDim)
    return set_error(RIA_ERR_INVALID, "ria_attn_prefill: row stride smaller than Hq*256");
  // q, gate and out move in 16-byte vectors
  if ((reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(gate) | reinterpret_cast<uintptr_t>(out)) % 16 ||
      q_row_stride % 8 || gate_row_stride % 8)
    return set_error(RIA_ERR_INVALID, "ria_attn_prefill: q, gate and out must be 16-byte aligned, row strides multiples of 8");
  if (length == 0) return RIA_OK;
  const int64_t blocks = (int64_t)((length + 15) / 16) * num_kv_heads;
  if (blocks > 0x7fffffff) return set_error(RIA_ERR_INVALID, "ria_attn_prefill: grid too large");
  // a prompt from slot 0 with a stage: its keys also go to fp16 tiles, which the attention reads
  const bool staged = stage && start_pos == 0;
  uint16_t* stage_k = nullptr;
  uint16_t* stage_v = nullptr;
  if (staged) {
    const int64_t half = stage_half_bytes(length, num_kv_heads);
    if (stage_bytes < 2 * half)
      return set_error(RIA_ERR_WORKSPACE, "ria_attn_prefill: stage %lld bytes < required %lld",
                       (long long)stage_bytes, (long long)(2 * half));
    if (reinterpret_cast<uintptr_t>(stage) % 16) return set_error(RIA_ERR_INVALID, "ria_attn_prefill: stage must be 16-byte aligned");
    stage_k = static_cast<uint16_t*>(stage);
    stage_v = stage_k + half / 2;
  }
  if (phase & RIA_PREFILL_APPEND) {
    int rc = kv_append_seq_impl(length, num_kv_heads, k, act_dtype, k_row_stride, v, act_dtype, v_row_stride,
                                k_cache, v_cache, kv_dtype, num_pages, page_table_row, page_capacity, start_pos,
                                inv_freq, rope_dim, k_norm_weight, stage_k, stage_v, stream);
    if (rc != RIA_OK) return rc;
  }
  if (!(phase & RIA_PREFILL_ATTEND)) return RIA_OK;
  PrefillAttnArgs a{};
  a.q = q;
  a.q_stride = q_row_stride;
  a.gate = gate;
  a.gate_stride = gate_row_stride;
  a.k_cache = static_cast<const uint16_t*>(k_cache);
  a.v_cache = static_cast<const uint16_t*>(v_cache);
  a.num_pages = num_pages;
  a.pt_len = page_capacity;
  a.start = start_pos;
  a.length = length;
  a.inv_freq = inv_freq;
  a.rope_dim = rope_dim;
  a.q_norm_w = q_norm_weight;
  a.scale = scale;
  a.num_q_heads = num_q_heads;
  a.num_kv_heads = num_kv_heads;
  a.group = group;
  a.out = out;
  int key_dtype = kv_dtype;
  if (staged) {  // the prompt's own fp16 tiles, logical page p at tile p
    a.k_cache = stage_k;
    a.v_cache = stage_v;
    a.num_pages = (length + kPageTokens - 1) / kPageTokens;
    a.staged = 1;
    key_dtype = RIA_DT_F16;
  }
  PrefillPlan plan = plan_prefill(length, start_pos, num_kv_heads, key_dtype == RIA_DT_F16, workspace ? kMaxPieces : 1);
  if (workspace) {
    if (reinterpret_cast<uintptr_t>(workspace) % 16)
      return set_error(RIA_ERR_INVALID, "ria_attn_prefill: workspace must be 16-byte aligned");
    if (partial_bytes(plan, group) > workspace_bytes)  // too small: no split
      plan = plan_prefill(length, start_pos, num_kv_heads, key_dtype == RIA_DT_F16, 1);
    a.chunk = plan.chunk;
    a.part = static_cast<float*>(workspace);
    a.part_ml = reinterpret_cast<float2*>(a.part + plan.pieces * group * plan.qt * kAttnHeadDim);
  }
  const dim3 grid(static_cast<unsigned>(plan.pieces));
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (act_dtype == RIA_DT_BF16)
    launch_prefill<RIA_DT_BF16>(a, page_table_row, key_dtype, plan.qt, grid, st);
  else if (act_dtype == RIA_DT_F16)
    launch_prefill<RIA_DT_F16>(a, page_table_row, key_dtype, plan.qt, grid, st);
  else
    launch_prefill<RIA_DT_F32>(a, page_table_row, key_dtype, plan.qt, grid, st);
  return check_launch("ria_attn_prefill");
}
}  // namespace ria

extern "C" int ria_attn_prefill_phase(int length, int num_q_heads, int num_kv_heads, const void* q,
                                      int64_t q_row_stride, const void* k, int64_t k_row_stride, const void* v,
                                      int64_t v_row_stride, const void* gate, int64_t gate_row_stride, int act_dtype,
                                      void* k_cache, void* v_cache, int kv_dtype, int num_pages,
                                      const int32_t* page_table_row, int64_t page_capacity, int32_t start_pos,
                                      const float* inv_freq, int rope_dim, const float* q_norm_weight,
                                      const float* k_norm_weight, float scale, void* out, int phase,
                                      void* stream) {
  return prefill_impl(length, num_q_heads, num_kv_heads, q, q_row_stride, k, k_row_stride, v, v_row_stride, gate,
                      gate_row_stride, act_dtype, k_cache, v_cache, kv_dtype, num_pages, page_table_row,
                      page_capacity, start_pos, inv_freq, rope_dim, q_norm_weight, k_norm_weight, scale, nullptr, 0,
                      nullptr, 0, out, phase, stream);
}

extern "C" int64_t ria_attn_prefill_stage_bytes(int length, int num_kv_heads) {
  if (length <= 0 || num_kv_heads <= 0) return 0;
  return 2 * stage_half_bytes(length, num_kv_heads);
}

extern "C" int ria_attn_prefill_staged(int length, int num_q_heads, int num_kv_heads, const void* q,
                                       int64_t q_row_stride, const void* k, int64_t k_row_stride, const void* v,
                                       int64_t v_row_stride, const void* gate, int64_t gate_row_stride,
                                       int act_dtype, void* k_cache, void* v_cache, int kv_dtype, int num_pages,
                                       const int32_t* page_table_row, int64_t page_capacity, int32_t start_pos,
                                       const float* inv_freq, int rope_dim, const float* q_norm_weight,
                                       const float* k_norm_weight, float scale, void* stage, int64_t stage_bytes,
                                       void* out, int phase, void* stream) {
  if (!stage) return set_error(RIA_ERR_INVALID, "ria_attn_prefill_staged: null stage");
  return prefill_impl(length, num_q_heads, num_kv_heads, q, q_row_stride, k, k_row_stride, v, v_row_stride, gate,
                      gate_row_stride, act_dtype, k_cache, v_cache, kv_dtype, num_pages, page_table_row,
                      page_capacity, start_pos, inv_freq, rope_dim, q_norm_weight, k_norm_weight, scale, stage,
                      stage_bytes, nullptr, 0, out, phase, stream);
}

extern "C" int64_t ria_attn_prefill_workspace_bytes(int length, int num_q_heads, int num_kv_heads, int32_t start_pos,
                                                    int fp16_keys) {
  if (length <= 0 || start_pos < 0 || num_kv_heads <= 0 || num_q_heads <= 0 || num_q_heads % num_kv_heads) return 0;
  return partial_bytes(plan_prefill(length, start_pos, num_kv_heads, fp16_keys != 0, kMaxPieces), num_q_heads / num_kv_heads);
}

extern "C" int ria_attn_prefill_split(int length, int num_q_heads, int num_kv_heads, const void* q,
                                      int64_t q_row_stride, const void* k, int64_t k_row_stride, const void* v,
                                      int64_t v_row_stride, const void* gate, int64_t gate_row_stride, int act_dtype,
                                      void* k_cache, void* v_cache, int kv_dtype, int num_pages,
                                      const int32_t* page_table_row, int64_t page_capacity, int32_t start_pos,
                                      const float* inv_freq, int rope_dim, const float* q_norm_weight,
                                      const float* k_norm_weight, float scale, void* stage, int64_t stage_bytes,
                                      void* workspace, int64_t workspace_bytes, void* out, int phase, void* stream) {
  return prefill_impl(length, num_q_heads, num_kv_heads, q, q_row_stride, k, k_row_stride, v, v_row_stride, gate,
                      gate_row_stride, act_dtype, k_cache, v_cache, kv_dtype, num_pages, page_table_row,
                      page_capacity, start_pos, inv_freq, rope_dim, q_norm_weight, k_norm_weight, scale, stage,
                      stage_bytes, workspace, workspace_bytes, out, phase, stream);
}

extern "C" int ria_attn_prefill(int length, int num_q_heads, int num_kv_heads, const void* q, int64_t q_row_stride,
                                const void* k, int64_t k_row_stride, const void* v, int64_t v_row_stride,
                                const void* gate, int64_t gate_row_stride, int act_dtype, void* k_cache,
                                void* v_cache, int kv_dtype, int num_pages, const int32_t* page_table_row,
                                int64_t page_capacity, int32_t start_pos, const float* inv_freq, int rope_dim,
                                const float* q_norm_weight, const float* k_norm_weight, float scale, void* out,
                                void* stream) {
  return ria_attn_prefill_phase(length, num_q_heads, num_kv_heads, q, q_row_stride, k, k_row_stride, v, v_row_stride,
                                gate, gate_row_stride, act_dtype, k_cache, v_cache, kv_dtype, num_pages,
                                page_table_row, page_capacity, start_pos, inv_freq, rope_dim, q_norm_weight,
                                k_norm_weight, scale, out, RIA_PREFILL_BOTH, stream);
}
