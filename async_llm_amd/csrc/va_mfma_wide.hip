// Wide matrix-core view attention: query tiles of 128 (head_dim 256) or 256 MFMA rows, for
// view-conditioned prefill (rows / G new tokens x G heads per workgroup).
//
// One workgroup of four waves per (slot, kv head), one wave per SIMD; a slot is one work item, or
// several pieces of tiles whose walks add up to the same number of tokens in every slot, run one
// after the other.  Wave w owns one
// (head_dim 256) or two blocks of 32 MFMA rows (row R = tile row R / G, head R % G).  All waves walk
// the same 32-token K/V tiles, which travel pool -> LDS directly (global_load_lds_dwordx4) into a
// ring of four buffers: two tiles are in flight while the scores of a third and the products of a
// fourth are computed, one barrier per tile.
//
//   S^T[32 tokens, 32 rows] = K . Q^T    v_mfma_f32_32x32x16, K from LDS as the A operand; each K
//                                        fragment is read once and used for all row blocks, whose
//                                        rotated queries are pinned in registers as B operands
//   softmax per row against a reference maximum that is raised only when a tile exceeds it by far
//   (row = lane % 32; the other half-wave holds the other 16 tokens)
//   O^T[D, 32 rows] += V^T . P^T         2 token steps x D/32 dim tiles; P is already laid out as
//                                        the B operand; V^T fragments come from transposing LDS
//                                        reads (ds_read_b64_tr_b16), each serving all row blocks
//
// The loop is a hand-ordered software pipeline: the scores of tile i + 1 run on the matrix pipe
// under the exponentials of tile i (each taken of scale * score - reference, formed in fp32 right
// in front of it), the products of tile i under the maxima of tile i + 1 and, at head dims under 256, some of its
// exponentials.  Interior tiles of a link take a branch-free ring step, in a loop of their own.
// V tiles keep whole rows in LDS, unpadded and swizzled (piece c of row r at position c ^ swz(r)); K
// tiles land in fragment order (8-token x 128-byte blocks, see the load pattern in the kernel), so
// that the K reads of a tile share one address register.  The query never goes through LDS: every
// lane loads its own rows in operand order and rotates them in registers, once per link.  Only the
// cosines and sines of an mRoPE tile pass through the ring buffers that are not yet in use (past the
// end of the ring at head dims under 256), and the pieces of rotary widths that no operand fits.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "va_internal.h"
#include "va_launch.h"
#include "va_mfma_common.h"
#include "va_stream_tile.h"

namespace va {

constexpr int kWideThreads = 256;
constexpr float kWideRaise = 14.f;  // a tile maximum this far above the reference (log2 units) raises it
constexpr int kWideWaves = 4;
constexpr int kWideTokens = 32;  // tokens per K/V tile
#ifndef VA_WIDE_BUFFERS
#define VA_WIDE_BUFFERS 4
#endif
constexpr int kWideBuffers = VA_WIDE_BUFFERS;  // ring depth: kWideBuffers - 2 tiles in flight
constexpr int kWideAhead = kWideBuffers - 2;    // a ring step requests the tile this far ahead

template <int kD>
struct WideShape {
  static constexpr int kChunks = kD / 8;     // 16-byte pieces of a head row
  static constexpr int kSteps = kD / 16;     // contraction steps of K.Q^T (32x32x16)
  static constexpr int kDimTiles = kD / 32;  // 32-dim tiles of the output
  static constexpr int kRowBytes = kChunks * 16;
  static constexpr int kRowsPerLoad = kWave / kChunks;              // tile rows one wave-level load covers
  static constexpr int kLoadsPerKind = kWideTokens / kRowsPerLoad;  // loads per K (or V) tile
  static constexpr int kLoadsPerWave = 2 * kLoadsPerKind / kWideWaves;
  static constexpr int kTileBytes = kWideTokens * kRowBytes;  // a K (or V) tile
  static constexpr int kBufferBytes = 2 * kTileBytes;
  // 32-row blocks per wave.  Two blocks halve the LDS bytes read per flop, but the state of a row
  // (D fp32 accumulators + D 16-bit query elements) then fills the register file at D = 256:
  // 64 rows need 256 + 128 of the 512 registers before any operand is staged, and the compiler
  // spills.  D = 256 therefore runs one block per wave.
  static constexpr int kBlocks = kD == 256 ? 1 : 2;
  static constexpr int kWaveRows = 32 * kBlocks;
  // Of the sixteen elements a lane has of a row block's tile, those whose exponentials are taken under the P.V products
  // of the tile before (steady part of a link).  Measured, attention and merge of a layer, 0 / 4 / 6 / 8 elements at 128
  // dims: 8 x 1500..2048 rows over 8000 tokens (32 q / 8 kv heads, bf16) 2500 / 2052 / 2013 / 2025 us, 4 of 300..1500
  // over up to six blocks (float16) 600 / 582 / 573 / 573, plain prefill of 6 356 / 332 / 332 / 334; 0 / 4 / 8 / 10
  // at 64 dims (64 q / 16 kv heads): 4 x 300..1000 over 4000 tokens 324 / 299 / 299 / 294, plain prefill 518 / 441 / 438
  // / 434.  At 256 dims the P.V products are twice as many per exponential, and full of V reads: 0 / 2 / 4 elements
  // 9950 / 10160 / 10260 us for 8 x 2048 rows over 41 k tokens.
  static constexpr int kEarly = kD == 256 ? 0 : kD == 128 ? 6 : 10;
  static constexpr int kTileRows = kWideWaves * kWaveRows;  // MFMA rows per workgroup
  // The cosines and sines of an mRoPE tile (at most one row per MFMA row, kD / 2 entries of four bytes)
  // lie behind the tiles requested during the set-up: at D = 256 in the rest of the ring (128 KB in all),
  // at smaller head dims past its end.
  static constexpr int kTurnBytes = kTileRows * (kD / 2) * 4;
  static constexpr int kRingBytes = kWideBuffers * kBufferBytes, kSetupBytes = kWideAhead * kBufferBytes + kTurnBytes;
  // Scattered rows: the index entries of eight tiles, for every wave its own (va_mfma_wide: gather)
  static constexpr int kIndexOffset = kRingBytes > kSetupBytes ? kRingBytes : kSetupBytes;
  static constexpr int lds_bytes(bool gather) { return kIndexOffset + (gather ? kWideWaves * 2 * kWave * 4 : 0); }
};

// Word of the cos|sin entry (row iq, pair dim) in LDS: rows of `half` words, their 16-byte pieces swizzled
// by the row so that the rows a wave reads side by side spread over the banks.
__device__ __forceinline__ int turn_word(int iq, int pair, int half) {
  return iq * half + 4 * ((pair >> 2) ^ (iq & min(7, (half >> 2) - 1))) + (pair & 3);
}

// Ring buffer of a tile (tile numbers are never negative: the unsigned remainder is one instruction
// for a power-of-two ring, the signed one five).
__device__ __forceinline__ uint32_t ring_slot(int tile) { return (uint32_t)tile % (uint32_t)kWideBuffers; }

// V tiles are read with transposing loads (16 lanes fetch 4 tokens x 16 dims, 32 bytes per token):
// moving token r's pieces by 2 (r % 4) puts the four rows of such a fetch side by side in one
// 128-byte window.
__device__ __forceinline__ int wide_vswz(int r) { return (r & 3) << 1; }

// max over the two half-waves (lanes l and l ^ 32) without touching LDS
__device__ __forceinline__ float half_wave_max(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

// kGather: every token of the launch has an index entry of its own (slot lists, pages of 1, 2, 4 or 8 tokens).
template <typename E, int kD, bool kGather>
__device__ __forceinline__ void wide_slot(const AttnArgs& a, unsigned workgroup, unsigned workgroups) {
  using S = typename E::storage;
  using Sh = WideShape<kD>;
  static_assert(!kGather || kWideAhead <= 2, "the entries of a tile are read a step after their request, behind its wait");
  constexpr int kChunks = Sh::kChunks, kSteps = Sh::kSteps, kDimTiles = Sh::kDimTiles;
  constexpr int kRowBytes = Sh::kRowBytes, kL = Sh::kLoadsPerWave, kB = Sh::kBlocks, kWaveRows = Sh::kWaveRows;

  extern __shared__ va_u32x4 smem[];
  const char* lds = (const char*)smem;

  // workgroup -> (slot, kv head); the slot's items are run one after the other
  // The slots of a die run in groups of up to 32 under ONE kv head at a time (a die has 32 compute
  // units): neighbouring slots hold neighbouring query tiles of one request, which walk the same
  // K/V rows, so the die's L2 holds one head's stream at a time instead of all of them.
  ItemHead where;
  {
    const unsigned die = workgroup & 7u, turn = workgroup >> 3, per_die = workgroups / (8u * a.num_kv_heads);
    unsigned g = 32;
    while (per_die % g) g >>= 1;
    const unsigned block = turn / (g * a.num_kv_heads), within = turn % (g * a.num_kv_heads);
    where = ItemHead{(int)((block * g + within % g) * 8u + die), (int)(within / g)};
  }
  // The plan is read through the constant address space: scalar loads, all words of an item or a link in one
  // trip (as ordinary loads they go out one after the other, each waiting for the one before it)
  using PlanWords = const __attribute__((address_space(4))) int32_t*;
  // mRoPE: threads per pair dim when cosines and sines are taken, the rows of a tile rounded up to a power of two
  int turn_lanes = 1;
  while (turn_lanes < Sh::kTileRows / (a.num_q_heads / a.num_kv_heads)) turn_lanes <<= 1;
  const int turn_iq = threadIdx.x & (turn_lanes - 1);
  const PlanWords slots_of = (PlanWords)a.wide_slots + where.item;
  const int item_begin = slots_of[0], item_end = slots_of[1];
  const int hk = where.head;
  const int G = a.num_q_heads / a.num_kv_heads;
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int lane = tid % kWave;
  const int j = lane % 32;         // row within a 32-row block / token within a tile / dim group
  const int h = lane / 32;         // half-wave: contraction group
  const int row0 = kWaveRows * wave + j;  // this lane's row in block 0; block 1 is 32 further
  int row_iq[kB];
#pragma unroll
  for (int b = 0; b < kB; ++b) row_iq[b] = (row0 + 32 * b) / G;
  const S* kp = (const S*)a.k_pool + (long long)hk * kD;
  const S* vp = (const S*)a.v_pool + (long long)hk * kD;
  const int P = a.page_size;
  const bool pow2_pages = (P & (P - 1)) == 0;
  const int p_shift = __builtin_ctz(P);  // t / P and t % P as shift and mask (power-of-two pages)
  const int row_bytes = (int)a.pool_row_stride * (int)sizeof(S);
  // bytes of a page, for the offsets of plain tiles: such tiles need the figure to fit 32 bits
  const bool page_fits = ((unsigned long long)(uint32_t)row_bytes << p_shift) <= 0xffffffffull;
  const uint32_t page_bytes = (uint32_t)row_bytes << p_shift;

  // This lane's part of a wave-level load (64 lanes x 16 bytes land as one 1 KB run in LDS; which
  // piece of the pool a lane fetches is free).  Waves 0 and 1 load K halves, waves 2 and 3 V halves.
  //   V: load u covers kRowsPerLoad whole rows, piece c of row r at position c ^ vswz(r).
  //   K: fragment order.  Load u of a half is the block (8 rows R, 128-byte column g) = the operands
  //      of four contraction steps for eight tokens: lane 16 s2 + 8 (h ^ R % 2) + j3 fetches row
  //      8 R + j3, piece 8 g + 2 s2 + h.  The block of step s = 4 g + s2 thus lies 256 s bytes into
  //      the 8-row region of R, and the fragment reads of a tile are ONE per-lane address plus
  //      immediates; 16 consecutive lanes (served together) read 256 consecutive bytes, the flip of
  //      h in odd R keeps the two regions they straddle on different banks.
  const bool wave_is_v = wave >= 2;
  constexpr int kColumns = kChunks / 8;  // 128-byte columns of a row
  const int ld_row0 = lane / kChunks;
  const int ld_x0 = (lane % kChunks) ^ wide_vswz(ld_row0);
  auto ld_row = [&](int u) __attribute__((always_inline)) {  // row within the wave's 16-token half
    return wave_is_v ? u * Sh::kRowsPerLoad + ld_row0 : 8 * (u / kColumns) + lane % 8;
  };
  auto ld_piece = [&](int u) __attribute__((always_inline)) {
    return wave_is_v ? (ld_x0 ^ wide_vswz(u * Sh::kRowsPerLoad))
                     : 8 * (u % kColumns) + 2 * (lane / 16) + (((lane / 8) ^ (u / kColumns)) & 1);
  };
  // The loads of a plain tile (uniform pages, inside the visible range) go out in groups of up to four
  // behind one setting of M0, as a wave-uniform base plus a per-lane offset that never changes.  A
  // group's immediate offsets move the pool address as well: the per-lane offsets have them taken
  // off beforehand (grouped_lane_offset) and carry a bias, which the base gives back, to stay positive.
  constexpr int kLoadBias = 3072;
  uint32_t ld_off[kL];
#pragma unroll
  for (int u = 0; u < kL; ++u)
    ld_off[u] = grouped_lane_offset((uint32_t)(ld_row(u) * row_bytes + 16 * ld_piece(u) + kLoadBias), u);
  constexpr int kLoadGroup = kL >= 4 ? 4 : kL;
  auto issue_plain = [&](const char* base, uint32_t dst) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < kL; u += kLoadGroup) load_group_to_lds<kLoadGroup>(base, ld_off + u, dst + u * 1024);
  };
  // LDS offsets of what this lane reads from a tile
  const int k_lane_byte = (j / 8) * 8 * kRowBytes + 128 * ((h ^ (j / 8)) & 1) + 16 * (j % 8);
  // V^T fragments come from transposing reads.  For dim tile t (dims 32t .. 32t+31) and 16-token
  // step kk the lane needs, as contraction elements 0..3 and 4..7, tokens 16kk + 4h + 0..3 and
  // 16kk + 8 + 4h + 0..3 of dim 32t + lane % 32 (the token order P^T has in its registers): two
  // reads, in each of which this lane points at token row `v_row` (+ 16kk, + 8) and at 4 dims of
  // the tile's 16-dim half lane / 16 % 2.  The swizzle folds into two per-lane bases, one for even
  // and one for odd t; everything else is an immediate offset.
  const int v_sub = lane % 16;
  const int v_row = 4 * h + v_sub / 4;
  const int v_swz = wide_vswz(v_row);
  const int v_piece = (2 * ((lane / 16) % 2) + (v_sub % 4) / 2) ^ (v_swz & 2);
  const int v_base = v_row * kRowBytes + 16 * v_piece + 8 * (v_sub % 2);
  const int v_even = v_base + 64 * (v_swz >> 2), v_odd = v_base + 64 * (1 ^ (v_swz >> 2));
  const uint32_t lds_base = lds_address(lds);

  for (int item_index = item_begin; item_index < item_end; ++item_index) {
  const PlanWords item = (PlanWords)a.items + (long long)item_index * VA_ITEM_WORDS;
  const int n_q = item[VA_I_N_Q];
  if (n_q == 0) continue;  // padding item
  const int part_base = item[VA_I_PART_BASE];
  const bool wave_active = (kWaveRows * wave) / G < n_q;  // the wave owns real rows
  // This lane's query rows: the links of an item serve the same output rows, so the first one tells them.
  // Rows past the tile repeat its last row.
  const S* q_row[kB];
  {
    const PlanWords link0 = item + VA_I_LINK0;
#pragma unroll
    for (int b = 0; b < kB; ++b) {
      const int at = link0[VA_L_QREF] + min(row_iq[b], n_q - 1);
      const long long src_row = a.sub_worker[(link0[VA_L_FLAGS] & VA_LINK_INDIRECT) ? a.qrefs[at] : at];
      const int g = row0 + 32 * b - row_iq[b] * G;
      q_row[b] = (const S*)a.q + src_row * a.q_row_stride + (long long)(hk * G + g) * kD + 8 * h;
    }
  }

  float m_ref[kB], m_tile[kB], l_run[kB];  // reference maximum (log2 units), last tile maximum, row sum
  float raise_above[kB];                    // m_ref + kWideRaise: what a tile's maximum is tested against
  va_f32x16 o[kB][kDimTiles];
#pragma unroll
  for (int b = 0; b < kB; ++b) {
    m_ref[b] = kNegBig;
    m_tile[b] = kNegBig;
    raise_above[b] = kNegBig + kWideRaise;
    l_run[b] = 0.f;
#pragma unroll
    for (int t = 0; t < kDimTiles; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) o[b][t][r] = 0.f;
  }

  const int wave_half = wave & 1;
  const bool table = a.rope.mode == VA_ROPE_TABLE;
  const int n_links = item[VA_I_N_LINKS];
  PlanWords link = (PlanWords)a.links + (long long)item[VA_I_LINK_BEGIN] * VA_LINK_WORDS;
  for (int li = 0; li < n_links; ++li, link += VA_LINK_WORDS) {
    const int lflags = link[VA_L_FLAGS];
    const int qref = link[VA_L_QREF];
    const int kv_begin = link[VA_L_KV_BEGIN];
    const int tok_begin = link[VA_L_TOK_BEGIN];
    const int tok_end = link[VA_L_TOK_END];
    const int causal_base = link[VA_L_CAUSAL_BASE];
    const bool slots = lflags & VA_LINK_SLOTS;
    // a 16-token half tile lies inside one page only if the link starts on a 16-token boundary
    const bool uniform_pages = !kGather && !slots && pow2_pages && page_fits && P >= 16 && (tok_begin % 16 == 0);

    const int t_stop = min(tok_end, causal_base + n_q);  // tokens any row of the tile sees
    const int t_last = t_stop - 1;
    int t_row[kB];
#pragma unroll
    for (int b = 0; b < kB; ++b) t_row[b] = min(tok_end, causal_base + row_iq[b] + 1);
    // tokens any row of this wave sees, and tokens EVERY real row of it sees (no masking below that)
    const int wave_iq_last = min(n_q - 1, (kWaveRows * wave + kWaveRows - 1) / G);
    const int t_wave = wave_active ? min(tok_end, causal_base + wave_iq_last + 1) : -0x7fffffff;
    const int t_wave_min = min(tok_end, causal_base + (kWaveRows * wave) / G + 1);
    const int n_tiles = t_stop > tok_begin ? (t_stop - tok_begin + kWideTokens - 1) / kWideTokens : 0;

    // Loads of a tile.  Wave w fetches one 16-token half of the K tile (w = 0, 1) or of the V tile
    // (w = 2, 3): kL wave-level loads of kRowsPerLoad rows each.  With uniform pages the half lies
    // in one page, so the wave needs ONE scalar page lookup per tile and every load is a
    // wave-uniform base plus a per-lane offset that never changes (ld_off); in tiles that reach past
    // the visible range rows past it re-read the last visible token (their scores are masked).  Links
    // of other page tables look every row up per lane.
    // Slot lists and pages under 16 tokens (kGather): looked up by the lanes in front of each request, the
    // entries cost a trip to memory per tile and drain the ring (6 requests of 60..4096 tokens over slot
    // lists, 32 q / 8 kv heads of 128 dims: 734 us a layer).  So they travel like the tiles do: one
    // wave-level load brings a wave's entries of four tiles to LDS, two to five ring steps ahead of their
    // requests, and a ring step reads the entries of the tile the NEXT step requests.
    const char* wave_pool = (const char*)(wave_is_v ? vp : kp);
    const char* wave_plain = wave_pool - kLoadBias;  // base of plain loads: the per-lane offsets carry the bias
    const uint32_t wave_lds = __builtin_amdgcn_readfirstlane(lds_address(lds)) + (wave_is_v ? Sh::kTileBytes : 0) +
                              wave_half * 16 * kRowBytes;
    // pool row of this wave's half of tile i (uniform pages, tile inside the visible range); read
    // through the constant address space so that the lookup stays a scalar load
    // (as a byte offset: page x bytes of a page + row in the page x bytes of a row, a 32 x 32 -> 64 bit
    // product and a 32-bit one; the row number times the row size would be a 64 x 32 bit product, six
    // scalar instructions in every ring step)
    auto half_offset = [&](int page, int t) __attribute__((always_inline)) {
      return (unsigned long long)(uint32_t)page * page_bytes + (uint32_t)(t & (P - 1)) * (uint32_t)row_bytes;
    };
    // (past the visible range: that of the last visible token)
    auto half_row = [&](int i) __attribute__((always_inline)) {
      const int t = min(tok_begin + i * kWideTokens + 16 * wave_half, t_last);
      return half_offset(((PlanWords)a.kv_indices)[kv_begin + (t >> p_shift)], t);
    };
    auto tile_is_plain = [&](int i) __attribute__((always_inline)) {
      return uniform_pages && tok_begin + (i + 1) * kWideTokens - 1 <= t_last;
    };
    // gather: entries of tiles 4 group .. 4 group + 3, this wave's half; lane -> (tile, token)
    const int g_shift = slots ? 0 : p_shift, g_mask = slots ? 0 : P - 1;
    const uint32_t wave_index_lds = __builtin_amdgcn_readfirstlane(lds_address(lds)) + Sh::kIndexOffset + wave * (2 * kWave * 4);
    const int32_t* wave_index = (const int32_t*)(lds + Sh::kIndexOffset + wave * (2 * kWave * 4));
    auto gather_token = [&](int i, int row) __attribute__((always_inline)) {
      return min(tok_begin + i * kWideTokens + 16 * wave_half + row, t_last);
    };
    auto request_entries = [&](int group) __attribute__((always_inline)) {
      const int t = gather_token(4 * group + lane / 16, lane % 16);
      load_word_to_lds(a.kv_indices + kv_begin + (t >> g_shift), wave_index_lds + (group & 1) * (kWave * 4));
    };
    // The rows of a wave's requests: lane % 8 and 8 + lane % 8 for every 128-byte column of K, another row per
    // request of V (ld_row).
    constexpr int kVBases = kD == 256 ? 2 : 1;  // the swizzle of V's pieces repeats every 1 or 2 requests
    const unsigned long long gather_base[2] = {(unsigned long long)(wave_pool + 16 * ld_piece(0)),
                                               (unsigned long long)(wave_pool + 16 * ld_piece(wave_is_v ? kVBases - 1 : kColumns))};
    auto gather_row = [&](int x) __attribute__((always_inline)) { return wave_is_v ? ld_row(x) : 8 * (x & 1) + lane % 8; };
    auto read_slots = [&](int i, int (&slot)[kL], auto entry_of) __attribute__((always_inline)) {
      auto one = [&](int x) __attribute__((always_inline)) {
        const int row = gather_row(x);
        slot[x] = (entry_of(i, row) << g_shift) + (gather_token(i, row) & g_mask);
      };
      one(0);
      one(1);
      if (wave_is_v)
#pragma unroll
        for (int x = 2; x < kL; ++x) one(x);
    };
    auto entry_in_lds = [&](int i, int row) __attribute__((always_inline)) { return wave_index[(i & 7) * 16 + row]; };
    auto entry_in_memory = [&](int i, int row) __attribute__((always_inline)) {
      return a.kv_indices[kv_begin + (gather_token(i, row) >> g_shift)];
    };
    auto issue_gather = [&](int i, const int (&slot)[kL]) __attribute__((always_inline)) {
      const uint32_t dst = wave_lds + ring_slot(i) * Sh::kBufferBytes;
      auto at = [&](int x, int base) __attribute__((always_inline)) {
        return (unsigned long long)(uint32_t)slot[x] * (uint32_t)row_bytes + gather_base[base];
      };
      if (wave_is_v) {
#pragma unroll
        for (int u = 0; u < kL; u += kLoadGroup) {
          unsigned long long rows[kLoadGroup];
#pragma unroll
          for (int x = 0; x < kLoadGroup; ++x) rows[x] = at(u + x, (u + x) % kVBases);
          load_rows_to_lds<kLoadGroup>(rows, dst + u * 1024);
        }
      } else {
        load_columns_to_lds<kColumns>(at(0, 0), dst);
        load_columns_to_lds<kColumns>(at(1, 1), dst + kColumns * 1024);
      }
    };
    auto issue = [&](int i, unsigned long long row) __attribute__((always_inline)) {
      const uint32_t dst = wave_lds + ring_slot(i) * Sh::kBufferBytes;
      if (tile_is_plain(i)) {
        const char* base = wave_plain + row;
        issue_plain(base, dst);
      } else if (uniform_pages) {
        // The last tile of a link: its visible rows lie in the page of the half's first token all the same, rows
        // past them repeat the last visible one.  (Looked up row by row, each request waited for an entry and
        // with it for the whole ring: 4 ragged requests of 300..1500 tokens over up to six blocks, 32 q / 8 kv
        // heads of 128 dims, two layers 1318 -> 1299 us; 8 of 2048 over eight blocks, 256 dims: no more than two
        // runs differ by.)
        const int left = max(0, t_last - (tok_begin + i * kWideTokens + 16 * wave_half));
#pragma unroll
        for (int u = 0; u < kL; ++u)
          load_to_lds(wave_pool + row, (uint32_t)(min(ld_row(u), left) * row_bytes + 16 * ld_piece(u)), dst + u * 1024);
      } else {
        const int t0 = tok_begin + i * kWideTokens + 16 * wave_half;
#pragma unroll
        for (int u = 0; u < kL; ++u) {
          const int t = min(t0 + ld_row(u), t_last);
          const int piece = 16 * ld_piece(u);
          load_to_lds(wave_pool + kv_slot(a.kv_indices, kv_begin, t, P, slots) * row_bytes + piece, dst + u * 1024);
        }
      }
    };
    // The pool row of the tile a ring step requests is looked up a whole step earlier (a scalar load whose
    // result is not touched before the next step): its latency never shows.
    auto row_of = [&](int tile) __attribute__((always_inline)) {
      return (uniform_pages && tile < n_tiles) ? half_row(tile) : 0ull;
    };

    // ---- set-up: the first two tiles on their way, the query rows rotated for this link ----
    // Every lane loads its own rows in operand order and rotates them in registers: a rotary pair
    // (dim d, dim d + half) is the same element of operands s and s + half / 16 of one lane, so nothing is
    // exchanged between lanes (staged through LDS the tile took two barriers and 13 300 cycles a link at D = 256
    // with the table, 21 200 under mRoPE; 11 900 and 13 300 like this).  What bounds it now is the L1's rate
    // for 64 KB of query pieces at 16 bytes a row and the table entries.  Positions, query rows and the page
    // numbers of the first tiles are requested together, ahead of the barrier; the tiles and the table entries,
    // which need them, behind it.
    va_u32x4 qf[kB][kSteps];  // B operands: row of block b, dims [16s + 8h, +8)
    uint32_t* turns = (uint32_t*)(lds + kWideAhead * Sh::kBufferBytes);
    const int half = a.rope.half, half_steps = a.rope.rotary_dim % 32 == 0 ? a.rope.rotary_dim / 32 : -1;
    const bool in_turn = half_steps > 0 && (half_steps == kSteps / 2 || half_steps == kSteps / 4 || half_steps == kSteps / 8);
    auto subrow_of = [&](int iq) __attribute__((always_inline)) {
      const int at = qref + min(iq, n_q - 1);
      return (lflags & VA_LINK_INDIRECT) ? a.qrefs[at] : at;
    };
    long long pos[kB < 3 ? 3 : kB];  // table: the positions of the lane's rows; mRoPE: that of row turn_iq, three axes
    if (table) {
#pragma unroll
      for (int b = 0; b < kB; ++b) pos[b] = a.sub_loc[subrow_of(row_iq[b])];
    } else {
      const Pos3 p = load_pos(a.sub_loc, a.sub_loc_axis_stride, subrow_of(turn_iq));
      pos[0] = p.t;
      pos[1] = p.h;
      pos[2] = p.w;
    }
    // Scattered rows: the entries of the first tiles in one load, a lane each, handed out by lane below (read where
    // they are needed, those of V rows past the first two were waited for one by one: 4 plain chunks of 144..197
    // tokens, 8 q / 2 kv heads of 128 dims, 28.3 -> 27.4 us).
    const int first_entries = kGather && n_tiles > 0 ? entry_in_memory(lane / 16, lane % 16) : 0;
#pragma unroll
    for (int b = 0; b < kB; ++b)
#pragma unroll
      for (int s = 0; s < kSteps; ++s) qf[b][s] = *(const va_u32x4*)(q_row[b] + 16 * s);
    unsigned long long first_rows[kWideAhead];
#pragma unroll
    for (int i = 0; i < kWideAhead; ++i) first_rows[i] = row_of(i);
    int first_slots[kWideAhead][kL];
    if (kGather && n_tiles > 0) {
#pragma unroll
      for (int i = 0; i < kWideAhead; ++i)
        read_slots(i, first_slots[i], [&](int tile, int row) __attribute__((always_inline)) {
          return __shfl(first_entries, 16 * tile + row);
        });
    }
    // (the positions are waited for before the tiles are requested: later they would have to wait for the tiles)
    if (table) {
#pragma unroll
      for (int b = 0; b < kB; ++b) asm volatile("" : "+v"(pos[b]));
    } else {
      asm volatile("" : "+v"(pos[0]), "+v"(pos[1]), "+v"(pos[2]));
    }
    ring_barrier<kAnyInFlight>();  // every wave has read the previous link's last tile
    if (kGather && n_tiles > 0) {
      request_entries(0);
#pragma unroll
      for (int i = 0; i < kWideAhead; ++i) issue_gather(i, first_slots[i]);  // (past the range: the last visible token)
    } else {
#pragma unroll
      for (int i = 0; i < kWideAhead; ++i)
        if (i < n_tiles) issue(i, first_rows[i]);
    }
    if (!table && in_turn) {
      // mRoPE: the cosines and sines of the tile's positions, each taken once and shared by the G query
      // heads of a row (an entry is cos | sin in the element type, as the rotation rounds them).  A thread
      // keeps to one row, so that its positions are loaded once, and the lanes of a wave to few pair dims, so
      // that their frequencies are a broadcast.
      const float axes[3] = {(float)pos[0], (float)pos[1], (float)pos[2]};
      const int first = tid / turn_lanes, step = kWideThreads / turn_lanes;
      if (turn_iq < n_q) {
        constexpr int kBatch = 8;  // frequencies requested together
#pragma unroll 1
        for (int pair0 = first; pair0 < half; pair0 += kBatch * step) {
          float freq[kBatch];
#pragma unroll
          for (int x = 0; x < kBatch; ++x) freq[x] = a.rope.inv_freq[min(pair0 + x * step, half - 1)];
#pragma unroll
          for (int x = 0; x < kBatch; ++x) {
            const int pair = pair0 + x * step;
            float c, sn;
            mrope_cos_sin(a.rope, axes, freq[x], pair, c, sn);
            if (pair < half) turns[turn_word(turn_iq, pair, half)] = Mma<E>::pack(c, sn);
          }
        }
      }
      ring_barrier<kAnyInFlight>();
    }
    auto rotate = [&](auto steps) __attribute__((always_inline)) {
      constexpr int kHalf = decltype(steps)::value;  // operands per rotary half
      if (table) {
        // table entries of up to four pairs of operands in flight before the first pair is rotated
        constexpr int kUnits = kB * kHalf, kAhead = kUnits < 4 ? kUnits : 4;
        TableTurn turn[kAhead];
        bool back[kB];
        const float* entry[kB];
#pragma unroll
        for (int b = 0; b < kB; ++b) {
          const int row = table_row(a.rope, pos[b]);
          back[b] = row < 0;
          entry[b] = a.rope.cos_sin + (long long)(back[b] ? ~row : row) * a.rope.rotary_dim + 8 * h;
        }
#pragma unroll
        for (int u = 0; u < kAhead; ++u) turn[u].load(entry[u / kHalf] + 16 * (u % kHalf), 16 * kHalf);
#pragma unroll
        for (int u = 0; u < kUnits; ++u) {
          const int b = u / kHalf, s = u % kHalf, next = u + kAhead;
          turn[u % kAhead].template apply<E>(back[b], qf[b][s], qf[b][s + kHalf]);
          if (next < kUnits) turn[u % kAhead].load(entry[next / kHalf] + 16 * (next % kHalf), 16 * kHalf);
        }
      } else {
#pragma unroll
        for (int b = 0; b < kB; ++b) {
          const int iq = min(row_iq[b], n_q - 1);
#pragma unroll
          for (int s = 0; s < kHalf; ++s) {
            va_u32x4 cs[2];
#pragma unroll
            for (int x = 0; x < 2; ++x)
              cs[x] = *(const va_u32x4*)(turns + turn_word(iq, 16 * s + 8 * h + 4 * x, 16 * kHalf));
            rotate_packed<E>(cs, qf[b][s], qf[b][s + kHalf]);
          }
        }
      }
    };
    if (wave_active && half_steps != 0) {
      if (half_steps == kSteps / 2) {
        rotate(std::integral_constant<int, kSteps / 2>{});
      } else if (half_steps == kSteps / 4) {
        rotate(std::integral_constant<int, kSteps / 4>{});
      } else if (kSteps >= 8 && half_steps == kSteps / 8) {
        rotate(std::integral_constant<int, (kSteps >= 8 ? kSteps / 8 : 1)>{});
      } else {
        // other rotary widths: piece by piece, through a slot per (lane, operand) of the same LDS
        va_u32x4* mine = (va_u32x4*)turns + tid;
        auto each = [&](int b, const S* row) __attribute__((always_inline)) {
          const Pos3 p = load_pos(a.sub_loc, a.sub_loc_axis_stride, subrow_of(row_iq[b]));
#pragma unroll 1
          for (int s = 0; s < kSteps; ++s) {
            const uint4 piece = rotated_query_piece<E>(a.rope, row - 8 * h, 16 * s + 8 * h, p);
            mine[kWideThreads * s] = va_u32x4{piece.x, piece.y, piece.z, piece.w};
          }
        };
        each(0, q_row[0]);
#pragma unroll
        for (int s = 0; s < kSteps; ++s) qf[0][s] = mine[kWideThreads * s];
        if constexpr (kB > 1) {
          each(kB - 1, q_row[kB - 1]);
#pragma unroll
          for (int s = 0; s < kSteps; ++s) qf[kB - 1][s] = mine[kWideThreads * s];
        }
      }
    }
    // The operands are waited for here: a load the compiler still knows of inside the tile loop would make
    // it wait for the loop's own requests as well, and drain the ring in every step.
#pragma unroll
    for (int b = 0; b < kB; ++b)
#pragma unroll
      for (int s = 0; s < kSteps; ++s) asm volatile("" : "+v"(qf[b][s]));

    // ---- the tile loop ----
    // Reference maximum.  The softmax runs against a per-row REFERENCE maximum m_ref that is
    // raised only when a tile's maximum exceeds it by more than kWideRaise (in log2 units):
    // p = exp2(s - m_ref) then stays below 2^kWideRaise, harmless for the 16-bit P operand and the
    // fp32 sums, and any consistent reference gives the same softmax.  Raising m_ref means
    // rescaling the D fp32 accumulators of every row, vector-ALU work on registers that otherwise
    // only the matrix pipe touches; it happens on the first tile and then hardly ever, so it is
    // kept out of the hot loop: the steady loop is left, the accumulators are rescaled, the tile is
    // computed, the steady loop is entered again.  (One wave per SIMD issues an instruction every four
    // clocks or so whatever its kind: the steady loop's own control being a counter and one test,
    // instead of the general loop's flags, is worth 2 % of the kernel.)
    //
    // Software pipeline.  One wave per SIMD means nothing but this wave's own instruction order
    // can keep the matrix pipe busy, so the loop body is written as pieces pinned in order with
    // scheduling barriers: while the scores of tile i+1 are computed (matrix pipe), the
    // exponentials of tile i run on the vector ALU; while the products P.V of tile i run, the V
    // fragments of the next product are transposed, the maxima of tile i+1 are taken and, at head dims under 256, its
    // first exponentials (kEarly).  A product takes 32 clocks and its issue four, an exponential with its multiply-add,
    // sum and half a packing 26: two under each score product, as 128 dims have them, do not fit, one does.
    //
    // Ring.  ring_step(k): wait until tile k has landed for the whole workgroup (one barrier) and
    // request tile k + 2 into the buffer of tile k - 2, which every wave has left by then.  Every
    // wave makes every step exactly once, in order; a step is made just before tile k is first
    // needed (its K, for the scores computed one iteration ahead).
    const int n_vis = t_wave > tok_begin ? min(n_tiles, (t_wave - tok_begin + kWideTokens - 1) / kWideTokens) : 0;
    int next_step = 0;
    unsigned long long row_ahead = row_of(kWideAhead);
    int slots_ahead[kL];  // gather: the same for scattered rows, read from LDS a step earlier
#pragma unroll
    for (int u = 0; u < kL; ++u) slots_ahead[u] = 0;
    auto ring_step = [&]() __attribute__((always_inline)) {
      const int k = next_step++;
      const bool refill = k + kWideAhead < n_tiles;
      const unsigned long long row = row_ahead;
      row_ahead = row_of(k + 1 + kWideAhead);
      // only the loads of the tiles requested after tile k (up to kWideAhead - 1 of them) may still be outstanding
      if (k + kWideAhead - 1 < n_tiles) {
        ring_barrier<(kWideAhead - 1) * kL>();
      } else if (kWideAhead > 2 && k + 1 < n_tiles) {
        ring_barrier<kL>();
      } else {
        ring_barrier<0>();
      }
      if constexpr (kGather) {
        if (k % 4 == 0) request_entries(k / 4 + 1);
        if (refill) {
          int slot[kL];
          read_slots(k + kWideAhead, slot, entry_in_lds);
          issue_gather(k + kWideAhead, slot);
        }
        read_slots(k + 1 + kWideAhead, slots_ahead, entry_in_lds);
      } else if (refill) {
        issue(k + kWideAhead, row);
      }
    };

    // The same step for the steady part of a link (uniform pages; the requested tile and the one
    // after it inside the visible range): no case distinctions, and the page lookup for the next
    // step is sent before the barrier and first touched after it, so its latency passes under the wait.
    const __attribute__((address_space(4))) char* link_pages =
        (const __attribute__((address_space(4))) char*)(a.kv_indices + kv_begin);
    auto ring_step_steady = [&]() __attribute__((always_inline)) {
      const int k = next_step++;
      const unsigned long long row = row_ahead;
      const int t = tok_begin + (k + 1 + kWideAhead) * kWideTokens + 16 * wave_half;
      // (base of the link's page list + an unsigned 32-bit byte offset: a scalar load with a register offset)
      const int page = *(const __attribute__((address_space(4))) int32_t*)(link_pages + ((uint32_t)(t >> p_shift) << 2));
      // The K half of the buffer refilled here was last read two steps ago (the scores of a tile are computed
      // an iteration ahead of its products), and every wave has passed a barrier since: the waves that load K
      // send their requests BEFORE the barrier, in the time they would otherwise only wait, and out of step
      // with the waves that load V, which must wait for the products of the previous iteration to end.
      int zero;
      const uint32_t dst = wave_lds + ring_slot(k + kWideAhead) * Sh::kBufferBytes;
      const char* base = wave_plain + row;
      if (!wave_is_v) {
        issue_plain(base, dst);
        zero = ring_barrier_zero<kWideAhead * kL>();
      } else {
        zero = ring_barrier_zero<(kWideAhead - 1) * kL>();
        issue_plain(base, dst);
      }
      row_ahead = half_offset(page + zero, t);
    };
    // The steady step of scattered rows (tiles past the range repeat the last visible token: only a next tile to
    // request must exist).  Entries requested in step 4m are complete behind the barrier of step 4m + 1, the
    // first of them is read there.
    auto ring_step_gather = [&]() __attribute__((always_inline)) {
      const int k = next_step++;
      if (k % 4 == 0) request_entries(k / 4 + 1);
      if (!wave_is_v) {
        issue_gather(k + kWideAhead, slots_ahead);
        ring_barrier<kWideAhead * kL>();
      } else {
        ring_barrier<(kWideAhead - 1) * kL>();
        issue_gather(k + kWideAhead, slots_ahead);
      }
      read_slots(k + 1 + kWideAhead, slots_ahead, entry_in_lds);
    };
    // iterations [1, i_steady_end) may take it: tiles i + 1 + kWideAhead and i + 2 + kWideAhead are plain,
    // tile i is unmasked for every row of the wave and a next tile exists
    int i_steady_end = 0;
    if (uniform_pages) {
      const int plain_tiles = (t_last + 1 - tok_begin) / kWideTokens;  // tiles 0 .. plain_tiles - 1 are plain
      const int unmasked_tiles = t_wave_min > tok_begin ? (t_wave_min - tok_begin) / kWideTokens : 0;
      i_steady_end = min(min(plain_tiles - 2 - kWideAhead, unmasked_tiles), n_vis - 1);
    } else if (kGather && P < 16) {
      const int unmasked_tiles = t_wave_min > tok_begin ? (t_wave_min - tok_begin) / kWideTokens : 0;
      i_steady_end = min(min(n_tiles - 1 - kWideAhead, unmasked_tiles), n_vis - 1);
    }

    // Scores of two tiles: the exponentials of one are taken in place while the products of the next
    // accumulate into the other; which is which alternates from tile to tile.
    va_f32x16 sc[kB];       // scores, then probabilities, of the current tile (between tiles)
    va_f32x16 sc_next[kB];  // scores of the next tile
    // K fragments: at most eight in registers; the fragment eight steps on is requested as one is consumed
    constexpr int kKRing = kSteps < 8 ? kSteps : 8;
    va_u32x4 kf[kKRing];
    auto read_k_fragment = [&](int tile, int s) __attribute__((always_inline)) {
      const char* kt = lds + ring_slot(tile) * Sh::kBufferBytes;
      kf[s % kKRing] = *(const va_u32x4*)(kt + k_lane_byte + 256 * s);
    };
    auto read_k = [&](int tile) __attribute__((always_inline)) {
#pragma unroll
      for (int s = 0; s < kKRing; ++s) read_k_fragment(tile, s);
    };
    auto score_step = [&](int tile, int s, auto& into) __attribute__((always_inline)) {
#pragma unroll
      for (int b = 0; b < kB; ++b) {
        // through the builtin: the compiler sees these products and keeps the wait states between
        // them and the vector-ALU instructions that feed them or read their results
        into[b] = Mma<E>::run32(kf[s % kKRing], qf[b][s], s == 0 ? va_f32x16{} : into[b]);
      }
      if (s + kKRing < kSteps) read_k_fragment(tile, s + kKRing);
    };

    if (n_vis > 0) {  // scores of tile 0
      ring_step();
      read_k(0);
#pragma unroll
      for (int s = 0; s < kSteps; ++s) score_step(0, s, sc);
    }
    // maximum of the (unmasked) scores of the next tile per lane, gathered piecewise between the
    // P.V products of the current one, whose matrix work leaves the vector ALU idle
    float early_max[kB];
    bool early_max_valid = false;
#pragma unroll
    for (int b = 0; b < kB; ++b) early_max[b] = 0.f;
    // One tile: phase A and phase B below, on the scores in `cur`, leaving those of the next tile in `nxt`.
    // The steady part of a link runs it in a loop of its own, whose control is a counter and the test for
    // a raised reference; every other tile (the first, masked ones, the last, the one after a raised
    // reference) goes through the general step further down.
    auto tile_body = [&](int i, auto& cur, auto& nxt) __attribute__((always_inline)) {

      // V^T fragments of this tile, kVAhead of them in flight: fragment idx = (step kk, dim tile t)
      const uint32_t vt = lds_base + ring_slot(i) * Sh::kBufferBytes + Sh::kTileBytes;
      const uint32_t vt_even = vt + v_even, vt_odd = vt + v_odd;
      constexpr int kFrags = 2 * kDimTiles;
      constexpr int kMaxFirst = kFrags > 2 ? 2 : kFrags - 1;  // first product the early maxima follow
      constexpr int kVAhead = kFrags < 4 ? kFrags : 4;
      va_u32x4 vfr[kVAhead];
      auto read_vfrag = [&](int idx) __attribute__((always_inline)) {
        const int kk = idx / kDimTiles, t = idx % kDimTiles;
        const uint32_t at = ((t & 1) ? vt_odd : vt_even) + 128 * (t / 2) + kk * 16 * kRowBytes;
        const va_u32x2 lo = lds_read_tr16(at), hi = lds_read_tr16(at + 8 * kRowBytes);
        vfr[idx % kVAhead] = va_u32x4{lo[0], lo[1], hi[0], hi[1]};
      };
      // ---- phase A: scores of tile i + 1 (matrix pipe) under the exponentials of tile i ----
      float sum[kB];
#pragma unroll
      for (int b = 0; b < kB; ++b) sum[b] = 0.f;
      // Piece r: the exponential of element r; the sum takes element r - 1 (an exponential's result
      // is not ready for the very next instruction) and odd pieces pack the finished pair into P.
      uint32_t pw[kB][8];
      auto exp_piece = [&](int r) __attribute__((always_inline)) {
#pragma unroll
        for (int b = 0; b < kB; ++b) {
          // raw score -> exponent in fp32, as the reference scales its scores.  (The multiply-add sits here,
          // in the shadow of a score product, rather than under the P.V products, whose slots are full: there
          // it costs 3.4 % of the kernel, here 0.8 %.  Staging the query times the scale instead makes it
          // free, but rounds other numbers than the reference does: out of tolerance once scores reach +-20.)
          cur[b][r] = __builtin_amdgcn_exp2f(fmaf(cur[b][r], a.scale_log2, -m_ref[b]));
          if (r > 0) sum[b] += cur[b][r - 1];
          if (r >= 2 && r % 2 == 0) pw[b][r / 2 - 1] = Mma<E>::pack(cur[b][r - 2], cur[b][r - 1]);
        }
      };
      constexpr int kPiecesPerStep = 16 / kSteps > 0 ? 16 / kSteps : 1;  // exponentials between two score steps
      // The last visible tile runs the same instructions: its "next scores" come from whatever
      // the following ring buffer holds and are never looked at (sixteen idle products per link
      // against a second copy of this phase and the register moves where the two would meet).
      read_k(i + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        if (r % kPiecesPerStep == 0) score_step(i + 1, r / kPiecesPerStep, nxt);
        __builtin_amdgcn_sched_barrier(0);
        exp_piece(r);
        // the first V fragments are requested once half of the K fragments have been consumed: the
        // counter of outstanding LDS reads holds fifteen, and a wait for the first K fragment
        // with more than that in flight becomes a wait for the excess as well
        if (r == 8) {
#pragma unroll
          for (int idx = 0; idx < kVAhead; ++idx) read_vfrag(idx);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int b = 0; b < kB; ++b) {
        l_run[b] += sum[b] + cur[b][15];
        pw[b][7] = Mma<E>::pack(cur[b][14], cur[b][15]);
      }

      // ---- phase B: O^T += V^T . P^T over two 16-token steps; a fragment serves all row blocks,
      // and once it has been used the fragment kVAhead further on is requested ----
      va_u32x4 pf[2][kB];
#pragma unroll
      for (int kk = 0; kk < 2; ++kk)
#pragma unroll
        for (int b = 0; b < kB; ++b)
          pf[kk][b] = va_u32x4{pw[b][4 * kk + 0], pw[b][4 * kk + 1], pw[b][4 * kk + 2], pw[b][4 * kk + 3]};
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int idx = 0; idx < kFrags; ++idx) {
        const int kk = idx / kDimTiles, t = idx % kDimTiles;
#pragma unroll
        for (int b = 0; b < kB; ++b) {
          Mma<E>::run32_acc(vfr[idx % kVAhead], pf[kk][b], o[b][t]);
        }
        __builtin_amdgcn_sched_barrier(0);
        if (idx + kVAhead < kFrags) read_vfrag(idx + kVAhead);
        // Elements of the next tile's scores folded into early_max after this product: the 15
        // comparisons are spread over the products from the third on (the last score product was
        // issued well before, so its results have been written).
        if (idx >= kMaxFirst) {
#pragma unroll
          for (int e = 1; e < 16; ++e) {
            if (kMaxFirst + (e - 1) * (kFrags - kMaxFirst) / 15 != idx) continue;
#pragma unroll
            for (int b = 0; b < kB; ++b)
              early_max[b] = fmaxf(e == 1 ? nxt[b][0] : early_max[b], nxt[b][e]);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    // The same tile in the steady part of a link at head dims under 256, whose two row blocks take twice the
    // exponentials per product: under the score products alone they do not fit, so the first kEarly elements of a tile
    // are taken under the P.V products of the tile before (`sum` and `pw` carry them), ahead of the test of its maxima.
    // Where the test then raises the reference they are dropped and the tile's scores are computed anew.
    constexpr int kEarly = Sh::kEarly;
    float sum[kB];
    uint32_t pw[kB][8];
    // element r of block b, part [first, end): exponential, the sum and the packing one element behind
    auto exp_element = [&](auto& of, int b, int r, int first) __attribute__((always_inline)) {
      of[b][r] = __builtin_amdgcn_exp2f(fmaf(of[b][r], a.scale_log2, -m_ref[b]));
      if (r > first) sum[b] += of[b][r - 1];
      if (r % 2 == 0 && r > first) pw[b][r / 2 - 1] = Mma<E>::pack(of[b][r - 2], of[b][r - 1]);
    };
    auto exp_finish = [&](auto& of, int b, int end) __attribute__((always_inline)) {
      sum[b] += of[b][end - 1];
      pw[b][end / 2 - 1] = Mma<E>::pack(of[b][end - 2], of[b][end - 1]);
    };
    auto early_exps = [&](auto& of) __attribute__((always_inline)) {  // (not under anything: the first tile of the part)
#pragma unroll
      for (int b = 0; b < kB; ++b) sum[b] = 0.f;
#pragma unroll
      for (int r = 0; r < kEarly; ++r)
#pragma unroll
        for (int b = 0; b < kB; ++b) exp_element(of, b, r, 0);
#pragma unroll
      for (int b = 0; b < kB; ++b) exp_finish(of, b, kEarly);
    };
    auto steady_body = [&](int i, auto& cur, auto& nxt) __attribute__((always_inline)) {
      const uint32_t vt = lds_base + ring_slot(i) * Sh::kBufferBytes + Sh::kTileBytes;
      const uint32_t vt_even = vt + v_even, vt_odd = vt + v_odd;
      constexpr int kFrags = 2 * kDimTiles, kVAhead = kFrags < 4 ? kFrags : 4;
      va_u32x4 vfr[kVAhead];
      auto read_vfrag = [&](int idx) __attribute__((always_inline)) {
        const int kk = idx / kDimTiles, t = idx % kDimTiles;
        const uint32_t at = ((t & 1) ? vt_odd : vt_even) + 128 * (t / 2) + kk * 16 * kRowBytes;
        const va_u32x2 lo = lds_read_tr16(at), hi = lds_read_tr16(at + 8 * kRowBytes);
        vfr[idx % kVAhead] = va_u32x4{lo[0], lo[1], hi[0], hi[1]};
      };
      // ---- phase A: scores of tile i + 1 under the rest of the exponentials of tile i ----
      constexpr int kPieces = kB * (16 - kEarly), kLead = 2, kSlots = kB * kSteps;
      auto piece = [&](int n) __attribute__((always_inline)) { exp_element(cur, n % kB, kEarly + n / kB, kEarly); };
      read_k(i + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int n = 0; n < kLead; ++n) piece(n);  // while the first K fragment is on its way
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int slot = 0; slot < kSlots; ++slot) {
        const int step = slot / kB, b = slot % kB;
        nxt[b] = Mma<E>::run32(kf[step % kKRing], qf[b][step], step == 0 ? va_f32x16{} : nxt[b]);
        if (b == kB - 1 && step + kKRing < kSteps) read_k_fragment(i + 1, step + kKRing);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int n = kLead; n < kPieces; ++n)
          if ((n - kLead) * kSlots / (kPieces - kLead) == slot) piece(n);
        if (slot == kSlots / 2) {
#pragma unroll
          for (int idx = 0; idx < kVAhead; ++idx) read_vfrag(idx);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int b = 0; b < kB; ++b) {
        exp_finish(cur, b, 16);
        l_run[b] += sum[b];
        sum[b] = 0.f;
      }
      va_u32x4 pf[2][kB];
#pragma unroll
      for (int kk = 0; kk < 2; ++kk)
#pragma unroll
        for (int b = 0; b < kB; ++b)
          pf[kk][b] = va_u32x4{pw[b][4 * kk + 0], pw[b][4 * kk + 1], pw[b][4 * kk + 2], pw[b][4 * kk + 3]};
      __builtin_amdgcn_sched_barrier(0);
      // ---- phase B: O^T += V^T . P^T under the first exponentials and the maxima of tile i + 1 (from the third
      // product on: the scores are written by then).  The maxima come first, the exponentials are taken in place. ----
      constexpr int kProducts = kB * kFrags, kFirst = 2;
      // of block b: eight maxima of three, ahead of the exponential of the first element each of them takes in
      auto max_piece = [&](int b, int e) __attribute__((always_inline)) {
        early_max[b] = e == 0 ? fmaxf(nxt[b][0], nxt[b][1]) : fmaxf(fmaxf(early_max[b], nxt[b][2 * e]), nxt[b][2 * e + 1]);
      };
      constexpr int kMaxes = kB * 8, kExps = kB * kEarly, kUnderB = kMaxes + kExps;
#pragma unroll
      for (int product = 0; product < kProducts; ++product) {
        const int idx = product / kB, b = product % kB, kk = idx / kDimTiles, t = idx % kDimTiles;
        Mma<E>::run32_acc(vfr[idx % kVAhead], pf[kk][b], o[b][t]);
        __builtin_amdgcn_sched_barrier(0);
        if (b == kB - 1 && idx + kVAhead < kFrags) read_vfrag(idx + kVAhead);
        if (product >= kFirst) {
#pragma unroll
          for (int n = 0; n < kUnderB; ++n) {
            // the maxima of the elements that are exponentiated here go ahead of them, the others behind
            if (kFirst + n * (kProducts - kFirst) / kUnderB != product) continue;
            constexpr int kHead = kB * kEarly / 2;
            if (n < kHead) {
              max_piece(n % kB, n / kB);
            } else if (n < kHead + kExps) {
              exp_element(nxt, (n - kHead) % kB, (n - kHead) / kB, 0);
            } else {
              max_piece((n - kExps) % kB, (n - kExps) / kB);
            }
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int b = 0; b < kB; ++b) exp_finish(nxt, b, kEarly);
    };
    // The reference of the rows is raised to the maxima of the tile in `cur` (m_tile, log2 units): what was
    // accumulated against the old reference is rescaled; the tile's raw scores stay as they are.
    auto raise_reference = [&](int i, auto& cur) __attribute__((always_inline)) {
      accumulator_fence<kB * kDimTiles>(&o[0][0]);
#pragma unroll
      for (int b = 0; b < kB; ++b) {
        const float m_new = fmaxf(m_ref[b], m_tile[b]);
        const float alpha = __builtin_amdgcn_exp2f(m_ref[b] - m_new);
        m_ref[b] = m_new;
        raise_above[b] = m_new + kWideRaise;
        l_run[b] *= alpha;
#pragma unroll
        for (int t = 0; t < kDimTiles; ++t) o[b][t] *= alpha;
        const int t0 = tok_begin + i * kWideTokens;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const bool visible = (t0 + (r / 4) * 8 + 4 * h + (r % 4)) < t_row[b];
          cur[b][r] = visible ? cur[b][r] : -INFINITY;
        }
      }
    };
    // the test of the steady part: the maxima were gathered under the previous products, nothing is masked
    auto steady_test = [&]() __attribute__((always_inline)) {
      bool raise = false;
#pragma unroll
      for (int b = 0; b < kB; ++b) {
        m_tile[b] = half_wave_max(early_max[b]) * a.scale_log2;
        raise = raise || m_tile[b] > raise_above[b];
      }
      return (bool)__any(raise);
    };

    int i = 0;
    while (i < n_vis) {
      bool raise = false;
      // (a part of one tile is not worth the exponentials and scores that entering and leaving it take)
      if (i >= 1 && i + (kEarly > 0) < i_steady_end && !steady_test()) {
        if constexpr (kEarly > 0) early_exps(sc);
        // (written without a break in the middle: with one the compiler keeps the accumulators of before and after the
        // products side by side, copies one to the other every tile and spills)
        do {
          if constexpr (kGather) {
            ring_step_gather();
          } else {
            ring_step_steady();
          }
          if constexpr (kEarly > 0) {
            steady_body(i, sc, sc_next);
          } else {
            tile_body(i, sc, sc_next);
          }
#pragma unroll
          for (int b = 0; b < kB; ++b) sc[b] = sc_next[b];
          ++i;
          raise = steady_test();
        } while (!raise && i < i_steady_end);
        early_max_valid = true;  // (a next tile exists throughout the steady part)
        if constexpr (kEarly > 0) {  // the general step wants the scores of its tile as they were
          read_k(i);
#pragma unroll
          for (int s = 0; s < kSteps; ++s) score_step(i, s, sc);
        }
        raise = false;  // (it makes the test again)
      }
      const int t0 = tok_begin + i * kWideTokens;
      if (i + 1 < n_tiles) ring_step();  // tile i + 1 has landed
      // mask and find the tile maxima; reg r of a block is token t0 + (r/4)*8 + 4h + r%4 of its row
      const bool masked = t0 + kWideTokens > t_wave_min;
#pragma unroll
      for (int b = 0; b < kB; ++b) {
        if (masked) {
#pragma unroll
          for (int r = 0; r < 16; ++r)
            sc[b][r] = (t0 + (r / 4) * 8 + 4 * h + (r % 4)) < t_row[b] ? sc[b][r] : -INFINITY;
        }
        // the tile maximum (raw): from the maxima found under the previous products, or, for a masked or
        // first tile, from sc
        float tile_max = early_max[b];
        if (masked || !early_max_valid) {
          tile_max = sc[b][0];
#pragma unroll
          for (int r = 1; r < 16; ++r) tile_max = fmaxf(tile_max, sc[b][r]);
        }
        m_tile[b] = half_wave_max(tile_max) * a.scale_log2;
        raise = raise || m_tile[b] > raise_above[b];
      }
      raise = __any(raise);
      if (raise) raise_reference(i, sc);
      tile_body(i, sc, sc_next);
#pragma unroll
      for (int b = 0; b < kB; ++b) sc[b] = sc_next[b];
      early_max_valid = i + 1 < n_vis;
      ++i;
    }
    while (next_step < n_tiles) ring_step();  // tiles this wave does not see: keep in step with the others
  }

  accumulator_fence<kB * kDimTiles>(&o[0][0]);
  // ---- emit: accumulator reg r of dim tile t is dim 32t + (r/4)*8 + 4h + r%4 of the lane's row ----
#pragma unroll
  for (int b = 0; b < kB; ++b) {
    float l = l_run[b];
    {
      const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(l), __float_as_uint(l), false, false);
      l = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    }
    const int my_row = row0 + 32 * b;
    const int iq = row_iq[b];
    if (iq >= n_q) continue;
    const int g = my_row - iq * G;
    const int hq = hk * G + g;
    const float inv = l > 0.f ? 1.f / l : 0.f;
    if (part_base < 0) {
      const PlanWords link0 = item + VA_I_LINK0;
      const int subrow = (link0[VA_L_FLAGS] & VA_LINK_INDIRECT) ? a.qrefs[link0[VA_L_QREF] + iq] : link0[VA_L_QREF] + iq;
      const long long out_row = a.sub_worker[subrow];
      S* orow = (S*)a.out + (out_row * a.num_q_heads + hq) * (long long)kD;
#pragma unroll
      for (int t = 0; t < kDimTiles; ++t)
#pragma unroll
        for (int r = 0; r < 16; r += 4) {  // four consecutive dims
          const int d0 = 32 * t + (r / 4) * 8 + 4 * h;
          *(uint2*)(orow + d0) = make_uint2(Mma<E>::pack(o[b][t][r] * inv, o[b][t][r + 1] * inv),
                                            Mma<E>::pack(o[b][t][r + 2] * inv, o[b][t][r + 3] * inv));
        }
      if (h == 0 && a.lse) {
        const float lse2 = l > 0.f ? m_ref[b] + log2f(l) : -INFINITY;
        a.lse[out_row * a.num_q_heads + hq] = a.lse_base2 ? lse2 : lse2 * kLn2;
      }
    } else {
      const long long slot = (long long)(part_base + iq) * a.num_q_heads + hq;
      float* prow = a.part_acc + slot * kD;
#pragma unroll
      for (int t = 0; t < kDimTiles; ++t)
#pragma unroll
        for (int r = 0; r < 16; r += 4)
          *(float4*)(prow + 32 * t + (r / 4) * 8 + 4 * h) = make_float4(o[b][t][r], o[b][t][r + 1], o[b][t][r + 2], o[b][t][r + 3]);
      if (h == 0) {
        a.part_ml[slot * 2 + 0] = m_ref[b];
        a.part_ml[slot * 2 + 1] = l;
      }
    }
  }
  }  // items of the slot
}

template <typename E, int kD, bool kGather>
__global__ __launch_bounds__(kWideThreads, 1) void attn_mfma_wide_kernel(AttnArgs a) {
  wide_slot<E, kD, kGather>(a, blockIdx.x, gridDim.x);
}

// Wide and narrow items in one launch: `wide` workgroups of wide slots, then one per narrow item and kv head.  The wide
// slots are bound by instruction issue and leave the memory idle, the streaming items are bound by memory and need few
// CUs (one takes in up to 58 GB/s, all 256 share 6.9 TB/s).  The wide slots start first; the planner lets them leave so
// many CUs that both kinds end together, and when they are done the remaining items have all CUs.  Attention and merge
// of a layer, two launches and this one: 48 decode rows and 4 chunks of 512 tokens, contexts of 1 k..32 k, 16 q / 4 kv
// heads of 256 dims 1229 -> 1090 us, 16 rows and 4 chunks of 256 503 -> 457, 24 rows and 4 chunks of 400, 32 q / 8 kv
// heads of 128 dims 441 -> 373; where the streaming items are a few tail rows it saves their launch (plain prefill of 6
// requests 0.7 %).  A streaming workgroup has a CU to itself here (registers of the wide kind): where many short ones
// want to share, at head dims under 256, the planner gives them a launch of their own.
template <typename E, int kD, bool kGather>
__global__ __launch_bounds__(kWideThreads, 1) void attn_mfma_joint_kernel(AttnArgs a, unsigned wide) {
  if (blockIdx.x < wide) {
    wide_slot<E, kD, kGather>(a, blockIdx.x, wide);
  } else {
    stream_block<E, kD, kGather>(a, blockIdx.x - wide);
  }
}

template <typename E, int kD, bool kGather>
static int launch_wide_one(const AttnArgs& a, int n_slots, int n_narrow, hipStream_t stream) {
  constexpr int wide_bytes = WideShape<kD>::lds_bytes(kGather), narrow_bytes = StreamShape<kD>::lds_bytes(kGather);
  constexpr int joint_bytes = wide_bytes > narrow_bytes ? wide_bytes : narrow_bytes;
  static_assert(kWideThreads == kStreamThreads, "one launch serves both kinds");
  const unsigned wide = (unsigned)n_slots * (unsigned)a.num_kv_heads, narrow = (unsigned)n_narrow * (unsigned)a.num_kv_heads;
  static std::atomic<unsigned long long> wide_devices{0}, joint_devices{0};
  const hipError_t allowed =
      narrow > 0 ? allow_lds(reinterpret_cast<const void*>(&attn_mfma_joint_kernel<E, kD, kGather>), joint_bytes, joint_devices)
                 : allow_lds(reinterpret_cast<const void*>(&attn_mfma_wide_kernel<E, kD, kGather>), wide_bytes, wide_devices);
  if (allowed != hipSuccess) return va_fail(VA_ERR_HIP, "raising the LDS limit: %s", hipGetErrorString(allowed));
  if (narrow > 0) {
    hipLaunchKernelGGL((attn_mfma_joint_kernel<E, kD, kGather>), dim3(wide + narrow), dim3(kWideThreads), joint_bytes, stream, a, wide);
  } else {
    hipLaunchKernelGGL((attn_mfma_wide_kernel<E, kD, kGather>), dim3(wide), dim3(kWideThreads), wide_bytes, stream, a);
  }
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? VA_OK : va_fail(VA_ERR_HIP, "wide attention launch: %s", hipGetErrorString(e));
}

template <typename E, int kD>
static int launch_wide_dim(const AttnArgs& a, int n_slots, int n_narrow, hipStream_t stream) {
  // Pages of at least 16 tokens take one lookup per half tile, smaller ones (a slot list has pages of one) an
  // entry per token; the choice hangs on the page size alone, so that a recorded launch keeps its kernel.
  // (Other page sizes, slot lists beside larger pages, and rings built deeper than the index entries allow go
  // through the first kernel's per-lane lookups.)
  if constexpr (kWideAhead <= 2) {
    if (a.page_size < 16 && (a.page_size & (a.page_size - 1)) == 0)
      return launch_wide_one<E, kD, true>(a, n_slots, n_narrow, stream);
  }
  return launch_wide_one<E, kD, false>(a, n_slots, n_narrow, stream);
}

template <typename E>
static int launch_wide_typed(const AttnArgs& a, int n_slots, int n_narrow, hipStream_t stream) {
  switch (a.head_dim) {
    case 64:
      return launch_wide_dim<E, 64>(a, n_slots, n_narrow, stream);
    case 128:
      return launch_wide_dim<E, 128>(a, n_slots, n_narrow, stream);
    case 256:
      return launch_wide_dim<E, 256>(a, n_slots, n_narrow, stream);
    default:
      return va_fail(VA_ERR_ARG, "matrix-core path supports head_dim 64, 128, 256");
  }
}

int launch_mfma_wide(const AttnArgs& a, int dtype, int n_slots, int n_narrow, hipStream_t stream) {
  return dtype == VA_BF16 ? launch_wide_typed<BF16>(a, n_slots, n_narrow, stream) : launch_wide_typed<F16>(a, n_slots, n_narrow, stream);
}

}  // namespace va
