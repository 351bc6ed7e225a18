// Streaming matrix-core view attention, device code: query tiles of up to 16 MFMA rows (decode and short
// prefill tiles), K/V streamed from the pool straight into LDS.
//
// The kernel is bound by HBM.  What the memory gives was measured with loads that fill LDS and nothing else, pages of
// 16 tokens in random order: 6.9 TB/s (read once, non-temporal) whether 256 or 2048 workgroups ask, 8 KB in
// flight per wave are enough, and one CU takes in up to 58 GB/s, twice its share.  So depth and occupancy are
// not what counts, but that no wave waits for another:
//   * the four waves of a workgroup are independent: each takes every fourth 16-token tile of the walk, brings
//     it global -> LDS (global_load_lds_dwordx4) into a ring of its own and waits for its own loads only.  There is no
//     barrier in the tile loop.  (One ring for all four, with two barriers a tile and every wave computing the
//     scores of every tile: 5.5 to 6.3 TB/s, the loads of a tile going out only when the slowest wave was done.)
//   * a tile goes from LDS to registers at once and its buffer is refilled before the softmax;
//   * a wave keeps its own softmax state; the four are folded through LDS at the end of the item;
//   * up to four items that walk the same tokens (the tiles of one run's many readers) share a workgroup: the tokens
//     are read once for all of them, where each used to read them from the die's L2.
// Launches of 16 q / 4 kv heads of 256 dims, bf16, us with one ring and with four: 64 requests over a shared prompt
// 353 -> 313 to 323 (1.96 GB = 6.1 to 6.3 TB/s), eight of 131072 tokens 678 -> 636 to 662 (4.3 GB = 6.5 to 6.8), 48 of
// 1 k..32 k 508 -> 487; 32 requests over token slots, 32 q / 8 kv heads of 128 dims, 92 -> 90 to 93.  An item costs about 5 us of set-up and fold, hence the few
// long items the planner makes (default_target).
//
//   S^T[16 tokens, 16 rows] = K . Q^T    v_mfma_f32_16x16x32, K from LDS as the A operand, the rotated query
//                                        rows as B operands
//   online softmax per row
//   O^T[D, 16 rows] += V^T . P^T         v_mfma_f32_16x16x16, V^T from transposing LDS reads (ds_read_b64_tr_b16),
//                                        P already laid out as the B operand
// LDS rows are not padded (the loads write 1 KB runs); bank conflicts are avoided by storing piece c of tile row r
// at position c ^ stream_swz(r), which costs nothing: the lane that fills position p fetches piece p ^ stream_swz(r).
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

#include "va_launch.h"
#include "va_mfma_common.h"

namespace va {

constexpr int kStreamThreads = 256;
constexpr int kStreamWaves = 4;
constexpr int kStreamTok = 16;  // tokens per tile

constexpr int kIndexSlots = 8;  // tiles whose index entries a wave's ring of entries holds

// kShort: launches of short items (stream_block_short), where an item's set-up and fold count and those of others have to
// run beside them: one tile a workgroup, and less LDS, for two to four workgroups on a CU.
template <int kD, bool kShort = false>
struct StreamShape {
  static constexpr int kChunks = kD / 8;                     // 16-byte pieces of a head row
  static constexpr int kSteps = kD / 32;                     // contraction steps of K.Q^T
  static constexpr int kDimTiles = kD / 16;                  // 16-dim tiles of the output
  static constexpr int kRowBytes = kChunks * 16;
  static constexpr int kRowsPerLoad = kWave / kChunks;       // tile rows one wave-level load covers
  static constexpr int kLoads = kStreamTok / kRowsPerLoad;   // loads of a K (or V) tile
  static constexpr int kTileBytes = kStreamTok * kRowBytes;  // a K (or V) tile
  // ring depth of a wave, in tiles, and workgroups per CU (as registers and LDS allow)
  static constexpr int kBuffers = kShort ? (kD == 64 ? 2 : 1) : kD == 64 ? 4 : 2;
  static constexpr int kMinBlocks = kShort ? (kD == 256 ? 2 : kD == 128 ? 3 : 4) : kD == 256 ? 1 : 2;
  // A wave's state at the end, in its own ring: accumulators (rows padded by 16 bytes, so that the sixteen rows of a
  // write spread over the banks), then maxima and sums.
  static constexpr int kFoldRowBytes = kD * 4 + 16;
  static constexpr int kFoldBytes = (16 * (kFoldRowBytes + 8) + 1023) / 1024 * 1024;
  static constexpr int kWaveRingBytes = kBuffers * 2 * kTileBytes > kFoldBytes ? kBuffers * 2 * kTileBytes : kFoldBytes;
  static constexpr int kRingBytes = kStreamWaves * kWaveRingBytes;
  // Behind the rings: the rotated query rows of the items that walk together, over scattered rows of fewer and for every
  // wave the index entries of kIndexSlots tiles.
  static constexpr int kIndexOffset = kRingBytes + (kShort ? 1 : VA_TOGETHER_SCATTERED) * 16 * kRowBytes;
  static constexpr int kIndexBytes = kIndexSlots * kStreamTok * 4;
  static constexpr int lds_bytes(bool gather) {
    return gather ? kIndexOffset + kStreamWaves * kIndexBytes : kRingBytes + (kShort ? 1 : VA_TOGETHER) * 16 * kRowBytes;
  }
};

// Piece c of tile row r lies at position c ^ stream_swz(r).  K fragments (16 rows, one piece of each) then hit sixteen
// different 16-byte columns of the banks, transposing V reads (8 rows, 32 bytes of each) eight different 32-byte ones.
template <int kD>
__device__ __forceinline__ int stream_swz(int r) {
  if constexpr (kD >= 128) return ((r & 7) << 1) | ((r >> 3) & 1);
  return ((r & 6) | ((r >> 3) & 1));  // (rows of 128 bytes: neighbouring rows lie side by side already)
}

// Wait until at most n of the wave's vector memory operations are outstanding.
template <int n>
__device__ __forceinline__ void wave_wait() {
  static_assert(n < kAnyInFlight, "the counter holds no more");
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(n) : "memory");
}

// max over the four lanes l, l ^ 16, l ^ 32, l ^ 48 (the contraction groups of an MFMA row) with the two
// row-swapping instructions of gfx950, no trip through the LDS crossbar: with both operands x,
// v_permlane16_swap leaves (rows 0 0 2 2, rows 1 1 3 3) of x and v_permlane32_swap (low low, high high).
__device__ __forceinline__ float max_over_contraction_groups(float x) {
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}

typedef int va_i32x4 __attribute__((ext_vector_type(4)));

// The whole item (its first link travels in it) in ONE round of scalar loads: fetched word by word where each was
// first needed, it cost three dependent trips to memory before the first tile could be requested.
__device__ __forceinline__ void load_item(const AttnArgs& a, int index, int (&item)[VA_ITEM_WORDS]) {
  const __attribute__((address_space(4))) va_i32x4* words =
      (const __attribute__((address_space(4))) va_i32x4*)(a.narrow_items + (long long)index * VA_ITEM_WORDS);
#pragma unroll
  for (int w = 0; w < VA_ITEM_WORDS / 4; ++w) {
    const va_i32x4 x = words[w];
#pragma unroll
    for (int k = 0; k < 4; ++k) item[4 * w + k] = x[k];
  }
}

// One work item for one kv head, or kB of them that walk the same tokens: a block of up to 16 MFMA rows each.
// kGather: pages hold less than a tile (1, 2, 4 or 8 tokens; a slot list has pages of one).
template <typename E, int kD, bool kGather, int kB, bool kShort = false>
__device__ __forceinline__ void stream_items(const AttnArgs& a, const int (&item)[kB][VA_ITEM_WORDS], int hk) {
  using S = typename E::storage;
  using Sh = StreamShape<kD, kShort>;
  static_assert(kB <= (kShort ? 1 : kGather ? VA_TOGETHER_SCATTERED : VA_TOGETHER), "room for the query rows of so many tiles");
  static_assert(Sh::kMinBlocks * Sh::lds_bytes(kGather) <= 160 * 1024, "the LDS of a CU");
  constexpr int kChunks = Sh::kChunks, kSteps = Sh::kSteps, kDimTiles = Sh::kDimTiles, kBuffers = Sh::kBuffers;
  constexpr int kLoads = Sh::kLoads, kRowBytes = Sh::kRowBytes, kTileBytes = Sh::kTileBytes;
  // the entries of tiles i + 1 .. i + 2 kBuffers of a wave are held or on their way at any time
  static_assert(!kGather || 2 * kBuffers <= kIndexSlots, "index entries of more tiles than their ring holds");

  extern __shared__ va_u32x4 smem[];
  char* lds = (char*)smem;

  const int G = a.num_q_heads / a.num_kv_heads;
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int lane = tid % kWave;
  const int j = lane % 16;   // MFMA row of this lane in a block of 16; also the token it supplies K of
  const int kg = lane / 16;  // contraction group
  const int row_iq = j / G;  // MFMA row j of an item: tile row j / G, head j % G
  const S* kp = (const S*)a.k_pool + (long long)hk * kD;
  const S* vp = (const S*)a.v_pool + (long long)hk * kD;
  const int P = a.page_size;
  const bool pow2_pages = (P & (P - 1)) == 0;
  const int p_shift = __builtin_ctz(P);  // t / P and t % P as shift and mask (power-of-two pages)
  const int row_bytes = (int)a.pool_row_stride * (int)sizeof(S);
  // bytes of a page, for the byte offsets of tiles inside a page: they need the figure to fit 32 bits
  const bool page_fits = ((unsigned long long)(uint32_t)row_bytes << p_shift) <= 0xffffffffull;
  const uint32_t page_bytes = (uint32_t)row_bytes << p_shift;

  // This lane's part of wave-level load u of a K or V tile: tile row, and the piece of it that belongs at
  // the lane's LDS position.  Tiles inside a page go out as a wave-uniform base plus a per-lane offset that
  // never changes, in groups of up to four behind one setting of M0 (a group's immediate offsets move the
  // pool address as well: grouped_lane_offset; the bias, which the base gives back, keeps the rest positive).
  constexpr int kLoadGroup = kLoads < 4 ? kLoads : 4;
  constexpr int kLoadBias = 1024 * (kLoadGroup - 1);
  const int ld_row0 = lane / kChunks;
  uint32_t ld_off[kLoads];
#pragma unroll
  for (int u = 0; u < kLoads; ++u) {
    const int row = u * Sh::kRowsPerLoad + ld_row0;
    ld_off[u] = grouped_lane_offset(
        (uint32_t)(row * row_bytes + 16 * ((lane % kChunks) ^ stream_swz<kD>(row)) + kLoadBias), u);
  }
  // LDS byte offsets (within a tile) of what this lane reads.  K: dims [32 s + 8 kg, +8) of token j; the
  // swizzle only touches the low four bits of a piece's position, so steps s and s + 4 are 256 bytes apart.
  // V: transposing reads; in dim tile q the lane points at dims 16 q + 4 (lane % 4) .. + 3 of token
  // 4 kg + lane % 16 / 4 and receives tokens 4 kg .. + 3 of dim 16 q + lane % 16.
  constexpr int kKBases = kSteps < 4 ? kSteps : 4, kVBases = kDimTiles < 8 ? kDimTiles : 8;
  int k_byte[kKBases], v_byte[kVBases];
#pragma unroll
  for (int s = 0; s < kKBases; ++s) k_byte[s] = j * kRowBytes + 16 * ((4 * s + kg) ^ stream_swz<kD>(j));
  {
    const int row = 4 * kg + (lane % 16) / 4;
#pragma unroll
    for (int q = 0; q < kVBases; ++q)
      v_byte[q] = kTileBytes + row * kRowBytes + 16 * ((2 * q + (lane % 4) / 2) ^ stream_swz<kD>(row)) + 8 * (lane % 2);
  }
  const uint32_t lds_base = __builtin_amdgcn_readfirstlane(lds_address(lds));
  const uint32_t wave_ring = lds_base + (uint32_t)wave * Sh::kWaveRingBytes;
  va_u32x4* q_stage = smem + Sh::kRingBytes / 16;

  float m_run[kB], l_run[kB];  // running maximum (log2 units) and row sum, of this wave's tokens
  va_f32x4 o[kB][kDimTiles];
#pragma unroll
  for (int b = 0; b < kB; ++b) {
    m_run[b] = kNegBig;
    l_run[b] = 0.f;
#pragma unroll
    for (int t = 0; t < kDimTiles; ++t) o[b][t] = va_f32x4{0.f, 0.f, 0.f, 0.f};
  }

  for (int li = 0; li < item[0][VA_I_N_LINKS]; ++li) {
    // the first link travels with the item
    int link[VA_LINK_WORDS];
    if (li == 0) {
#pragma unroll
      for (int w = 0; w < VA_LINK_WORDS; ++w) link[w] = item[0][VA_I_LINK0 + w];
    } else {
      const __attribute__((address_space(4))) va_i32x4* words = (const __attribute__((address_space(4))) va_i32x4*)(
          a.links + (long long)(item[0][VA_I_LINK_BEGIN] + li) * VA_LINK_WORDS);
#pragma unroll
      for (int w = 0; w < VA_LINK_WORDS / 4; ++w) {
        const va_i32x4 x = words[w];
        link[4 * w + 0] = x[0];
        link[4 * w + 1] = x[1];
        link[4 * w + 2] = x[2];
        link[4 * w + 3] = x[3];
      }
    }
    const int lflags = link[VA_L_FLAGS];
    const int kv_begin = link[VA_L_KV_BEGIN];
    const int tok_begin = link[VA_L_TOK_BEGIN];
    const int tok_end = link[VA_L_TOK_END];
    const int causal_base = link[VA_L_CAUSAL_BASE];
    const bool slots = lflags & VA_LINK_SLOTS;
    // no other query tile reads these rows: they are requested as lines to evict first
    const bool read_once = lflags & VA_LINK_ONCE;
    // a 16-token tile lies inside one page: one wave-uniform page read per tile
    const bool uniform_pages = !kGather && !slots && pow2_pages && page_fits && P >= 16 && (tok_begin % 16 == 0);

    const int t_stop = min(tok_end, causal_base + item[0][VA_I_N_Q]);  // tokens any row of the tile sees
    const int t_row = min(tok_end, causal_base + row_iq + 1);          // tokens this lane's row sees (partners are not causal)
    const int t_last = t_stop - 1;
    const int n_all = t_stop > tok_begin ? (t_stop - tok_begin + kStreamTok - 1) / kStreamTok : 0;
    const int n_tiles = n_all > wave ? (n_all - wave + kStreamWaves - 1) / kStreamWaves : 0;  // this wave's
    auto first_token = [&](int i) __attribute__((always_inline)) {  // of this wave's tile i
      return tok_begin + (i * kStreamWaves + wave) * kStreamTok;
    };

    // page of tile i (uniform page tables).  Read through the constant address space: the table is
    // read-only for the kernel, and this keeps the lookup a scalar load (a vector load would have
    // to be waited for together with every tile load in flight).
    auto page_of = [&](int i) __attribute__((always_inline)) {
      return ((const __attribute__((address_space(4))) int32_t*)a.kv_indices)[kv_begin + (first_token(i) >> p_shift)];
    };
    // kGather.  Looked up by the lanes in front of each request, the entries cost a trip to memory per tile and
    // the wait for it drains the ring.  So they travel like the tiles do: a load per tile brings its sixteen entries
    // to LDS, sent kBuffers iterations before the tile is requested, just ahead of the tile that the wait in front of
    // that request is for.
    const int g_shift = slots ? 0 : p_shift, g_mask = slots ? 0 : P - 1;
    auto token_of = [&](int i, int row) __attribute__((always_inline)) { return min(first_token(i) + row, t_last); };
    auto slot_of = [&](int entry, int t) __attribute__((always_inline)) { return (entry << g_shift) + (t & g_mask); };
    const uint32_t index_lds = lds_base + Sh::kIndexOffset + (uint32_t)wave * Sh::kIndexBytes;
    const int32_t* index = (const int32_t*)(lds + Sh::kIndexOffset + wave * Sh::kIndexBytes);
    auto request_entries = [&](int i) __attribute__((always_inline)) {
      if (lane < kStreamTok)
        load_word_to_lds(a.kv_indices + kv_begin + (token_of(i, lane) >> g_shift),
                         index_lds + (uint32_t)(i % kIndexSlots) * (kStreamTok * 4));
    };
    // Request tile i of this wave into buffer i % kBuffers of its ring.  Rows past the visible range re-read
    // the last visible token (their scores are masked).  (The kinds of page table and of cache policy are told apart
    // here, by scalar branches: with a tile loop for each the kernel is three times as long, and a launch of few
    // tokens waits for its instructions.)
    auto issue_offsets = [&](const char* k_base, const char* v_base, const uint32_t* off, uint32_t dst, auto once) __attribute__((always_inline)) {
#pragma unroll
      for (int u = 0; u < kLoads; u += kLoadGroup)
        load_group_to_lds<kLoadGroup, decltype(once)::value>(k_base, off + u, dst + u * 1024);
#pragma unroll
      for (int u = 0; u < kLoads; u += kLoadGroup)
        load_group_to_lds<kLoadGroup, decltype(once)::value>(v_base, off + u, dst + kTileBytes + u * 1024);
    };
    auto issue_rows = [&](const int* slot, uint32_t dst, auto once) __attribute__((always_inline)) {
      unsigned long long at[kLoads];
#pragma unroll
      for (int u = 0; u < kLoads; ++u)
        at[u] = (unsigned long long)kp + (unsigned long long)(uint32_t)slot[u] * (uint32_t)row_bytes +
                16 * ((lane % kChunks) ^ stream_swz<kD>(u * Sh::kRowsPerLoad + ld_row0));
#pragma unroll
      for (int u = 0; u < kLoads; u += kLoadGroup)
        load_rows_to_lds<kLoadGroup, decltype(once)::value>(at + u, dst + u * 1024);
#pragma unroll
      for (int u = 0; u < kLoads; ++u) at[u] += (unsigned long long)vp - (unsigned long long)kp;
#pragma unroll
      for (int u = 0; u < kLoads; u += kLoadGroup)
        load_rows_to_lds<kLoadGroup, decltype(once)::value>(at + u, dst + kTileBytes + u * 1024);
    };
    auto issue = [&](int i, int page, const int* slot) __attribute__((always_inline)) {
      const uint32_t dst = wave_ring + (uint32_t)(i % kBuffers) * (2 * kTileBytes);
      const int t0 = first_token(i);
      if constexpr (kGather) {
        if (read_once) {
          issue_rows(slot, dst, std::true_type{});
        } else {
          issue_rows(slot, dst, std::false_type{});
        }
      } else if (uniform_pages) {
        const unsigned long long base =
            (unsigned long long)(uint32_t)page * page_bytes + (uint32_t)(t0 & (P - 1)) * (uint32_t)row_bytes - kLoadBias;
        const char *k_base = (const char*)kp + base, *v_base = (const char*)vp + base;
        const int last_row = t_last - t0;
        if (last_row < kStreamTok - 1) {
          uint32_t off[kLoads];
#pragma unroll
          for (int u = 0; u < kLoads; ++u)
            off[u] = ld_off[u] - (uint32_t)(max(0, u * Sh::kRowsPerLoad + ld_row0 - last_row) * row_bytes);
          issue_offsets(k_base, v_base, off, dst, std::false_type{});
        } else if (read_once) {
          issue_offsets(k_base, v_base, ld_off, dst, std::true_type{});
        } else {
          issue_offsets(k_base, v_base, ld_off, dst, std::false_type{});
        }
      } else {  // each lane looks a token up, and the rows go round the lanes
        const int mine = (int)kv_slot(a.kv_indices, kv_begin, min(t0 + lane % kStreamTok, t_last), P, slots);
        int each[kLoads];
#pragma unroll
        for (int u = 0; u < kLoads; ++u) each[u] = __shfl(mine, u * Sh::kRowsPerLoad + ld_row0, kWave);
        issue_rows(each, dst, std::false_type{});
      }
    };

    // ---- set-up: first tiles on their way, then the query tile ----
    // (no barrier: a wave's ring and index entries are its own, and it has read the previous link's tiles)
    if constexpr (kGather) {
      wave_wait<0>();  // entries requested past the end of the previous link
      if (n_tiles > 0) {
        int first[kBuffers][kLoads];
#pragma unroll
        for (int i = 0; i < kBuffers; ++i)
#pragma unroll
          for (int u = 0; u < kLoads; ++u) {
            const int t = token_of(i, u * Sh::kRowsPerLoad + ld_row0);
            first[i][u] = slot_of(a.kv_indices[kv_begin + (t >> g_shift)], t);
          }
#pragma unroll
        for (int i = kBuffers; i < 2 * kBuffers; ++i) request_entries(i);
#pragma unroll
        for (int i = 0; i < kBuffers; ++i)
          if (i < n_tiles) issue(i, 0, first[i]);
      }
    } else {
      int page[kBuffers];
#pragma unroll
      for (int i = 0; i < kBuffers; ++i) page[i] = uniform_pages && i < n_tiles ? page_of(i) : 0;
#pragma unroll
      for (int i = 0; i < kBuffers; ++i)
        if (i < n_tiles) issue(i, page[i], nullptr);
    }

    if (li > 0) ring_barrier<kAnyInFlight>();  // every wave has read the previous link's query tile
    // the query rows, rotated, in LDS, swizzled like a K tile
    for (int idx = tid; idx < kB * 16 * (kChunks / 2); idx += kStreamThreads) {  // two pieces per step
      const int R = idx / (kChunks / 2), x = idx - R * (kChunks / 2);
      const int jr = R % 16, iq = jr / G, g = jr - iq * G;
      int n_q = item[0][VA_I_N_Q], qref = link[VA_L_QREF];
#pragma unroll
      for (int b = 1; b < kB; ++b) {
        if (R / 16 == b) {
          n_q = item[b][VA_I_N_Q];
          qref = item[b][VA_I_LINK0 + VA_L_QREF];
        }
      }
      int c0 = 2 * x, c1 = 2 * x + 1;
      uint4 p0 = make_uint4(0, 0, 0, 0), p1 = p0;
      if (iq < n_q) {
        // indirect links find sub-row and query row side by side in the plan; direct ones ask sub_worker
        const bool indirect = lflags & VA_LINK_INDIRECT;
        const int subrow = indirect ? a.qrefs[qref + iq] : qref + iq;
        const long long src_row = indirect ? (long long)a.qref_rows[qref + iq] : a.sub_worker[subrow];
        const S* qh = (const S*)a.q + src_row * a.q_row_stride + (long long)(hk * G + g) * kD;
        const Pos3 p = load_pos(a.sub_loc, a.sub_loc_axis_stride, subrow);
        if (a.rope.mode == VA_ROPE_TABLE && x < a.rope.rotary_dim / 16) {
          // the table entries of the unit in four 16-byte loads
          TableQueryUnit<E> unit;
          unit.load(a.rope, qh, x, p);
          unit.finish(a.rope, p, p0, p1);
          c0 = x;
          c1 = x + a.rope.rotary_dim / 16;
        } else {
          rotated_query_unit<E>(a.rope, qh, x, p, c0, c1, p0, p1);
        }
      }
      q_stage[R * kChunks + (c0 ^ stream_swz<kD>(jr))] = va_u32x4{p0.x, p0.y, p0.z, p0.w};
      q_stage[R * kChunks + (c1 ^ stream_swz<kD>(jr))] = va_u32x4{p1.x, p1.y, p1.z, p1.w};
    }
    ring_barrier<kAnyInFlight>();
    // B operands: row j of a block, dims [32s + 8kg, +8).  Up to two blocks hold them in registers; four read them anew
    // for every tile (the accumulators fill the registers, and the LDS has the time: a tile of D = 256 is 48 KB of
    // reads, 400 cycles, where memory delivers one in 1400)
    constexpr bool kKeepQuery = kB <= 2;
    auto read_query = [&](int b, int s) __attribute__((always_inline)) {
      return *(const va_u32x4*)((const char*)q_stage + b * 16 * kRowBytes + k_byte[s % 4] + 256 * (s / 4));
    };
    va_u32x4 qf[kKeepQuery ? kB : 1][kSteps];
    if constexpr (kKeepQuery) {
#pragma unroll
      for (int b = 0; b < kB; ++b)
#pragma unroll
        for (int s = 0; s < kSteps; ++s) qf[b][s] = read_query(b, s);
#pragma unroll
      for (int b = 0; b < kB; ++b)
#pragma unroll
        for (int s = 0; s < kSteps; ++s) asm volatile("" : "+v"(qf[b][s]));
    }

    // ---- the tile loop ----
    {
      int next_page = uniform_pages && kBuffers < n_tiles ? page_of(kBuffers) : 0;
      for (int i = 0; i < n_tiles; ++i) {
        // The tile has landed once at most the loads of the kBuffers - 1 tiles requested after it are outstanding.
        if (i + kBuffers - 1 < n_tiles) {
          constexpr int kNewer = (kBuffers - 1) * 2 * kLoads;
          wave_wait<(kNewer < kAnyInFlight ? kNewer : kAnyInFlight - 1)>();
        } else {
          wave_wait<0>();
        }
        const bool refill = i + kBuffers < n_tiles;
        // (waited for here, where nothing else is outstanding on its counter: behind the reads of K it would have to
        // be waited for together with all of them)
        if constexpr (!kGather) asm volatile("" ::"s"(next_page));
        const char* kt = lds + wave * Sh::kWaveRingBytes + (i % kBuffers) * (2 * kTileBytes);
        const uint32_t tile_lds = wave_ring + (uint32_t)(i % kBuffers) * (2 * kTileBytes);
        int next_rows[kLoads];  // gather: entries, then rows, of the tile requested below
#pragma unroll
        for (int u = 0; u < kLoads; ++u)
          next_rows[u] = kGather ? index[((i + kBuffers) % kIndexSlots) * kStreamTok + u * Sh::kRowsPerLoad + ld_row0] : 0;
        // scores: S^T = K . Q^T; lane (j, kg) supplies dims [32s + 8kg, +8) of token j
        // (every K fragment is requested before the first product, the first V fragments behind them)
        va_u32x4 kfr[kSteps];
        va_u32x2 vfr[kDimTiles];
        auto read_v = [&](int q) __attribute__((always_inline)) {
          vfr[q] = lds_read_tr16(tile_lds + v_byte[q % kVBases] + 256 * (q / kVBases));
        };
        constexpr int kVFirst = kDimTiles < 6 ? kDimTiles : 6;
#pragma unroll
        for (int s = 0; s < kSteps; ++s) kfr[s] = *(const va_u32x4*)(kt + k_byte[s % 4] + 256 * (s / 4));
#pragma unroll
        for (int q = 0; q < kVFirst; ++q) read_v(q);
        __builtin_amdgcn_sched_barrier(0);
        va_f32x4 sc[kB];
#pragma unroll
        for (int s = 0; s < kSteps; ++s)
#pragma unroll
          for (int b = 0; b < kB; ++b) {
            va_u32x4 query;
            if constexpr (kKeepQuery) query = qf[b][s]; else query = read_query(b, s);
            sc[b] = Mma<E>::run(kfr[s], query, s == 0 ? va_f32x4{0.f, 0.f, 0.f, 0.f} : sc[b]);
          }
#pragma unroll
        for (int q = kVFirst; q < kDimTiles; ++q) read_v(q);
        __builtin_amdgcn_sched_barrier(0);
        // the buffer is refilled as soon as its tile is in registers
        if (refill) {
          asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
          if constexpr (kGather) {
#pragma unroll
            for (int u = 0; u < kLoads; ++u)
              next_rows[u] = slot_of(next_rows[u], token_of(i + kBuffers, u * Sh::kRowsPerLoad + ld_row0));
            request_entries(i + 2 * kBuffers);
          }
          issue(i + kBuffers, next_page, next_rows);
          if (uniform_pages && i + 1 + kBuffers < n_tiles) next_page = page_of(i + 1 + kBuffers);
        }
        __builtin_amdgcn_sched_barrier(0);

        // Online softmax; this lane holds tokens 4 kg + r of row j.  The accumulators are rescaled only in tiles that
        // raise a maximum.  (Raising it by leaps only, as the wide kernel does, would spare most of these -- but the
        // weight of a row's largest score is then no longer exactly 1, and is rounded: error against 64-bit attention
        // 2.03e-3 -> 2.25e-3, with scores three times as large 1.69e-3 -> 2.2e-3, 16 requests of 100..8000 tokens in bf16.)
        const int t0 = first_token(i);
        float most[kB];
        bool raise = false;
#pragma unroll
        for (int b = 0; b < kB; ++b) {
          most[b] = -INFINITY;
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float v = (t0 + 4 * kg + r) < t_row ? sc[b][r] * a.scale_log2 : -INFINITY;
            sc[b][r] = v;
            most[b] = fmaxf(most[b], v);
          }
          raise = raise || most[b] > m_run[b];
        }
        if (__any(raise)) {
#pragma unroll
          for (int b = 0; b < kB; ++b) {
            const float m_new = fmaxf(m_run[b], max_over_contraction_groups(most[b]));
            // (the bare instruction: results below 2^-126 become 0 instead of denormal)
            const float alpha = __builtin_amdgcn_exp2f(m_run[b] - m_new);
            m_run[b] = m_new;
            l_run[b] *= alpha;
#pragma unroll
            for (int t = 0; t < kDimTiles; ++t) o[b][t] *= alpha;
          }
        }
        va_u32x2 pf[kB];
#pragma unroll
        for (int b = 0; b < kB; ++b) {
          float pr[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) pr[r] = __builtin_amdgcn_exp2f(sc[b][r] - m_run[b]);
          l_run[b] += (pr[0] + pr[1]) + (pr[2] + pr[3]);
          pf[b] = va_u32x2{Mma<E>::pack(pr[0], pr[1]), Mma<E>::pack(pr[2], pr[3])};
        }

        // O^T += V^T . P^T
#pragma unroll
        for (int q = 0; q < kDimTiles; ++q)
#pragma unroll
          for (int b = 0; b < kB; ++b) o[b][q] = Mma<E>::run16(vfr[q], pf[b], o[b][q]);
      }
    }
  }

  // ---- the four waves' states are folded through LDS, block by block: o[q][r] is dim 16 q + 4 kg + r of row j ----
  wave_wait<0>();  // (index entries requested past the end)
#pragma unroll
  for (int b = 0; b < kB; ++b) {
    if (b > 0) __syncthreads();  // the block before has been read
    // row sums live spread over the four contraction groups
    l_run[b] += __shfl_xor(l_run[b], 16, kWave);
    l_run[b] += __shfl_xor(l_run[b], 32, kWave);
    {
      char* mine = lds + wave * Sh::kWaveRingBytes;
  #pragma unroll
      for (int q = 0; q < kDimTiles; ++q) *(va_f32x4*)(mine + j * Sh::kFoldRowBytes + 16 * kg + 64 * q) = o[b][q];
      if (kg == 0) *(float2*)(mine + 16 * Sh::kFoldRowBytes + 8 * j) = make_float2(m_run[b], l_run[b]);
    }
    __syncthreads();
    const int row = tid / 16, seg = tid % 16;
    const int iq = row / G, part_base = item[b][VA_I_PART_BASE];
    if (iq >= item[b][VA_I_N_Q]) continue;
    float weight[kStreamWaves], m = kNegBig, l = 0.f;
    {
      float2 state[kStreamWaves];
  #pragma unroll
      for (int w = 0; w < kStreamWaves; ++w) {
        state[w] = *(const float2*)(lds + w * Sh::kWaveRingBytes + 16 * Sh::kFoldRowBytes + 8 * row);
        m = fmaxf(m, state[w].x);
      }
  #pragma unroll
      for (int w = 0; w < kStreamWaves; ++w) {
        weight[w] = __builtin_amdgcn_exp2f(state[w].x - m);
        l += state[w].y * weight[w];
      }
    }
    const int hq = hk * G + row - iq * G;
    va_f32x4 sum[kD / 64];
  #pragma unroll
    for (int x = 0; x < kD / 64; ++x) {
      sum[x] = va_f32x4{0.f, 0.f, 0.f, 0.f};
  #pragma unroll
      for (int w = 0; w < kStreamWaves; ++w)
        sum[x] += *(const va_f32x4*)(lds + w * Sh::kWaveRingBytes + row * Sh::kFoldRowBytes + 16 * (seg + 16 * x)) * weight[w];
    }
    if (part_base < 0) {
      const int qref0 = item[b][VA_I_LINK0 + VA_L_QREF];
      const long long out_row = (item[b][VA_I_LINK0 + VA_L_FLAGS] & VA_LINK_INDIRECT) ? (long long)a.qref_rows[qref0 + iq]
                                                                                   : a.sub_worker[qref0 + iq];
      S* orow = (S*)a.out + (out_row * a.num_q_heads + hq) * (long long)kD;
      const float inv = l > 0.f ? 1.f / l : 0.f;
  #pragma unroll
      for (int x = 0; x < kD / 64; ++x)
        *(uint2*)(orow + 4 * (seg + 16 * x)) = make_uint2(Mma<E>::pack(sum[x][0] * inv, sum[x][1] * inv),
                                                         Mma<E>::pack(sum[x][2] * inv, sum[x][3] * inv));
      if (seg == 0 && a.lse) {
        const float lse2 = l > 0.f ? m + log2f(l) : -INFINITY;
        a.lse[out_row * a.num_q_heads + hq] = a.lse_base2 ? lse2 : lse2 * kLn2;
      }
    } else {
      const long long slot = (long long)(part_base + iq) * a.num_q_heads + hq;
      float* prow = a.part_acc + slot * kD;
  #pragma unroll
      for (int x = 0; x < kD / 64; ++x) *(va_f32x4*)(prow + 4 * (seg + 16 * x)) = sum[x];
      if (seg == 0) {
        a.part_ml[slot * 2 + 0] = m;
        a.part_ml[slot * 2 + 1] = l;
      }
    }
  }
}

// The item (and its partners) of workgroup `block` of the narrow items.
template <typename E, int kD, bool kGather>
__device__ __forceinline__ void stream_block(const AttnArgs& a, unsigned block) {
  const ItemHead where = item_and_head(block, a.num_kv_heads);
  int item[1][VA_ITEM_WORDS];
  load_item(a, where.item, item[0]);
  const int partners = item[0][VA_I_PARTNERS];
  // padding items keep the launch order aligned with the die round-robin; partners are served by the item before them
  if (item[0][VA_I_N_Q] == 0 || partners < 0) return;
  auto together = [&](auto blocks) __attribute__((always_inline)) {
    constexpr int kB = decltype(blocks)::value;
    int items[kB][VA_ITEM_WORDS];
#pragma unroll
    for (int b = 0; b < kB; ++b) load_item(a, where.item + 8 * min(b, partners), items[b]);
#pragma unroll
    for (int b = 1; b < kB; ++b)
      if (b > partners) items[b][VA_I_N_Q] = 0;
    stream_items<E, kD, kGather, kB>(a, items, where.head);
  };
  static_assert(VA_TOGETHER == 4 && VA_TOGETHER_SCATTERED == 2, "the tiles served together below");
  if (partners == 0) {
    stream_items<E, kD, kGather, 1>(a, item, where.head);
  } else if (kGather || partners == 1) {
    together(std::integral_constant<int, 2>{});
  } else if constexpr (!kGather) {
    together(std::integral_constant<int, 4>{});
  }
}

// The same where items are short: its workgroups serve a tile each, also one that a plan would have walk with others.
template <typename E, int kD, bool kGather>
__device__ __forceinline__ void stream_block_short(const AttnArgs& a, unsigned block) {
  const ItemHead where = item_and_head(block, a.num_kv_heads);
  int item[1][VA_ITEM_WORDS];
  load_item(a, where.item, item[0]);
  if (item[0][VA_I_N_Q] == 0) return;
  stream_items<E, kD, kGather, 1, true>(a, item, where.head);
}

}  // namespace va
