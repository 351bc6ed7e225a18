// Plan blob layout shared by the host planner and the kernels.
//
// A plan turns the sub-request tables of one launch into work items.  One work
// item is one workgroup per kv head: a tile of query rows walking a chain of
// KV ranges ("links").  Each link is a token range of one sub-request; the
// query tile is re-rotated at every link start because each sub-request has
// its own rotation offset per row.
#pragma once
#include <stdint.h>

#define VA_PLAN_MAGIC 0x56415031  // "VAP1"
#define VA_PLAN_HEADER_WORDS 24
#define VA_ITEM_WORDS 16
#define VA_LINK_WORDS 8

// header word indices
enum {
  VA_H_MAGIC = 0,
  VA_H_KERNEL,
  VA_H_Q_TILE,
  VA_H_KV_CHUNK,
  VA_H_N_ITEMS,
  VA_H_N_LINKS,
  VA_H_N_QREFS,
  VA_H_N_PARTIALS,
  VA_H_N_ROW_PARTS,
  VA_H_N_ROWS,
  VA_H_OFF_ITEMS,
  VA_H_OFF_LINKS,
  VA_H_OFF_QREFS,
  VA_H_OFF_ROW_INDPTR,
  VA_H_OFF_ROW_IDS,
  VA_H_OFF_ROW_FLAGS,
  VA_H_N_EMPTY_ROWS,   // rows no sub-request serves
  VA_H_N_SUBROWS,
  VA_H_N_WIDE,     // items [0, n_wide) are wide tiles, the rest narrow
  VA_H_WIDE_TILE,
  VA_H_OFF_QREF_ROWS,  // parallel to qrefs: the query/output row of each entry (sub_worker[qrefs[k]])
  VA_H_N_WIDE_SLOTS,   // workgroups per kv head of the wide launch (a multiple of 8)
  VA_H_OFF_WIDE_SLOTS, // [n_wide_slots + 1]: slot s runs the wide items [indptr[s], indptr[s + 1]) one after the other
  VA_H_MERGE_WAVES,    // merge launch: 4, 8 or 16 = waves of a workgroup per (row, q head); 1 = the kernel for many
                       // rows, a workgroup per row of few states (its own waves have nothing to do with the word)
};

// item word indices
enum {
  VA_I_LINK_BEGIN = 0,
  VA_I_N_LINKS,
  VA_I_N_Q,        // query rows in the tile
  VA_I_PART_BASE,  // first partial slot (one per query row), or -1: write `out` directly
  VA_I_TOKENS,     // KV tokens the item walks (scheduling weight)
  VA_I_KIND,       // 1: wide tile (more rows than the streaming kernel's tile)
  VA_I_PARTNERS,   // narrow tiles that walk the same tokens: the first of up to VA_TOGETHER of them holds how many
                   // follow at the next turns of its die (8 items apart) and its workgroup serves them all; they hold -1
  VA_I_LINK0 = 8,  // words 8..15: a copy of the item's first link, so that a kernel finds it with the
                   // same load as the item (one level less in the chain of dependent loads at its start)
};

// narrow tiles of the matrix-core path that one workgroup serves: fewer over scattered rows, whose index entries share
// the LDS with the query rows
#define VA_TOGETHER 4
#define VA_TOGETHER_SCATTERED 2

// Flags beside the chunk in its header word (a multiple of 64; 0 in plans of fixed capacity).
// Narrow items of a launch of their own that are short: their set-up and fold take as long as their walk, so several
// workgroups share a CU and serve a tile each (attn_stream_short_kernel, whose workgroups take no notice of VA_I_PARTNERS).
// 64 requests over 64 shared tokens and one or two private blocks, us a layer, in the kernel before independent waves / in
// the ordinary kernel / now: blocks of 300..900, 16 q / 4 kv heads of 256 dims 48.9 / 60.3 / 47.1, 32 / 8 of 128
// 51.7 / 53.6 / 49.9, 64 / 16 of 64 61.3 / 61.9 / 50.9; of 100..400 26.9 / 31.6 / 24.8, 28.4 / 29.4 / 26.2, 36.5 / 40.1 / 28.0.
#define VA_CHUNK_SHORT_ITEMS 1
// Wide and narrow items get a launch each (one launch serves both otherwise).  In a plan of fixed capacity a matter of the
// capacity and the shape alone.
#define VA_CHUNK_APART 2

// link word indices
enum {
  VA_L_KV_BEGIN = 0,  // first entry of the sub-request's page (or slot) list in kv_indices
  VA_L_TOK_BEGIN,     // token range within the sub-request
  VA_L_TOK_END,
  VA_L_QREF,          // base sub-row id, or offset into qrefs when VA_LINK_INDIRECT
  VA_L_CAUSAL_BASE,   // token t is visible to tile row i iff t <= causal_base + i
  VA_L_FLAGS,
};

#define VA_LINK_INDIRECT 1  // sub-row of tile row i is qrefs[qref + i], else qref + i
#define VA_LINK_SLOTS 2     // kv_indices entries are token slots (page size 1)
#define VA_LINK_ONCE 4      // no other query tile of the launch reads this token range (per kv head the rows are
                            // fetched exactly once): the streaming kernel requests them non-temporally

#define VA_NO_CAUSAL 0x3fffffff

// row flags
#define VA_ROW_DIRECT 1  // an item writes this row's output itself
#define VA_ROW_EMPTY 2   // nothing serves the row: merge kernel writes zeros
