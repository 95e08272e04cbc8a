// Contract between the runtime's MIR executor and the per-rule join kernels
// that the Python emitter generates for a program.
//
// A pipeline (one `execute-pipeline` MIR node) runs as:
//   root   one thread per distinct key of the driver root source: look the
//          key up in every root source, record the ranges, and size the
//          first nested level's iteration space (key_work);
//   then the per-key work is flattened into one global item space (an
//   exclusive scan of key_work) cut into slices -- `grain` items each, or,
//   after a weigh launch, of about equal level-2 cost -- that persistent
//   waves pull from per-XCD counters, so a slice may span many small keys
//   or a fraction of one huge key.  The traversal runs in one of these modes:
//   direct (3)  the rule emits exactly one tuple per item (last level is a
//               filter-free cartesian product or scan): tuple i goes to row
//               base+i of NEW, one pass, no counting;
//   fused  (2)  one pass; each slice appends its tuples to segments of a
//               staging buffer (bump-allocated with an atomic) and logs
//               (slice, local offset, source, count) records; after the
//               scan of the per-slice counts a gather kernel moves every
//               segment to its slice's offset in NEW;
//   count  (0)  counts only (count-only rules; fallback when staging
//               overflows);
//   write  (1)  re-runs the traversal writing at the scanned offsets;
//   probe  (5)  traverses like count but writes nothing except the number
//               of searches, root-map lookups and bitmap tests it made
//               (probe_ctr); run once, untimed, to report join probes;
//   weigh  (4)  rules with two or more nested levels: writes each level-1
//               item's cost (its level-2 candidates + SRD_ITEM_COST) so the
//               runtime can cut slices of equal cost instead of equal item
//               counts (slice_start); a few items of two hub keys can carry
//               more level-2 work than whole slices of ordinary ones.
// Output order depends only on the item order, never on which wave ran a
// slice, so every mode yields the same NEW rows in the same order.
//
// Reference counterpart: the JitRunner_<rule> phases setup / launch_count /
// scan_and_resize / launch_materialize of
// src/srdatalog/codegen/jit/complete_runner.py:929-1523 and the block-group
// work partition of complete_runner.py:377-736.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "srd_device.h"

#define SRD_MAX_VIEWS 8
#define SRD_MAX_COLS 8
#define SRD_MAX_DESTS 2

enum SrdVersion : uint32_t { SRD_FULL = 0, SRD_DELTA = 1, SRD_NEW = 2 };
enum SrdRootKind : uint32_t { SRD_ROOT_JOIN = 0, SRD_ROOT_SCAN = 1 };

struct SrdViewSpec {
  const char* rel;
  uint32_t ncols;
  uint32_t cols[SRD_MAX_COLS];  // index column order
  uint32_t ver;                 // SrdVersion
  uint32_t want_bitmaps;        // a nested level searches this two-column view at depth 1
  uint32_t want_root_pos;       // a nested level looks keys up among this view's root values
};

struct SrdDestSpec {
  const char* rel;
  uint32_t arity;
  uint32_t cols[SRD_MAX_COLS];  // dedup index (column order written to NEW)
};

struct SrdViews {
  srd::IndexView v[SRD_MAX_VIEWS];
};

struct SrdOut {
  uint32_t* cols;   // NEW buffer, column c at cols + c*stride
  uint64_t stride;
  uint64_t base;    // first row this launch writes
};

struct SrdDyn;

struct SrdLaunchArgs {
  SrdViews views;
  uint32_t n_root;             // driver root keys (join) or 1 (scan)
  uint32_t drv_view;           // view whose root_vals enumerate the keys
  uint32_t grain;              // level-1 items per slice
  uint32_t grid_blocks;        // persistent blocks for count / write
  uint64_t n_slices;           // ceil(total work / grain)
  uint64_t total_work;
  uint32_t* key_rng;           // per key: 2 u32 per root slot
  uint32_t* key_aux;           // per key: level-1 driver choice
  uint64_t* key_work;          // per key: level-1 item count
  uint64_t* work_start;        // exclusive scan of key_work, n_root+1 entries
  uint32_t* counts;            // per slice tuple count
  uint64_t* offsets;           // exclusive scan of counts
  uint32_t* work_ctr;          // SRD_XCDS slice counters, SRD_CTR_STRIDE words apart (zeroed per launch)
  SrdOut out[SRD_MAX_DESTS];
  // fused mode staging (column c of dest d at stage + (d*SRD_MAX_COLS + c)*stage_cap)
  uint32_t* stage;
  uint64_t stage_cap;          // tuples
  unsigned long long* stage_ctr;   // bump allocator (tuples)
  uint64_t* recs;              // 3 u64 per segment record
  uint64_t rec_cap;
  uint32_t* rec_ctr;
  uint32_t* overflow;          // set when staging or the record log ran out
  // cost-balanced slicing: slice s covers items [slice_start[s], slice_start[s+1])
  // (nullptr: [s*grain, min((s+1)*grain, total_work)))
  const uint64_t* slice_start;
  uint64_t* item_cost;         // weigh mode output, one entry per item
  uint64_t slice_lo;           // the launch takes slices [slice_lo, n_slices)
  uint32_t n_ranges;           // slice ranges, 1..SRD_XCDS (0 is taken as 1)
  uint32_t window_min;         // nested column joins narrow the driving range of items with
                               // at least this many candidates (0: never)
  // probe runs only (else nullptr): the root launch and the probe mode add
  // their lower/upper-bound searches, root-map lookups and bitmap tests
  unsigned long long* probe_ctr;
  // mark mode (6) only: the destination's NEW as a dense bitmap over its
  // key space, a tuple (v0 .. vk-1) in index order at bit
  // sum(v_c << mark_shift * (k-1-c)); mark_sum has a byte per block
  // of 2^18 keys, set to 1 when a bit of the block is set, so extraction
  // reads only marked blocks
  uint32_t* mark_bits;
  uint8_t* mark_sum;
  uint32_t mark_shift;
  // rules whose last level is a product marked row by row (srdj::prod_mark):
  // SrdPipelineExt::mark_prod, the root launch and the weigh mode price large
  // products in row steps and the mark mode walks them so (0: by tuples)
  uint32_t mark_prod;
  // device-sized mark launches: tuples derived, summed into SRD_ROW_CTRS
  // counters SRD_ROW_CTR_STRIDE words apart (nullptr: not counted)
  unsigned long long* mark_rows;
  // weighed mark launches of rules with mark_prod 2: slice s covers the cost
  // range [srd_cost_cut(s), srd_cost_cut(s+1)) of the items' cost prefix
  // (nullptr: whole items), slice_start[s] being the item that holds its first
  // unit; a large product is split by rows where a cut falls inside it
  const uint64_t* item_pref;
  uint64_t n_items;
  uint64_t cost_q, cost_rem;
  // device-sized launches (the *_dyn entry points) only: views, key and
  // slice counts and output bases are read from this device struct, which
  // kernels of the same iteration fill in, instead of the fields above
  const SrdDyn* dyn;
};

// Cost at which slice s of a launch of S slices over w cost units starts
// (q = w / S, rem = w % S).
__host__ __device__ inline uint64_t srd_cost_cut(uint64_t s, uint64_t q, uint64_t rem) {
  return s * q + (s < rem ? s : rem);
}

// Device-resident part of a device-sized launch.  skip != 0 turns every
// launch reading it into a no-op (an iteration after convergence, or one
// abandoned because a buffer would overflow).
struct SrdDyn {
  SrdViews views;
  uint64_t total_work;
  uint64_t n_slices;
  uint64_t out_base[SRD_MAX_DESTS];
  uint32_t n_root;
  uint32_t drv_view;
  uint32_t skip;
  uint32_t grain;               // items per slice, decided with n_slices
};

// Slices are split into SRD_XCDS contiguous ranges, one per XCD (workgroups
// are dispatched to the XCDs round-robin, so block b runs on XCD b % 8):
// the waves of one XCD work through neighbouring slices, whose keys (and
// their index ranges and bitmaps) then stay in that XCD's L2, and take
// slices of the other ranges once their own is done.
#define SRD_XCDS 8u
#define SRD_CTR_STRIDE 32u     // one 128-byte line per counter: atomics on one line serialise

#define SRD_ROW_CTRS 64u
#define SRD_ROW_CTR_STRIDE 16u // u64 words: a 128-byte line per counter

#define SRD_ITEM_COST 4u       // level-1 cost of an item, in level-2 candidates
// A product is marked row by row when it has at least this many tuples and
// its row steps, 64 lanes each, are no more than its tuples.
#define SRD_PROD_MIN 256u
// Two-source cartesian products at a nested last level with at least this
// many tuples, and a source of at least SRD_CART_TILE_DIM rows, are walked in
// register tiles (one 64-row tile per lane register, the other broadcast a
// row at a time) instead of the flattened per-tuple decode.
#ifndef SRD_CART_TILE_MIN
#define SRD_CART_TILE_MIN 1024u
#endif
#ifndef SRD_CART_TILE_DIM
#define SRD_CART_TILE_DIM 48u
#endif
#define SRD_BM_MIN 512u        // default shortest range given a heavy-key bitmap

#define SRD_SEG 2048u          // staging segment size (tuples)

// Items per uniform slice of a launch over `total` items: the rule's default
// (4096, or 256 with a nested level) once that gives every wave of the full
// grid (2048 blocks of 4) a slice, else an equal share of the items for
// each wave, in whole 64-item batches.  A wave walks its slice serially, a
// dozen dependent loads per batch, so with 4096 items a slice the 5,000 rows
// of a small relation ran on two waves: 83 us against 31 us for the load of
// 5,000 pairs, 254 us against 70 us for 260,000 pairs (21 and 22 us since waves
// own their first slices), and 133 us against
// 95 us (mean over the iterations) for the recursive join of the closure of
// 5,000 pairs over 1,000 vertices.
#define SRD_GRID_WAVES 8192u
// A launch whose products are marked row by row counts 64 units a step and
// folds a product's values anew in every slice that holds some of its rows:
// its slices hold at least SRD_PROD_GRAIN units.  Few slices leave a small
// launch's products to a few dozen waves, one after the other; many fold the
// same values again: sessions of the closure of 1,200 pairs over 400 vertices
// run in 1.32 / 1.11 / 1.02 / 0.96 ms with 1024 / 512 / 256 / 128, of 5,000
// pairs over 1,000 in 1.15 / 1.01 / 0.93 / 1.10, Andersen at 1/30 in 10.5 /
// 10.4 / 10.2 / 10.6.  Long closures of sparse graphs go on gaining below it:
// runs over 2,000 vertices and 4,000 pairs 2.42 / 1.97 / 1.71 / 1.61 ms, over
// 6,000 and 6,300 6.85 / 5.45 / 4.53 / 4.02.
#define SRD_PROD_GRAIN 256u
__host__ __device__ inline uint32_t srd_grain(uint64_t total, uint32_t dflt, uint32_t least = 64u) {
  if (dflt <= least) return dflt;
  const uint64_t share = (total + SRD_GRID_WAVES - 1) / SRD_GRID_WAVES;
  if (share >= dflt) return dflt;
  const uint32_t g = (uint32_t(share) + 63u) & ~63u;
  return g < least ? least : (g < dflt ? g : dflt);
}

typedef void (*SrdLaunchFn)(const SrdLaunchArgs* args, hipStream_t stream);

struct SrdPipelineDesc {
  const char* rule;
  uint32_t n_views;
  SrdViewSpec views[SRD_MAX_VIEWS];
  uint32_t root_kind;                // SrdRootKind
  uint32_t n_root_src;               // root sources (join) / 1 (scan)
  uint32_t root_view[SRD_MAX_VIEWS];
  uint32_t n_dest;
  SrdDestSpec dest[SRD_MAX_DESTS];
  uint32_t count_only;               // rule carries .with_count()
  uint32_t default_grain;
  uint32_t direct_ok;                // one tuple per level-1 item (mode 3 valid)
  SrdLaunchFn root;
  SrdLaunchFn count;
  SrdLaunchFn write;
  SrdLaunchFn fused;
  SrdLaunchFn direct;
  SrdLaunchFn weigh;                 // nullptr unless the rule has >= 2 nested levels
  // The rule writes its single destination's rows strictly increasing in
  // the destination's index order: every level is a column join binding the
  // next index column, so tuples come out in (root key, level 1, level 2 ...)
  // order with no repeats, in every mode.
  uint32_t sorted_output;
  SrdLaunchFn probe;                 // mode 5 (search counting)
  // device-sized variants (SrdLaunchArgs::dyn set; grid_blocks fixed);
  // nullptr outside recursive steps, and direct_dyn unless direct_ok
  SrdLaunchFn root_dyn;
  SrdLaunchFn count_dyn;
  SrdLaunchFn write_dyn;
  SrdLaunchFn direct_dyn;
  // mode 6: set the bit of every derived tuple in the destination's dense
  // bitmap instead of writing rows; nullptr unless the rule has a single
  // destination whose terms are all variables
  SrdLaunchFn mark;
};

// What a rule's mark mode can do beyond marking tuple by tuple, by rule name.
struct SrdPipelineExt {
  const char* rule;
  // large products of the rule's last level are walked row by row: 1 = the
  // product is the level under the root (its keys are the items), 2 = the
  // second level, whose items are weighed, 3 = a deeper one, 0 = no such level
  uint32_t mark_prod;
  SrdLaunchFn mark_dyn;   // device-sized mark mode; nullptr outside recursive steps
  // two-level rules whose product splits into a source that depends on the
  // level-1 variable and one (view uni_view, its column 1) that depends on
  // the root key alone: the pipeline that derives (root key, value of the
  // first), marked in a bitmap of its own and multiplied out by
  // union_products.  uni_minor: the first source's variable is the
  // destination's last column (else its row column); uni_row_col, uni_root_col:
  // index columns of the row variable and, or -1, of the root variable.
  const struct SrdPipelineDesc* uni;
  uint32_t uni_view, uni_minor, uni_row_col;
  int32_t uni_root_col;
  // the rule copies one relation: its row, in the destination's index order, is
  // the scanned index's row
  uint32_t copy;
};

#ifdef __cplusplus
extern "C" {
#endif

struct srd_engine;

// Engine entry points used by the generated extern "C" shim of a program.
// program_text: relation declarations followed by the MIR program in the
// reference's S-expression form.
struct srd_engine* srd_engine_create(const char* program_text, const SrdPipelineDesc* pipelines,
                                     uint32_t n_pipelines);
// The same with the rules' mark-mode extensions.
struct srd_engine* srd_engine_create_ext(const char* program_text, const SrdPipelineDesc* pipelines,
                                         uint32_t n_pipelines, const SrdPipelineExt* exts,
                                         uint32_t n_exts);
void srd_engine_destroy(struct srd_engine* e);
const char* srd_engine_last_error(struct srd_engine* e);

#ifdef __cplusplus
}
#endif
