// Which grouped GEMMs an expert call runs: the few-rows ones (afd_gemm_rows.hip), the large-tile
// ones (afd_gemm_mx.hip, afd_gemm_fp8.hip, afd_gemm_a16.hip), or whichever the router's counts call
// for. The results are the same bits, so the choice is one of time alone. Host code,
// but for rows_few, which the router runs on the GPU.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/afd.h"

namespace afd {

// Pairs per local expert up to which the few-rows GEMMs run. The line lies where the large tiles
// catch up (large tiles -> few rows): 64 FP8 experts, all local, hidden 4096, inter 1536, top-8: at
// 37 pairs per expert 278 -> 234 us (uniform routing) and 328 -> 283 (Zipf 1.2), at 64 285 -> 339
// and 343 -> 346; MXFP4 experts, hidden 4096, inter 2048: at 32 200 -> 189 us (uniform) and
// 236 -> 222 (Zipf 1.2), at 48 210 -> 225 and 245 -> 259. With bf16 activations they catch up a
// little later: MXFP4 at 40 250 -> 235 and 369 -> 253, at 65 300 -> 319 and 386 -> 320; FP8 at 40
// 275 -> 249 and 322 -> 276, at 65 318 -> 347 and 347 -> 344; and so they do in narrow layers.
constexpr int kFewRowsPerExpert = 40;
// A call knows its own pairs, not how many of them are local: with at most 40 pairs per local
// expert if all were, the few-rows GEMMs run. An MXFP4 rank that owns a quarter of a model's experts
// has the line at four times as many tokens, so nearly up to there, 35 expected pairs per local
// expert, both forms are launched and the router's count of local pairs decides between them: 64 of
// 256 experts, 512 tokens 233 -> 185 us, 750 tokens 237 -> 207 (Zipf 1.2), 194 -> 179 (uniform), with
// bf16 activations 512 tokens 334 -> 219, 1024 362 -> 274. Where the large tiles then run after all,
// the two launches that return at once cost 2 to 5 us (2% at 1200 tokens), which is why this ends a
// little before 40; and a rank that owns all experts, which would always pay them (64 of 64, 560
// tokens 209 -> 215 us; 32 of 32 of hidden 2048, 800 tokens 101 -> 105), never launches both for
// this. A call whose descriptor holds the token count (a graph of that capacity) does: it may have
// few tokens (64 of 64, hidden 4096, inter 1024, room for 500: 60 tokens 125 -> 91 us), and so does a
// call that doesn't say the model's experts: missing the few rows costs more than launching them.
// Measured up to a quarter, hence the second bound. FP8 experts gain nothing there (32 of 128
// experts, 512 tokens: 68 -> 74 us) and take the large tiles.
constexpr int kGatedRowsPerModelExpert = 35, kGatedRowsPerExpert = 140;
// Groups of 32 rows run three workgroups a CU instead of two, groups of 64 read the weights of an
// expert of 33 to 64 rows once: 32 while few experts have more rows. At most 16 pairs per expert:
// -6 to +0.6% over the four formats and two routings (64 FP8 experts, bf16 activations, 8 tokens
// 121 -> 117 us; 32 local of hidden 2048, 64 tokens 46 -> 43); at 25 219 -> 236 us (FP8 experts, all
// local), at 37 224 -> 353.
constexpr int kNarrowRowsPerExpert = 16;
// Routing may put the pairs on a few of the experts, so that these have many row groups each,
// which read the weights again (from the caches) and fill the chip with work that the large tiles
// do better. Up to this many pairs (in groups of 64 and of 32 rows) the few-rows GEMMs run whatever
// the routing is: over 8 to 48 hot experts they were at most 11% slower than the large tiles (half of
// 64 FP8 experts hot, fp8 activations, 174 -> 193 us) and up to 60% faster. Above, the router's counts
// decide. There it was (large tiles -> few rows): 128 FP8 experts, 640 tokens, 32 hot 224 -> 306 us;
// 256, 510 tokens, 32 hot 213 -> 303; 128 MXFP4 experts, 640 tokens, 64 hot 211 -> 280; and 256 FP8
// experts, 510 tokens, uniform 1340 -> 1008 (hidden 4096, inter 2048, top-8). The two launches that
// return at once cost 2 to 6 us: 256 MXFP4 experts, hidden 2048, inter 1024, 800 tokens, uniform 232
// (large tiles) and 192 (few rows alone) -> 198; 128 of hidden 4096, inter 2048, 640 tokens, 64 hot
// 218 (large tiles) -> 224.
constexpr int kFewPairs = 2560, kFewPairsNarrow = 2048;
// What the counts have to be for the few-rows GEMMs to run: the row groups of gate_up make at most
// two rounds of the workgroups that the chip holds, or there are at most 3/2 groups per expert with
// rows, so the reading of each expert's weights bounds the call. Over 128 and 256 experts, hidden 4096
// / inter 2048 and 2048 / 1024, the four formats, 480 to 1280 tokens and 8 to 128 hot experts or
// Zipf routing this takes the faster form but for 0.4% on average, 12% at worst (64 of 128 MXFP4
// experts hot, 204 -> 228 us).
constexpr int kRowsCus = 256;  // compute units
constexpr int kRowsRounds = 2;

enum RowsForm { kRowsLarge = 0, kRowsFew = 1, kRowsBoth = 2 };
// kRowsBoth: both are launched, and all but the form that the router chose return at once.
struct RowsPlan {
  int32_t form;         // RowsForm
  int32_t group_shift;  // the few-rows GEMMs' groups have 1 << group_shift rows
  int32_t max_pairs;    // kRowsBoth: bounds of rows_few
  int32_t max_groups;
  int32_t grid_groups;  // the few-rows GEMMs are launched for so many row groups, the most there can be
};

// The plan of a call of n tokens; capacity: of at most n, the job's descriptor holds how many.
inline RowsPlan rows_plan(const afd_moe_cfg& cfg, int64_t n, bool capacity) {
  const int64_t pairs = n * cfg.topk, local = cfg.num_local;
  const int64_t experts = cfg.tile_walk >> AFD_NUM_EXPERTS_SHIFT;  // the model's; 0: not said
  RowsPlan p;
  const bool narrow = pairs <= kNarrowRowsPerExpert * local;
  p.group_shift = narrow ? 5 : 6;
  p.max_pairs = static_cast<int32_t>(kFewRowsPerExpert * local);
  p.max_groups = kRowsRounds * (narrow ? 3 : 2) * kRowsCus / (2 * cfg.inter / 256);
  // The counts say large tiles only if 2 groups > 3 active; with groups <= active + pairs / rows that
  // takes more than max_groups <= groups < 3 pairs / rows.
  const bool always_few = 3 * pairs <= int64_t(p.max_groups) << p.group_shift;
  if (pairs <= kFewRowsPerExpert * local)
    p.form = always_few || pairs <= (narrow ? kFewPairsNarrow : kFewPairs) ? kRowsFew : kRowsBoth;
  else
    p.form = cfg.weight_fmt == AFD_W_MXFP4 && pairs <= kGatedRowsPerExpert * local &&
                     (capacity || experts == 0 || pairs <= kGatedRowsPerModelExpert * experts)
                 ? kRowsBoth
                 : kRowsLarge;
  // groups of the pairs that the few-rows GEMMs run for: at most one per pair, and one per expert
  // plus one per full group
  const int64_t most = pairs < p.max_pairs ? pairs : p.max_pairs, groups = local + (most >> p.group_shift);
  p.grid_groups = static_cast<int32_t>(most < groups ? most : groups);
  return p;
}

// The router's choice for a kRowsBoth call: `pairs` local pairs in `groups` row groups of `active`
// experts.
__host__ __device__ __forceinline__ bool rows_few(const RowsPlan& p, int pairs, int groups, int active) {
  return pairs <= p.max_pairs && (groups <= p.max_groups || 2 * groups <= 3 * active);
}

}  // namespace afd
