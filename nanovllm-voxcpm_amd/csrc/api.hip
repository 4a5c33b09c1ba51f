// Entry points declared in include/mlora.h.  mlora_add_lora stands where the reference's backend
// method stands (nanovllm_voxcpm/lora.py:241-381); its slice grouping plan (lora.py:65-90, 195-239)
// and pointer tables (lora_ops/triton_ops/utils.py:15-116) have no counterpart: one launch takes a
// table of slices with their own widths, and pointers travel by value.
//
// C-ABI front door: argument checks, form selection, error text.
#include <stdarg.h>
#include <stdio.h>
#include <stdlib.h>

#include <mutex>

#include "common.h"
#include "launch.h"
#include "mlora_diag.h"

namespace mlora {

namespace {
thread_local char g_error[512] = "";
}

void set_error(const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_error, sizeof(g_error), fmt, ap);
  va_end(ap);
}

int check_launch(const char* what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    set_error("%s: launch failed: %s", what, hipGetErrorString(e));
    return static_cast<int>(e);
  }
  return 0;
}

namespace {
int g_knob_generation = 0;
}
int knob_generation() { return g_knob_generation; }

int env_int(const char* name, int fallback) {
  const char* v = getenv(name);
  if (!v || !*v) return fallback;
  return atoi(v);
}

}  // namespace mlora

using namespace mlora;

namespace {

// Both matrix-core forms step through K in units of 32.
bool mfma_supported(const MloraAddArgs* a) { return a->k % 32 == 0 && a->k >= 32; }

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

// The vectorised kernels move eight 16-bit elements per lane: every row they touch has to
// start on a 16-byte boundary.
bool vector_ok(const MloraAddArgs* a) {
  if (a->dtype != MLORA_DTYPE_F16 && a->dtype != MLORA_DTYPE_BF16) return false;
  if (!a->plan) return false;
  if (!padded_rank(a->r)) return false;  // 8, 16, 24, ... 64: rows of B start on 16-byte boundaries
  if (a->k % 8 || a->x_stride % 8 || a->y_stride % 8) return false;
  if (!aligned16(a->x) || !aligned16(a->y)) return false;
  for (int i = 0; i < a->num_slices; ++i) {
    const MloraSlice& s = a->slices[i];
    if (s.n % 8 || s.y_col % 8 || !aligned16(s.a) || !aligned16(s.b)) return false;
  }
  return true;
}

}  // namespace

namespace {

// Diagnostic knobs, read from the environment once per process.
struct ApiKnobs {
  int generation = -1, small_batch_tokens, force_form, no_split, split_min_rk, split_max_tokens, auto_fused, slot_max_slots, no_wide, no_pair;
  void read() {
    generation = knob_generation();
    small_batch_tokens = env_int("MLORA_SMALL_BATCH_TOKENS", 0);
    force_form = env_int("MLORA_FORCE_FORM", 0);
    no_split = env_int("MLORA_NO_SPLIT", 0);
    // Measured on the prefill batch (7605 tokens, rank 64) and the mixed one: the one-launch
    // long-segment form takes 4060 us per step against 3586 for two launches (mixed: 6090 against
    // 4992).  Its workgroups are all resident at once, so the whole grid first shrinks (a chain of
    // dependent slab fetches per workgroup, HBM nearly idle) and then expands; the saved launch
    // does not pay for the wait on the slowest role of each unit.  AUTO keeps the two launches.
    auto_fused = env_int("MLORA_AUTO_FUSED", 0);
    no_wide = env_int("MLORA_NO_WIDE", 0);
    no_pair = env_int("MLORA_NO_PAIR", 0);
    // The split form pays when A[slot], which every workgroup of a tile would otherwise fetch whole,
    // is large: rank x K >= 131072 elements (256 KB).  Measured on the decode batch (256 tokens, 32
    // adapters), one workgroup per (tile, column range) against the split form, us per call: rank 16,
    // K = 4096: 6.9 / 8.0 (what producers publish reaches the consumers 1.6 us later, two trips
    // through the memory system; more than spreading 128 KB saves); rank 32, K = 4096: 15.5 / 10.5;
    // rank 32, K = 1024: 4.9-10.0 / 8.1-17.1; rank 16, K = 8192: the K range of a workgroup no
    // longer fits its registers as one batch of loads.
    split_min_rk = env_int("MLORA_SPLIT_MIN_RK", 131072);
    // ... and while the batch has few tiles: K = 4096, rank 32 / 64, 1011 tokens: 12.0 / 17.7 us against
    // 14.8 / 23.1; 1620 tokens: 17.6 / 26.8 against 15.8 / 24.7
    split_max_tokens = env_int("MLORA_SPLIT_MAX_TOKENS", 1280);
    // The slot-major grid launches a workgroup per (slot id, column range) whether the slot has
    // tokens or not; with many more slot ids than adapters in the batch those requests are waste.
    slot_max_slots = env_int("MLORA_SLOT_MAX_SLOTS", 64);
  }
};
const ApiKnobs& knobs() {
  static ApiKnobs k;
  if (k.generation != knob_generation()) k.read();
  return k;
}

}  // namespace

static bool slot_major_pays(const MloraAddArgs* a, const Batch& batch);

// Fewer than sixteen tokens to a slot that has any: one small tile each.
static bool short_segments(const Batch& batch) { return batch.tokens < 16ll * batch.slots; }

// Where 16-token tiles stop paying.  Their cost per token grows with the
// rank (every tile fetches A[slot] and B[slot] again, every column range repeats its tile's shrink)
// while 64-token tiles pay more before they move any data (one launch over small tiles 3.5 us, two
// about 10).  The forms meet where tokens (with a slot) x width does not depend on the shape: width = slices x K x max(1, K / 1024) +
// columns x max(1, columns / 4096), for long K and wide outputs cost the small tiles more than their share.  What it does depend on: whether the
// small tiles' kernel asks for all of K at once (decode_one_batch) or walks K batch by batch (above rank 16 the pair stands in for it then), and whether the other form
// is one launch (`one_launch`), which pays about half as much before it moves data.  The lines lie where 22166 random calls (K 512 to
// 16384, every rank, 100 to 9392 tokens of 1 to 128 slots, even and uneven, up to half of the tokens without adapter) take the least time together, and they are flat there: time of the forms on the lines' sides over the
// fastest form's, on gate_ups by two launches, at 7e6, 1e7, 1.4e7, 1.8e7, 2.2e7, 2.6e7: rank 24 all of K at once 1.033, 1.019, 1.017, 1.017, 1.019, 1.017, batch by batch 1.039, 1.047, 1.061, 1.078, 1.102,
// 1.120; rank 32 1.029, 1.023, 1.024, 1.027, 1.034, 1.036 and 1.025, 1.037, 1.059, 1.081, 1.107, 1.129; rank 64 1.023, 1.033, 1.057, 1.079, 1.102, 1.126 and 1.037, 1.070, 1.107, 1.151, 1.170, 1.208; one slice with outputs
// that are not wide at 5.5e6, 7.7e6, 1e7, 1.3e7: ranks 24 and 32, K 1100 to 1700 1.034, 1.047, 1.053, 1.061, 1700 to 1950 1.066, 1.065, 1.072, 1.088, 2100 to 3000 1.083, 1.082, 1.089, 1.101, above rank 32 1.079, 1.093,
// 1.113, 1.141, 1.099, 1.098, 1.108, 1.119 and 1.014, 1.013, 1.013, 1.011; K = 2048 and rank 32, all of K at once, at 1e7, 1.3e7, 1.7e7, 2.1e7 1.027, 1.019, 1.029, 1.031.  Against one launch, us per call over
// small tiles / 64-token tiles, K = 1024: rank 64, q|k|v 14.8 / 14.3 at 1620 tokens, 18.0 / 15.0 at 3250; o 10.5 / 14.8 at 4511, 18.1 / 15.2 at 6648; rank 32, o of 3 slots 7.7 / 10.2 at
// 4000, 12.4 / 10.2 at 5000; up to rank 16 they meet at 19000 tokens for q|k|v, 4500 for gate_up, 4800 for down of K = 4096.
// MLORA_SMALL_BATCH_TOKENS, when set, replaces the rule by a plain token count.
static double small_work(const MloraAddArgs* a, const Batch& batch) {
  double cols = 0;
  for (int i = 0; i < a->num_slices; ++i) cols += a->slices[i].n;
  return batch.tokens * (static_cast<double>(a->num_slices) * a->k * (a->k > 1024 ? a->k / 1024.0 : 1.0) + cols * (cols > 4096 ? cols / 4096.0 : 1.0));
}
static bool small_batch(const MloraAddArgs* a, bool one_launch, double work) {
  const int fixed = knobs().small_batch_tokens;
  if (fixed > 0) return a->num_tokens <= fixed;
  const bool whole = decode_one_batch(a);
  double limit;
  if (a->r <= 16) limit = (whole ? 8.3e7 : 3.5e7) * (one_launch ? 0.65 : 1.0);
  else limit = one_launch ? 9.4e6 : !whole ? 8.5e6 : a->r <= 32 ? 2.1e7 : 1.1e7;
  return work <= limit;
}
// Over the slots with K shared out (slot.hip) small tiles pay for longer (25 such calls between the lines: 0.872 of the time; K = 4096, rank 32, 558 tokens of 25 slots 7.1 / 11.2).
static bool small_batch_in_parts(const MloraAddArgs* a, const Batch& batch, double work) {
  return knobs().small_batch_tokens <= 0 && work <= (a->r <= 16 ? 8.3e7 : a->r <= 32 ? 2.6e7 : 1.5e7) && slot_supported(a) && slot_k_parts(a) > 1 &&
         slot_major_pays(a, batch);
}

// About how many 16-token tiles a batch has: its segments end anywhere inside their last tile.
int mlora::small_tiles_about(const Batch& batch) {
  const int tiles = static_cast<int>((batch.tokens + 7ll * batch.slots) / MLORA_TILE_SMALL);
  return tiles > batch.slots ? tiles : batch.slots;
}

// Where the slot-major grid pays.  Its workgroups request the weights of EVERY slot id, with or
// without tokens, so what it costs grows with the slot ids nobody uses: measured on decode batches of
// 4..256 tokens over 32 slot ids (us per call, slot-major / tile-major): gate_up, whose slots weigh
// 327 KB each, 5.9 / 3.9 at 4 tokens, 5.6 / 5.2 at 64, 6.1 / 6.0 at 128, 6.7 / 6.8 at 256; o (64 KB per
// slot) 3.5 / 3.4 at 4 tokens, 3.7 / 3.8 at 64, 3.8 / 4.1 at 256; over 8 slot ids it is the faster
// grid at every batch size and every projection; with 128 slot ids of which 32 are in use it
// takes 967 us per decode step against 629.  With K shared out between a tile's workgroups the lines are others
// (below).  So, without: while all slots together weigh at most 3 MB, or when the batch has four tokens per slot id.
// All of this was measured on decode batches; on batches of many tiles per slot (a prefill of
// 2098 tokens over 8 slot ids, o: 15.4 us per call against 10.1 tile-major) the grid over the slots
// is the slower one: it is taken up to 32 tokens per slot id.
// (Where the number of slots with tokens was counted.)  Prompts are few long
// segments: most of the grid is then workgroups without a tile, and the tiles behind a slot's first one learn
// their slot from a record after all (rank 32, 37 tokens of one slot of 8: gate_up 7.4 / 4.9; 100 tokens
// of 4 slots: gate_up 7.7 / 5.0; rank 64, 200 tokens of 3 slots of 32: qkv 9.0 / 6.5, gate_up 12.9 / 10.0,
// down 10.2 / 9.1; rank 16, 250 tokens of 4 slots of 8: 4.05 / 4.11, 3.86 / 3.97, 5.67 / 5.58).
static bool slot_major_pays(const MloraAddArgs* a, const Batch& batch) {
  if (a->num_slots > knobs().slot_max_slots) return false;
  if (batch.tokens > 32 * a->num_slots) return false;
  const bool sparse = batch.slots_counted && 2 * batch.slots <= a->num_slots;
  const int parts = slot_k_parts(a);
  // Buffers of a rank between 32 and 64 run rank 64's code masked: K = 2048 gains like rank 64's (rank 48, slot-major / pair: 7.0 /
  // 7.4 at 16 tokens of 8 slot ids, 8.3 / 9.8 at 128 of 32, 10.6 / 12.3 at 256 of 64), eight parts of 1024 columns do not fit
  // the registers (K = 8192: 11.4 / 7.9 at one token of 8, 20.3 / 13.4 at 128 of 32), and K = 4096 stays with the pair.
  if (parts > 1 && a->r > 32 && !exact_rank(a->r) && a->k != 2048) return false;
  if (parts > 1) {
    // K shared out: the lines lie where the requests for slots without tokens, and at K = 8192 more workgroups than fit
    // the chip together, cost what the second launch does.  us per call, slot-major / the best other form, at
    // one and four tokens per slot id unless said:
    const int tiles = small_tiles_about(batch), slots = a->num_slots, rank = compute_rank(a->r);
    const bool few = sparse || 2 * batch.tokens <= slots;
    // K = 2048: rank 64 8 slot ids 6.3 / 6.8, 32 8.0 / 10.4 and 8.6 / 11.4, 64 11.1 / 13.5; 8 tokens of 64 8.8 / 7.6.  Rank 32 16 ids
    // 5.2 / 5.3, 48 6.2 / 7.0, 64 7.4 / 8.3; 8 tokens of 32 5.2 / 5.1, 37 of one slot of 8 5.3 / 5.2.  Rank 16 40 ids 4.6 / 4.5, 48 4.7 /
    // 4.8, 64 5.3 / 5.4, 512 tokens of 32 (46 tiles) 5.2 / 5.2, 1000 (76) 6.2 / 7.6; rank 8 alike.
    // Three slices (rank 64): twelve workgroups a tile, which have to fit the chip together: 8 ids 6.6 / 7.2 and 7.4 / 8.4, 16 8.5 / 9.9 and
    // 8.9 / 10.4, 256 tokens of 16 (23 tiles) 9.4 / 11.0, 4 tokens of 16 8.0 / 7.6, 24 14.2 / 14.6, 32 16.1 / 13.5 (rank 32, without an instance: 8 ids 5.2 / 5.4, 16 6.0 / 5.8).
    if (a->num_slices == 3) return slots <= (few ? 8 : 16) && tiles <= 24;
    if (a->k == 2048) return rank <= 16 ? !few && tiles >= 48 : !(few && (rank == 32 || rank * slots >= 2048));
    // K = 4096: 64 slot ids 5.1 / 5.7 at rank 8, 5.7 / 6.1, 8.7 / 10.3, 13.6 / 14.4 at rank 64; 8 tokens of 64 4.8 / 5.3, 5.3 / 5.4, 7.2 /
    // 6.8, 11.7 / 7.9; 64 tokens of 4 slots of 32 4.6 / 4.7, 4.6 / 4.8, 5.6 / 5.7, 9.2 / 8.0.
    if (a->k == 4096) return !(few && rank * slots >= 2048);
    // K = 8192: rank 8 48 ids 8.7 / 9.3 and 9.4 / 15.0, 64 10.5 / 10.2 and 11.4 / 15.5, 64 tokens of 8 slots of 64 10.3 / 15.0.  Rank 16 64
    // ids 9.2 / 9.9 and 10.1 / 11.1, 64 tokens of 4 slots of 32 6.0 / 6.9, 250 of 8 8.4 / 7.7.  Rank 32 40 ids 12.7 / 13.2, 48 13.4 / 12.1,
    // 512 tokens of 32 (46 tiles) 11.3 / 13.1, 1000 (76) 17.5 / 16.9, 8 of 32 7.6 / 7.4.  Rank 64 32 ids 13.7 / 15.0, 40 20.2 / 20.0, 512
    // tokens of 32 16.5 / 17.8, 2 of 16 9.3 / 9.2 (rank 32 6.0 / 7.2), 37 of one slot of 8 8.0 / 8.3.
    if (few) return slots <= 8 || rank <= 8 || (rank <= 32 && slots <= 16) || (rank <= 16 && slots <= 32 && tiles <= 16);
    if (rank <= 8) return slots <= 48 || batch.tokens >= 2 * slots;
    return rank <= 16 || (tiles <= 48 && slots <= (rank <= 32 ? 40 : 32));
  }
  if (sparse || (batch.slots_counted && batch.tokens > MLORA_TILE_SMALL * batch.slots)) return false;
  double cols = 0;
  for (int i = 0; i < a->num_slices; ++i) cols += a->slices[i].n;
  const double per_slot = 2.0 * a->r * (static_cast<double>(a->num_slices) * a->k + cols);
  if (a->num_slots * per_slot <= 3.0e6) return true;
  // Where A[slot] and B[slot] are light the line lies at two tokens per slot id: tokens at random, us per call, slot-major / tile-major:
  // 64 of 32 ids, rank 16 qkv 3.68 / 3.82, gate_up 4.91 / 5.00, rank 8 gate_up 4.51 / 4.74, rank 24 o 4.33 / 4.61, rank 32 o 4.17 / 4.31, but gate_up
  // 7.5 / 7.4, rank 64 qkv 7.9 / 7.5, o 6.0 / 5.8; 128 of 64, rank 8 gate_up 7.20 / 7.38, rank 16 o 3.61 / 3.86, gate_up 8.03 / 8.24, rank 24 o 4.45 /
  // 4.70, rank 32 o 4.46 / 4.51.  At two, three and 3.9 tokens of 12 to 64 ids, ranks 8 to 32, 69 of 69 such calls are 0.4 to 7 % faster.
  const bool light = a->k == 1024 && (compute_rank(a->r) <= 16 || (compute_rank(a->r) == 32 && a->num_slices == 1 && cols <= 2048));
  return batch.tokens >= (light ? 2 : 4) * a->num_slots;
}

// Where the shrink and the expand as two launches over 16-token tiles (pair.hip) beat the form that
// `form` names.  A second launch costs about 3 us; what it saves is the repeated intake of A[slot] by
// every column range of a tile, which grows with rank x K and with the number of ranges.  Measured, us per
// call, that form / the pair (replayed graphs; 201 tokens over 48 slots of mixed rank 8..64, K = 2048:
// qkv 27.6 / 17.0, o 23.6 / 11.8, gate_up 43.5 / 31.9, down 38.7 / 17.5):
//  - split form (rank x K >= 131072, few tokens): 4 of 4 shapes at 1..512 tokens, rank 16..64 (one token:
//    rank 64, K = 2048: 10.9 / 7.1; rank 16, K = 8192: 7.3 / 7.1; 64 tokens, rank 32, K = 8192: 15.3 / 10.7);
//  - one workgroup per (tile, column range): from rank x K = 131072 on (1234 tokens, rank 32, K = 4096: 19.1 /
//    13.9; it loses below: rank 16, K = 4096, 2000 tokens 11.5 / 12.5, and ties at rank 32, K = 2048), and for
//    buffers of a rank between the instances', whose code is the general one away from K = 1024 (64 tokens, rank 48, K = 2048:
//    14.5 / 12.1, 12.5 / 9.4, 29.4 / 19.3, 35.7 / 12.9; at 1500 tokens and rank 24 qkv and o are
//    still the faster ones in one launch: 12.7 / 13.3, 8.1 / 11.2);
//  - 64-token tiles, where A is as large (between the instances' ranks from rank x K = 49152 on: K = 3072, rank 24, 1565 tokens 11.9 / 8.3) and the outputs are not
//    wide: while two K parts of every (tile, slice) find a compute unit, tiles x slices <= 128.  The shrink is
//    one workgroup per compute unit, and a second round of them costs what the first one does.  64-token tiles /
//    pair, at 1900 and 2200 tokens of 4 slots (123 and 141 tiles): rank 64, K = 4096 16.8 / 13.1, 17.1 / 19.0, K = 2048
//    14.9 / 12.8, 15.2 / 17.7, K = 8192 23.4 / 20.0, 24.4 / 29.9; rank 32, K = 4096 12.8 / 11.2, 13.2 / 15.2; rank 16, K =
//    8192 15.7 / 13.8, 16.5 / 17.2.  At 1300 and 1600 tokens of 100 slots (125 and 144 tiles): rank 64, K = 4096 23.4 / 22.3,
//    23.7 / 28.5; rank 32, K = 4096 16.0 / 15.3, 16.7 / 18.8.  (One slice above rank 16 and segments counted at 16 to 127 tokens stop at 96 tiles: 1500 tokens of 16 and 64 slots, 100
//    and 121 tiles, 64-token tiles / pair: rank 64, K = 4096 16.1 / 20.1, 19.5 / 25.3, rank 32 13.3 / 15.1, 13.1 / 17.9);
//  - wide outputs above rank 16: while tiles x slices x rank <= 2048, since the tiles' B rows are what the second launch takes in, and 3600 between the
//    instances' ranks, whose 64-token tiles take in as many as the next instance's.  Pair's time over 64-token tiles' on random gate_ups by that product (to 1024, 2048, 3000, 4500),
//    even segments: rank 24 0.87, 0.98, 1.02, 1.03, rank 32 0.92, 1.00, 1.03, 1.09, rank 40 to 56 0.78, 0.90, 0.98, 1.05, rank 64 0.82, 0.97, 1.05, 1.11; a few popular slots: -, 0.94, 0.92, 0.97, -, 0.91,
//    0.95, 1.03, -, 0.89, 0.89, 0.93, -, -, -, 1.04;
//  - segments of few tokens, whose 64-token tiles are mostly copies of their last row: two launches over 64-token tiles up to 22 tokens to a slot that has any (pair's time over theirs
//    by tokens per slot, below 8, to 16, to 20, to 26, to 34: rank 24 and 32 0.82, 0.86, 0.98, 1.04, 1.08; rank 40 to 56 0.78, 0.82, 1.01, 1.05, 1.06; rank 64 0.86, 0.88, 1.08, 1.12,
//    1.14; 540 calls); one launch over them below 16, unless its ranges repeat little of the shrink (K > 1100, below 8, to 12, to 16, to 22: rank 24 and 32 0.88, 0.88, 1.02, 1.09; rank 40 to 56
//    0.89, -, 0.78, 1.00; rank 64 0.94, 0.97, 0.94, 0.98; at K = 1024 1.10 and more); one launch over small tiles below 16, where A and B of the slots are 60 MB and the outputs wide (128 slots, gate_up, K = 1024, rank 64, 600, 1000, 1500 tokens
//    43.9 / 36.5, 47.2 / 38.1, 50.8 / 40.6; K = 2048, rank 16 32.7 / 28.2, 51.2 / 39.6).  Where nobody counted the slots in use, below 8 tokens to a slot id: with all,
//    half and a quarter of the ids in use 0.78, 0.78 and 0.93 of 64-token tiles' time, and beyond, up to 16, 0.79, 0.90 and 1.02 (up to rank 16 0.68, 0.70 and 0.80).
static bool pair_pays(const MloraAddArgs* a, int form, const Batch& batch) {
  const long long rk = static_cast<long long>(a->r) * a->k;
  long long cols = 0;
  for (int i = 0; i < a->num_slices; ++i) cols += a->slices[i].n;
  const bool few_tokens = short_segments(batch), middling = !few_tokens && batch.slots_counted && a->r > 16 && exact_rank(a->r) && batch.tokens < 128ll * batch.slots;
  const double weights = 2.0 * batch.slots * a->r * (static_cast<double>(a->num_slices) * a->k + cols);
  if (form == MLORA_FORM_SGMV && batch.tokens < (batch.slots_counted ? 22ll : a->r <= 16 ? 16ll : 8ll) * batch.slots) return true;
  if (form == MLORA_FORM_WIDE && few_tokens && batch.slots_counted && !wide_repeats_little(a)) return true;
  if (form == MLORA_FORM_MFMA && batch.tokens < (batch.slots_counted ? 16ll : 8ll) * batch.slots && weights >= 6.0e7 && cols >= 2ll * a->num_slices * a->k) return true;
  if (form == MLORA_FORM_SGMV && a->r > 16 && cols > 2ll * a->k && static_cast<long long>(small_tiles_about(batch)) * a->num_slices * a->r <= (exact_rank(a->r) ? 2048 : 3600)) return true;
  switch (form) {
    case MLORA_FORM_SPLIT: return true;  // (AUTO keeps the split form for workspaces without room for the pair's partial sums)
    case MLORA_FORM_MFMA: {
      if (!exact_rank(a->r)) {
        const double width = static_cast<double>(a->num_slices) * a->k + cols * (cols > 4096 ? cols / 4096.0 : 1.0);
        return a->k != 1024 || batch.tokens * width > (a->r > 32 ? 1.0e7 : 2.0e7);
      }
      return rk >= 131072;
    }
    case MLORA_FORM_SGMV:
    case MLORA_FORM_WIDE:
      return rk >= (exact_rank(a->r) ? 131072 : 49152) && (a->k >= 4096 || cols <= 2ll * a->k) && static_cast<long long>(small_tiles_about(batch)) * a->num_slices <= (a->num_slices == 1 && middling ? 96 : 128);
    default: return false;
  }
}

// Where three slices, or one above rank 16, over 16-token tiles (one workgroup per tile and column range) give way to one launch over 64-token
// tiles although the batch is small: once the tiles' workgroups, tile t on XCD t % 8, no longer fit the 32 compute
// units of an XCD, they run in two rounds, each of which shrinks its tile anew.  16-token / 64-token tiles, us per call, q|k|v
// at workgroups per XCD: K = 1024, rank 64: 11.7 / 13.7 at 32, 16.6 / 13.8 at 36, 17.5 / 12.8 at 44, 17.7 / 13.6 at 48; rank
// 32: 7.5 / 9.3 at 32, 10.4 / 10.9 at 36, 10.9 / 9.1 at 44; K = 768, rank 64: 10.7 / 12.6 at 32, 17.3 / 12.5 at 36; rank 32: 7.0 /
// 8.7 and 10.9 / 9.9; K = 512, rank 64: 7.7 / 9.7 and 11.8 / 10.8; between the instances' ranks the gain begins further on (K = 1024, rank 24 8.1 / 10.8 at
// 36, 12.5 / 10.8 at 48, rank 48 11.4 / 14.6 and 18.0 / 14.6), but the tiles' number is an estimate: 32 for them too takes no more time than 40, counted or not.  One slice, o, K = 1024, in one range of 1024 columns (decode_ranges has made the most of the
// ranges): 2800 / 4000 / 4700 tokens of 48 slots rank 64 13.0 / 13.6, 22.8 / 13.6, 23.4 / 14.1, rank 24 8.7 / 10.9, 14.2 / 10.7, 14.7 / 11.0, of 128 slots rank 48 14.2
// / 12.2, 15.1 / 14.1, 23.3 / 16.2.  With a smaller A the rounds are too short to matter (K = 512,
// rank 32: 7.2 / 8.8 at 36).  The two-launch pair lies above both nearly throughout (K = 1024, rank 32 / 64, 1500 tokens
// of 8 slots: 11.0 / 13.3 / 11.0 and 17.7 / 17.3 / 13.8 over 16-token tiles, as a pair, over 64-token tiles).
static bool wide_instead(const MloraAddArgs* a, const Batch& batch) {
  if (a->num_slices == 2 || a->r <= 16 || a->r * static_cast<long long>(a->k) < 24576) return false;
  const int layers = (small_tiles_about(batch) + 7) / 8;
  int columns = 0;
  for (int i = 0; i < a->num_slices; ++i) columns += a->slices[i].n;
  if (layers * (columns / 64ll + a->num_slices) <= 32) return false;  // (a range has 64 columns at least)
  return layers * decode_ranges(a, batch, &columns) > 32 && wide_supported(a) && wide_pays(a, batch);
}

namespace {

int add_lora_impl(const MloraAddArgs* a, bool trusted_workspace, int active_slots, int active_tokens);

}  // namespace

extern "C" int mlora_add_lora(const MloraAddArgs* a) { return add_lora_impl(a, false, 0, 0); }
extern "C" int mlora_add_lora_active(const MloraAddArgs* a, int32_t active_slots) { return add_lora_impl(a, false, active_slots, 0); }
extern "C" int mlora_add_lora_counts(const MloraAddArgs* a, int32_t active_slots, int32_t active_tokens) {
  return add_lora_impl(a, false, active_slots, active_tokens);
}

namespace {

}  // namespace

int mlora::check_args(const MloraAddArgs* a) {
  if (!a) { set_error("mlora_add_lora: NULL args"); return MLORA_E_INVALID; }
  if (a->num_tokens < 0 || a->k < 0 || a->r < 0 || a->num_slots < 0 || a->num_slices < 0) {
    set_error("mlora_add_lora: negative size"); return MLORA_E_INVALID;
  }
  if (a->dtype != MLORA_DTYPE_F32 && a->dtype != MLORA_DTYPE_F16 && a->dtype != MLORA_DTYPE_BF16) {
    set_error("mlora_add_lora: unknown dtype %d", a->dtype); return MLORA_E_INVALID;
  }
  if (a->form < MLORA_FORM_AUTO || a->form > MLORA_FORM_PAIR) { set_error("mlora_add_lora: unknown form %d", a->form); return MLORA_E_INVALID; }
  if (a->num_slices > MLORA_MAX_SLICES) { set_error("mlora_add_lora: %d slices exceed %d", a->num_slices, MLORA_MAX_SLICES); return MLORA_E_TOO_LARGE; }
  if (a->r > MLORA_MAX_RANK) { set_error("mlora_add_lora: rank %d exceeds %d", a->r, MLORA_MAX_RANK); return MLORA_E_TOO_LARGE; }
  if (a->num_slots > MLORA_MAX_SLOTS) { set_error("mlora_add_lora: %d slots exceed %d", a->num_slots, MLORA_MAX_SLOTS); return MLORA_E_TOO_LARGE; }
  if (a->num_tokens == 0 || a->num_slices == 0 || a->num_slots == 0 || a->r == 0) return kNothingToDo;
  if (!a->x || !a->y || !a->token_to_slot) { set_error("mlora_add_lora: NULL tensor pointer"); return MLORA_E_INVALID; }
  bool any = false;
  for (int i = 0; i < a->num_slices; ++i) {
    const MloraSlice& s = a->slices[i];
    if (s.n < 0 || s.y_col < 0) { set_error("mlora_add_lora: slice %d has negative extent", i); return MLORA_E_INVALID; }
    if (s.n > 0 && (!s.a || !s.b)) { set_error("mlora_add_lora: slice %d has NULL weights", i); return MLORA_E_INVALID; }
    if (static_cast<int64_t>(s.y_col) + s.n > a->y_stride) {
      set_error("mlora_add_lora: slice %d ends at column %lld, beyond the y row stride %lld", i, static_cast<long long>(s.y_col) + s.n,
                static_cast<long long>(a->y_stride));
      return MLORA_E_INVALID;
    }
    any |= s.n > 0;
  }
  if (a->x_stride < a->k) { set_error("mlora_add_lora: x row stride %lld is below K = %d", static_cast<long long>(a->x_stride), a->k); return MLORA_E_INVALID; }
  if (!any) return kNothingToDo;
  if (reinterpret_cast<uintptr_t>(a->plan) & 15) { set_error("mlora_add_lora: plan must be 16-byte aligned"); return MLORA_E_INVALID; }
  return 0;
}

int mlora::chosen_form(const MloraAddArgs* a, const Batch& batch) {
  int form = a->form;
  const bool vec = vector_ok(a);
  const ApiKnobs& kn = knobs();
  if (form == MLORA_FORM_AUTO) {
    const int forced = kn.force_form;
    if (forced >= MLORA_FORM_TOKEN && forced <= MLORA_FORM_PAIR && (forced == MLORA_FORM_TOKEN || vec)) form = forced;
  }
  if (form == MLORA_FORM_AUTO) {
    // Small batches (decode) are one launch over 16-token tiles; large ones split into 64-token
    // tiles for the long segments and 16-token tiles for the rest: one launch whose workgroups do
    // both products where a tile's column ranges repeat little of its shrink, else two launches.
    // (What the two kinds of large ones cost is looked at only where small tiles do not win over both.)
    const bool mfma = mfma_supported(a), small_tiles = mfma && decode_supported(a);
    const double work = small_work(a, batch);
    const bool small = small_tiles && small_batch(a, true, work) && small_batch(a, false, work);
    const bool two_launches = !small && mfma && sgmv_supported(a) && sgmv_workspace_ok(a);
    const bool one_launch = !small && mfma && !kn.no_wide && wide_supported(a) && wide_pays(a, batch);
    // (fp32 rows and anything else the 128-bit kernels for 16-bit elements do not take: one workgroup per token,
    // which fetches A and B per token and walks K in chained steps, except where the pair of launches has the
    // element type: config 1's batch, 64 tokens over 4 slots, rank 16, fp32, qkv / o / gate_up / down 25 / 25 / 27 /
    // 70 us per call in one workgroup per token, 7.0 / 6.7 / 8.0 / 7.6 in two launches; rank 24, 36 / 16 / 39 / 104 and 9.5 / 9.2 / 10.7 /
    // 10.9, rank 56, 81 / 80 / 90 / 243 and 12.6 / 12.1 / 14.3 / 15.5, one token of rank 24 15.3 / 15.4 / 15.8 / 43 and 8.5 / 8.5 / 9.2 / 9.9)
    if (!vec) form = a->dtype == MLORA_DTYPE_F32 && !kn.no_pair && pair_supported(a) ? MLORA_FORM_PAIR : MLORA_FORM_TOKEN;
    else if (small_tiles && !small && small_batch_in_parts(a, batch, work)) form = MLORA_FORM_SPLIT;
    else if (one_launch && !(small_tiles && small_batch(a, true, work))) form = MLORA_FORM_WIDE;
    else if (!one_launch && two_launches && !(small_tiles && small_batch(a, false, work))) form = MLORA_FORM_SGMV;
    else if (small_tiles) form = MLORA_FORM_SPLIT;
    else form = MLORA_FORM_BGMV;
  }
  // the split form where it pays (a large A[slot]) and shape and workspace allow it, else one
  // workgroup per (tile, column range)
  if (form == MLORA_FORM_SPLIT && a->form != MLORA_FORM_SPLIT &&
      (kn.no_split || ((static_cast<long long>(a->r) * a->k < kn.split_min_rk || batch.tokens > kn.split_max_tokens) && kn.force_form != MLORA_FORM_SPLIT) || !split_supported(a)))
    form = MLORA_FORM_MFMA;
  // small tiles with the grid laid over the slots where the shape allows it and slot ids are few.
  // Also where the split form would be taken: at K = 4096 the slot-major kernel shares K out between
  // the workgroups of a tile itself (down, decode batch, us per call, slot-major / split form:
  // rank 32: 6.3 / 10.6, rank 64: 9.8 / 17.0).
  if ((form == MLORA_FORM_MFMA || form == MLORA_FORM_SPLIT) && a->form == MLORA_FORM_AUTO && kn.force_form != MLORA_FORM_MFMA &&
      kn.force_form != MLORA_FORM_SPLIT && slot_supported(a) && slot_major_pays(a, batch))
    form = MLORA_FORM_SLOT;
  if (a->form == MLORA_FORM_AUTO && kn.force_form == 0 && !kn.no_pair && !kn.auto_fused && vec && pair_pays(a, form, batch) && pair_supported(a))
    form = MLORA_FORM_PAIR;
  if (form == MLORA_FORM_MFMA && a->form == MLORA_FORM_AUTO && kn.force_form == 0 && !kn.no_wide && kn.small_batch_tokens <= 0 &&
      wide_instead(a, batch))
    form = MLORA_FORM_WIDE;
  // long-segment batches in one launch, on request
  if (form == MLORA_FORM_SGMV && a->form == MLORA_FORM_AUTO && kn.force_form != MLORA_FORM_SGMV && kn.auto_fused && fused_supported(a))
    form = MLORA_FORM_FUSED;
  return form;
}

namespace {

int add_lora_impl(const MloraAddArgs* a, bool trusted_workspace, int active_slots, int active_tokens) {
  const int rc = check_args(a);
  if (rc) return rc == kNothingToDo ? 0 : rc;
  const Batch batch = batch_of(a, active_slots, active_tokens);
  const bool vec = vector_ok(a);
  const int form = chosen_form(a, batch);
  switch (form) {
    case MLORA_FORM_TOKEN:
      return launch_token_add(a);
    case MLORA_FORM_BGMV:
      if ((a->effective_rank || !exact_rank(a->r)) && a->form == MLORA_FORM_AUTO) return launch_token_add(a);  // the vector-ALU tiles read whole rank-r rows
      if (!exact_rank(a->r)) { set_error("mlora_add_lora: the BGMV form takes ranks 8, 16, 32 and 64"); return MLORA_E_UNSUPPORTED; }
      if (a->effective_rank) { set_error("mlora_add_lora: the BGMV form does not take effective_rank"); return MLORA_E_UNSUPPORTED; }
      if (!vec) { set_error("mlora_add_lora: BGMV form needs 16-bit elements, a plan, rank in {8,16,32,64} and 16-byte aligned rows"); return MLORA_E_UNSUPPORTED; }
      return launch_bgmv(a, /*include_long=*/true);
    case MLORA_FORM_WIDE:
      if (!vec || !mfma_supported(a) || !wide_supported(a)) {
        set_error("mlora_add_lora: the one-launch form over 64-token tiles needs 16-bit elements, a plan, a rank of 8, 16, 32 or 64, K %% 128 == 0 "
                  "and no empty slice");
        return MLORA_E_UNSUPPORTED;
      }
      return launch_wide(a, batch);
    case MLORA_FORM_PAIR:
      if (!pair_supported(a)) {
        set_error("mlora_add_lora: the pair form needs a plan, a workspace, rows of x of a multiple of 128 bytes, B rows of 16 to 128 (fp32: 256) bytes "
                  "in steps the kernels have, 16-byte aligned rows and no empty slice");
        return MLORA_E_UNSUPPORTED;
      }
      return launch_pair(a, batch);
    case MLORA_FORM_SGMV:
    case MLORA_FORM_FUSED:
    case MLORA_FORM_SPLIT:
    case MLORA_FORM_SLOT:
    case MLORA_FORM_MFMA: {
      if (!vec || !mfma_supported(a)) { set_error("mlora_add_lora: MFMA forms need 16-bit elements, a plan, a rank that is a multiple of 8 up to 64 and K %% 32 == 0"); return MLORA_E_UNSUPPORTED; }
      if (form == MLORA_FORM_MFMA) return launch_decode(a, /*include_long=*/true, batch);
      if (form == MLORA_FORM_SLOT) {
        if (!slot_supported(a)) {
          set_error("mlora_add_lora: the slot-major form needs one or two non-empty slices and K = 1024 (three at an exact rank with column "
                    "ranges of at most 512 columns), or K = 4096 with rank <= 16 or (2048, 4096 and 8192; 2048 at rank 64 with three too) with one slice of at most 4096 columns and an "
                    "initialised workspace");
          return MLORA_E_UNSUPPORTED;
        }
        return launch_slot(a, trusted_workspace);
      }
      if (form == MLORA_FORM_SPLIT) {
        if (!split_supported(a)) {
          set_error("mlora_add_lora: the split form needs a rank of 8, 16, 32 or 64, K %% 512 == 0, at most 8 K parts, no empty slice and a 256-byte aligned "
                    "workspace of at least %d bytes whose exchange area holds every tile's partial sums", MLORA_WORKSPACE_HEAD_BYTES);
          return MLORA_E_UNSUPPORTED;
        }
        return launch_split(a, /*include_long=*/true, trusted_workspace);
      }
      if (!sgmv_supported(a)) { set_error("mlora_add_lora: SGMV form needs K %% 128 == 0 and a rank of 8, 16, 32 or 64"); return MLORA_E_UNSUPPORTED; }
      if (!sgmv_workspace_ok(a)) {
        set_error("mlora_add_lora: SGMV form needs a 16-byte aligned workspace of %zu bytes and no empty slice",
                  sgmv_workspace_bytes(a->num_tokens, a->num_slices, a->r, a->dtype));
        return MLORA_E_INVALID;
      }
      if (form == MLORA_FORM_FUSED) {
        if (!fused_supported(a)) {
          set_error("mlora_add_lora: the one-launch long-segment form needs K %% 256 == 0, at most %d groups of tiles and a workspace "
                    "whose head holds their seals", kWsTiles);
          return MLORA_E_UNSUPPORTED;
        }
        return launch_fused(a, trusted_workspace);
      }
      return launch_sgmv(a, batch);
    }
  }
  set_error("mlora_add_lora: unreachable form %d", form);
  return MLORA_E_INVALID;
}

}  // namespace

// ---- the entry point that allocates nothing --------------------------------------------------
// Scratch of mlora_add_lora_static: part of the library's device image, so every GPU the
// library runs on holds its own copy at its own address from module load until the process ends.
// In host code the name `scratch` is only a handle for hipGetSymbolAddress; the address kernels
// and copies may use is the one that call returns, looked up once per device.
static __device__ __align__(256) unsigned char scratch[MLORA_STATIC_SCRATCH_BYTES];

namespace {
constexpr int kMaxDevices = 64;
void* g_scratch_ptr[kMaxDevices];  // device address of `scratch` on each GPU (nullptr: not looked up yet)
std::mutex g_scratch_mutex;

// Address of the current device's copy of `scratch`; nullptr (and the error text set) on failure.
void* static_scratch(hipStream_t stream) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess || dev < 0 || dev >= kMaxDevices) {
    set_error("mlora_add_lora_static: cannot identify the current device (%s)", e != hipSuccess ? hipGetErrorString(e) : "index out of range");
    return nullptr;
  }
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (!g_scratch_ptr[dev]) {
    // The look-up may load the code object, which a stream capture in progress does not survive:
    // the first call on a device has to be made outside any capture (one with num_tokens = 0 will do).
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(stream, &status) == hipSuccess && status == hipStreamCaptureStatusActive) {
      set_error("mlora_add_lora_static: the first call on a device must be made outside stream capture (call once with num_tokens = 0 before capturing)");
      return nullptr;
    }
    (void)hipGetLastError();
    void* ptr = nullptr;
    e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !ptr) {
      set_error("mlora_add_lora_static: hipGetSymbolAddress failed on device %d: %s", dev, hipGetErrorString(e));
      return nullptr;
    }
    g_scratch_ptr[dev] = ptr;
  }
  return g_scratch_ptr[dev];
}
}  // namespace

extern "C" int mlora_add_lora_static(const MloraAddArgs* a) {
  if (!a) { set_error("mlora_add_lora_static: NULL args"); return MLORA_E_INVALID; }
  if (a->num_tokens < 0 || a->num_slices < 0 || a->r < 0) { set_error("mlora_add_lora_static: negative size"); return MLORA_E_INVALID; }
  const unsigned long long one_copy = 4ull * static_cast<unsigned long long>(a->num_tokens) * static_cast<unsigned long long>(a->num_slices) *
                                      static_cast<unsigned long long>(a->r);
  if (one_copy > MLORA_STATIC_SCRATCH_BYTES - MLORA_WORKSPACE_HEAD_BYTES) {
    set_error("mlora_add_lora_static: num_tokens x num_slices x r x 4 = %llu bytes exceed the static scratch of %u bytes behind its head (use mlora_add_lora with a workspace)",
              one_copy, static_cast<unsigned>(MLORA_STATIC_SCRATCH_BYTES - MLORA_WORKSPACE_HEAD_BYTES));
    return MLORA_E_TOO_LARGE;
  }
  void* ptr = static_scratch(static_cast<hipStream_t>(a->stream));
  if (!ptr) return MLORA_E_INVALID;
  MloraAddArgs b = *a;
  b.workspace = ptr;
  b.workspace_bytes = MLORA_STATIC_SCRATCH_BYTES;
  // The array starts out zeroed (it is part of the loaded image) and only this library's kernels
  // ever write it, so its head is always either in the initial state or as a launch left it.
  return add_lora_impl(&b, /*trusted_workspace=*/true, 0, 0);
}

extern "C" size_t mlora_add_workspace_bytes(int32_t num_tokens, int32_t num_slices, int32_t r, int32_t dtype) {
  if (num_tokens <= 0 || num_slices <= 0 || r <= 0) return 0;
  return sgmv_workspace_bytes(num_tokens, num_slices, r, dtype);  // head + room for every K part of the intermediate
}

extern "C" int mlora_workspace_init(void* workspace, int64_t workspace_bytes, void* stream) {
  if (!workspace || (reinterpret_cast<uintptr_t>(workspace) & 255)) { set_error("mlora_workspace_init: workspace must be 256-byte aligned"); return MLORA_E_INVALID; }
  if (workspace_bytes < MLORA_WORKSPACE_HEAD_BYTES) {
    set_error("mlora_workspace_init: %lld bytes are fewer than MLORA_WORKSPACE_HEAD_BYTES = %d", static_cast<long long>(workspace_bytes), MLORA_WORKSPACE_HEAD_BYTES);
    return MLORA_E_INVALID;
  }
  return workspace_init(workspace, static_cast<hipStream_t>(stream));
}

extern "C" uint64_t mlora_stream_capture_id(void* stream) {
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  unsigned long long id = 0;
  if (hipStreamGetCaptureInfo(static_cast<hipStream_t>(stream), &status, &id) != hipSuccess) {
    (void)hipGetLastError();
    return 0;
  }
  return status == hipStreamCaptureStatusActive ? static_cast<uint64_t>(id) : 0;
}

extern "C" void mlora_reload_knobs(void) { ++g_knob_generation; }

extern "C" int mlora_abi_version(void) { return MLORA_ABI_VERSION; }

extern "C" const char* mlora_last_error(void) { return g_error; }

extern "C" const char* mlora_build_info(void) {
  return "mlora gfx950 (wave64; small tiles: MFMA 16x16x32 or dot2 + wave reductions; big tiles: MFMA 16x16x32 shrink + expand) built " __DATE__ " " __TIME__;
}
