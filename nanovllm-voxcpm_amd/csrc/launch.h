// Internal launch entry points shared by the C-ABI front door.
#pragma once

#include <hip/hip_runtime.h>

#include "mlora.h"

namespace mlora {

int env_int(const char* name, int fallback);

// Ranks the kernels are instantiated for.  Buffers of another rank that is a multiple of eight and
// at most 64 (24, 40, 48, 56) run on the next instance up in the small-tile kernels, with the
// buffers' rank as the run-time stride and everything beyond it masked as for an adapter of lower
// rank; the other forms take exact ranks only.
inline bool exact_rank(int r) { return r == 8 || r == 16 || r == 32 || r == 64; }
inline bool padded_rank(int r) { return r >= 8 && r <= 64 && r % 8 == 0; }
// What the host knows of a batch beyond its size: how many slots have tokens and how many tokens a slot, each as counted, else (a captured call, a
// caller who does not say) the most there can be.
struct Batch {
  int slots, tokens;
  bool slots_counted, tokens_counted;
};
inline Batch batch_of(const MloraAddArgs* a, int active_slots, int active_tokens) {
  Batch b;
  b.slots_counted = active_slots > 0;
  b.tokens_counted = active_tokens > 0;
  b.slots = a->num_slots < a->num_tokens ? a->num_slots : a->num_tokens;
  if (b.slots_counted && active_slots < b.slots) b.slots = active_slots;
  b.tokens = b.tokens_counted && active_tokens < a->num_tokens ? active_tokens : a->num_tokens;
  return b;
}
// The 64-token tiles serve buffers of every padded rank; by name only those of the instances' own, as ever.
inline bool tiles64_rank(const MloraAddArgs* a) { return a->form == MLORA_FORM_AUTO ? padded_rank(a->r) : exact_rank(a->r); }
inline int compute_rank(int r) { return r <= 8 ? 8 : r <= 16 ? 16 : r <= 32 ? 32 : 64; }
// Diagnostic knobs are read from the environment once and kept; mlora_reload_knobs() advances
// this number, and a holder whose copy is older reads its variables again.
int knob_generation();

// api.hip: the checks on a call's arguments (0, kNothingToDo or an error code), and the form that serves it.
constexpr int kNothingToDo = INT32_MIN;
int check_args(const MloraAddArgs* a);
int chosen_form(const MloraAddArgs* a, const Batch& batch);

// token.hip: one workgroup per token; needs only token_to_slot.
int launch_token_add(const MloraAddArgs* a);

// bgmv.hip: small tiles (<= 16 tokens of one slot) on the vector ALU.  include_long selects
// whether the small tiles of segments at or above the threshold are walked too.
int launch_bgmv(const MloraAddArgs* a, bool include_long);

// decode.hip: the same small tiles with both products on the matrix cores, one workgroup per
// (tile, column range).
bool decode_one_batch(const MloraAddArgs* a);  // its wavefronts ask for all of their K at once
bool decode_supported(const MloraAddArgs* a);  // x and y below 2 GiB each
int launch_decode(const MloraAddArgs* a, bool include_long, const Batch& batch);
int decode_ranges(const MloraAddArgs* a, const Batch& batch, int* columns);  // column ranges of that launch, and columns per range

// slot.hip: the same small tiles, the grid laid over the slots: weights are requested from the
// workgroup index alone, before the slot's record has arrived.
bool slot_supported(const MloraAddArgs* a);
int slot_k_parts(const MloraAddArgs* a);  // 4 or 8 when the workgroups of a tile would share K out, else 1
int launch_slot(const MloraAddArgs* a, bool trusted_workspace);
// How often the fullest of 256 compute units has the time of a workgroup, of which two fit side by side and take the price of both: between the whole
// rounds and the share of one that the workgroups come to, since tiles that end early let others in and the number of tiles is an estimate.
inline double rounds_of(long long workgroups) {
  const double share = workgroups / 256.0;
  return 0.5 * (static_cast<double>((workgroups + 255) / 256) + (share > 1 ? share : 1));
}

// How a launch over 64-token tiles is cut, into `count` K parts or into ranges of `count` columns, and how many columns (of K, of a range) the fullest compute
// unit then streams.
struct Cut {
  int count;
  double columns;
};
int big_tiles_about(const Batch& batch, int tokens);  // 64-token tiles and short segments of a batch with that many tokens with a slot (sgmv.hip)
Cut ring_cut(const MloraAddArgs* a, const Batch& batch, int most_parts);  // the shrink of two launches (sgmv.hip)
Cut wide_cut(const MloraAddArgs* a, const Batch& batch, int widest_range = 2048);  // both products in one (wide.hip)
int sgmv_parts(const MloraAddArgs* a, const Batch& batch);  // K parts of launch_sgmv

int small_tiles_about(const Batch& batch);  // 16-token tiles of a batch (api.hip)

// split.hip: the same small tiles, producers and consumers of the intermediate in one launch.
// trusted_workspace: the head of the workspace is known to be in its initial or a left-behind
// state without carrying the signature (the library's own zero-initialised array).
bool split_supported(const MloraAddArgs* a);
int launch_split(const MloraAddArgs* a, bool include_long, bool trusted_workspace);
int workspace_init(void* workspace, hipStream_t stream);

// sgmv.hip: 64-token MFMA tiles of the segments at or above the threshold, as a shrink launch
// and an expand launch that meet in the caller's workspace.
bool sgmv_supported(const MloraAddArgs* a);
bool sgmv_workspace_ok(const MloraAddArgs* a);
size_t sgmv_workspace_bytes(int num_tokens, int num_slices, int r, int dtype);
int launch_sgmv(const MloraAddArgs* a, const Batch& batch);

// slab.hip: the shrink launch of that form, operands through LDS by direct loads.
struct PlanLayout;
bool slab_supported(const MloraAddArgs* a);
void launch_slab_shrink(const MloraAddArgs* a, const PlanLayout& lay, int big_cap, int tiles8, int parts, const void* const* slices);

// fused.hip: the same tiles, shrink and expand in one launch (workgroups of a unit exchange the
// intermediate through the workspace under seals kept in its head).
bool fused_supported(const MloraAddArgs* a);
int launch_fused(const MloraAddArgs* a, bool trusted_workspace);

// wide.hip: the same tiles, one launch, one workgroup per (tile, column range) doing both products.
bool wide_supported(const MloraAddArgs* a);
bool wide_repeats_little(const MloraAddArgs* a);  // of a tile's shrink: at most 1024 columns of K over all its ranges of 512
bool wide_pays(const MloraAddArgs* a, const Batch& batch);  // against the two launches
int launch_wide(const MloraAddArgs* a, const Batch& batch);

// pair.hip: a shrink launch and an expand launch over the 16-token tiles, operands through LDS by
// direct loads; 16- and 32-bit elements.
bool pair_supported(const MloraAddArgs* a);
// Under AUTO fp32 takes one launch where that is the faster one.
int launch_pair(const MloraAddArgs* a, const Batch& batch);

// group.hip: the low-level shrink and expand over tiles of a slot; `supported` says where they are the faster ones too.
bool group_shrink_supported(const MloraShrinkArgs* a);
int launch_group_shrink(const MloraShrinkArgs* a);
bool group_expand_supported(const MloraExpandArgs* a);
int launch_group_expand(const MloraExpandArgs* a);

// in-kernel timeline of trace builds (no-ops otherwise)
void decode_trace_set(void* buf);
void slot_trace_set(void* buf);
void split_trace_set(void* buf);
void fused_trace_set(void* buf);
void sgmv_trace_set(void* buf);
void wide_trace_set(void* buf);
void pair_trace_set(void* buf);

}  // namespace mlora
