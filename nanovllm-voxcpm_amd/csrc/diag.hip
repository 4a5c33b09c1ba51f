// Entry points of the diagnostic variants of the library (include/mlora_diag.h): none of them has a
// counterpart in the reference and none is part of the product library.
#include "common.h"
#include "group_layout.h"
#include "launch.h"
#include "mlora_diag.h"

using namespace mlora;

extern "C" int mlora_trace_set(void* buf) {
#ifdef MLORA_TRACE
  decode_trace_set(buf);
  slot_trace_set(buf);
  split_trace_set(buf);
  fused_trace_set(buf);
  sgmv_trace_set(buf);
  wide_trace_set(buf);
  pair_trace_set(buf);
  return 0;
#else
  (void)buf;
  set_error("mlora_trace_set: this library was built without MLORA_TRACE (make trace builds the variant that records timelines)");
  return MLORA_E_UNSUPPORTED;
#endif
}

extern "C" int mlora_choice(const MloraAddArgs* a, int32_t active_slots, int32_t active_tokens, int32_t* out) {
  out[0] = out[1] = out[2] = 0;
  const int rc = check_args(a);
  if (rc) return rc == kNothingToDo ? 0 : rc;
  const Batch batch = batch_of(a, active_slots, active_tokens);
  out[0] = chosen_form(a, batch);
  if (out[0] == MLORA_FORM_SGMV) out[1] = sgmv_parts(a, batch);
  if (out[0] == MLORA_FORM_WIDE) out[2] = wide_cut(a, batch).count;
  if (out[0] == MLORA_FORM_MFMA) decode_ranges(a, batch, &out[2]);
  return 0;
}

extern "C" void mlora_group_layout(int32_t num_tokens, int32_t num_slots, int64_t parts, int32_t extra, int32_t count, int32_t* out) {
  GroupPlaces p = {};
  p.T = num_tokens; p.num_slots = num_slots;
  out[1] = lay_out(p, &out[0], parts, extra);
  out[2] = p.slots8; out[3] = p.tiles; out[4] = p.width;
  out[5] = out[0] == kBySlot ? tile_width(p, count) : p.width;
  out[6] = out[0] == kBySlot ? tiles_beyond(p, count) : 0;
}
