/*
 * mlora_diag.h - measurement and test aids of the MI355X multi-LoRA library.  Nothing here has a
 * counterpart in the reference and nothing here is needed to use the library: include/mlora.h is
 * the product's C-ABI.
 *
 * mlora_probe_launch, mlora_trace_set, mlora_group_layout and mlora_choice are exported by the diagnostic variants only
 * (libmlora_gfx950_diag.so from `make diag`, libmlora_gfx950_trace.so from `make trace`).
 * mlora_reload_knobs is exported by every variant: the test-suite changes MLORA_* variables
 * between tests of one process.
 */
#ifndef MLORA_DIAG_H_
#define MLORA_DIAG_H_

#include <stdint.h>

#include "mlora.h"

#ifdef __cplusplus
extern "C" {
#endif

/* Diagnostic knobs (the MLORA_* environment variables) are read once per process and kept;
 * this makes the next call read them again. */
void mlora_reload_knobs(void);

/* Launches of known cost: kind 0 enqueues a kernel that does nothing with the given grid and
 * workgroup size (what a launch costs by itself); kind 1 a read-modify-write stream over `bytes`
 * of 16-bit elements at `buf` (every element read, incremented, written back once: the access
 * pattern of y); kind 2 a read-only stream over them; kind 3 a kernel of the given grid whose
 * workgroups each write the number of the XCD they run on to `buf` (int32 per workgroup, linear
 * workgroup order: the placement the kernels' grids of x extent 8 rely on can be checked). */
int mlora_probe_launch(void* stream, int32_t kind, void* buf, int64_t bytes, int32_t grid_x, int32_t grid_y, int32_t grid_z,
                       int32_t threads);

/* In-kernel timelines.  The variant built with `make trace` records, per workgroup of the apply
 * kernels, up to 16 readings of the 100 MHz clock at fixed points of the kernel into `buf`
 * (uint64 [workgroups][16], device memory the caller zeroes; NULL switches recording off).  The
 * diag variant returns MLORA_E_UNSUPPORTED. */
int mlora_trace_set(void* buf);

/* How the low-level ops over tiles of a slot are laid over a grid of `parts` workgroups per place (host
 * arithmetic, nothing is launched; num_tokens and num_slots at least 1, parts at least 1): out[0] 1 if
 * over the tokens, 0 if over the slots, out[1] places, out[2] slot ids rounded up to eight, out[3]
 * tiles of a slot with a place of their own, out[4] tokens of a narrow tile; of a slot that has
 * `count` tokens, out[5] tokens of its tiles, out[6] tiles beyond those with a place of their own.
 * `extra` is 1 where the tokens without a slot need places (the shrink), else 0. */
void mlora_group_layout(int32_t num_tokens, int32_t num_slots, int64_t parts, int32_t extra, int32_t count, int32_t* out);

/* What mlora_add_lora_counts would take for a call (host arithmetic, nothing is launched; the same error codes): out[0] the form,
 * 0 where there is nothing to do, out[1] the K parts of MLORA_FORM_SGMV, out[2] the columns per range of MLORA_FORM_WIDE and
 * MLORA_FORM_MFMA. */
int mlora_choice(const MloraAddArgs* args, int32_t active_slots, int32_t active_tokens, int32_t* out);

#ifdef __cplusplus
}
#endif
#endif /* MLORA_DIAG_H_ */
