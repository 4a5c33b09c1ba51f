// Computes, for decode-sized batches, what the reference computes with a shrink launch, a
// temporary [slices, T, r] tensor and one or two expand launches
// (nanovllm_voxcpm/lora.py:291-381 driving lora_ops/triton_ops/lora_shrink_op.py:16-173,
// lora_expand_op.py:11-91 and kernel_utils.py:7-228; its small-batch dispatch:
// lora_shrink_op.py:10-13, 176-210): y_i[t] += (x[t] . A_i[s_t]^T) . B_i[s_t]^T * scaling.
//
// Small-tile form: one workgroup per (small tile, slice, column range).  A small tile is up
// to sixteen tokens of one slot, described by a self-contained 128-byte record.
//
// A launch of this size (a few MB) is bound by fixed latencies and by how fast one compute
// unit takes data in (about 20 bytes per cycle, cache-resident or not), not by HBM bandwidth,
// so the kernel is built around the number of dependent round trips to memory and the launch
// around the number of workgroups:
//   0. the scalar launch arguments arrive preloaded in SGPRs (the kernel takes them as plain
//      leading arguments for that purpose), so no fetch of the argument block comes first;
//   1. the plan header, the tile record, the token indices and the column-range entry are
//      fetched together — their addresses depend on nothing but the workgroup index — and one
//      branch-free test decides whether the workgroup has work;
//   2. every global load the workgroup needs — its K-range of the x rows and of A[slot], the
//      B[slot] rows and the y rows of its output spans — is issued before any arithmetic;
//   3. column ranges are sized on the host so that a launch spreads over 150-250 workgroups.
// Both products run on the matrix cores (v_mfma_f32_16x16x32, fp32 accumulate): the sixteen
// token rows are one MFMA dimension, so a half-empty tile costs nothing but idle multiplier
// lanes.  The eight wavefronts split K for the shrink, sum their partial tiles through LDS,
// keep the rank-r intermediate there as a hi + lo pair of operand-precision values, and then
// each take 64-column spans of the expand; the B rows of a span are interleaved across its
// four MFMAs so that a lane owns consecutive columns and y is updated with wide accesses.
#include "common.h"
#include "launch.h"

#include <type_traits>

namespace mlora {

namespace {

constexpr int kMaxSplits = 32;
constexpr int kNW = 8;          // wavefronts per workgroup
constexpr int kSpansAheadMax = 2;  // output spans per wavefront whose loads are issued up front (SA: 1 or 2)

MLORA_TRACE_DECL

struct DecodeSplit {
  const void* a;
  const void* b;
  int n, y_col, n0, n1;
};

struct DecodeSplits {
  DecodeSplit split[kMaxSplits];
};

// KSPW: k-steps (32 elements of K) each wavefront covers when that is known at compile time
// (K = 32 * kNW * KSPW), 0 when it has to be worked out from K at run time.
//
// eff_rank (may be null): rank of the adapter resident in each slot.  16-rank blocks of A[slot] at
// or above it are neither fetched nor multiplied, the intermediate is zero from that rank on, and
// B[slot] elements from that rank on are replaced by zeros before they reach a multiplier.
//
// TR (KSPW a multiple of four): a compute unit's vector L1 handles a 128-bit load whose consecutive
// lanes touch different rows (what the MFMA operand layout asks for) at about a quarter of the
// rate of one whose lanes walk along a row, and even cache-resident operands showed up as
// 3-4 us per launch.  With TR the x rows and A rows of a wavefront's K range are fetched
// row-contiguously (sixteen lanes per 256 bytes of a row) and turned into operand layout through
// a private LDS block per wavefront, and the expand runs with the tokens as MFMA rows, so that
// sixteen consecutive lanes cover 128 contiguous bytes of one y row.
//
// SA: spans per wavefront requested up front.  A launch whose column ranges are at most 512 columns
// wide (one span per wavefront) takes the instance with SA = 1: the second span's requests, though
// clamped to a line or two, cost 0.2 us per launch (o 4.31 -> 4.07, qkv 4.44 -> 4.25, down 7.02 -> 6.81).
//
// GR (with MASKED): the buffers' rank is `rbuf_arg` < R, a multiple of eight (24 in the instance for
// 32; 40, 48, 56 in the one for 64): rows of A[slot] are rbuf * K apart, B rows rbuf elements long, and
// whatever lies beyond rbuf is treated like the ranks beyond an adapter's own (requests clamped
// into the buffers, values masked).
// Two workgroups per compute unit (at most 128 registers) where the LDS holds two: up to rank 16 and K = 2048, where the last text alone stays
// below that by itself and three texts with two spans (rank 8 150 registers, rank 16 146) would not, nor the last with y leaving at once (masked, rank 16, two spans: 129
// registers, q|k|v of 3001 tokens at K = 2048 17.7 -> 19.5 us).  us per call with one / two, every tile short, K = 2048,
// rank 8: gate_up of 64 tokens of 32 slots 8.3 / 6.8, of 256 of 64 16.6 / 13.5, q|k|v of 128 of 64 5.4 / 4.8; rank 16: 9.3 / 7.7, 19.1 / 16.2, 6.6 / 6.4.
// Nothing at K = 3072, rank 8, where the bound spills (o of 16 tokens of 16 slots 4.27 / 4.39).  (Rank 32 in 72 KB, its blocks of A staged one by one, and
// 128 registers: q|k|v of 1234 tokens at K = 2048 15.4 -> 14.9, but gate_up of 600 at K = 1024 12.5 -> 13.4, o of 2000 8.2 -> 8.7.)
constexpr int decode_waves(int r, int kspw, bool bound) { return bound && r <= 16 && kspw <= 8 ? 4 : 2; }

// SHORT (staged form): with a text each for tiles of up to four, up to eight and more tokens (below); without, the last one alone.
// THROUGH (staged form): y leaves at once (store_through), in instances of its own: a branch on it around every store costs calls with plain stores
// 1 to 3 % (0.1 us; a prompt of 37 tokens, 96 calls, 500 -> 507 us), one around a span's 0.3 to 1 %.
template <typename T, int R, int KSPW, bool TR, bool MASKED, int SA, bool GR, bool SHORT, bool THROUGH>
__global__ __launch_bounds__(kNW* kWave, decode_waves(R, KSPW, SHORT || THROUGH)) void decode_kernel(const int32_t* __restrict__ plan, const void* __restrict__ xv,
                                                            void* __restrict__ yv_, int64_t xs, int64_t ys, int small_off,
                                                            int include_long, int T_, int K, int num_slots, float scaling,
                                                            const int32_t* __restrict__ eff_rank, int rbuf_arg, DecodeSplits splits) {
  static_assert(!GR || (MASKED && R >= 32), "buffers of a rank between the instances' take the masked code of the next instance up");
  constexpr int RB = (R + 15) / 16;      // 16-rank blocks of the shrink output
  constexpr int KSTEPS = (R + 31) / 32;  // MFMA k-steps of the expand
  constexpr int HSTRIDE = R + 8;         // padded LDS row of the intermediate
  constexpr int NT = kNW * kWave;
  constexpr int CH = TR ? 4 : KSPW > 0 ? KSPW : 4;  // k-steps whose operands are in registers together
  constexpr int ROUNDS = TR ? KSPW / 4 : 1;          // staged form: groups of four k-steps per wavefront

  __shared__ __attribute__((aligned(16))) float s_red[kNW * RB * 64 * 4];
  __shared__ __attribute__((aligned(16))) T s_hi[16 * HSTRIDE];
  __shared__ __attribute__((aligned(16))) T s_lo[16 * HSTRIDE];
  constexpr int kStageRow = 17;  // 16 chunks of 16 bytes + one of padding: operand reads hit every bank once
  constexpr int SB = RB < 2 ? RB : 2;  // 16-rank blocks of A staged together (rank 64 goes through in two passes)
  __shared__ __attribute__((aligned(16))) i32x4 s_stage[TR ? kNW * (1 + SB) * 16 * kStageRow : 1];
  static_assert(!TR || (KSPW >= 4 && KSPW % 4 == 0), "the staged form takes the k-steps of a wavefront four at a time");

  const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
  const int lr = lane & 15, lg = lane >> 4;
  const int rbuf = GR ? rbuf_arg : R;  // rank of the buffers: row count of A[slot], row length of B
  MLORA_STAMP(0);  // first instruction

  // grid (8, column ranges, tiles / 8): linear workgroup ids advance along x first and
  // consecutive ids go to consecutive XCDs, so blockIdx.x is the XCD: the column ranges of one
  // tile share an XCD and its L2.
  const int split_id = blockIdx.y;
  const int tile = blockIdx.z * 8 + blockIdx.x;

  // URGENT: up to the x and A rows a wavefront goes before those that are at their B rows and y: 64 tokens of 32 slots, rank 32, q|k|v 4.47 -> 4.31 us per call,
  // o of 100 tokens of 60 4.36 -> 4.19.  Not with two spans each (gate_up of 200 tokens of 30, rank 24, 8.15 -> 8.37) and not with two
  // workgroups on a compute unit (3001 tokens, K = 2048, rank 16, q|k|v 14.0 -> 16.4); nothing at the other ranks.
  constexpr bool URGENT = TR && KSPW == 4 && SA == 1 && R == 32;
  if constexpr (URGENT) __builtin_amdgcn_s_setprio(3);

  // ---- round trip 1 ---------------------------------------------------------------------------
  const int32_t* rec = plan + small_off + tile * MLORA_SMALL_TILE_WORDS;  // tile < capacity: in bounds
  const int row = rec[MLORA_SMALL_TILE_ROWS + lr];
  // staged form: row 4 * lg + i of the products is token lg + 4 * i of the tile, so that the tokens of a tile of up to four or
  // eight are the rows i = 0 or i < 2 of every lane group and the requests of the others are left out (64 tokens of 32 slots, rank 32, us per
  // call: q|k|v 4.70 -> 4.48, gate_up 7.55 -> 7.15)
  i32x4 rows4;
  if constexpr (SHORT) {
#pragma unroll
    for (int i = 0; i < 4; ++i) rows4[i] = rec[MLORA_SMALL_TILE_ROWS + 4 * i + lg];
  } else {
    rows4 = *reinterpret_cast<const i32x4*>(rec + MLORA_SMALL_TILE_ROWS + 4 * lg);  // tokens 4 * lg .. + 3
  }
  const i32x4 rec0 = *reinterpret_cast<const i32x4*>(rec);       // slot, count, start, 0
  typedef int i32x16 __attribute__((ext_vector_type(16)));
  const DecodeSplit sp = splits.split[split_id];
  const i32x16 hdr = *reinterpret_cast<const i32x16*>(plan);  // the whole header in one scalar load
  const RankPrefetch ranks = rank_prefetch(MASKED ? eff_rank : nullptr, num_slots, lane);
  // (everything above is requested before anything below is scheduled: left to itself the
  // compiler requests this launch's column range only after the header has arrived)
  __builtin_amdgcn_sched_barrier(0);
  const int slot = rec0[0], m = rec0[1];
  const int n_tiles = hdr[MLORA_PLAN_TILES_SHORT] + hdr[MLORA_PLAN_TILES_LONG_SMALL] * include_long;
  // One exit test, evaluated without short-circuit, that consumes everything fetched above
  // (the token index through its first lane), so that all of it is requested here, together,
  // instead of piece by piece behind a chain of branches.
  const int usable = int(hdr[MLORA_PLAN_MAGIC] == MLORA_PLAN_MAGIC_VALUE) & int(hdr[MLORA_PLAN_NUM_TOKENS] == T_) &
                     int(hdr[MLORA_PLAN_MAX_SLOTS] == num_slots) & int(tile < n_tiles) & int(m > 0) &
                     int(slot < num_slots) & int(sp.n0 < sp.n1) & int(sp.a != nullptr) & int(sp.b != nullptr) &
                     int(sp.n > 0) & int(sp.y_col >= 0) & int(__builtin_amdgcn_readfirstlane(row) >= 0) &
                     int(__builtin_amdgcn_readfirstlane(SHORT ? rows4[0] | rows4[1] | rows4[2] | rows4[3] : rows4[0]) >= 0);
  if (!usable) {
    count_rejected_plan(plan, hdr[MLORA_PLAN_MAGIC] == MLORA_PLAN_MAGIC_VALUE && hdr[MLORA_PLAN_NUM_TOKENS] == T_ &&
                                  hdr[MLORA_PLAN_MAX_SLOTS] == num_slots);
    return;
  }
  MLORA_STAMP(1);  // tile record and plan header are here

  // rank of the adapter in this slot (requested together with the record, see rank_prefetch)
  // (MASKED = false is the instance for callers that gave no rank vector: eff is the constant R
  // there and every test on it below folds away)
  int eff = MASKED ? rank_pick(ranks, eff_rank, num_slots, slot, R) : R;
  if (GR && eff > rbuf) eff = rbuf;
  if (MASKED && eff == 0) return;
  const int rb_n = MASKED ? (eff + 15) >> 4 : RB;  // 16-rank blocks of A in use

  const bool live = lr < m;  // this lane's token exists
  const T* xrow = static_cast<const T*>(xv) + static_cast<int64_t>(row) * xs + lg * 8;
  const T* A = static_cast<const T*>(sp.a) + static_cast<int64_t>(slot) * rbuf * K;
  const T* arow[RB];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
    const int rr = rb * 16 + lr;
    arow[rb] = A + static_cast<int64_t>(rr < rbuf ? rr : rbuf - 1) * K + lg * 8;
  }
  const T* B = static_cast<const T*>(sp.b) + static_cast<int64_t>(slot) * sp.n * rbuf;
  T* yrow = static_cast<T*>(yv_) + static_cast<int64_t>(row) * ys + sp.y_col + 16 * lg;

  // XI: rows of a lane group that hold tokens.  What follows is written once per XI (a test in front of single requests would cost more than the
  // requests), in the text of decode_rest.h.
  if constexpr (SHORT) {
    auto rest = [&](auto xi) __attribute__((always_inline)) {
      constexpr int XI = decltype(xi)::value;
#include "decode_rest.h"
    };
    const int tokens = __builtin_amdgcn_readfirstlane(m);
    if (tokens <= 4) rest(std::integral_constant<int, 1>{});
    else if (tokens <= 8) rest(std::integral_constant<int, 2>{});
    else rest(std::integral_constant<int, 4>{});
  } else {
    // (the text itself: as a lambda its code comes out in another order, 2 % slower for 155 tokens of 3 slots)
    constexpr int XI = 4;
#include "decode_rest.h"
  }
}

struct Launch {
  const MloraAddArgs* a;
  int small_off, include_long, staged, short_tiles, through;
  int widest;  // columns of the widest column range
  dim3 grid;
  const DecodeSplits* splits;
};

template <typename T, int R, int KSPW, bool TR, bool MASKED, int SA, bool GR, bool SHORT, bool THROUGH>
void launch_texts(const Launch& l) {
  const MloraAddArgs* a = l.a;
  hipLaunchKernelGGL((decode_kernel<T, R, KSPW, TR, MASKED, SA, GR, SHORT, THROUGH>), l.grid, dim3(kNW * kWave), 0, static_cast<hipStream_t>(a->stream),
                     a->plan, a->x, a->y, a->x_stride, a->y_stride, l.small_off, l.include_long, a->num_tokens, a->k,
                     a->num_slots, a->scaling, a->effective_rank, a->r, *l.splits);
}

template <typename T, int R, int KSPW, bool TR, bool MASKED, int SA, bool GR = false>
void launch_spans(const Launch& l) {
  if constexpr (TR) {
    if (l.short_tiles) return launch_texts<T, R, KSPW, TR, MASKED, SA, GR, true, false>(l);
    if constexpr (KSPW <= 8) {
      if (l.through) return launch_texts<T, R, KSPW, TR, MASKED, SA, GR, false, true>(l);
    }
  }
  launch_texts<T, R, KSPW, TR, MASKED, SA, GR, false, false>(l);
}

// One span per wavefront up front when no column range holds more (staged form; the other form
// keeps its two).
template <typename T, int R, int KSPW, bool TR, bool MASKED>
void launch_masked(const Launch& l) {
  if constexpr (TR) {
    if (l.widest <= kNW * 64) return launch_spans<T, R, KSPW, TR, MASKED, 1>(l);
  }
  launch_spans<T, R, KSPW, TR, MASKED, kSpansAheadMax>(l);
}

// With a rank vector the instance that reads it; without, the one that has no such code at all.
template <typename T, int R, int KSPW, bool TR = false>
void launch_one(const Launch& l) {
  if (l.a->effective_rank) launch_masked<T, R, KSPW, TR, true>(l);
  else launch_masked<T, R, KSPW, TR, false>(l);
}

// The steps-per-wavefront specialisations kept: 1, 2 and 4 (K = 256, 512, 1024) for every rank
// and 16 (K = 4096) where the loads of sixteen steps still fit the register file.
template <typename T, int R>
void launch_kspw(const Launch& l, int kspw) {
  if constexpr (R >= 32) {
    if (l.a->r != R) {
      // buffers of a rank between the instances' (24; 40, 48, 56): the masked code of this instance
      // with the buffers' rank as stride, in the staged form for K = 1024 and the general one else
      if (l.staged && kspw == 4) {
        if (l.widest <= kNW * 64) return launch_spans<T, R, 4, true, true, 1, true>(l);
        return launch_spans<T, R, 4, true, true, kSpansAheadMax, true>(l);
      }
      return launch_spans<T, R, 0, false, true, kSpansAheadMax, true>(l);
    }
  }
  if (l.staged) {
    // staged operands, the k-steps of a wavefront four at a time (rank 64 in two passes of 32 ranks
    // through the same LDS block); how many k-steps fit is a matter of registers: every load of
    // the workgroup's K range is issued before the first is used
    if (kspw == 4) return launch_one<T, R, 4, true>(l);
    if constexpr (R <= 32) {
      if (kspw == 8) return launch_one<T, R, 8, true>(l);
    }
    if constexpr (R <= 16) {
      if (kspw == 12) return launch_one<T, R, 12, true>(l);
      if (kspw == 16) return launch_one<T, R, 16, true>(l);
    }
  }
  if (kspw == 4) return launch_one<T, R, 4>(l);
  if (kspw == 2) return launch_one<T, R, 2>(l);
  if (kspw == 1) return launch_one<T, R, 1>(l);
  if constexpr (R <= 16) {
    if (kspw == 16) return launch_one<T, R, 16>(l);
  }
  launch_one<T, R, 0>(l);
}

template <typename T>
void launch_rank(const Launch& l, int r, int kspw) {
  switch (compute_rank(r)) {
    case 8: launch_kspw<T, 8>(l, kspw); break;
    case 16: launch_kspw<T, 16>(l, kspw); break;
    case 32: launch_kspw<T, 32>(l, kspw); break;
    default: launch_kspw<T, 64>(l, kspw); break;
  }
}

// Diagnostic knobs, read from the environment once per process.
struct DecodeKnobs {
  int generation = -1, staged, nt, short_tiles, through;
  void read() {
    generation = knob_generation();
    staged = env_int("MLORA_DECODE_STAGED", 1);
    nt = env_int("MLORA_DECODE_NT", 0);
    short_tiles = env_int("MLORA_DECODE_SHORT", -1);
    through = env_int("MLORA_DECODE_THROUGH", -1);
  }
};
const DecodeKnobs& decode_knobs() {
  static DecodeKnobs k;
  if (k.generation != knob_generation()) k.read();
  return k;
}

}  // namespace

// Columns per range of a launch, and the number of ranges (0: no columns).  Every range repeats the
// shrink of its tile, but a compute unit takes in only 30-60 bytes per cycle even from the L2, so a
// launch is fastest when its bytes are spread over 150-250 workgroups: ranges shrink down to 128
// columns for narrow projections and stay at 1024 (two 64-column spans per wavefront, all loads still
// in registers) for wide ones.  Measured per launch at 32 tiles: o 6.2 us at 1024 columns, 5.1 at 512,
// 4.7 at 256; gate_up 8.2 / 8.9 / 11.1.
// Above rank 16 a workgroup has its compute unit to itself, 32 on an XCD, and what does not fit runs in a second round that shrinks its tile
// anew: one slice whose ranges spill takes as many fewer as fit (o, K = 1024, 2000 / 2400 / 2800 tokens of 32 slots, in ranges of 832, 960 and 1024 columns: rank 64 11.5 / 18.3 /
// 13.2, rank 24 8.3 / 12.2 / 8.8; 2400 tokens in one range 12.2 and 8.3).
int decode_ranges(const MloraAddArgs* a, const Batch& batch, int* columns) {
  int nt = decode_knobs().nt;
  if (nt <= 0) {
    long long cols = 0;
    for (int i = 0; i < a->num_slices; ++i) cols += a->slices[i].n;
    const int segs = a->num_slots < a->num_tokens ? a->num_slots : a->num_tokens;
    const int by_tokens = (a->num_tokens + MLORA_TILE_SMALL - 1) / MLORA_TILE_SMALL;
    const long long tiles = segs > by_tokens ? segs : by_tokens;  // about the number of tiles in use
    nt = static_cast<int>(cols * tiles / 160);
    if (nt > 1024) nt = 1024;
    if (nt < 128) nt = 128;
    if (a->num_slices == 1 && a->r > 16) {
      const int n = a->slices[0].n, fit = 32 / ((small_tiles_about(batch) + 7) / 8);
      if ((n + nt - 1) / nt > fit && fit > 0 && (n + fit - 1) / fit <= 1024) nt = (n + fit - 1) / fit;
    }
  }
  if (nt < 64) nt = 64;
  nt = (nt + 63) & ~63;
  int total;
  for (;;) {
    total = 0;
    for (int i = 0; i < a->num_slices; ++i) total += (a->slices[i].n + nt - 1) / nt;
    if (total <= kMaxSplits) break;
    nt *= 2;
  }
  *columns = nt;
  return total;
}

// Whether there is an instance that asks for all of this K at once (launch_kspw); the general text walks K batch by batch.
bool decode_one_batch(const MloraAddArgs* a) {
  if (a->k == 1024) return true;
  return exact_rank(a->r) && (a->k == 256 || a->k == 512 || (a->k == 2048 && a->r <= 32) || ((a->k == 3072 || a->k == 4096) && a->r <= 16));
}

// Nothing in the kernel limits the size of x or y.
bool decode_supported(const MloraAddArgs*) { return true; }

void decode_trace_set(void* buf) {
#ifdef MLORA_TRACE
  (void)hipMemcpyToSymbol(HIP_SYMBOL(trace_buf), &buf, sizeof(buf));
#else
  (void)buf;
#endif
}

int launch_decode(const MloraAddArgs* a, bool include_long, const Batch& batch) {
  DecodeSplits splits;
  const PlanLayout lay = plan_layout(a->num_tokens, a->num_slots);
  int cap = lay.cap_small;
  if (!include_long) {  // a segment below the threshold is exactly one small tile
    const int segs = a->num_slots < a->num_tokens ? a->num_slots : a->num_tokens;
    if (segs < cap) cap = segs;
  }
  if (cap == 0) return 0;
  cap = (cap + 7) & ~7;

  Launch l;
  l.a = a; l.small_off = lay.small_off; l.include_long = include_long ? 1 : 0; l.splits = &splits;
  l.staged = decode_knobs().staged;
  // The texts for short tiles pay where there are some: prompts fill their tiles, and the launch's workgroups then run the last of three texts
  // for the price of the others (155 tokens of 3 slots, us per call without / with them: rank 48 q|k|v 8.4 / 8.6, gate_up 9.7 / 10.0, rank 32 5.5 / 5.6;
  // 64 tokens of 32 slots, rank 32, 4.8 / 4.5 and 7.5 / 7.1): up to twelve tokens per slot with tokens.  With two spans per wavefront, whose texts
  // are longer, up to four (128 tokens of 16 slots, K = 2048, rank 16, gate_up 7.4 / 7.9; 200 of 30, rank 24, 8.2 / 8.2; 100 of 60, rank 32, 12.1 / 11.3).
  // Behind a capture the slots of the buffers count for those with tokens: a graph is captured for batches of about one token per slot, and one that
  // then brings full tiles loses up to 3 % of a call (64 tokens of 3 of 48 slots, without / with the texts: rank 16, K = 2048, q|k|v 5.1 / 5.2, o 4.9 / 4.8; rank 32, K =
  // 1024, 4.4 / 4.5 and 4.2 / 4.3; rank 48 6.9 / 6.9, gate_up 9.3 / 9.5), less than short tiles would lose without.

  int nt;
  const int total = decode_ranges(a, batch, &nt);
  if (total == 0) return 0;
  int s = 0;
  l.widest = 0;
  for (int i = 0; i < a->num_slices; ++i) {
    const MloraSlice& sl = a->slices[i];
    for (int n0 = 0; n0 < sl.n; n0 += nt) {
      DecodeSplit& d = splits.split[s++];
      d.a = sl.a; d.b = sl.b; d.n = sl.n; d.y_col = sl.y_col;
      d.n0 = n0; d.n1 = n0 + nt < sl.n ? n0 + nt : sl.n;
      if (d.n1 - d.n0 > l.widest) l.widest = d.n1 - d.n0;
    }
  }
  l.short_tiles = decode_knobs().short_tiles < 0 ? batch.tokens <= (l.widest <= kNW * 64 ? 12 : 4) * batch.slots : decode_knobs().short_tiles != 0;
  long long cols = 0;
  for (int i = 0; i < a->num_slices; ++i) cols += a->slices[i].n;
  // (three slices above rank 16 lose by it, q|k|v of 2 to 8 MB 1 %, of more 1.5 %; the line itself stands at store_through)
  l.through = decode_knobs().through < 0 ? batch.tokens * cols * 2 >= kThroughBytes && (a->num_slices < 3 || a->r <= 16) : decode_knobs().through != 0;
  for (; s < kMaxSplits; ++s) splits.split[s] = DecodeSplit{nullptr, nullptr, 0, 0, 0, 0};
  l.grid = dim3(8, static_cast<unsigned>(total), static_cast<unsigned>(cap / 8));
  const int nks = a->k / 32;
  const int kspw = (nks % kNW == 0) ? nks / kNW : 0;
  if (a->dtype == MLORA_DTYPE_BF16) launch_rank<__bf16>(l, a->r, kspw);
  else launch_rank<_Float16>(l, a->r, kspw);
  return check_launch("mlora_add_lora(small tiles, one workgroup per column range)");
}

}  // namespace mlora
