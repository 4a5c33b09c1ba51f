// The small-tile fused apply of decode.hip (one workgroup per (<= 16 tokens of one slot, column
// range), both products on the matrix cores; same arithmetic, same order, same bits) with the grid
// laid over the SLOTS instead of over the tiles.  Computes what the reference computes with a
// shrink launch, a temporary [slices, T, r] tensor and one or two expand launches
// (nanovllm_voxcpm/lora.py:291-381, lora_ops/triton_ops/lora_shrink_op.py:16-173,
// lora_expand_op.py:11-91).
//
// Why a second grid.  A decode launch lives for three to five trips to memory, and in the
// tile-major kernel the first of them fetches nothing but the 128-byte tile record: which slot a
// workgroup serves is written there, so not one operand can be requested before it has arrived.
// More than half of a decode launch's bytes are A[slot] and B[slot], and their addresses need the
// slot id only.  Here the slot id IS the workgroup index: workgroup (x, range, z) serves slot
// 8 z + x, so it requests the slot's record (its first sixteen tokens) and right behind it, without
// waiting, every A line it will need; the record is waited for while they are on their way, and
// only the x and y rows (whose addresses are token indices) hang on it.  The B rows, which need the
// slot id alone as well, go out behind the x rows: nothing uses them before the expand, and a
// compute unit hands over only so many requests at a time, so in front of the record's wait they
// held the x rows up (gate_up: 32 KB of A and 32 KB of B per workgroup).  For that
// to be true the weight pointers must not need a fetch either: they are leading kernel arguments,
// which arrive preloaded in scalar registers with the wavefront (14 dwords: the record list, two
// slices' A and B, their widths, and a packed word).  A slot without tokens costs its workgroups
// the A lines they requested in vain; they leave as soon as the record says so.
//
// Tiles behind a slot's first sixteen tokens are taken by further workgroups of the same launch
// (z beyond the slot layers), which learn their slot from their record like the tile-major
// kernel: a batch with every token on one adapter spreads over as many workgroups as before.
//
// Long K (KP > 1: four or eight parts of 512 or 1024 columns).  What a compute unit can take in per unit of time is what bounds a decode
// launch (about 35 bytes per cycle, whether the lines come from HBM or from the L2), and with one
// workgroup per column range every range pulls ALL of x's tile and of A[slot]: at K = 4096 that is
// 256 KB per workgroup against 16 KB of B and y.  With KP > 1 the KP workgroups of a tile each take
// one K part AND one column range: a workgroup multiplies its part, publishes the 16 x r partial
// sums as tagged 64-bit words in the workspace's exchange area, picks up the other parts'
// words, adds all parts in part order (so every workgroup of the tile holds the same bits) and
// expands its columns.  The hand-over follows the protocol of split.hip: words are valid when
// their tag is the workspace's generation + 1, every workgroup of the grid reports once, which
// advances the generation, nothing is ever cleared.  Waiting is bounded: a workgroup
// whose partners' words are not there in time multiplies their parts itself, in their order.
#include "common.h"
#include "launch.h"

#include <type_traits>

namespace mlora {

namespace {

constexpr int kNW = 8;  // wavefronts per workgroup (NW: of those that share K out in parts of 512 columns, four)

MLORA_TRACE_DECL

// What a workgroup needs to know of its column range.
struct Range {
  const void* a;
  const void* b;
  int n, y_col, n0, n1;
};

// One tile.  EARLY: the slot is known from the workgroup index (slot_early) and A[slot] is
// requested before the record has arrived; otherwise the record names the slot.
// The operand path is the staged one of decode.hip: x rows and A rows of a wavefront's K range are
// fetched row-contiguously (sixteen lanes per 256 bytes of a row), turned into MFMA operand layout
// through a private LDS block per wavefront, and the expand runs with the tokens as MFMA rows.
// What the workgroups of a tile need to hand each other partial sums (KP > 1).
struct Exchange {
  uint32_t* ws;    // workspace head
  int spin_ticks;  // bound of the wait for the partners' words, in ticks of the 100 MHz clock (< 0: never accept any)
  int trusted;     // the head is known to be in a launch's or the initial state without carrying the signature
  int part;        // this workgroup's K part
  int64_t tile;    // which of the area's (tile, slice) places is theirs
};

typedef unsigned long long u64;

// GR (with MASKED): the buffers' rank is `rbuf` < R, a multiple of eight: rows of A[slot] are rbuf * K
// apart and B rows rbuf elements long; whatever lies beyond rbuf is treated like the ranks beyond
// an adapter's own (requests clamped into the buffers, values masked).
template <typename T, int NW, int R, int KSPW, int KP, bool MASKED, bool GR, int SA, bool EARLY>
__device__ __forceinline__ void slot_tile(const int32_t* __restrict__ rec, const int slot_early, const int early_ok, const int rbuf_arg, const Range sp,
                                          const int y_col0, const int y_col1, const int y_col2, const int slice, const void* __restrict__ xv,
                                          void* __restrict__ yv_, const int64_t xs, const int64_t ys,
                                          const int num_slots, const float scaling, const int32_t* __restrict__ eff_rank,
                                          const uint32_t check, int32_t* __restrict__ plan_hdr, const Exchange xc, float* __restrict__ s_red,
                                          T* __restrict__ s_hi, T* __restrict__ s_lo, i32x4* __restrict__ s_stage, int* __restrict__ s_ok) {
  constexpr int RB = (R + 15) / 16;      // 16-rank blocks of the shrink output
  constexpr int KSTEPS = (R + 31) / 32;  // MFMA k-steps of the expand
  constexpr int HSTRIDE = R + 8;         // padded LDS row of the intermediate
  constexpr int NT = NW * kWave;
  constexpr int ROUNDS = KSPW / 4;       // groups of four k-steps per wavefront
  constexpr int KPART = 32 * NW * KSPW;  // columns of x and A one workgroup multiplies
  constexpr int K = KPART * KP;           // row length of A[slot]
  constexpr int WORDS = RB * 256;         // partial sums of one (tile, K part), in the order of the shared sum below
  constexpr int EPT = (WORDS + NT - 1) / NT;  // of which a thread holds this many
  constexpr int kStageRow = 17;          // 16 chunks of 16 bytes + one of padding
  constexpr int SB = RB < 2 ? RB : 2;    // 16-rank blocks of A staged together
  constexpr bool K16 = R == 16;          // expand on the 16x16x16 MFMA: 64-bit operand pieces
  static_assert(!GR || (MASKED && R >= 32), "buffers of a rank between the instances' take the masked code of the next instance up");
  static_assert(KSPW >= 4 && KSPW % 4 == 0, "the k-steps of a wavefront are taken four at a time");

  const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
  const int lr = lane & 15, lg = lane >> 4;
  const int rbuf = GR ? rbuf_arg : R;  // rank of the buffers: row count of A[slot], row length of B

  // URGENT: up to the x rows a wavefront goes before those that are at their B rows and y.  With two spans each those are half of what a compute
  // unit hands over: 256 tokens of 32 slots, rank 16, gate_up 6.44 -> 6.21 us per call; with one span it costs more than it brings (o of 64 tokens
  // of 32, rank 32, 3.9 -> 4.1), and above rank 16 too (352 of 28, rank 32, gate_up 12.7 -> 13.0).
  constexpr bool URGENT = KP == 1 && SA == 2 && R <= 16;
  if constexpr (URGENT) __builtin_amdgcn_s_setprio(3);

  // ---- requests that depend on nothing but the workgroup index --------------------------------
  // (the token rows as a vector load, four per lane group: all sixteen through the scalar cache
  // into scalar registers measured slower, 556 -> 598 us per decode step in the tile-major kernel)
  // SPREAD: row 4 * lg + i of the products is token lg + 4 * i of the tile, so the tokens of a tile of up to four or eight are the rows i = 0
  // or i < 2 of every lane group, and what the others would fetch (the tile's tokens once more) is left out instruction by
  // instruction: handing requests over is what a wavefront spends its first microsecond on.  us per call, before / after: one token of 8 slot
  // ids, rank 32, q|k|v 3.87 / 3.54, o 3.65 / 3.31; 64 tokens of 32, o 4.30 / 3.87; 256 of 32, rank 16, q|k|v 3.98 / 3.91, o 3.65 / 3.57.
  // Not for K parts, which wait for each other rather than for their requests (64 of 32 6.04 / 6.06), nor for two spans per wavefront (256 of
  // 32, gate_up 6.44 / 6.64: workgroups of three texts side by side).
  constexpr bool SPREAD = EARLY && KP == 1 && SA == 1;
  i32x4 rows4;
  if constexpr (SPREAD) {
#pragma unroll
    for (int i = 0; i < 4; ++i) rows4[i] = rec[MLORA_SMALL_TILE_ROWS + 4 * i + lg];
  } else {
    rows4 = *reinterpret_cast<const i32x4*>(rec + MLORA_SMALL_TILE_ROWS + 4 * lg);
  }
  const i32x4 rec0 = *reinterpret_cast<const i32x4*>(rec);                                     // slot, count, start, check
  int eff_early = R;
  if constexpr (MASKED && EARLY) {
    if (eff_rank) eff_early = eff_rank[slot_early];
  }
  const RankPrefetch ranks = rank_prefetch((MASKED && !EARLY) ? eff_rank : nullptr, num_slots, lane);
  if constexpr (EARLY) __builtin_amdgcn_sched_barrier(0);  // the record's requests go out first

  const int kp = KP > 1 ? xc.part : 0;  // this workgroup's K part (and column range)
  const int ks0 = kp * (KPART / 32) + wave * KSPW;
  // the workspace's state and signature (KP > 1): requested with the record (requested behind the A rows, or behind
  // the record, they cost up to 0.7 us more: 64 tokens of 32 slots, K = 2048, rank 64 masked 8.4 / 9.2 / 9.1 us per call)
  uint32_t signature = 0;
  WsState state = {0, 0, 0, 0};
  if constexpr (KP > 1) {
    signature = xc.ws[0];
    state = ws_state(xc.ws, blockIdx.x);
  }
  i32x4 ast[RB][4 * ROUNDS];
  Pack8 bop[SA][4][KSTEPS];
  // every A line of this wavefront's K range
  auto request_a = [&](const int slot, const int rb_n) {
    const T* A = static_cast<const T*>(sp.a) + static_cast<int64_t>(slot) * rbuf * K;
#pragma unroll
    for (int r = 0; r < ROUNDS; ++r) {
      const int64_t koff = static_cast<int64_t>(ks0 + 4 * r) * 32 + (lane & 15) * 8;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) {
          const int rr = rb * 16 + 4 * lg + i;
          if (!MASKED || EARLY || RB == 1 || rb < rb_n) ast[rb][4 * r + i] = load128(A + static_cast<int64_t>(rr < rbuf ? rr : rbuf - 1) * K + koff);
          else ast[rb][4 * r + i] = i32x4{0, 0, 0, 0};
        }
      }
    }
  };
  // the B rows of its spans
  auto request_b = [&](const int slot) {
    const T* B = static_cast<const T*>(sp.b) + static_cast<int64_t>(slot) * sp.n * rbuf;
#pragma unroll
    for (int s = 0; s < SA; ++s) {
      const int c0 = sp.n0 + (wave + s * NW) * 64;
      // requested whether the span exists or not (addresses clamped into the range)
      if constexpr (K16) {
        // a span's 64 B rows of 32 bytes are 2 KB of contiguous memory: fetched as such
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          int n = c0 + 32 * h + (lane >> 1);
          n = n < sp.n1 ? n : sp.n1 - 1;
          bop[s][h][0].raw = load128(B + static_cast<int64_t>(n) * R + (lane & 1) * 8);
        }
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          int n = c0 + 4 * lr + j;
          n = n < sp.n1 ? n : sp.n1 - 1;
#pragma unroll
          for (int ks = 0; ks < KSTEPS; ++ks) {
            int kc = (lg + 4 * ks) & (R / 8 - 1);
            if (GR && kc * 8 >= rbuf) kc = rbuf / 8 - 1;  // (masked where it is used)
            bop[s][j][ks].raw = load128(B + static_cast<int64_t>(n) * rbuf + kc * 8);
          }
        }
      }
    }
  };
  // The requests made in vain by a workgroup that turns out to have no work: waited for, and named
  // as used on that path too, so that the compiler cannot move them behind the test on the record
  // (left to itself it sinks every load into the only path that uses it).
  auto settle_requests = [&]() {
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
      for (int j = 0; j < 4 * ROUNDS; ++j) asm volatile("" ::"v"(ast[rb][j]));
  };
  if constexpr (EARLY) request_a(slot_early, RB);
  // (everything above is requested before anything below is scheduled)
  __builtin_amdgcn_sched_barrier(0);

  // ---- the record is here (the weights, when requested early, are still on their way) ---------
  const int slot = EARLY ? slot_early : rec0[0];
  const int m = rec0[1];
  const int matches = int(static_cast<uint32_t>(rec0[3]) == check);
  // (every word of the record takes part in the test: a word that nothing reads is a register the
  // compiler hands out again while the request is still on its way, and the write to it then
  // waits for the record in the middle of the requests for the weights)
  const int usable = matches & early_ok & int(m > 0) & int(slot >= 0) & int(slot < num_slots) & int(sp.n0 < sp.n1) &
                     int(__builtin_amdgcn_readfirstlane(SPREAD ? rows4[0] | rows4[1] | rows4[2] | rows4[3] : rows4[0]) >= 0) & int(rec0[2] >= 0) & int(!EARLY || rec0[0] == slot_early);
  // KP > 1: the exchange area can be used when the head is in the state a launch (or the
  // initialisation) left it in.  Every workgroup of the grid, with or without work, reports once
  // that it reads the area no more.
  const uint32_t generation = ws_generation(state), tag = generation + 1u;
  const bool xok = KP > 1 && (xc.trusted | ws_state_ok(signature, state));
  // (by the last wavefront, which has the fewest spans to expand)
  auto report = [&]() {
    if constexpr (KP > 1) {
      if (xok && tid == NT - kWave) ws_report(xc.ws, generation);
    }
  };
  if (!usable) {
    report();
    // a plan that was built for another batch shape (or never built): count the launch that found
    // it so, once (the first workgroup's record exists in every plan)
    if (!matches && EARLY && blockIdx.x == 0 && blockIdx.y == 0 && blockIdx.z == 0 && tid == 0 && plan_hdr)
      atomicAdd(plan_hdr + MLORA_PLAN_REJECTED, 1);
    if constexpr (EARLY) settle_requests();
    return;
  }
  MLORA_STAMP(1);
  // (the column offset of the slice inside y comes with the arguments that are not preloaded:
  // selected here, behind the wait for the record, it holds nothing up)
  const int y_col = slice == 0 ? y_col0 : slice == 1 ? y_col1 : y_col2;

  int eff = R;
  if constexpr (MASKED) {
    if constexpr (EARLY) {
      const int e = __builtin_amdgcn_readfirstlane(eff_early);
      eff = e < 0 ? 0 : e > R ? R : e;
    } else {
      eff = rank_pick(ranks, eff_rank, num_slots, slot, R);
    }
    if (GR && eff > rbuf) eff = rbuf;
    if (eff == 0) {
      report();
      if constexpr (EARLY) settle_requests();
      return;
    }
  }
  const int rb_n = MASKED ? (eff + 15) >> 4 : RB;  // 16-rank blocks of A in use
  if constexpr (!EARLY) request_a(slot, rb_n);

  // XI: rows of a lane group that hold tokens.  What follows the record is written once per XI (a test in front of single
  // requests would cost more than the requests), in the text of slot_rest.h.
  if constexpr (SPREAD) {
    auto rest = [&](auto xi) __attribute__((always_inline)) {
      constexpr int XI = decltype(xi)::value;
#include "slot_rest.h"
    };
    const int tokens = __builtin_amdgcn_readfirstlane(m);
    if (tokens <= 4) rest(std::integral_constant<int, 1>{});
    else if (tokens <= 8) rest(std::integral_constant<int, 2>{});
    else rest(std::integral_constant<int, 4>{});
  } else {
    // (the text itself, not the lambda: as a lambda the K parts' code comes out in another order, 4.85 -> 5.03 us for 37 tokens of one
    // slot, rank 32, K = 4096)
    constexpr int XI = 4;
#include "slot_rest.h"
  }
}

// Leading arguments up to `rbuf` (14 dwords) arrive preloaded in scalar registers: everything the
// early requests need.  packed = columns per range / 64 | ranges of slice 0 << 8 | slots << 16.
// A launch of one slice passes n1 = 0 (blockIdx.y never reaches a second slice).
// KP > 1: one slice, blockIdx.y is the workgroup's K part and column range alike (ranges of slice 0 = KP).
template <typename T, int NW, int R, int KSPW, int KP, bool MASKED, bool GR, int SA>
__global__ __launch_bounds__(NW* kWave) void slot_kernel(const int32_t* __restrict__ recs, const void* __restrict__ a0,
                                                          const void* __restrict__ b0, const void* __restrict__ a1,
                                                          const void* __restrict__ b1, int n0, int n1, uint32_t packed, int rbuf,
                                                          const void* __restrict__ xv, void* __restrict__ yv_, int64_t xs, int64_t ys,
                                                          int y_col0, int y_col1, uint32_t check, float scaling,
                                                          const int32_t* __restrict__ eff_rank, int32_t* __restrict__ plan_hdr,
                                                          uint32_t* __restrict__ ws, int spin_ticks, int trusted) {
  constexpr int RB = (R + 15) / 16;
  constexpr int HSTRIDE = R + 8;
  constexpr int kStageRow = 17;
  constexpr int SB = RB < 2 ? RB : 2;
  __shared__ __attribute__((aligned(16))) float s_red[NW * RB * 64 * 4];
  __shared__ __attribute__((aligned(16))) T s_hi[16 * HSTRIDE];
  __shared__ __attribute__((aligned(16))) T s_lo[16 * HSTRIDE];
  __shared__ __attribute__((aligned(16))) i32x4 s_stage[NW * (1 + SB) * 16 * kStageRow];
  __shared__ int s_ok;
  MLORA_STAMP(0);

  const int nt = static_cast<int>(packed & 255u) * 64, ranges0 = static_cast<int>((packed >> 8) & 255u);
  const int num_slots = static_cast<int>(packed >> 16);
  const int ri = blockIdx.y;
  const bool second = ri >= ranges0;
  Range sp;
  sp.a = second ? a1 : a0;
  sp.b = second ? b1 : b0;
  sp.n = second ? n1 : n0;
  sp.y_col = 0;  // (selected inside, late)
  sp.n0 = (second ? ri - ranges0 : ri) * nt;
  sp.n1 = sp.n0 + nt < sp.n ? sp.n0 + nt : sp.n;

  // grid (8, column ranges, slot layers + layers of further tiles): blockIdx.x is the XCD, so a
  // slot's column ranges share an L2
  const int zslots = (num_slots + 7) >> 3;
  const Exchange xc{ws, spin_ticks, trusted, static_cast<int>(blockIdx.y), static_cast<int64_t>(blockIdx.z * 8 + blockIdx.x)};
  if (static_cast<int>(blockIdx.z) < zslots) {
    const int s = blockIdx.z * 8 + blockIdx.x;  // its record exists: the list is rounded up to eight
    const int slot = s < num_slots ? s : num_slots - 1;
    slot_tile<T, NW, R, KSPW, KP, MASKED, GR, SA, true>(recs + s * MLORA_SMALL_TILE_WORDS, slot, int(s < num_slots), rbuf, sp, y_col0, y_col1, 0, int(second), xv, yv_,
                                                xs, ys, num_slots, scaling, eff_rank, check, plan_hdr, xc, s_red, s_hi, s_lo, s_stage, &s_ok);
  } else {
    const int q = zslots * 8 + (blockIdx.z - zslots) * 8 + blockIdx.x;
    slot_tile<T, NW, R, KSPW, KP, MASKED, GR, SA, false>(recs + q * MLORA_SMALL_TILE_WORDS, 0, 1, rbuf, sp, y_col0, y_col1, 0, int(second), xv, yv_, xs, ys, num_slots,
                                                 scaling, eff_rank, check, plan_hdr, xc, s_red, s_hi, s_lo, s_stage, &s_ok);
  }
}

// Three slices (the stacked q | k | v projection): six pointers do not fit the fourteen preloaded
// dwords, so the second and third slice's travel as 40-bit offsets from the first one's, in units of
// 16 bytes (+-8 TiB: the slices of a projection are allocations of their own and may lie far apart;
// the launcher takes this kernel only when they fit): their low 32 bits as four arguments, their
// high 8 bits together in a fifth; the widths as 16-bit counts of eight columns.  widths01 = n0 / 8 | n1 / 8 << 16; widths2 = n2 / 8 | ranges of slice 0 << 16 |
// ranges of slices 0 and 1 << 24; packed = columns per range / 64 | slots << 16.  KP > 1: KP ranges and K parts of
// every slice, of a width of its own.
template <typename T, int NW, int R, int KP, int SA, bool MASKED>
__global__ __launch_bounds__(NW* kWave) void slot_kernel3(const int32_t* __restrict__ recs, const void* __restrict__ a0,
                                                           const void* __restrict__ b0, uint32_t aoff1, uint32_t aoff2, uint32_t boff1, uint32_t boff2,
                                                           uint32_t off_high, uint32_t widths01, uint32_t widths2, uint32_t packed,
                                                           const void* __restrict__ xv, void* __restrict__ yv_, int64_t xs, int64_t ys,
                                                           int y_col0, int y_col1, int y_col2, uint32_t check, float scaling,
                                                           const int32_t* __restrict__ eff_rank, int32_t* __restrict__ plan_hdr,
                                                           uint32_t* __restrict__ ws, int spin_ticks, int trusted) {
  constexpr int RB = (R + 15) / 16;
  constexpr int HSTRIDE = R + 8;
  constexpr int kStageRow = 17;
  constexpr int SB = RB < 2 ? RB : 2;
  __shared__ __attribute__((aligned(16))) float s_red[NW * RB * 64 * 4];
  __shared__ __attribute__((aligned(16))) T s_hi[16 * HSTRIDE];
  __shared__ __attribute__((aligned(16))) T s_lo[16 * HSTRIDE];
  __shared__ __attribute__((aligned(16))) i32x4 s_stage[NW * (1 + SB) * 16 * kStageRow];
  __shared__ int s_ok;
  MLORA_STAMP(0);

  const int num_slots = static_cast<int>(packed >> 16);
  const int cum1 = static_cast<int>((widths2 >> 16) & 255u), cum2 = static_cast<int>(widths2 >> 24);
  const int ri = blockIdx.y;
  const int slice = KP > 1 ? ri / KP : int(ri >= cum1) + int(ri >= cum2);
  // (offset i: low word off_i, bits 32..39 in byte i of off_high, sign-extended)
  const uint32_t alo = slice == 1 ? aoff1 : aoff2, blo = slice == 1 ? boff1 : boff2;
  const int32_t ahi = static_cast<int8_t>(off_high >> (slice == 1 ? 0 : 8)), bhi = static_cast<int8_t>(off_high >> (slice == 1 ? 16 : 24));
  const int64_t ao = slice == 0 ? 0 : (static_cast<int64_t>(ahi) << 32) | alo, bo = slice == 0 ? 0 : (static_cast<int64_t>(bhi) << 32) | blo;
  Range sp;
  sp.a = static_cast<const char*>(a0) + ao * 16;
  sp.b = static_cast<const char*>(b0) + bo * 16;
  sp.n = 8 * static_cast<int>(slice == 0 ? widths01 & 0xffffu : slice == 1 ? widths01 >> 16 : widths2 & 0xffffu);
  sp.y_col = 0;  // (selected inside, late)
  const int part = KP > 1 ? ri % KP : ri - (slice == 0 ? 0 : slice == 1 ? cum1 : cum2);
  const int nt = KP > 1 ? ((sp.n + KP - 1) / KP + 63) & ~63 : static_cast<int>(packed & 255u) * 64;
  sp.n0 = part * nt;
  sp.n1 = sp.n0 + nt < sp.n ? sp.n0 + nt : sp.n;

  const int zslots = (num_slots + 7) >> 3;
  const Exchange xc{ws, spin_ticks, trusted, part, static_cast<int64_t>(blockIdx.z * 8 + blockIdx.x) * 3 + slice};
  if (static_cast<int>(blockIdx.z) < zslots) {
    const int s = blockIdx.z * 8 + blockIdx.x;
    const int slot = s < num_slots ? s : num_slots - 1;
    slot_tile<T, NW, R, 4, KP, MASKED, false, SA, true>(recs + s * MLORA_SMALL_TILE_WORDS, slot, int(s < num_slots), R, sp, y_col0, y_col1, y_col2, slice, xv,
                                                  yv_, xs, ys, num_slots, scaling, eff_rank, check, plan_hdr, xc, s_red, s_hi, s_lo, s_stage, &s_ok);
  } else {
    const int q = zslots * 8 + (blockIdx.z - zslots) * 8 + blockIdx.x;
    slot_tile<T, NW, R, 4, KP, MASKED, false, SA, false>(recs + q * MLORA_SMALL_TILE_WORDS, 0, 1, R, sp, y_col0, y_col1, y_col2, slice, xv, yv_, xs, ys,
                                                   num_slots, scaling, eff_rank, check, plan_hdr, xc, s_red, s_hi, s_lo, s_stage, &s_ok);
  }
}

// How a tile's K is shared out: between kp workgroups of nw wavefronts.
struct Parts { int kp, nw; };

struct Launch {
  const MloraAddArgs* a;
  dim3 grid;
  uint32_t packed;
  int widest;
  int spin_ticks, trusted;
};

// Offsets of slice i's A and B from slice 0's, in units of 16 bytes, when they fit 40 bits.
bool offsets16(const MloraAddArgs* a, int i, long long* ao, long long* bo) {
  const long long da = static_cast<const char*>(a->slices[i].a) - static_cast<const char*>(a->slices[0].a);
  const long long db = static_cast<const char*>(a->slices[i].b) - static_cast<const char*>(a->slices[0].b);
  if ((da & 15) || (db & 15)) return false;
  const long long qa = da / 16, qb = db / 16, lim = 1ll << 39;
  if (qa < -lim || qa >= lim || qb < -lim || qb >= lim) return false;
  *ao = qa;
  *bo = qb;
  return true;
}

template <typename T, int NW, int R, int KP, int SA>
void launch_three(const Launch& l, int nt, int cum1, int cum2) {
  const MloraAddArgs* a = l.a;
  const PlanLayout lay = plan_layout(a->num_tokens, a->num_slots);
  long long o[4] = {0, 0, 0, 0};  // A of slices 1 and 2, B of slices 1 and 2
  (void)offsets16(a, 1, &o[0], &o[2]);
  (void)offsets16(a, 2, &o[1], &o[3]);
  const uint32_t ao1 = static_cast<uint32_t>(o[0]), ao2 = static_cast<uint32_t>(o[1]), bo1 = static_cast<uint32_t>(o[2]), bo2 = static_cast<uint32_t>(o[3]);
  uint32_t high = 0;
  for (int i = 0; i < 4; ++i) high |= static_cast<uint32_t>((o[i] >> 32) & 0xff) << (8 * i);
  const uint32_t w01 = static_cast<uint32_t>(a->slices[0].n / 8) | (static_cast<uint32_t>(a->slices[1].n / 8) << 16);
  const uint32_t w2 = static_cast<uint32_t>(a->slices[2].n / 8) | (static_cast<uint32_t>(cum1) << 16) | (static_cast<uint32_t>(cum2) << 24);
  const uint32_t packed = static_cast<uint32_t>(nt / 64) | (static_cast<uint32_t>(a->num_slots) << 16);
  const uint32_t check = static_cast<uint32_t>(MLORA_PLAN_CHECK(a->num_tokens, a->num_slots));
  auto launch = [&](auto* kernel) {
    hipLaunchKernelGGL(kernel, l.grid, dim3(NW * kWave), 0, static_cast<hipStream_t>(a->stream), a->plan + lay.slotrec_off, a->slices[0].a,
                       a->slices[0].b, ao1, ao2, bo1, bo2, high, w01, w2, packed, a->x, a->y, a->x_stride, a->y_stride, a->slices[0].y_col,
                       a->slices[1].y_col, a->slices[2].y_col, check, a->scaling, a->effective_rank, const_cast<int32_t*>(a->plan),
                       static_cast<uint32_t*>(a->workspace), l.spin_ticks, l.trusted);
  };
  if (a->effective_rank) launch(slot_kernel3<T, NW, R, KP, SA, true>);
  else launch(slot_kernel3<T, NW, R, KP, SA, false>);
}

template <typename T, int NW, int R, int KSPW, int KP, bool MASKED, bool GR, int SA>
void launch_spans(const Launch& l) {
  const MloraAddArgs* a = l.a;
  const PlanLayout lay = plan_layout(a->num_tokens, a->num_slots);
  const MloraSlice& s0 = a->slices[0];
  const MloraSlice s1 = a->num_slices > 1 ? a->slices[1] : MloraSlice{nullptr, nullptr, 0, 0};
  hipLaunchKernelGGL((slot_kernel<T, NW, R, KSPW, KP, MASKED, GR, SA>), l.grid, dim3(NW * kWave), 0, static_cast<hipStream_t>(a->stream),
                     a->plan + lay.slotrec_off, s0.a, s0.b, s1.a, s1.b, s0.n, s1.n, l.packed, a->r, a->x, a->y, a->x_stride, a->y_stride,
                     s0.y_col, s1.y_col, static_cast<uint32_t>(MLORA_PLAN_CHECK(a->num_tokens, a->num_slots)), a->scaling,
                     a->effective_rank, const_cast<int32_t*>(a->plan), static_cast<uint32_t*>(a->workspace), l.spin_ticks, l.trusted);
}

// Instances of one span per wavefront alone for eight parts, of two alone for four parts of 512 columns.
template <typename T, int NW, int R, int KSPW, int KP>
void launch_one(const Launch& l) {
  constexpr int kTwo = KP == 8 ? 1 : 2, kOne = NW == 4 && KP == 4 ? 2 : 1;
  const bool one_span = KP == 8 || l.widest <= NW * 64;
  if constexpr (R >= 32) {
    if (l.a->r != R) {  // buffers of a rank between the instances': the masked code with the buffers' rank as stride
      if (one_span) launch_spans<T, NW, R, KSPW, KP, true, true, kOne>(l);
      else launch_spans<T, NW, R, KSPW, KP, true, true, kTwo>(l);
      return;
    }
  }
  if (l.a->effective_rank) {
    if (one_span) launch_spans<T, NW, R, KSPW, KP, true, false, kOne>(l);
    else launch_spans<T, NW, R, KSPW, KP, true, false, kTwo>(l);
  } else {
    if (one_span) launch_spans<T, NW, R, KSPW, KP, false, false, kOne>(l);
    else launch_spans<T, NW, R, KSPW, KP, false, false, kTwo>(l);
  }
}

template <typename T, int NW, int KSPW, int KP>
bool launch_ranks(const Launch& l, int r) {
  switch (r) {
    case 8: launch_one<T, NW, 8, KSPW, KP>(l); return true;
    case 16: launch_one<T, NW, 16, KSPW, KP>(l); return true;
    case 32: launch_one<T, NW, 32, KSPW, KP>(l); return true;
    case 64: launch_one<T, NW, 64, KSPW, KP>(l); return true;
  }
  return false;
}

// parts: of K (one: every workgroup multiplies the whole of it).
template <typename T>
bool launch_rank(const Launch& l, int rank, int k, Parts parts) {
  const int r = compute_rank(rank), each = k / parts.kp;
  if (parts.nw == 4 && each == 512) {
    if (parts.kp == 4) return launch_ranks<T, 4, 4, 4>(l, r);
    if (parts.kp == 8) return launch_ranks<T, 4, 4, 8>(l, r);
  } else if (parts.nw == kNW && each == 1024) {
    if (parts.kp == 1) return launch_ranks<T, kNW, 4, 1>(l, r);
    if (parts.kp == 4) return launch_ranks<T, kNW, 4, 4>(l, r);
    if (parts.kp == 8) return launch_ranks<T, kNW, 4, 8>(l, r);
  } else if (parts.nw == kNW && each == 4096 && parts.kp == 1) {
    switch (r) {
      case 8: launch_one<T, kNW, 8, 16, 1>(l); return true;
      case 16: launch_one<T, kNW, 16, 16, 1>(l); return true;
    }
  }
  return false;
}

// Columns per range: as in the tile-major launch, sized for 150-250 workgroups; at most 1024 (two
// 64-column spans per wavefront, all loads in registers).
int range_columns(const MloraAddArgs* a) {
  long long cols = 0;
  for (int i = 0; i < a->num_slices; ++i) cols += a->slices[i].n;
  const int segs = a->num_slots < a->num_tokens ? a->num_slots : a->num_tokens;
  const int by_tokens = (a->num_tokens + MLORA_TILE_SMALL - 1) / MLORA_TILE_SMALL;
  const long long tiles = segs > by_tokens ? segs : by_tokens;  // about the number of tiles in use
  int nt = static_cast<int>(cols * tiles / 160);
  if (nt > 1024) nt = 1024;
  if (nt < 128) nt = 128;
  nt = (nt + 63) & ~63;
  while (nt < 1024) {
    int total = 0;
    for (int i = 0; i < a->num_slices; ++i) total += (a->slices[i].n + nt - 1) / nt;
    if (total <= 32) break;
    nt *= 2;
  }
  return nt > 1024 ? 1024 : nt;
}

int kspw_of(const MloraAddArgs* a) { return a->k % (32 * kNW) == 0 ? a->k / (32 * kNW) : 0; }

// Diagnostic knobs, read from the environment once per process.
struct SlotKnobs {
  int generation = -1, kparts, spin_ticks;
  void read() {
    generation = knob_generation();
    kparts = env_int("MLORA_SLOT_KPARTS", 0);          // 1: never share K out between workgroups
    spin_ticks = env_int("MLORA_SLOT_SPIN_TICKS", 20000);  // 200 us; 0: do not wait; < 0: never accept a partner's words
  }
};
SlotKnobs& slot_knobs() {
  static SlotKnobs k;
  if (k.generation != knob_generation()) k.read();
  return k;
}

// Whether a tile's workgroups can hand each other the partial sums of these parts: columns for every part, an
// instance for their ranges, an exchange area that holds every tile's.
bool parts_fit(const MloraAddArgs* a, Parts p) {
  for (int i = 0; i < a->num_slices; ++i) {
    const int n = a->slices[i].n, nt = ((n + p.kp - 1) / p.kp + 63) & ~63;
    if (n < p.kp * 64 || (p.kp - 1) * nt >= n) return false;  // (a part without columns would leave the tile)
    const int spans = (nt + 64 * p.nw - 1) / (64 * p.nw);
    if (spans > 2 || (spans == 2 && (p.kp == 8 || (p.nw == kNW && a->r > 32)))) return false;  // (instances; registers beside the parts)
  }
  const PlanLayout lay = plan_layout(a->num_tokens, a->num_slots);
  const long long words = static_cast<long long>(lay.cap_slotrec + lay.cap_over) * a->num_slices * p.kp * ((compute_rank(a->r) + 15) / 16) * 256;
  return words * 8 <= kWsXchgBytes;
}

// K parts of a launch (one slice, or q | k | v at K = 2048 and rank 64; an initialised workspace), else one.  Of 1024 columns for eight wavefronts or of
// 512 for four: smaller parts take in less per compute unit, and there are twice as many workgroups that wait
// for each other, so K = 4096 is cut into eight while parts x tiles (or slot ids) are few (us per call in four parts / in
// eight: rank 16, 16 slot ids 4.7 / 4.4, 32 4.8 / 4.6, 40 4.9 / 5.0, 64 5.7 / 5.8; rank 32, 16 5.3 / 4.9, 24 5.5 / 5.4, 32 6.0 / 6.0, 40
// 6.3 / 7.8; rank 64, 16 7.5 / 7.1, 24 8.5 / 8.2, 32 9.2 / 10.5; 250 tokens of 8 slots of 32, rank 32 6.4 / 7.3).
// K = 2048 in four, 8192 in eight of 1024.
Parts k_parts(const MloraAddArgs* a) {
  const Parts one = {1, kNW};
  const bool three = a->num_slices == 3 && a->k == 2048 && a->r == 64;
  if (!(a->num_slices == 1 || three) || slot_knobs().kparts == 1) return one;
  if (!a->workspace || (reinterpret_cast<uintptr_t>(a->workspace) & 255) || a->workspace_bytes < MLORA_WORKSPACE_HEAD_BYTES) return one;
  const Parts small = {a->k / 512, 4}, large = {a->k / 1024, kNW};
  const int tiles = small_tiles_about(batch_of(a, 0, 0)), most = tiles > a->num_slots ? tiles : a->num_slots;
  if ((a->k == 2048 || (a->k == 4096 && 8 * most <= (a->r <= 16 ? 256 : 192))) && parts_fit(a, small)) return small;
  if ((a->k == 4096 || a->k == 8192) && parts_fit(a, large)) return large;
  return one;
}

}  // namespace

// K = 1024 at every rank; one slice of K = 2048, 4096 and 8192 at every rank with the K parts of a tile shared out between its
// workgroups, K = 4096 without up to rank 16 (what fits the register file as one batch of loads); one or two
// slices with their pointers as arguments, three (K = 1024 at the exact ranks, K = 2048 in K parts at rank 64) with the later
// two's as offsets from the first one's; 16-bit elements.
bool slot_supported(const MloraAddArgs* a) {
  if (a->dtype != MLORA_DTYPE_BF16 && a->dtype != MLORA_DTYPE_F16) return false;
  if (a->num_slices < 1 || a->num_slices > 3 || !a->plan) return false;
  long long cols = 0;
  for (int i = 0; i < a->num_slices; ++i) {
    if (a->slices[i].n <= 0) return false;
    cols += a->slices[i].n;
  }
  if (cols > 200 * 1024) return false;  // at most 255 column ranges of up to 1024 columns
  if (!padded_rank(a->r)) return false;
  const int kspw = kspw_of(a);
  if (a->num_slices == 3) {
    // q | k | v: an exact rank, offsets that fit 40 bits, widths that fit 16-bit counts of eight columns; K = 1024
    // with column ranges of at most 512 columns (one span per wavefront), or K = 2048 at rank 64 in K parts
    long long ao, bo;
    if (!exact_rank(a->r) || !offsets16(a, 1, &ao, &bo) || !offsets16(a, 2, &ao, &bo)) return false;
    for (int i = 0; i < 3; ++i)
      if (a->slices[i].n % 8 || a->slices[i].n / 8 > 0xffff) return false;
    if (kspw != 4) return k_parts(a).kp > 1;
    return range_columns(a) <= kNW * 64;
  }
  if (kspw == 4) return true;
  return k_parts(a).kp > 1 || (kspw == 16 && a->r <= 16);
}

int slot_k_parts(const MloraAddArgs* a) { return k_parts(a).kp; }

void slot_trace_set(void* buf) {
#ifdef MLORA_TRACE
  (void)hipMemcpyToSymbol(HIP_SYMBOL(trace_buf), &buf, sizeof(buf));
#else
  (void)buf;
#endif
}

int launch_slot(const MloraAddArgs* a, bool trusted_workspace) {
  const PlanLayout lay = plan_layout(a->num_tokens, a->num_slots);
  const Parts parts = k_parts(a);
  const int kp = parts.kp;
  // with K parts a (tile, slice)'s workgroups are its K parts and its column ranges alike
  const int nt = kp > 1 ? ((a->slices[0].n + kp - 1) / kp + 63) & ~63 : range_columns(a);
  const int ranges0 = kp > 1 ? kp : (a->slices[0].n + nt - 1) / nt;
  const int ranges1 = a->num_slices > 1 ? (a->slices[1].n + nt - 1) / nt : 0;
  const int total = kp > 1 ? a->num_slices * kp : ranges0 + ranges1 + (a->num_slices > 2 ? (a->slices[2].n + nt - 1) / nt : 0);
  if (total > 255) {
    set_error("mlora_add_lora(slot-major): %d column ranges exceed 255", total);
    return MLORA_E_UNSUPPORTED;
  }
  Launch l;
  l.a = a;
  l.packed = static_cast<uint32_t>(nt / 64) | (static_cast<uint32_t>(ranges0) << 8) | (static_cast<uint32_t>(a->num_slots) << 16);
  l.widest = 0;
  for (int i = 0; i < a->num_slices; ++i) {
    const int w = a->slices[i].n < nt ? a->slices[i].n : nt;
    if (w > l.widest) l.widest = w;
  }
  l.spin_ticks = slot_knobs().spin_ticks;
  l.trusted = trusted_workspace ? 1 : 0;
  l.grid = dim3(8, static_cast<unsigned>(total), static_cast<unsigned>((lay.cap_slotrec + lay.cap_over) / 8));
  if (a->num_slices == 3 && kp > 1) {
    if (a->dtype == MLORA_DTYPE_BF16) launch_three<__bf16, 4, 64, 4, 2>(l, nt, 0, 0);
    else launch_three<_Float16, 4, 64, 4, 2>(l, nt, 0, 0);
    return check_launch("mlora_add_lora(small tiles, K parts of three slices)");
  }
  if (a->num_slices == 3) {
    switch (a->r) {
#define MLORA_THREE(R)                                                                                      \
  case R:                                                                                                   \
    if (a->dtype == MLORA_DTYPE_BF16) launch_three<__bf16, kNW, R, 1, 1>(l, nt, ranges0, ranges0 + ranges1);   \
    else launch_three<_Float16, kNW, R, 1, 1>(l, nt, ranges0, ranges0 + ranges1);                              \
    break;
      MLORA_THREE(8)
      MLORA_THREE(16)
      MLORA_THREE(32)
      MLORA_THREE(64)
#undef MLORA_THREE
      default: set_error("mlora_add_lora(slot-major): unsupported rank %d for three slices", a->r); return MLORA_E_UNSUPPORTED;
    }
    return check_launch("mlora_add_lora(small tiles, one workgroup per slot and column range, three slices)");
  }
  const bool ok = a->dtype == MLORA_DTYPE_BF16 ? launch_rank<__bf16>(l, a->r, a->k, parts) : launch_rank<_Float16>(l, a->r, a->k, parts);
  if (!ok) {
    set_error("mlora_add_lora(slot-major): unsupported rank %d / K %d", a->r, a->k);
    return MLORA_E_UNSUPPORTED;
  }
  return check_launch("mlora_add_lora(small tiles, one workgroup per slot and column range)");
}

}  // namespace mlora
