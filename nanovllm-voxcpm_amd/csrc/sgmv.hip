// Computes, for prefill-sized batches, what the reference computes with its segment-grouped
// shrink and expand kernels (nanovllm_voxcpm/lora_ops/triton_ops/lora_shrink_op.py:16-101, 257-341,
// lora_expand_op.py:11-170, kernel_utils.py:7-228, launched from nanovllm_voxcpm/lora.py:291-381):
// y_i[t] += (x[t] . A_i[s_t]^T) . B_i[s_t]^T * scaling, tokens grouped by slot.
//
// SGMV form for batches above the small-batch limit: two launches that meet in a small
// workspace, both on the matrix cores (v_mfma_f32_16x16x32 bf16 / f16, fp32 accumulate).  Work
// units are the 64-token tiles of the long segments and, behind them in the same grids, the
// short segments (one small-tile record each).
//
//   shrink — H^T[rank x tokens] = A[slot] . X_tile^T for a (tile, slice, K part).  What bounds
//            this product is what a compute unit takes in (down of the prefill batch: 117 MB of x and A, 13.4 us as loads
//            alone), so each operand element is fetched once per workgroup, in whole row pieces straight to LDS, through a
//            ring of up to eight stages that the four wavefronts fill and read together.  No wavefront shares a sum with
//            another, so the accumulators go straight to the
//            workspace as fp32; when K is split across workgroups each part writes its own
//            partial.  (Before, the wavefronts streamed their x rows into registers in the matrix cores' operand layout, at a third of the
//            rate out of the L2, and A slab by slab through LDS: us per call, before / now, in the parts that were cut then: 7000 tokens, rank 64, K = 4096
//            30.4 / 29.4, gate_up 66.2 / 65.4; with parts that need not divide K 9000 tokens 43.4 / 39.4 and 76.8 / 72.1, K = 8192, 4500
//            47.5 / 38.0; 5000 mixed tokens down 34.1 / 32.4, gate_up 78.5 / 75.7.)
//   expand — OUT[tokens x cols] = H . B[slot]^T for a (group of tiles, column range).  The H
//            tiles are staged in LDS once (K partials summed, scaled, and split into a hi + lo
//            pair of operand-precision values, about 16 significant bits: the expand loses
//            nothing that would show after the final rounding of y).  A wavefront owns spans of
//            64 or 128 columns: it fetches the span's B rows once per slot, then for every tile
//            of the group the y rows of two or four 16-token blocks at a time, runs the MFMAs
//            and writes y back.  Tokens are the MFMA rows and the B rows fed to the MFMAs of a
//            span are interleaved, so a lane ends up with consecutive output columns of four
//            tokens and sixteen consecutive lanes cover a contiguous piece of one y row: y moves
//            in fully coalesced accesses with no transposition pass.
// Splitting the two products means no column range repeats the shrink of its tile, and each
// kernel keeps only its own operands in registers.
#include "dma.h"
#include "lds.h"
#include "sgmv_body.h"

namespace mlora {

namespace {

// ---- shrink -------------------------------------------------------------------------------------
constexpr int kRingWaves = 4;
constexpr int kRingThreads = kRingWaves * kWave;
constexpr int kRing = kMostLds / 2;  // of LDS, so that two workgroups fit a compute unit
constexpr int kRingStage = 24;       // KB of a stage at most

// NA8: groups of eight ranks, TB: blocks of sixteen tokens; both operands in groups of eight rows, 1 KB (128 bytes of K) each.
template <int NA8, int TB> struct RingShape {
  static constexpr int RB = (NA8 + 1) / 2;
  static constexpr int PIECE = NA8 + 2 * TB;                                                   // direct loads of 128 bytes of K
  static constexpr int P = PIECE * 4 <= kRingStage ? 4 : PIECE * 2 <= kRingStage ? 2 : 1;      // such pieces of a stage
  static constexpr int BYTES = P * PIECE * 1024;
  static constexpr int NST = kRing / BYTES > 8 ? 8 : kRing / BYTES;                            // stages of the ring
  static constexpr int LO = PIECE / kRingWaves, HI = (PIECE + kRingWaves - 1) / kRingWaves;    // a wavefront's loads of a piece
  static constexpr int WT = RB > 1 ? (TB < 2 ? TB : 2) : TB;                                   // wavefronts across the tokens
  static constexpr int WR = RB < kRingWaves / WT ? RB : kRingWaves / WT;                       // and across the ranks
  static constexpr int BR = RB / WR, BT = TB / WT;
  static_assert(NST >= 3 && (NST - 2) * HI * P <= 63, "the wait for a stage counts what is younger");
};

// The sums of a tile over pieces [c0, c1) of K.  The wavefronts share out the loads of a stage and the blocks of sixteen tokens by sixteen ranks; every
// block adds K up in two chains, the even and the odd 32 columns, as the one-launch form (fused.hip) does.  In one chain the sums' error against 64
// bits was larger than what slab.hip leaves (rms, one part / slab.hip's or this: K = 1024 1.84e-7 / 1.27e-7; three parts, K = 4096 2.2e-7 / 1.5e-7, 8192
// 3.2e-7 / 2.2e-7), and 0.4 % faster (4346 calls; K = 10240 at rank 24 and 600 tokens 16.4 / 16.7 us).
template <typename T, int NA8, int TB>
__device__ __forceinline__ void ring_tile(char* lds, const char* abase, uint32_t arow, const char* const (&xrow)[2], int c0, int c1, float* __restrict__ dst,
                                          int64_t hrow, int r_all, int m) {
  typedef RingShape<NA8, TB> S;
  constexpr int NST = S::NST, BR = S::BR, BT = S::BT, P = S::P;
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int lr = lane & 15, lg = lane >> 4;
  // which groups of eight rows a wavefront asks for: of tokens `wave` and `wave + 4`, of ranks the same, where there are fewer from the last wavefront down
  constexpr int NX = TB == 4 ? 2 : 1, NA = NA8 == 8 ? 2 : 1;
  const bool has_x = TB > 1 || wave < 2, has_a = NA8 >= 4 || wave >= 4 - NA8;
  const int a0 = NA8 >= 4 ? wave : has_a ? wave - (4 - NA8) : 0;
  const uint32_t swz = static_cast<uint32_t>((lane & 7) ^ (lane >> 3)) * 16;  // chunk p of a row goes to place p ^ (row & 7)
  uint32_t aoff[NA];
#pragma unroll
  for (int g = 0; g < NA; ++g) {
    const int rank = (a0 + 4 * g) * 8 + (lane >> 3);  // (buffers of a rank in between: the last row again, whose sums are not stored)
    aoff[g] = static_cast<uint32_t>(rank < r_all ? rank : r_all - 1) * arow + swz;
  }
  const uint32_t to0 = __builtin_amdgcn_readfirstlane(lds_address(lds));
  auto issue = [&](int s, int stage) {
#pragma unroll
    for (int p = 0; p < P; ++p) {
      int c = c0 + s * P + p;
      if (P > 1) c = c < c1 ? c : c1 - 1;  // (a repeated piece is not multiplied)
      const uint32_t to = to0 + stage * S::BYTES + p * (S::PIECE * 1024);
      if (has_x) {
#pragma unroll
        for (int g = 0; g < NX; ++g) dma16v(xrow[g] + static_cast<int64_t>(c) * 128 + swz, to + (NA8 + wave + 4 * g) * 1024);
      }
      if (has_a) {
#pragma unroll
        for (int g = 0; g < NA; ++g) dma16(abase + static_cast<int64_t>(c) * 128, aoff[g], to + (a0 + 4 * g) * 1024);
      }
    }
  };
  const bool hi = S::HI == S::LO || (has_x ? NX : 0) + (has_a ? NA : 0) == S::HI;
  const int wt = wave % S::WT, wr = wave / S::WT;
  const bool works = wr < S::WR;
  f32x4 acc[2][BR][BT];
#pragma unroll
  for (int ks = 0; ks < 2; ++ks)
#pragma unroll
    for (int rb = 0; rb < BR; ++rb)
#pragma unroll
      for (int tb = 0; tb < BT; ++tb) acc[ks][rb][tb] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int n = (c1 - c0 + P - 1) / P;
#pragma unroll
  for (int s = 0; s < NST - 1; ++s)
    if (s < n) issue(s, s);
  MLORA_STAMP(2);  // shrink: first stages requested
  const uint32_t read = lr * 128 + ((lg ^ (lr & 7)) * 16);
  int stage = 0, into = NST - 1;
  for (int s = 0; s < n; ++s) {
    const int younger = n - 1 - s < NST - 2 ? n - 1 - s : NST - 2;
    wait_lds();  // this wavefront's operand reads of the stage before are through
    if (hi) wait_stages<S::HI * P, NST - 2>(younger);
    else wait_stages<S::LO * P, NST - 2>(younger);
    stage_barrier();  // the stage is whole, and the one before has been read by all
    if (s + NST - 1 < n) issue(s + NST - 1, into);
    if (works) {
#pragma unroll
      for (int p = 0; p < P; ++p) {
        if (P > 1 && c0 + s * P + p >= c1) break;
        Pack8 xa[2][BT], aw[2][BR];
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
          const char* at = lds + stage * S::BYTES + p * (S::PIECE * 1024) + (read ^ (ks * 64));  // chunk lg, then chunk lg + 4, of the swizzled row
#pragma unroll
          for (int tb = 0; tb < BT; ++tb) xa[ks][tb].raw = *reinterpret_cast<const i32x4*>(at + (NA8 + 2 * (wt * BT + tb)) * 1024);
#pragma unroll
          for (int rb = 0; rb < BR; ++rb) aw[ks][rb].raw = *reinterpret_cast<const i32x4*>(at + (wr * BR + rb) * 2048 - (NA8 == 1 ? (lr & 8) * 128 : 0));
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
#pragma unroll
          for (int rb = 0; rb < BR; ++rb)
#pragma unroll
            for (int tb = 0; tb < BT; ++tb) acc[ks][rb][tb] = Mma<T>::run(aw[ks][rb], xa[ks][tb], acc[ks][rb][tb]);
      }
    }
    stage = stage + 1 == NST ? 0 : stage + 1;
    into = into + 1 == NST ? 0 : into + 1;
  }
#pragma unroll
  for (int ks = 0; ks < 2; ++ks)
#pragma unroll
    for (int rb = 0; rb < BR; ++rb) mfma_settle(acc[ks][rb]);  // (the last products and the reads of the sums lie on two sides of branches)
  MLORA_STAMP(5);  // shrink: multiplied
  if (!works) return;
  // acc[.][rb][tb]: lane holds ranks 16 rb + 4 lg .. + 3 of token lr of the block
#pragma unroll
  for (int rb = 0; rb < BR; ++rb)
#pragma unroll
    for (int tb = 0; tb < BT; ++tb) {
      const int tok = (wt * BT + tb) * 16 + lr, r = (wr * BR + rb) * 16 + 4 * lg;
      if (tok < m && r < r_all) *reinterpret_cast<f32x4*>(dst + tok * hrow + r) = acc[0][rb][tb] + acc[1][rb][tb];
    }
}

// grid (8, slices * K parts, tiles / 8): blockIdx.x is the XCD
template <typename T>
__global__ __launch_bounds__(kRingThreads, 2) void sgmv_shrink_kernel(const int32_t* __restrict__ plan, const void* __restrict__ xv, float* __restrict__ hws,
                                                                      int64_t xs, int big_off, int small_off, int big_cap, int bigrows_off, int T_, int K,
                                                                      int num_slots, int num_slices, int parts, int R, const int32_t* __restrict__ eff_rank,
                                                                      ShrinkSlices sl) {
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int tile = tile_position(big_cap);
  MLORA_STAMP(0);  // first instruction
  int row[2];
#pragma unroll
  for (int g = 0; g < 2; ++g) row[g] = tile_row(plan, bigrows_off, small_off, big_cap, tile, (wave + 4 * g) * 8 + (lane >> 3));
  const TileRef tr = fetch_tile(plan, big_off, small_off, big_cap, tile, T_, num_slots);
  const RankPrefetch ranks = rank_prefetch(eff_rank, num_slots, lane);
  __builtin_amdgcn_sched_barrier(0);
  if (!tr.ok) {
    count_rejected_plan(plan, tr.plan_ok);
    return;
  }
  MLORA_STAMP(1);  // tile record here
  const int slot = __builtin_amdgcn_readfirstlane(tr.slot), m = __builtin_amdgcn_readfirstlane(tr.m), start = __builtin_amdgcn_readfirstlane(tr.start);
  const int eff = __builtin_amdgcn_readfirstlane(rank_pick(ranks, eff_rank, num_slots, slot, R));
  if (eff == 0) return;
  const int slice = blockIdx.y / parts, part = blockIdx.y - slice * parts;
  const int chunks = K / 64, c0 = part * chunks / parts, c1 = (part + 1) * chunks / parts;
  const uint32_t arow = static_cast<uint32_t>(K) * sizeof(T);
  const char* abase = uniform(static_cast<const char*>(sl.a[slice]) + static_cast<int64_t>(slot) * R * arow);
  const char* xrow[2];
#pragma unroll
  for (int g = 0; g < 2; ++g) xrow[g] = reinterpret_cast<const char*>(static_cast<const T*>(xv) + static_cast<int64_t>(row[g]) * xs);
  const int64_t hrow = static_cast<int64_t>(num_slices) * R;
  float* dst = hws + (static_cast<int64_t>(part) * T_ + start) * hrow + slice * R;
  const int groups = (eff + 7) >> 3;  // (ranks beyond the adapter's in its last block: the expand does not use them)
  auto by_groups = [&](auto tb) __attribute__((always_inline)) {
    constexpr int TB = decltype(tb)::value;
    if (groups <= 1) ring_tile<T, 1, TB>(lds, abase, arow, xrow, c0, c1, dst, hrow, R, m);
    else if (groups == 2) ring_tile<T, 2, TB>(lds, abase, arow, xrow, c0, c1, dst, hrow, R, m);
    else if (groups <= 4) ring_tile<T, 4, TB>(lds, abase, arow, xrow, c0, c1, dst, hrow, R, m);
    else ring_tile<T, 8, TB>(lds, abase, arow, xrow, c0, c1, dst, hrow, R, m);
  };
  if (m <= 16) by_groups(std::integral_constant<int, 1>{});
  else if (m <= 32) by_groups(std::integral_constant<int, 2>{});
  else by_groups(std::integral_constant<int, 4>{});
#ifdef MLORA_TRACE
  MLORA_STAMP(6);  // partial sums issued
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  MLORA_STAMP(7);  // ... and acknowledged
#endif
}

// ---- expand -------------------------------------------------------------------------------------
template <typename T, int R, int CPL, int TPF, int G, bool STREAM>
__global__ __launch_bounds__(kExpandWaves* kWave, 2) void sgmv_expand_kernel(const int32_t* __restrict__ plan, const float* __restrict__ hws,
                                                                             void* __restrict__ yv_, int64_t ys, int big_off, int small_off,
                                                                             int big_units, int bigrows_off, int T_, int num_slots, int r,
                                                                             int num_slices, int ksplit, float scaling,
                                                                             const int32_t* __restrict__ eff_rank, ExpandSplits splits) {
  constexpr int HSTRIDE = 2 * R + 8;     // padded LDS row: R leading parts, R remainders
  __shared__ __attribute__((aligned(16))) T s_h[G * MLORA_TILE_BIG * HSTRIDE];
  __shared__ __attribute__((aligned(16))) int s_row[G * MLORA_TILE_BIG];
  __shared__ int s_slot[G], s_m[G], s_eff[G];

  const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
  const int lr = lane & 15, lg = lane >> 4;
  // A workgroup takes G consecutive 64-token tiles (consecutive tiles mostly belong to one slot,
  // whose B rows then stay in registers across them), or, past `big_units`, one short segment.
  const int unit = tile_position(big_units);  // blockIdx.x is the XCD; a block of the list of units is G positions of the XCD's block of tiles
  MLORA_STAMP(8);  // expand: first instruction
  const bool is_big = unit < big_units;
  const int sidx = is_big ? 0 : unit - big_units;

  // header and every candidate record are requested together (all addresses are in bounds for
  // the whole grid)
  const i32x4 hdr0 = *reinterpret_cast<const i32x4*>(plan);
  const i32x4 hdr1 = *reinterpret_cast<const i32x4*>(plan + 4);
  const i32x4 hdr2 = *reinterpret_cast<const i32x4*>(plan + 8);
  const i32x4 small = *reinterpret_cast<const i32x4*>(plan + small_off + sidx * MLORA_SMALL_TILE_WORDS);
  i32x4 big[G];
#pragma unroll
  for (int g = 0; g < G; ++g) big[g] = reinterpret_cast<const i32x4*>(plan + big_off)[is_big ? unit * G + g : 0];
  // the token rows of the tiles: where they lie follows from the unit's number, so they are
  // requested here, with the records (threads 0..63 hold one position of every tile each)
  int rowv[G];
#pragma unroll
  for (int g = 0; g < G; ++g) {
    rowv[g] = 0;
    if (tid < MLORA_TILE_BIG) {
      if (is_big) rowv[g] = plan[bigrows_off + (unit * G + g) * MLORA_TILE_BIG + tid];
      else if (g == 0) rowv[g] = plan[small_off + sidx * MLORA_SMALL_TILE_WORDS + MLORA_SMALL_TILE_ROWS + (tid & (MLORA_TILE_SMALL - 1))];
    }
  }
  const ExpandSplit sp = splits.split[blockIdx.y];
  const int n_short = hdr1[MLORA_PLAN_TILES_SHORT - 4];
  int slot[G], start[G], m[G], any = 0;
#pragma unroll
  for (int g = 0; g < G; ++g) {
    const bool have = is_big ? true : (g == 0 && sidx < n_short);  // (places of the list of 64-token tiles that hold none carry count 0)
    slot[g] = is_big ? big[g][0] : small[0];
    start[g] = is_big ? big[g][1] : small[2];
    m[g] = is_big ? big[g][2] : small[1];
    if (!have || m[g] <= 0 || slot[g] < 0 || slot[g] >= num_slots) m[g] = 0;
  }
  // rank of the adapter in each tile's slot (a second, dependent fetch, only with the vector
  // given): ranks at or above it are left out of the intermediate, of the B rows and of the MFMAs
  int eff[G];
#pragma unroll
  for (int g = 0; g < G; ++g) {
    eff[g] = r;
    if (eff_rank && m[g] > 0) {
      const int e = eff_rank[slot[g]];
      eff[g] = e < 0 ? 0 : e > r ? r : e;
      if (eff[g] == 0) m[g] = 0;  // nothing resident: the tile is skipped
    }
    any |= m[g];
  }
  const int usable = int(hdr0[MLORA_PLAN_MAGIC] == MLORA_PLAN_MAGIC_VALUE) & int(hdr0[MLORA_PLAN_NUM_TOKENS] == T_) &
                     int(hdr0[MLORA_PLAN_MAX_SLOTS] == num_slots) & int(any > 0) & int(sp.n0 < sp.n1);
  if (!usable) {
    count_rejected_plan(plan, hdr0[MLORA_PLAN_MAGIC] == MLORA_PLAN_MAGIC_VALUE && hdr0[MLORA_PLAN_NUM_TOKENS] == T_ &&
                                  hdr0[MLORA_PLAN_MAX_SLOTS] == num_slots);
    return;
  }
  MLORA_STAMP(9);  // expand: tile records here

  bool masked = false;
#pragma unroll
  for (int g = 0; g < G; ++g) masked |= m[g] > 0 && eff[g] < R;
  if (masked)
    expand_body<T, R, CPL, TPF, G, true, false, STREAM>(s_h, s_row, s_slot, s_m, s_eff, plan, hws, yv_, ys, T_, r, num_slices, ksplit, scaling, sp, slot, start,
                                         m, eff, rowv);
  else
    expand_body<T, R, CPL, TPF, G, false, false, STREAM>(s_h, s_row, s_slot, s_m, s_eff, plan, hws, yv_, ys, T_, r, num_slices, ksplit, scaling, sp, slot, start,
                                          m, eff, rowv);
}

template <typename T> void launch_shrink(const MloraAddArgs* a, const SgmvShape& sh) {
  allow_lds<sgmv_shrink_kernel<T>>(kRing);
  hipLaunchKernelGGL((sgmv_shrink_kernel<T>), dim3(8, static_cast<unsigned>(a->num_slices * sh.ksplit), static_cast<unsigned>(sh.tiles8)), dim3(kRingThreads), kRing,
                     static_cast<hipStream_t>(a->stream), a->plan, a->x, partials_of(a), a->x_stride, sh.lay.big_off, sh.lay.small_off, sh.big_cap,
                     sh.lay.bigrows_off, a->num_tokens, a->k, a->num_slots, a->num_slices, sh.ksplit, a->r, a->effective_rank, sh.sl);
}

template <typename T, int R>
void launch_expand_group(const MloraAddArgs* a, const PlanLayout& lay, int big_units, dim3 grid, int ksplit, int cpl, int group,
                         bool stream, const ExpandSplits& sp) {
  hipStream_t st = static_cast<hipStream_t>(a->stream);
  const float* h = partials_of(a);
#define MLORA_EXPAND(CPL_, TPF_, G_, S_)                                                                                       \
  hipLaunchKernelGGL((sgmv_expand_kernel<T, R, CPL_, TPF_, G_, S_>), grid, dim3(kExpandWaves* kWave), 0, st, a->plan, h, a->y, \
                     a->y_stride, lay.big_off, lay.small_off, big_units, lay.bigrows_off, a->num_tokens, a->num_slots, a->r, \
                     a->num_slices, ksplit, a->scaling, a->effective_rank, sp)
  if (cpl == 4) {
    if (group == 4) MLORA_EXPAND(4, 4, 4, false); else if (group == 2) MLORA_EXPAND(4, 4, 2, false); else MLORA_EXPAND(4, 4, 1, false);
  } else if (stream) {
    if (group == 2) MLORA_EXPAND(8, 2, 2, true); else MLORA_EXPAND(8, 2, 1, true);
  } else {
    if (group == 4) MLORA_EXPAND(8, 2, 4, false); else if (group == 2) MLORA_EXPAND(8, 2, 2, false); else MLORA_EXPAND(8, 2, 1, false);
  }
#undef MLORA_EXPAND
}

template <typename T>
void launch_expand_rank(const MloraAddArgs* a, const PlanLayout& lay, int big_units, dim3 grid, int ksplit, int cpl, int group,
                        bool stream, const ExpandSplits& sp) {
  switch (compute_rank(a->r)) {
    case 8: launch_expand_group<T, 8>(a, lay, big_units, grid, ksplit, cpl, group, stream, sp); break;
    case 16: launch_expand_group<T, 16>(a, lay, big_units, grid, ksplit, cpl, group, stream, sp); break;
    case 32: launch_expand_group<T, 32>(a, lay, big_units, grid, ksplit, cpl, group, stream, sp); break;
    default: launch_expand_group<T, 64>(a, lay, big_units, grid, ksplit, cpl, group, stream, sp); break;
  }
}

}  // namespace

size_t sgmv_workspace_bytes(int num_tokens, int num_slices, int r, int dtype) {
  (void)dtype;
  if (num_tokens <= 0 || num_slices <= 0 || r <= 0) return 0;
  return MLORA_WORKSPACE_HEAD_BYTES + kMaxKSplit * partial_bytes(num_tokens, num_slices, r);
}

void sgmv_trace_set(void* buf) {
#ifdef MLORA_TRACE
  (void)hipMemcpyToSymbol(HIP_SYMBOL(trace_buf), &buf, sizeof(buf));
#else
  (void)buf;
#endif
}

bool sgmv_supported(const MloraAddArgs* a) { return a->k % 128 == 0 && a->k >= 128 && tiles64_rank(a); }

// A workspace that holds at least one partial can be used (fewer K parts are taken then).
bool sgmv_workspace_ok(const MloraAddArgs* a) {
  if (!a->workspace || (reinterpret_cast<uintptr_t>(a->workspace) & 255)) return false;
  for (int i = 0; i < a->num_slices; ++i)
    if (a->slices[i].n <= 0) return false;  // every slice owns a workspace column block
  return partials_room(a) >= partial_bytes(a->num_tokens, a->num_slices, a->r);
}

// About how many 64-token tiles and short segments a batch has: its segments end anywhere inside their last tile.
int big_tiles_about(const Batch& batch, int tokens) {
  if (!batch.slots_counted) return tokens / MLORA_TILE_BIG + batch.slots / 4 + 1;  // (half of the slot ids, half a tile each)
  const int tiles = static_cast<int>((tokens + 31ll * batch.slots) / MLORA_TILE_BIG);
  return tiles > batch.slots ? tiles : batch.slots;
}

// The ring's parts need not divide K.  What counts is how many of its workgroups come to a compute unit of the fullest XCD, whose block of the tile list
// is whole runs (big_tile_run: 81 tiles of three slots are runs of 11, and three parts of them 33 workgroups on 32 compute units: K = 8192, rank 32, 5051
// tokens 43.7 us, in four parts 40.8), times the columns of a part.  A part also costs its sums, which every column range of the second launch
// reads: as much as 40 columns a slice and, by tiles x columns of the outputs, 0.3 r / (r + 64) a range (gate_up of 9392 tokens, a quarter without adapter, rank 64, one / three parts 62.9 / 67.6).
// Against the best of one to four parts, each measured, on 5800 calls of K = 384 to 16384, every rank, 200 to 9392 tokens of 1 to 128 slots, this takes 1.010 of
// the time for one slice, 1.004 for two, 1.012 for three; parts that divide K, as many as powers of two, took 1.122, 1.054 and 1.079 (one
// slice, rank 48, K = 2560, 2384 tokens of a slot, one part / four 20.7 / 13.8 us; K = 2048, rank 40, 1436 of 3 13.4 / 9.6).
// us per call with one / two / three / four parts, rank 64: K = 4096, 4000 tokens of 3 slots 31.0 / 24.1 / 21.9 / 20.4, 5500 33.5 / 27.4 / 30.3 / 27.5, 7000
// 35.1 / 29.7 / 31.9 / 29.4, 9000 42.7 / 45.6 / 39.1 / 41.3; K = 8192, 5500 58.9 / 45.5 / 51.3 / 47.2, 7000 63.8 / 52.1 / 57.3 / 54.1, 9000 72.4 / 77.4 / 64.9 / 69.4; gate_up, K = 1024,
// 2500 34.6 / 33.1 / 34.9 / 34.0, 4000 43.4 / 41.9 / 44.0 / 44.8, 5500 52.6 / 54.4, 7000 62.7 / 65.4; K = 2048, 1500 42.2 / 38.5 / 37.5 / 37.0, 2500 56.6 / 52.3
// / 54.9 / 54.9, 4000 77.0 / 73.9 / 76.9 / 77.1.
Cut ring_cut(const MloraAddArgs* a, const Batch& batch, int most_parts) {
  const int tiles = big_tiles_about(batch, batch.tokens), run = big_tile_run(tiles, batch.slots < tiles ? batch.slots : tiles);
  const long long wgs = static_cast<long long>((tiles + 8 * run - 1) / (8 * run)) * 8 * run * a->num_slices;
  long long cols = 0;
  for (int i = 0; i < a->num_slices; ++i) cols += a->slices[i].n;
  const double sums = 40.0 * a->num_slices + 0.3 * a->r / (a->r + 64) * tiles * cols / 512;
  constexpr double share[] = {1.0, 1.0 / 2, 1.0 / 3, 1.0 / 4};
  static_assert(kMaxKSplit == 4, "a share of K for every number of parts");
  Cut best = {1, 0};
  for (int p = 1; p <= most_parts; ++p) {
    const double columns = rounds_of(wgs * p) * a->k * share[p - 1] + sums * p;
    if (p == 1 || columns < best.columns) best = {p, columns};
  }
  return best;
}

int sgmv_parts(const MloraAddArgs* a, const Batch& batch) { return sgmv_shape(a, batch).ksplit; }

// Every segment of the batch: 64-token tiles of the long ones, one short tile each for the rest.
int launch_sgmv(const MloraAddArgs* a, const Batch& batch) {
  const SgmvShape sh = sgmv_shape(a, batch);
  if (sh.empty) return 0;
  if (sh.slab) launch_slab_shrink(a, sh.lay, sh.big_cap, sh.tiles8, sh.ksplit, sh.sl.a);
  else if (a->dtype == MLORA_DTYPE_BF16) launch_shrink<__bf16>(a, sh);
  else launch_shrink<_Float16>(a, sh);
  int rc = check_launch("mlora_add_lora(sgmv shrink)");
  if (rc) return rc;

  dim3 grid(8, static_cast<unsigned>(sh.nsplit), static_cast<unsigned>(sh.units / 8));
  if (a->dtype == MLORA_DTYPE_BF16) launch_expand_rank<__bf16>(a, sh.lay, sh.big_units, grid, sh.ksplit, sh.cpl, sh.group, sh.stream, sh.splits);
  else launch_expand_rank<_Float16>(a, sh.lay, sh.big_units, grid, sh.ksplit, sh.cpl, sh.group, sh.stream, sh.splits);
  return check_launch("mlora_add_lora(sgmv expand)");
}

}  // namespace mlora
