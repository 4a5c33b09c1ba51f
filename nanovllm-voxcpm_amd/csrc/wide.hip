// Computes, for prefill-sized batches, what the reference computes with its segment-grouped
// shrink and expand kernels (nanovllm_voxcpm/lora_ops/triton_ops/lora_shrink_op.py:16-101, 257-341,
// lora_expand_op.py:11-170, kernel_utils.py:7-228, launched from nanovllm_voxcpm/lora.py:291-381):
// y_i[t] += (x[t] . A_i[s_t]^T) . B_i[s_t]^T * scaling, tokens grouped by slot.
//
// One launch over the work units of the two-launch form (sgmv.hip): the 64-token tiles of the long
// segments and, behind them in the same grid, the short segments.  A workgroup takes one (tile,
// column range): it multiplies the tile's x rows by A[slot] of the range's slice over the whole of
// K, then expands the result into its column range.  Nothing passes
// between workgroups and nothing between launches: no workspace, no second launch with its
// launch-to-first-byte latency, and no K parts.  The price is that every column range of a tile
// repeats the tile's shrink: its x rows and the slot's A rows come from the XCD's L2 after the
// first range has fetched them (a tile's ranges are dispatched together on one XCD), so the
// repeats cost compute-unit intake, not HBM traffic.  The library takes this form where the
// repeats are few or it streams less than two launches would (wide_pays): projections of few, narrow slices over a short K.
// Buffers of a rank between the instances' (24, 40, 48, 56) take the next instance up: their B rows lie in LDS at its pitch, and what their rank does
// not have is fetched from their last row or piece and masked.  Steps of 24 layers, K = 1024, over 16-token tiles / this and sgmv.hip: rank 48, 9392 tokens
// 4320 / 2941 us, 8192 mixed 5144 / 4288, rank 24 3359 / 2692 and 4171 / 3860.
//
// What bounds it is the intake of a compute unit (o at rank 64: 256 KB of x and A and 128 KB of B and y per workgroup; loads alone bring 55 GB/s) and
// what stands still meanwhile.  Both products are therefore one stream: 64 columns of K (128 bytes of every x and A row) or 64 columns
// of the range (128 bytes of every y row and the B rows) make up stages of up to 24 KB, asked for one after the other by a wavefront
// that does nothing else, as direct loads of whole row pieces to LDS, two to seven stages ahead of the four wavefronts that multiply.  So B and y are on
// their way while the last of K is multiplied, and no register holds what has not arrived.  Before, x came in the matrix
// cores' operand layout (37 GB/s per compute unit out of the L2, along rows 107 and more) through registers, A slab by slab between barriers, and B and y were
// first asked for when the intermediate was there.  us per call, before (with store_through) / now: 9392 tokens, a quarter without adapter, rank 64, K = 1024, q|k|v 22.9 /
// 18.3, o 14.8 / 13.6; 8192 mixed tokens of 128 slots of ranks 8-64 35.0 / 33.1, 20.6 / 19.5; 6000 such 30.9 / 27.4, 19.9 / 19.1; rank 32, q|k|v, 4000
// tokens 11.7 / 9.9, 1234 13.6 / 12.2, 4000 mixed 21.4 / 18.7; rank 16, 8000 tokens 13.8 / 13.7.  Loads alone, without products and stores, take 13.4 and 10.8 of
// the first call's 18.3 and 13.6.
// A wavefront for the requests, because a wait then counts its own loads and nothing else: stores take part in
// the count of a wavefront that also stores, and how many of them a partly filled tile issues differs.
#include "dma.h"
#include "lds.h"
#include "sgmv_body.h"

namespace mlora {

namespace {

constexpr int kWorkers = 4;                           // wavefronts that multiply
constexpr int kWideThreads = (kWorkers + 1) * kWave;  // and one that asks
// Two workgroups on a compute unit: one streams while the other starts or ends.  52 KB and three of them: o of prefill 13.4 -> 13.0, mixed 19.9 ->
// 19.6, but q|k|v 34.7 -> 35.8 and 12.9 -> 15.7 (rank 32, 1234 tokens); 152 KB and one: q|k|v 17.8 -> 25.8.  (A build that spilled four registers took 34.7
// where this takes 33.1.)
constexpr int kRing = kMostLds / 2;
// Bytes of a stage at most, in KB.  A stage costs a barrier and a trip through LDS whatever it holds, so small pieces share one: one piece a stage, rank
// 32 q|k|v of 1234 tokens 12.9 -> 16.3, mixed 34.7 -> 36.7.
constexpr int kStage = 24;

// C: 16-byte pieces of a B row in LDS (the buffers' rank / 8, or the next power of two); NA8: groups of eight ranks of the adapter, likewise; TB: blocks of sixteen tokens
template <int C, int NA8, int TB> struct WideShape {
  static constexpr int RB = (NA8 + 1) / 2;
  static constexpr int PIECE = NA8 + 2 * TB;                  // direct loads of 128 bytes of K
  static constexpr int SPAN = C + 2 * TB;                     // of 64 columns
  static constexpr int Q = 4 * SPAN <= kStage ? 4 : 2 * SPAN <= kStage ? 2 : 1;  // spans of a stage
  static constexpr int P = PIECE * 4 <= kStage ? 4 : PIECE * 2 <= kStage ? 2 : 1;
  static constexpr int STEP = 4 / TB;                         // a wavefront's spans lie that far apart
  static constexpr int KND = PIECE * P, END = SPAN * Q;       // of a stage of K, of spans
  static constexpr int LEAST = KND < END ? KND : END, LARGEST = KND < END ? END : KND;
  static constexpr int SLOT = LARGEST * 1024;
  static constexpr int MOST = 2 + 63 / LARGEST < 8 ? 2 + 63 / LARGEST : 8, NST = kRing / SLOT > MOST ? MOST : kRing / SLOT;
  static constexpr int WT = RB > 1 ? (TB < 2 ? TB : 2) : TB;  // wavefronts across the tokens
  static constexpr int WR = RB < 4 / WT ? RB : 4 / WT;        // and across the ranks
  static constexpr int BR = RB / WR, BT = TB / WT;
  static constexpr int KSE = (NA8 + 3) / 4;                   // k-steps of the expand
  static constexpr int HROW = KSE * 128;                      // bytes of a row of the intermediate: leading parts, remainders
  static constexpr int SH = C == 8 ? 5 : C == 4 ? 4 : 3;      // the swizzle of the B pieces
  static_assert(NST >= 3 && (NST - 2) * LARGEST <= 63 && TB * 16 * HROW <= SLOT, "");
};

template <int C, int NA8, int TB>
__device__ __forceinline__ void wide_ask(char* lds, const char* abase, uint32_t arow, const char* const (&xrow)[8], int chunks, const char* bbase,
                                         const char* const (&yrow)[8], int ncols, int spans, int eff, int R) {
  typedef WideShape<C, NA8, TB> F;
  constexpr int NST = F::NST;
  const int lane = threadIdx.x & (kWave - 1);
  const uint32_t swz = static_cast<uint32_t>((lane & 7) ^ (lane >> 3)) * 16;
  uint32_t aoff[NA8];
#pragma unroll
  for (int g = 0; g < NA8; ++g) {
    const int rank = g * 8 + (lane >> 3);  // (buffers of a rank in between: the last row again, whose products are not used)
    aoff[g] = static_cast<uint32_t>(rank < R ? rank : R - 1) * arow + swz;
  }
  const uint32_t brow = static_cast<uint32_t>(R) * 2;
  uint32_t boff[C], bwant = 0;  // where a lane's pieces of a span come from, and which of them the adapter has
#pragma unroll
  for (int i = 0; i < C; ++i) {
    const uint32_t u = i * 64 + lane, piece = u ^ ((u >> F::SH) & 7), c = piece % C;
    boff[i] = piece / C * brow + (c * 16 < brow ? c * 16 : brow - 16);  // (beyond the rank: the last piece again, and masked)
    bwant |= static_cast<uint32_t>(static_cast<int>(c) * 8 < eff) << i;
  }
  const uint32_t to0 = __builtin_amdgcn_readfirstlane(lds_address(lds));
  const uint32_t lasty = static_cast<uint32_t>(ncols) * 2 - 16, lastb = static_cast<uint32_t>(ncols) * brow - 16;
  const int n = (chunks + F::P - 1) / F::P;
  // Stages are asked for in order; the pointers walk along (an address computed from a stage's number would be kept in registers of its own).
  const char *xp[2 * TB], *yp[2 * TB], *ap = abase, *bp = bbase;
#pragma unroll
  for (int g = 0; g < 2 * TB; ++g) xp[g] = xrow[g], yp[g] = yrow[g];
  int chunk = 0, span = 0;
  uint32_t yoff = swz < lasty ? swz : lasty, left = lastb;
#pragma unroll
  for (int g = 0; g < 2 * TB; ++g) yp[g] += yoff;
  auto issue = [&](int s) {
    const uint32_t to = to0 + static_cast<uint32_t>(s % NST) * F::SLOT;
    if (s < n) {
#pragma unroll
      for (int p = 0; p < F::P; ++p) {
        const uint32_t at = to + p * (F::PIECE * 1024);
        const int step = ++chunk < chunks ? 128 : 0;  // (the last chunk is repeated to the end of its stage, and not multiplied again)
#pragma unroll
        for (int g = 0; g < 2 * TB; ++g) {
          dma16v(xp[g], at + g * 1024);
          xp[g] += step;
        }
#pragma unroll
        for (int g = 0; g < NA8; ++g) dma16(ap, aoff[g], at + (2 * TB + g) * 1024);
        ap += step;
      }
    } else if (s > n) {
#pragma unroll
      for (int j = 0; j < F::Q; ++j) {
        const uint32_t at = to + j * (F::SPAN * 1024);
#pragma unroll
        for (int i = 0; i < C; ++i) {
          // (piece 0 of a row is always fetched, so every one of these requests is made by some lane and counts)
          if (NA8 >= C || (bwant >> i & 1)) dma16(bp, boff[i] < left ? boff[i] : left, at + (2 * TB + i) * 1024);
        }
        const bool more = ++span < spans;
        uint32_t next = static_cast<uint32_t>(span) * 128 + swz;
        next = next < lasty ? next : lasty;
        if (!more) next = yoff;
#pragma unroll
        for (int g = 0; g < 2 * TB; ++g) {
          dma16v(yp[g], at + g * 1024);
          yp[g] += next - yoff;
        }
        yoff = next;
        bp += more ? 64 * brow : 0;
        left -= more ? 64 * brow : 0;
      }
    }
  };
  const int S = n + 1 + (spans + F::Q - 1) / F::Q;
#pragma nounroll
  for (int s = 1 - NST; s < S; ++s) {
    if (s >= 0) {
      if (s < n) {
        // (what may be on its way behind stage s: the window's stages, less the one of the intermediate)
        const int young = S - 1 - s < NST - 2 ? S - 1 - s : NST - 2;
        if (s + young < n) wait_stages<F::KND, NST - 2>(young);
        else wait_stages<F::LEAST, NST - 2>(young - 1);
      } else if (s > n) {
        wait_stages<F::END, NST - 2>(S - 1 - s);
      }
      stage_barrier();
      if (s == n + 1) stage_barrier();  // the intermediate is in registers
    }
    if (s + NST - 1 < S) issue(s + NST - 1);
  }
}

template <typename T, int C, int NA8, int TB>
__device__ __forceinline__ void wide_work(char* lds, int wave, int chunks, int spans, T* __restrict__ ycols, int64_t ys, const i32x4 rows, int ncols, int m, int eff,
                                          float scaling) {
  typedef WideShape<C, NA8, TB> F;
  constexpr int NST = F::NST, BR = F::BR, BT = F::BT, KSE = F::KSE;
  const int lane = threadIdx.x & (kWave - 1), lr = lane & 15, lg = lane >> 4;
  const int wt = wave % F::WT, wr = wave / F::WT;
  const bool works = wr < F::WR;
  f32x4 acc[2][BR][BT];
#pragma unroll
  for (int ks = 0; ks < 2; ++ks)
#pragma unroll
    for (int rb = 0; rb < BR; ++rb)
#pragma unroll
      for (int tb = 0; tb < BT; ++tb) acc[ks][rb][tb] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int n = (chunks + F::P - 1) / F::P;
  const uint32_t kread = lr * 128 + ((lg ^ (lr & 7)) * 16);
  int slot = 0;
  auto next = [&]() { slot = slot + 1 == NST ? 0 : slot + 1; };
  for (int s = 0; s < n; ++s) {
    wait_lds();
    stage_barrier();
    if (works) {
#pragma unroll
      for (int p = 0; p < F::P; ++p) {
        if (F::P > 1 && s * F::P + p >= chunks) break;
        const uint32_t st = slot * F::SLOT + p * (F::PIECE * 1024);
        Pack8 xa[2][BT], aw[2][BR];
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
          const char* at = lds + st + (kread ^ (ks * 64));  // chunk lg, then chunk lg + 4, of the swizzled row
#pragma unroll
          for (int tb = 0; tb < BT; ++tb) xa[ks][tb].raw = *reinterpret_cast<const i32x4*>(at + (2 * (wt * BT + tb)) * 1024);
#pragma unroll
          for (int rb = 0; rb < BR; ++rb) {
            // (eight ranks fill half a block: the other half repeats them and is masked out below)
            const char* ar = at + 2 * TB * 1024 + (wr * BR + rb) * 2048;
            if (NA8 == 1) ar -= (lr & 8) * 128;
            aw[ks][rb].raw = *reinterpret_cast<const i32x4*>(ar);
          }
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
    next();
  }
#pragma unroll
  for (int ks = 0; ks < 2; ++ks)
#pragma unroll
    for (int rb = 0; rb < BR; ++rb) mfma_settle(acc[ks][rb]);
  wait_lds();
  stage_barrier();
  char* const h = lds + slot * F::SLOT;
  auto place = [&](int t, int piece) { return h + t * F::HROW + ((piece ^ (t & 7)) * 16); };
  if (works) {
#pragma unroll
    for (int rb = 0; rb < BR; ++rb)
#pragma unroll
      for (int tb = 0; tb < BT; ++tb) {
        const int t = (wt * BT + tb) * 16 + lr, r0 = (wr * BR + rb) * 16 + 4 * lg;
        const float live = t < m ? scaling : 0.f;
        T hi[4], lo[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float v = r0 + i < eff ? (acc[0][rb][tb][i] + acc[1][rb][tb][i]) * live : 0.f;
          hi[i] = from_f32<T>(v);
          lo[i] = from_f32<T>(v - to_f32(hi[i]));
        }
        u32x2 h2, l2;
        __builtin_memcpy(&h2, hi, 8);
        __builtin_memcpy(&l2, lo, 8);
        *reinterpret_cast<u32x2*>(place(t, r0 >> 3) + (r0 & 4) * 2) = h2;
        *reinterpret_cast<u32x2*>(place(t, KSE * 4 + (r0 >> 3)) + (r0 & 4) * 2) = l2;
        if (F::RB == 1) {  // the second half of the k-step
          *reinterpret_cast<u32x2*>(place(t, 2 + (r0 >> 3)) + (r0 & 4) * 2) = u32x2{0, 0};
          *reinterpret_cast<u32x2*>(place(t, KSE * 4 + 2 + (r0 >> 3)) + (r0 & 4) * 2) = u32x2{0, 0};
        }
      }
  }
  next();
  wait_lds();
  stage_barrier();
  const int tb = wave % TB, mq = wave / TB;
  int last = -1;  // the span whose sums are in out
  Pack8 hop[KSE], hlo[KSE];
#pragma unroll
  for (int ks = 0; ks < KSE; ++ks) {
    const int t = tb * 16 + lr;
    hop[ks].raw = *reinterpret_cast<const i32x4*>(place(t, ks * 4 + lg));
    hlo[ks].raw = *reinterpret_cast<const i32x4*>(place(t, KSE * 4 + ks * 4 + lg));
  }
  wait_lds();
  stage_barrier();
  const uint32_t bu = lr * (4 * C) + (C % 4 && lg >= C ? C - 1 : lg);
  const uint32_t bread = (bu ^ ((bu >> F::SH) & 7)) * 16;
  const uint32_t yread = (tb * 16 + 4 * lg) * 128 + (((lr >> 1) ^ (4 * (lg & 1))) * 16) + (lr & 1) * 8;
  const bool mask = eff < KSE * 32, whole = m >= tb * 16 + 16;
  f32x4 out[4];
  u32x2 yq[4];
  T* yp[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) yp[i] = ycols + static_cast<int64_t>(rows[i]) * ys + 4 * lr;
  auto put = [&](int e, int i) {
    union { u32x2 raw; T e[4]; unsigned long long w; } v;
    v.raw = yq[i];
#pragma unroll
    for (int j = 0; j < 4; ++j) v.e[j] = from_f32<T>(to_f32(v.e[j]) + out[j][i]);
    T* p = yp[i] + e * 64;
    store_through(p, v.raw);
  };
  auto finish = [&](int e) {
    if (whole && e * 64 + 64 <= ncols) {
#pragma unroll
      for (int i = 0; i < 4; ++i) put(e, i);
    } else if (e * 64 + 4 * lr < ncols) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (tb * 16 + 4 * lg + i < m) put(e, i);
    }
  };
  const int stages = (spans + F::Q - 1) / F::Q;
  for (int q = 0; q < stages; ++q) {
    if (q > 0) {
      wait_lds();
      stage_barrier();
    }
#pragma unroll
    for (int first = 0; first < F::Q; first += F::STEP) {
      const int e = q * F::Q + first + mq;
      if ((F::Q < F::STEP && mq >= F::Q) || e >= spans) continue;
      const char* sy = lds + slot * F::SLOT + (first + mq) * (F::SPAN * 1024);
      const char* sb = sy + 2 * TB * 1024;
      Pack8 bo[4][KSE];
      u32x2 yn[4];
      // (a piece's number is a sum without carries, so its place is the parts' places put together)
#pragma unroll
      for (int ks = 0; ks < KSE; ++ks)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int part = (j * C + (C % 4 ? 0 : ks * 4)) * 16;
          bo[j][ks].raw = *reinterpret_cast<const i32x4*>(sb + (bread ^ (part & 127)) + (part & ~127));
        }
#pragma unroll
      for (int i = 0; i < 4; ++i) yn[i] = *reinterpret_cast<const u32x2*>(sy + (yread ^ (i * 16)) + i * 128);
      __builtin_amdgcn_sched_barrier(0);
      if (last >= 0) finish(last);  // the span before, while this one's operands come
      __builtin_amdgcn_sched_barrier(0);
      if (mask) {
        int e8 = eff;
        asm volatile("" : "+s"(e8));  // (or the masks are kept in registers all the time)
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int ks = 0; ks < KSE; ++ks) mask_ranks(bo[j][ks], (ks * 4 + lg) * 8, e8);
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) out[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < KSE; ++ks) {
#pragma unroll
        for (int j = 0; j < 4; ++j) out[j] = Mma<T>::run(hlo[ks], bo[j][ks], out[j]);
#pragma unroll
        for (int j = 0; j < 4; ++j) out[j] = Mma<T>::run(hop[ks], bo[j][ks], out[j]);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) yq[i] = yn[i];
      last = e;
    }
    next();
  }
  if (last >= 0) finish(last);
}

// grid (8, column ranges, tiles / 8): blockIdx.x is the XCD.  At most 128 registers: two workgroups of five wavefronts need three or four on a SIMD.
template <typename T, int C>
__global__ __launch_bounds__(kWideThreads, 4) void wide_kernel(const int32_t* __restrict__ plan, const void* __restrict__ xv, void* __restrict__ yv_,
                                                               int64_t xs, int64_t ys, int big_off, int small_off, int big_cap, int bigrows_off,
                                                               int T_, int K, int R, int num_slots, float scaling, const int32_t* __restrict__ eff_rank,
                                                               ShrinkSlices sl, ExpandSplits splits) {
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const bool asks = wave == kWorkers;
  const int tile = tile_position(big_cap);
  MLORA_STAMP(0);  // first instruction
  // the asking wavefront's token rows, eight to a request, with the record (their place follows from the tile's)
  int row[8];
  if (asks) {
#pragma unroll
    for (int g = 0; g < 8; ++g) row[g] = tile_row(plan, bigrows_off, small_off, big_cap, tile, g * 8 + (lane >> 3));
  }
  const TileRef tr = fetch_tile(plan, big_off, small_off, big_cap, tile, T_, num_slots);
  const RankPrefetch ranks = rank_prefetch(eff_rank, num_slots, lane);
  const ExpandSplit sp = splits.split[blockIdx.y];
  __builtin_amdgcn_sched_barrier(0);
  if (!tr.ok || sp.n0 >= sp.n1) {
    count_rejected_plan(plan, tr.plan_ok);
    return;
  }
  MLORA_STAMP(1);  // tile record here
  const int slot = __builtin_amdgcn_readfirstlane(tr.slot), m = __builtin_amdgcn_readfirstlane(tr.m);
  const int eff = __builtin_amdgcn_readfirstlane(rank_pick(ranks, eff_rank, num_slots, slot, R));
  if (eff == 0) return;
  const int chunks = K / 64, ncols = sp.n1 - sp.n0, spans = (ncols + 63) / 64;
  const int groups = (eff + 7) >> 3;
  T* const ycols = static_cast<T*>(yv_) + sp.y_col + sp.n0;
  // one text per number of rank groups and of token blocks
  auto by_groups = [&](auto blocks, auto run) __attribute__((always_inline)) {
    if (C > 1 && groups <= 1) run(std::integral_constant<int, 1>{}, blocks);
    else if (C > 2 && groups <= 2) run(std::integral_constant<int, 2>{}, blocks);
    else if (C > 4 && groups <= 4) run(std::integral_constant<int, 4>{}, blocks);
    else run(std::integral_constant<int, C>{}, blocks);
  };
  auto by_tile = [&](auto run) __attribute__((always_inline)) {
    if (m <= 16) by_groups(std::integral_constant<int, 1>{}, run);
    else if (m <= 32) by_groups(std::integral_constant<int, 2>{}, run);
    else by_groups(std::integral_constant<int, 4>{}, run);
  };
  if (asks) {
    __builtin_amdgcn_s_setprio(3);
    const char *xrow[8], *yrow[8];
    const int swz = ((lane & 7) ^ (lane >> 3)) * 16;
#pragma unroll
    for (int g = 0; g < 8; ++g) {
      xrow[g] = reinterpret_cast<const char*>(static_cast<const T*>(xv) + static_cast<int64_t>(row[g]) * xs) + swz;
      yrow[g] = reinterpret_cast<const char*>(ycols + static_cast<int64_t>(row[g]) * ys);
    }
    const uint32_t arow = static_cast<uint32_t>(K) * sizeof(T);
    const char* abase = uniform(static_cast<const char*>(sl.a[sp.slice]) + static_cast<int64_t>(slot) * R * arow);
    const char* bbase = uniform(static_cast<const char*>(sp.b) + (static_cast<int64_t>(slot) * sp.n + sp.n0) * (R * sizeof(T)));
    by_tile([&](auto na8, auto tb) __attribute__((always_inline)) {
      wide_ask<C, decltype(na8)::value, decltype(tb)::value>(lds, abase, arow, xrow, chunks, bbase, yrow, ncols, spans, eff, R);
    });
  } else {
    // (the rows of the tokens it stores: a wavefront's block of tokens follows from the tile's count, and they are wanted at the end only)
    const int block = m <= 16 ? 0 : m <= 32 ? wave & 1 : wave;
    i32x4 rows;
#pragma unroll
    for (int i = 0; i < 4; ++i) rows[i] = tile_row(plan, bigrows_off, small_off, big_cap, tile, block * 16 + 4 * (lane >> 4) + i);
    by_tile([&](auto na8, auto tb) __attribute__((always_inline)) {
      wide_work<T, C, decltype(na8)::value, decltype(tb)::value>(lds, wave, chunks, spans, ycols, ys, rows, ncols, m, eff, scaling);
    });
  }
}

struct WideLaunch {
  const MloraAddArgs* a;
  PlanLayout lay;
  ShrinkSlices sl;
  ExpandSplits splits;
  dim3 grid;
  int big_cap;
};

template <typename T, int C>
void launch_wide_one(const WideLaunch& l) {
  const MloraAddArgs* a = l.a;
  allow_lds<wide_kernel<T, C>>(kRing);
  hipLaunchKernelGGL((wide_kernel<T, C>), l.grid, dim3(kWideThreads), kRing, static_cast<hipStream_t>(a->stream), a->plan, a->x, a->y, a->x_stride,
                     a->y_stride, l.lay.big_off, l.lay.small_off, l.big_cap, l.lay.bigrows_off, a->num_tokens, a->k, a->r, a->num_slots, a->scaling,
                     a->effective_rank, l.sl, l.splits);
}

template <typename T>
void launch_wide_rank(const WideLaunch& l) {
  switch (compute_rank(l.a->r)) {
    case 8: launch_wide_one<T, 1>(l); break;
    case 16: launch_wide_one<T, 2>(l); break;
    case 32: launch_wide_one<T, 4>(l); break;
    default: launch_wide_one<T, 8>(l); break;
  }
}

// Diagnostic knob, read from the environment once and again after mlora_reload_knobs().
struct WideKnobs {
  int generation = -1, nt;
  void read() {
    generation = knob_generation();
    nt = env_int("MLORA_WIDE_NT", 0);  // columns per range (0: wide_cut)
  }
};
const WideKnobs& wide_knobs() {
  static WideKnobs k;
  if (k.generation != knob_generation()) k.read();
  return k;
}

}  // namespace

void wide_trace_set(void* buf) {
#ifdef MLORA_TRACE
  (void)hipMemcpyToSymbol(HIP_SYMBOL(trace_buf), &buf, sizeof(buf));
#else
  (void)buf;
#endif
}

// Columns of a range.  Wider ranges repeat less of a tile's shrink, narrower ones are more workgroups: the width (512, 1024, 2048) whose fullest compute
// unit has the fewest columns of K and of ranges to stream, by the tiles the two launches count.  Against the best of the three, each measured, on
// 6900 calls where this form is a fast one 1.020 of the time, 512 columns throughout 1.10; where nobody counted the tokens with a slot, the mean
// of all of them and half of them 1.033 (all of them alone 1.046: o of 9392 tokens, a quarter without adapter, rank 64, K = 1024, then takes one range of 1024 columns,
// 17.0 us for 16.3).  us per call with 512 / 1024 columns, rank 64, K = 1024, 3 slots: q|k|v 6000 tokens 22.3 / 24.9, 9000
// 34.8 / 26.7, o 13.6 / 17.3 and 22.9 / 18.9; rank 32, 9000 29.7 / 23.0 and 20.0 / 16.5; rank 64, K = 2048, q|k|v 2500 23.9 / 23.1, 4000 30.9 /
// 25.0, 6000 48.5 / 41.4, o 4000 20.0 / 22.9, 6000 31.9 / 24.2; rank 64, K = 1024, 128 slots, 8192
// tokens: q|k|v 34.5 / 29.8, 5000 tokens 28.7 / 24.3, o 19.5 / 24.4.
Cut wide_cut(const MloraAddArgs* a, const Batch& batch, int widest_range) {
  // of `ranges` ranges over the tiles of so many tokens with a slot
  auto rounds = [&](int tokens, long long ranges) {
    const int tiles = big_tiles_about(batch, tokens);
    if (tokens >= 128ll * batch.slots) return rounds_of(tiles * ranges);
    // Short segments are tiles of any number of tokens, which end at different times and let the next ones in: no whole rounds, and a workgroup of `fill` of a
    // full one's rows counts for two thirds of those and a third of a full one.
    const double fill = (a->r + static_cast<double>(tokens) / tiles) / (a->r + MLORA_TILE_BIG), share = tiles * ranges / 256.0 * (1 + 2 * (fill < 1 ? fill : 1)) / 3;
    return share > 1 ? share : 1.0;
  };
  int longest = 0;
  for (int i = 0; i < a->num_slices; ++i)
    if (a->slices[i].n > longest) longest = a->slices[i].n;
  Cut best = {512, 0};
  for (int log2 = 9, columns = 512; columns <= widest_range && (columns == 512 || columns < 2 * longest); columns = 1 << ++log2) {
    long long ranges = 0;
    int widest = 0;
    for (int i = 0; i < a->num_slices; ++i) {
      ranges += (a->slices[i].n + columns - 1) >> log2;
      const int n = a->slices[i].n < columns ? a->slices[i].n : columns;
      if (n > widest) widest = n;
    }
    double streamed = rounds(batch.tokens, ranges);
    if (!batch.tokens_counted) streamed = 0.5 * (streamed + rounds(batch.tokens / 2, ranges));
    streamed *= a->k + widest;
    if (columns == 512 || streamed <= best.columns * (1 + 1e-9)) best = {columns, streamed};  // (of equals the fewer workgroups)
  }
  return best;
}

// Whether this form beats the two-launch one.  What it saves is a launch with its latency from launch to first byte and the partial sums' trip
// through the workspace, as much as streaming 1200 columns, and the second launch's own stream of y and B, 1.6 columns for each of its; what it adds is the intake of x and A
// rows by every column range of a tile beyond the first of its slice, and a stage costs 1.2 of the ring's, which two launches' workgroups fill in fours.  So by what the fullest compute unit
// streams in either, where the outputs are not wide; these (gate_up) stay with
// two launches (rank 64, K = 1024, 1100 tokens of 16 slots), and where nobody counted the tokens only repeats of at most 1024 columns of K a tile count.  Against the
// best cut of either form this takes 1.018 of the time (8700 calls of K 512 to 16384, every rank, 100 to 9392 tokens, even and uneven, outputs not wide; the repeats alone
// 1.036).  us per call, this form / two launches, rank 64: K = 1024, q|k|v of 2500, 5000, 7500 tokens of 3 slots 13.8 / 15.7, 18.6 / 21.4,
// 23.6 / 29.1, o 13.5 / 14.0, 13.6 / 14.4, 13.9 / 15.7; K = 2048, o of 158 to 250 workgroups of 1024 columns 24.2 / 26.6, 24.6 / 28.1, 26.7 / 31.3 (with 126 19.3 / 16.9, with 284 37.2 /
// 38.9); q|k|v of 252 25.2 / 30.3, of 210 33.9 / 30.9, of 344 42.0 / 33.1; 8192 tokens of 126 slots, K = 4096, 55.2 / 40.9.  Ranges of 2048 columns stay out of the comparison: of three slices only the widest fills
// them (q|k|v that one launch in such ranges would win by its cost took 1.10 of two launches' time).
bool wide_repeats_little(const MloraAddArgs* a) {
  long long repeats = 0;
  for (int i = 0; i < a->num_slices; ++i) repeats += (a->slices[i].n + 511) / 512 - 1;
  return repeats * a->k <= 1024;
}
bool wide_pays(const MloraAddArgs* a, const Batch& batch) {
  long long cols = 0;
  for (int i = 0; i < a->num_slices; ++i) cols += a->slices[i].n;
  if (wide_repeats_little(a)) return true;
  if (!batch.tokens_counted || cols > 2ll * a->k) return false;
  return 1.2 * wide_cut(a, batch, 1024).columns <= ring_cut(a, batch, most_parts(a)).columns + 1200.0 + 1.6 * big_tiles_about(batch, batch.tokens) * cols / 256.0;
}

bool wide_supported(const MloraAddArgs* a) {
  if (!(a->k % 128 == 0 && a->k >= 128 && tiles64_rank(a))) return false;
  for (int i = 0; i < a->num_slices; ++i)
    if (a->slices[i].n <= 0) return false;
  return true;
}

int launch_wide(const MloraAddArgs* a, const Batch& batch) {
  const TileShape sh = tile_shape(a);
  if (sh.empty) return 0;
  WideLaunch l;
  l.a = a; l.lay = sh.lay; l.sl = sh.sl; l.big_cap = sh.big_cap;
  const int nsplit = fill_splits(a, wide_knobs().nt > 0 ? wide_knobs().nt : wide_cut(a, batch).count, l.splits.split);
  l.grid = dim3(8, static_cast<unsigned>(nsplit), static_cast<unsigned>(sh.tiles8));
  if (a->dtype == MLORA_DTYPE_BF16) launch_wide_rank<__bf16>(l);
  else launch_wide_rank<_Float16>(l);
  return check_launch("mlora_add_lora(64-token tiles, one launch)");
}

}  // namespace mlora
