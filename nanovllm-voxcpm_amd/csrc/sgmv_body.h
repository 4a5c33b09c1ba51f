// Shared by the two-launch and the one-launch form of the long-segment kernels: tile lookup, the
// shrink of one (tile, slices, K part) and the expand of one (group of tiles, column range) as
// device functions, and the host-side helpers both launchers use.
#pragma once
#include <type_traits>

#include "common.h"
#include "launch.h"

namespace mlora {

namespace {

MLORA_TRACE_DECL

constexpr int kMaxSplits = 64;
constexpr int kExpandWaves = 4;
// Bytes of y from which on the expand launch touches it with the non-temporal hint.  The line is drawn between a launch that has
// written y and one that reads it, as in a model, for what the hint saves here (y evicts neither A nor B nor the sums) it costs there: what
// the writer left in the memory-side cache and what the reader would find in it.  gate_up, us, plain and what the hint adds, in a matrix product +
// apply + SwiGLU / a copy + apply + a copy / the apply by itself (MB = 2^20 bytes; the first within 0.5 to 1, the others within 0.2):
//   rank 64, K = 1024, 8 slots    78 MB 190 +1.5 / 106 +1.0 / 50 -2.4   102 MB 212 +1.4 / 129 -2.2 / 58 -4.5   125 MB 246 -1.9 / 158 +0.4 / 67 -4.9
//                                147 MB 317 -1.7 / 194 -1.8 / 82 -7.2
//   rank 64, K = 2048, 5 slots   100 MB 301 -3.1 / 137 +1.5 / 68 -7.4   138 MB 447 -2.0 / 180 +0.1 / 79 -9.0   188 MB 486 -2.6 / 240 -6.1 / 98 -10
//   mixed ranks of 128 slots     109 MB 261 +1.8 / 174 -1.5 / 93 -2.5   128 MB 284 +3.3 / 190 -0.9 / 98 -3.1   147 MB 350 +1.5 / 220 -7.3 / 107 -4.6
//   rank 32, K = 1024            125 MB 239 -1.3 / 147 +0.3 / 60 -4.8   147 MB 313 -1.3 / 181 -0.9 / 74 -8.2   256 MB 475 -9.4 / 316 -9.2 / 123 -13
//   rank 16, K = 2048             78 MB 247 +1.3 / 98 +2.9 / 42 -2.9     94 MB 247 +0.2 / 115 -0.2 / 49 -3.9   128 MB 325 +3.1 / 154 -0.7 / 65 -5.2
//                                138 MB 433 +3.2 / 167 +2.6 / 68 -6.0   188 MB 476 -0.1 / 226 -3.2 / 88 -8.6   256 MB 636 -2.9 / 317 -8.6 / 122 -12
// Up to 138 MB one or the other of the two pays for it somewhere, from 147 MB on they gain or stay within half a percent.
// (The figures are of plain stores without the hint.  With store_through instead, copies' way, hint / without: rank 64, K = 2048, 140 MB 49.2 / 51.4, K = 1024, 147 MB
// 55.7 / 55.3, rank 16, 147 MB 47.7 / 48.3, and 125 MB of 64 slots 39.9 / 39.8 without by the line.)
constexpr long long kStreamBytes = 140ll << 20;
constexpr int kMaxKSplit = 4;  // most K parts the shrink ever uses (the workspace has room for them)

struct ShrinkSlices {
  const void* a[MLORA_MAX_SLICES];
};

struct ExpandSplit {
  const void* b;
  int n, y_col, n0, n1, slice, pad;
};

struct ExpandSplits {
  ExpandSplit split[kMaxSplits];
};

// A unit of work of either kernel: up to 64 tokens of one slot.  Workgroups below `big_cap` take
// the 64-token tiles of the long segments; the ones above take the short segments (fewer than
// sixteen tokens, one small-tile record each), so that one pair of launches covers the batch.
struct TileRef {
  int slot, start, m, ok;
  int plan_ok;  // the plan's header is that of this call's batch shape
};

// Position in the tile lists of workgroup (x, ., z) of a grid (8, ., big_cap / 8 + short segments / 8):
// the first big_cap / 8 layers take the 64-token tiles, XCD x its own block of the list; the layers
// behind them take the short segments, eight abreast.  Positions from big_cap on are short segments.
__device__ __forceinline__ int tile_position(int big_cap) {
  const int blk = big_cap >> 3, z = blockIdx.z, x = blockIdx.x;
  return z < blk ? x * blk + z : big_cap + (z - blk) * 8 + x;
}

__device__ __forceinline__ TileRef fetch_tile(const int32_t* __restrict__ plan, int big_off, int small_off, int big_cap, int tile,
                                              int T_, int num_slots) {
  // both candidate records and the header are requested together (every address is in bounds
  // for the whole grid); the choice between them costs no second round trip
  const int sidx = tile >= big_cap ? tile - big_cap : 0;
  const i32x4 big = reinterpret_cast<const i32x4*>(plan + big_off)[tile < big_cap ? tile : 0];
  const i32x4 small = *reinterpret_cast<const i32x4*>(plan + small_off + sidx * MLORA_SMALL_TILE_WORDS);
  const i32x4 hdr0 = *reinterpret_cast<const i32x4*>(plan);
  const i32x4 hdr1 = *reinterpret_cast<const i32x4*>(plan + 4);
  const i32x4 hdr2 = *reinterpret_cast<const i32x4*>(plan + 8);
  const bool is_big = tile < big_cap;
  TileRef t;
  t.slot = is_big ? big[0] : small[0];
  t.start = is_big ? big[1] : small[2];
  t.m = is_big ? big[2] : small[1];
  // the position holds a tile of this plan: places of the list of 64-token tiles that hold none carry count 0
  const bool present = is_big ? true : sidx < hdr1[MLORA_PLAN_TILES_SHORT - 4];
  t.ok = int(hdr0[MLORA_PLAN_MAGIC] == MLORA_PLAN_MAGIC_VALUE) & int(hdr0[MLORA_PLAN_NUM_TOKENS] == T_) &
         int(hdr0[MLORA_PLAN_MAX_SLOTS] == num_slots) & int(present) & int(t.m > 0) & int(t.slot >= 0) &
         int(t.slot < num_slots);
  t.plan_ok = int(hdr0[MLORA_PLAN_MAGIC] == MLORA_PLAN_MAGIC_VALUE) & int(hdr0[MLORA_PLAN_NUM_TOKENS] == T_) &
              int(hdr0[MLORA_PLAN_MAX_SLOTS] == num_slots);
  return t;
}

// Token row at position `ti` of tile `tile`.  Where it lies follows from the tile's number alone (a
// 64-token tile has its row list behind the big-tile records, a short segment carries its rows in
// its record), so it is requested together with the record instead of after it.  Positions past
// the tile's count hold a valid row as well (a tile's own in a short segment's record, row 0 in a
// big tile's list): read, never written.
__device__ __forceinline__ int tile_row(const int32_t* __restrict__ plan, int bigrows_off, int small_off, int big_cap, int tile, int ti) {
  const bool is_big = tile < big_cap;
  const int at = is_big ? bigrows_off + tile * MLORA_TILE_BIG + ti
                        : small_off + (tile - big_cap) * MLORA_SMALL_TILE_WORDS + MLORA_SMALL_TILE_ROWS + (ti & (MLORA_TILE_SMALL - 1));
  return plan[at];
}

// ---- shrink -------------------------------------------------------------------------------------
// Of the one-launch form (fused.hip): four wavefronts of sixteen tokens each walk a K part in batches of KR columns (a wavefront holds the batch of its
// sixteen token rows in registers) and A slabs of as many columns that pass through LDS.  Both
// streams run one step ahead of the MFMAs: the next slab sits in registers and the next x batch
// is in flight while the current slab is multiplied.  (The two launches' shrink is a kernel of its own, in sgmv.hip.)
constexpr int kShrinkWaves = 4;

// Body of the shrink for one tile.  MASKED: the adapter in the tile's slot has fewer ranks than
// the buffers (eff < R): 16-rank blocks of A[slot] at or above its rank are neither copied to LDS
// nor multiplied, and their partial sums are not written (the expand does not read them).  The
// unmasked instance is the code without any of those tests.
template <typename T, int R, int KR, bool MASKED>
__device__ __forceinline__ void shrink_body(T* __restrict__ s_a, const void* __restrict__ xv, float* __restrict__ hws, int64_t xs, int T_, int K,
                                            int num_slices, int krange, const ShrinkSlices& sl, int slice, int kpart, int slot, int start, int m,
                                            int eff, int row) {
  constexpr int RB = (R + 15) / 16;      // 16-rank blocks
  constexpr int NT = kShrinkWaves * kWave;
  constexpr int ASTRIDE = KR + 8;        // padded LDS row: 16 rows x 16 bytes cover all banks once
  constexpr int CPR = KR / 8;            // 16-byte chunks per slab row
  constexpr int TOTAL = R * CPR;         // chunks per slab
  constexpr int CHUNKS = (TOTAL + NT - 1) / NT;  // chunks each thread copies per slab
  constexpr int KS = KR / 32;            // k-steps per slab

  const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
  const int lr = lane & 15, lg = lane >> 4;
  const int rb_n = MASKED ? (eff + 15) >> 4 : RB;          // 16-rank blocks of A[slot] in use
  const int rows_used = MASKED ? (rb_n * 16 < R ? rb_n * 16 : R) : R;

  const int k0 = kpart * krange;
  const int nbatch = krange / KR;
  const bool active = wave * 16 < m;  // this wavefront's token block exists
  // `row`: token row of this lane, position wave * 16 + lane % 16 of the tile (positions past the
  // end of the tile name valid rows too: they feed the MFMA harmlessly and are never
  // written back)
  const int ti = wave * 16 + lr;
  MLORA_STAMP(2);  // shrink: body entered (the token rows were requested with the record)
  const T* xptr = static_cast<const T*>(xv) + static_cast<int64_t>(row) * xs + k0 + lg * 8;
  const int64_t aoff = static_cast<int64_t>(slot) * R * K + k0;

  i32x4 v[CHUNKS];
  auto request_slab = [&](const T* Aslab) {
#pragma unroll
    for (int i = 0; i < CHUNKS; ++i) {
      const int c = i * NT + tid;
      if constexpr (MASKED) {
        if (i * (NT / CPR) >= rows_used) continue;  // these rows lie beyond the adapter's rank (the same for every thread)
      }
      if (TOTAL % NT == 0 || c < TOTAL) v[i] = load128(Aslab + static_cast<int64_t>(c / CPR) * K + (c % CPR) * 8);
    }
  };
  auto store_slab = [&]() {
#pragma unroll
    for (int i = 0; i < CHUNKS; ++i) {
      const int c = i * NT + tid;
      if constexpr (MASKED) {
        if (i * (NT / CPR) >= rows_used) continue;
      }
      if (TOTAL % NT == 0 || c < TOTAL) *reinterpret_cast<i32x4*>(&s_a[(c / CPR) * ASTRIDE + (c % CPR) * 8]) = v[i];
    }
  };
  auto request_x = [&](Pack8(&buf)[KS], int kc) {
#pragma unroll
    for (int i = 0; i < KS; ++i) buf[i].raw = load128(xptr + kc + i * 32);
  };

  // D layout: lane holds H[rank 16*rb + 4*(lane/16) + i][token lane%16]: four consecutive ranks
  auto write_partials = [&](const f32x4(&part)[RB]) {
    if (active && ti < m) {
      float* dst = hws + ((static_cast<int64_t>(kpart) * T_ + start + ti) * num_slices + slice) * R;
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) {
        const int r0 = rb * 16 + 4 * lg;
        if (r0 < R && (!MASKED || rb < rb_n)) *reinterpret_cast<f32x4*>(dst + r0) = part[rb];
      }
    }
  };

  // (Written once for wavefronts whose token block exists and once for those without one, which
  // only help with the slabs: a branch on `active` around the x requests keeps the compiler from
  // counting the loads in flight, and the wait for a slab then is a wait for the x batch requested
  // after it as well.)
  auto batches = [&](auto act_tag) {
  constexpr bool ACT = decltype(act_tag)::value;
  Pack8 xa[KS], xb[KS];
  f32x4 acc[2][RB];
  const T* A = static_cast<const T*>(sl.a[slice]) + aoff;
  request_slab(A);
  if (ACT) request_x(xa, 0);
  MLORA_STAMP(3);  // shrink: first slab and first x batch requested (the token rows are here)
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) acc[0][rb] = acc[1][rb] = f32x4{0.f, 0.f, 0.f, 0.f};
  // Two x buffers, one slab per batch.  A batch that has a successor (MORE) requests the
  // successor's x batch, waits for its own slab alone, and requests the successor's slab
  // after the barrier; the last batch of the K part is a copy of its own without those
  // requests.  Written that way (instead of tests on b inside one body) every wait counts
  // the requests younger than what it waits for: the x batch that was just requested stays
  // in flight while the current one is multiplied.
  auto batch = [&](auto more_tag, Pack8(&cur)[KS], Pack8(&nxt)[KS], int b) __attribute__((always_inline)) {
    constexpr bool MORE = decltype(more_tag)::value;
    if (MORE && ACT) request_x(nxt, (b + 1) * KR);
    __syncthreads();  // everyone is done reading the previous slab
    store_slab();
    if (b == 0) MLORA_STAMP(4);  // shrink: first slab arrived and is on its way to LDS
    __syncthreads();
    if constexpr (MORE) request_slab(A + (b + 1) * KR);
    if (ACT) {
#pragma unroll
      for (int i = 0; i < KS; ++i) {
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) {
          if constexpr (MASKED) {
            if (rb >= rb_n) continue;
          }
          const int rr = rb * 16 + lr;
          Pack8 aw;
          aw.raw = *reinterpret_cast<const i32x4*>(&s_a[(rr < R ? rr : R - 1) * ASTRIDE + i * 32 + lg * 8]);
          acc[i & 1][rb] = Mma<T>::run(aw, cur[i], acc[i & 1][rb]);
        }
      }
      if constexpr (MASKED && !MORE) {  // rank blocks were skipped by branches
        mfma_settle(acc[0]);
        mfma_settle(acc[1]);
      }
    }
  };
  int b = 0;
  for (; b + 2 < nbatch; b += 2) {
    batch(std::true_type{}, xa, xb, b);
    batch(std::true_type{}, xb, xa, b + 1);
  }
  if (b + 1 < nbatch) {
    batch(std::true_type{}, xa, xb, b);
    batch(std::false_type{}, xb, xa, b + 1);
  } else {
    batch(std::false_type{}, xa, xb, b);
  }
  MLORA_STAMP(5);  // shrink: multiplied
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) acc[0][rb] += acc[1][rb];
  if (ACT) write_partials(acc[0]);
  };
  if (active) batches(std::true_type{});
  else batches(std::false_type{});
}

// ---- expand -------------------------------------------------------------------------------------
// grid (8, column ranges, tiles / 8), four wavefronts.  OUT[tokens x cols] = H . B[slot]^T with
// the tokens as MFMA rows: in the accumulator layout a lane then holds four tokens of one column,
// and with the B rows of the CPL MFMAs of a span of 16 * CPL columns interleaved (MFMA j takes
// column CPL * (lane % 16) + j) it holds CPL consecutive columns of each of those tokens.
// Sixteen consecutive lanes therefore cover 32 * CPL contiguous bytes of one y row: y is read
// and written in fully coalesced accesses (128-bit for CPL = 8, 64-bit for CPL = 4; the narrower
// span needs half the registers, so more wavefronts and more of their loads are in flight).
// TPF: token blocks whose y rows are requested together.
template <typename T, int N> union alignas(N * sizeof(T)) YVec {
  T e[N];
  uint32_t u[N / 2];
};

template <int N> struct YRaw;
template <> struct YRaw<4> { typedef u32x2 type; };
template <> struct YRaw<8> { typedef u32x4 type; };

// y is touched once per launch.  STREAM: its loads and stores carry the non-temporal hint (kStreamBytes says when
// and what it gives); without, the stores leave at once (store_through; hinted loads with such stores are slower than either: 9392 tokens, rank
// 64, gate_up 57.5 -> 60.6).  An item
// stays the raw vectors it was fetched as until it is used: unpacked where it is requested, its
// arithmetic is scheduled ahead of the barrier that ends the staging of the intermediate, and the
// wavefront waits for the item in front of work that could have run meanwhile.
template <typename T, int N, bool STREAM>
__device__ __forceinline__ typename YRaw<N>::type load_y(const T* p) {
  const typename YRaw<N>::type* q = reinterpret_cast<const typename YRaw<N>::type*>(p);
  if constexpr (STREAM) return __builtin_nontemporal_load(q);
  else return *q;
}
template <typename T, int N>
__device__ __forceinline__ YVec<T, N> unpack_y(const typename YRaw<N>::type& r) {
  YVec<T, N> v;
  __builtin_memcpy(&v, &r, sizeof(r));
  return v;
}
template <typename T, int N, bool STREAM>
__device__ __forceinline__ void store_y(T* p, const YVec<T, N>& v) {
  typedef typename YRaw<N>::type Raw;
  Raw r;
  __builtin_memcpy(&r, &v, sizeof(r));
  if constexpr (STREAM) __builtin_nontemporal_store(r, reinterpret_cast<Raw*>(p));
  else store_through(p, r);
}

// Body of the expand for the tiles of one workgroup.  MASKED: some tile's slot holds an adapter of
// fewer ranks than the kernel's R, which the buffers' `rank` may be too: chunks of the intermediate the shrink did not write are not read,
// ranks at or above the adapter's are zero in the intermediate, B columns from that rank on are
// not fetched (zeros take their place in the operand).  The unmasked instance is the code without
// any of those tests.
//
// SC1: the partial sums are fetched with agent-scope loads (past the compute unit's and the XCD's
// caches): they were written by other workgroups of the same launch.
template <typename T, int R, int CPL, int TPF, int G, bool MASKED, bool SC1 = false, bool STREAM = false>
__device__ __forceinline__ void expand_body(T* __restrict__ s_h, int* __restrict__ s_row, int* __restrict__ s_slot, int* __restrict__ s_m,
                                            int* __restrict__ s_eff, const int32_t* __restrict__ plan, const float* __restrict__ hws,
                                            void* __restrict__ yv_, int64_t ys, int T_, int rank, int num_slices, int ksplit,
                                            float scaling, const ExpandSplit& sp, const int (&slot)[G], const int (&start)[G],
                                            const int (&m)[G], const int (&eff)[G], const int (&rowv)[G]) {
  constexpr int TB = MLORA_TILE_BIG / 16;
  constexpr int NB = TB / TPF;           // y batches per tile
  constexpr int STEPS = G * NB;          // (tile, batch) steps of a span
  constexpr int KSTEPS = (R + 31) / 32;  // MFMA k-steps
  constexpr int HSTRIDE = 2 * R + 8;     // padded LDS row: R leading parts, R remainders
  constexpr int NT = kExpandWaves * kWave;
  constexpr int CPR = R / 8;             // groups of eight ranks per token
  constexpr int SPAN = 16 * CPL;         // columns of one span
  constexpr int HC = (MLORA_TILE_BIG * CPR + NT - 1) / NT;  // H chunks per thread and tile

  const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
  const int lr = lane & 15, lg = lane >> 4;

  // The partial sums of a tile's intermediate: requested (every K part together), then summed,
  // scaled, split and written to LDS.  The first tile's are requested before anything else: they
  // depend on the tile record alone, and are on their way while the token rows make theirs.
  const int r = MASKED ? rank : R;  // of the buffers
  const int64_t hrow = static_cast<int64_t>(num_slices) * r;
  const int64_t part = static_cast<int64_t>(T_) * hrow;
  f32x4 t[HC][kMaxKSplit][2];
  auto request_h = [&](int g) {
    const float* src = hws + static_cast<int64_t>(start[g]) * hrow + sp.slice * r;
#pragma unroll
    for (int h = 0; h < HC; ++h) {
      const int c = h * NT + tid;
      int tok = c / CPR;
      tok = tok < m[g] ? tok : m[g] - 1;
      const float* q = src + tok * hrow + (c % CPR) * 8;
      const bool used = !MASKED || (c % CPR) * 8 < eff[g];  // the shrink wrote this chunk
#pragma unroll
      for (int kp = 0; kp < kMaxKSplit; ++kp) {
        if (kp < ksplit) {
          if (used && SC1) {
            const uint64_t* q8 = reinterpret_cast<const uint64_t*>(q + kp * part);
#pragma unroll
            for (int w = 0; w < 4; ++w) {
              const uint64_t pair = __hip_atomic_load(q8 + w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
              t[h][kp][w >> 1][2 * (w & 1)] = __uint_as_float(static_cast<uint32_t>(pair));
              t[h][kp][w >> 1][2 * (w & 1) + 1] = __uint_as_float(static_cast<uint32_t>(pair >> 32));
            }
          } else if (used) {
            t[h][kp][0] = *reinterpret_cast<const f32x4*>(q + kp * part);
            t[h][kp][1] = *reinterpret_cast<const f32x4*>(q + kp * part + 4);
          } else {
            t[h][kp][0] = f32x4{0.f, 0.f, 0.f, 0.f};
            t[h][kp][1] = f32x4{0.f, 0.f, 0.f, 0.f};
          }
        }
      }
    }
  };
  auto stage_h = [&](int g) {
#pragma unroll
    for (int h = 0; h < HC; ++h) {
      const int c = h * NT + tid, tok = c / CPR, ch = c % CPR;
      if ((MLORA_TILE_BIG * CPR) % NT != 0 && c >= MLORA_TILE_BIG * CPR) continue;
      f32x4 s0 = t[h][0][0], s1 = t[h][0][1];
#pragma unroll
      for (int kp = 1; kp < kMaxKSplit; ++kp) {
        if (kp < ksplit) {
          s0[0] += t[h][kp][0][0]; s0[1] += t[h][kp][0][1]; s0[2] += t[h][kp][0][2]; s0[3] += t[h][kp][0][3];
          s1[0] += t[h][kp][1][0]; s1[1] += t[h][kp][1][1]; s1[2] += t[h][kp][1][2]; s1[3] += t[h][kp][1][3];
        }
      }
      Pack8 hi, lo;
      float v[8], back[8], rem[8];
      const float live = tok < m[g] ? scaling : 0.f;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        v[i] = (!MASKED || ch * 8 + i < eff[g]) ? s0[i] * live : 0.f;  // ranks the adapter does not have contribute nothing
        v[4 + i] = (!MASKED || ch * 8 + 4 + i < eff[g]) ? s1[i] * live : 0.f;
      }
      pack8<T>(v, hi);
      unpack8<T>(hi, back);
#pragma unroll
      for (int i = 0; i < 8; ++i) rem[i] = v[i] - back[i];
      pack8<T>(rem, lo);
      *reinterpret_cast<i32x4*>(&s_h[(g * MLORA_TILE_BIG + tok) * HSTRIDE + ch * 8]) = hi.raw;
      *reinterpret_cast<i32x4*>(&s_h[(g * MLORA_TILE_BIG + tok) * HSTRIDE + R + ch * 8]) = lo.raw;
    }
  };

  // A wavefront's work is a sequence of items: for each of its spans of 16 * CPL columns, the
  // (tile, y batch) steps that hold tokens.  The y rows of the item after the current one are
  // always in flight, and those of the first item (and its B rows) go out before the H tiles
  // are staged, so that the stream of y never waits for anything but itself.
  T* const ybase = static_cast<T*>(yv_) + sp.y_col;
  auto next_step = [&](int st) {
    for (++st; st < STEPS; ++st)
      if (s_m[st / NB] > (st % NB) * TPF * 16) break;
    return st;
  };
  int first_step = 0;  // (set once the tiles' sizes are in LDS)
  auto column = [&](int c0) {  // first of this lane's CPL columns, clamped into the range
    const int c = c0 + CPL * lr;
    return c < sp.n1 ? c : sp.n1 - 8;
  };
  typedef typename YRaw<CPL>::type YItem[TPF][4];  // a y item as it was fetched: 16 * TPF tokens x 16 * CPL columns of a wavefront
  auto issue_y = [&](YItem& buf, int c0, int st) {
    const int g = st / NB, tp = (st % NB) * TPF, cl = column(c0);
#pragma unroll
    for (int u = 0; u < TPF; ++u) {
      const i32x4 rows = *reinterpret_cast<const i32x4*>(&s_row[g * MLORA_TILE_BIG + (tp + u) * 16 + 4 * lg]);
#pragma unroll
      for (int i = 0; i < 4; ++i) buf[u][i] = load_y<T, CPL, STREAM>(ybase + static_cast<int64_t>(rows[i]) * ys + cl);
    }
  };
  Pack8 bop[CPL][KSTEPS];
  int b_slot = -1, b_c0 = -1;  // what bop holds
  auto load_b = [&](int c0, int sg, int eg) {
    // the B rows of the span (lanes whose chunk lies beyond the rank fetch a valid chunk anyway,
    // their H operand is zero; columns past the range repeat the last one and are never stored)
    const T* B = static_cast<const T*>(sp.b) + static_cast<int64_t>(sg) * sp.n * r;
    if (!MASKED || eg >= R) {
#pragma unroll
      for (int j = 0; j < CPL; ++j) {
        int n = c0 + CPL * lr + j;
        n = n < sp.n1 ? n : sp.n1 - 1;
#pragma unroll
        for (int ks = 0; ks < KSTEPS; ++ks) {
          const int kc = (lg + 4 * ks) & (R / 8 - 1);
          bop[j][ks].raw = load128(B + static_cast<int64_t>(n) * R + kc * 8);
        }
      }
    } else if constexpr (MASKED) {
      // an adapter of lower rank: only its own chunks of eight ranks are fetched, the rest of the
      // operand is zero, and what the boundary chunk holds beyond the rank is masked out
      const int eg8 = (eg + 7) >> 3;
#pragma unroll
      for (int j = 0; j < CPL; ++j) {
        int n = c0 + CPL * lr + j;
        n = n < sp.n1 ? n : sp.n1 - 1;
#pragma unroll
        for (int ks = 0; ks < KSTEPS; ++ks) {
          const int kc = lg + 4 * ks;
          if (kc < eg8) {
            bop[j][ks].raw = load128(B + static_cast<int64_t>(n) * r + kc * 8);
            if (eg & 7) mask_ranks(bop[j][ks], kc * 8, eg);
          } else {
            bop[j][ks].raw = i32x4{0, 0, 0, 0};
          }
        }
      }
    }
    b_slot = sg;
    b_c0 = c0;
  };
  auto process = [&](YItem& buf, int c0, int st) {
    const int g = st / NB, tp = (st % NB) * TPF;
    const int mg = s_m[g];
    const T* hg = s_h + g * MLORA_TILE_BIG * HSTRIDE;
    const int c = c0 + CPL * lr;
    const bool col_ok = c < sp.n1;
#pragma unroll
    for (int u = 0; u < TPF; ++u) {
      const int tb = tp + u;
      if (tb * 16 >= mg) continue;
      Pack8 hop[KSTEPS], hlo[KSTEPS];
#pragma unroll
      for (int ks = 0; ks < KSTEPS; ++ks) {
        const int kc = lg + 4 * ks;
        if (kc * 8 < R) {
          hop[ks].raw = *reinterpret_cast<const i32x4*>(&hg[(tb * 16 + lr) * HSTRIDE + kc * 8]);
          hlo[ks].raw = *reinterpret_cast<const i32x4*>(&hg[(tb * 16 + lr) * HSTRIDE + R + kc * 8]);
        } else {
          hop[ks].raw = i32x4{0, 0, 0, 0};
          hlo[ks].raw = i32x4{0, 0, 0, 0};
        }
      }
      f32x4 out[CPL];
#pragma unroll
      for (int j = 0; j < CPL; ++j) {
        out[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < KSTEPS; ++ks) {
          out[j] = Mma<T>::run(hlo[ks], bop[j][ks], out[j]);
          out[j] = Mma<T>::run(hop[ks], bop[j][ks], out[j]);
        }
      }
      // lane holds out[token 16*tb + 4*lg + i][column c0 + CPL*lr + j]
      const i32x4 rows = *reinterpret_cast<const i32x4*>(&s_row[g * MLORA_TILE_BIG + tb * 16 + 4 * lg]);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (col_ok && tb * 16 + 4 * lg + i < mg) {
          const YVec<T, CPL> yv = unpack_y<T, CPL>(buf[u][i]);
          YVec<T, CPL> r;
#pragma unroll
          for (int j = 0; j < CPL; ++j) r.e[j] = from_f32<T>(to_f32(yv.e[j]) + out[j][i]);
          store_y<T, CPL, STREAM>(ybase + static_cast<int64_t>(rows[i]) * ys + c, r);
        }
      }
    }
  };

  YItem ya, yb;
  int c0 = sp.n0 + wave * SPAN;
  const bool has_work = c0 < sp.n1;

  // `rowv[g]` (threads 0..63): token row at position tid of tile g, requested by the caller
  // together with the tile records.  Entries past the end of a tile name valid rows too (a
  // valid row to read, never written).  The partial sums of the first tile hang on the tile
  // record alone; they are requested before the barrier the rows pass through, so that they and
  // the y rows are on their way together.  (The B rows of the first span could go out there too,
  // but they are 16 KB per wavefront and hold everything behind them up: prefill 3748 -> 3858 us.)
#pragma unroll
  for (int g = 0; g < G; ++g) {
    if (tid == 0) { s_slot[g] = slot[g]; s_m[g] = m[g]; s_eff[g] = eff[g]; }
    if (m[g] > 0 && tid < MLORA_TILE_BIG) s_row[g * MLORA_TILE_BIG + tid] = rowv[g];
  }
  if (m[0] > 0) request_h(0);
  __syncthreads();
  if constexpr (!SC1) MLORA_STAMP(10);  // expand: token rows (and the first partial sums) here
  first_step = next_step(-1);  // exists: some tile holds tokens
  int st = first_step;
  auto advance = [&](int fc0, int fst, int& nc0, int& nst) {  // item after (fc0, fst); false when there is none
    nst = next_step(fst);
    nc0 = fc0;
    if (nst >= STEPS) {
      nst = first_step;
      nc0 = fc0 + kExpandWaves * SPAN;
    }
    return nc0 < sp.n1;
  };
  // H tiles -> LDS: K partials summed (always in the same order), scaled, split into leading
  // part and remainder; absent tokens get zeros.  All loads of a tile are in flight together.
  auto stage_all = [&]() {
#pragma unroll
    for (int g = 0; g < G; ++g) {
      if (m[g] == 0) continue;
      if (g > 0) request_h(g);
      stage_h(g);
    }
  };
  // the B rows of an item's span and slot, if the registers do not hold them already
  auto ensure_b = [&](int c0, int st) {
    const int g = st / NB, sg = s_slot[g];
    if (sg != b_slot || c0 != b_c0) load_b(c0, sg, s_eff[g]);
  };
  // The B rows and the first two y items go out, then the intermediate is staged while they are
  // on their way.  The staging is written out once per path (no work / one item / two items) so
  // that each is straight-line code from the requests to the staging: the compiler then waits for
  // the partial sums alone, not for everything requested after them.
  // (Every path passes the one barrier that ends the staging in its own copy: a wavefront counts
  // at the barrier wherever its program counter is.  The markers keep the compiler from merging
  // the ends of the copies into one block, where it would have to wait for every load again.)
  if (!has_work) {
    stage_all();
    asm volatile("; staged, no item" ::: "memory");
    __syncthreads();
    if constexpr (!SC1) MLORA_STAMP(11);  // expand: intermediate in LDS
    return;
  }
  int c1 = 0, st1 = 0;
  load_b(c0, s_slot[st / NB], s_eff[st / NB]);
  issue_y(ya, c0, st);
  if (!advance(c0, st, c1, st1)) {
    stage_all();
    asm volatile("; staged behind one item" ::: "memory");
    __syncthreads();
    if constexpr (!SC1) MLORA_STAMP(11);
    process(ya, c0, st);
    if constexpr (!SC1) MLORA_STAMP(14);  // expand: wavefront 0 has stored its first item
    if constexpr (!SC1) MLORA_STAMP(12);  // expand: wavefront 0 has stored an item (the last stamp taken stays)
  } else {
    issue_y(yb, c1, st1);
    stage_all();
    asm volatile("; staged behind two items" ::: "memory");
    __syncthreads();
    if constexpr (!SC1) MLORA_STAMP(11);
    // Two y buffers, used in turn, both on their way whenever the wavefront has two more items.
    // The order inside the loop is what lets the compiler count the loads in flight instead of
    // waiting for all of them: an item's B rows are looked after (a reload only when span or slot
    // change, behind a branch) BEFORE the item after it is requested, so whatever waits for B
    // rows or for a y item knows how many requests are younger; the paths that run out of items
    // leave the loop where they find out, with their own copy of the last step.
    process(ya, c0, st);
    if constexpr (!SC1) MLORA_STAMP(14);
    if constexpr (!SC1) MLORA_STAMP(12);
    for (;;) {
      // here: (c1, st1) is on its way in yb; ya is free
      int c2, st2;
      const bool more2 = advance(c1, st1, c2, st2);
      ensure_b(c1, st1);
      if (!more2) {
        process(yb, c1, st1);
        if constexpr (!SC1) MLORA_STAMP(12);
        break;
      }
      issue_y(ya, c2, st2);
      process(yb, c1, st1);
      if constexpr (!SC1) MLORA_STAMP(12);
      // here: (c2, st2) is on its way in ya; yb is free
      const bool more3 = advance(c2, st2, c1, st1);
      ensure_b(c2, st2);
      if (!more3) {
        process(ya, c2, st2);
        if constexpr (!SC1) MLORA_STAMP(12);
        break;
      }
      issue_y(yb, c1, st1);
      process(ya, c2, st2);
      if constexpr (!SC1) MLORA_STAMP(12);
    }
  }
#ifdef MLORA_TRACE
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  if constexpr (!SC1) MLORA_STAMP(13);  // expand: wavefront 0's stores acknowledged
#endif
}

// The fp32 partials of the intermediate live behind the head of the workspace.
float* partials_of(const MloraAddArgs* a) { return reinterpret_cast<float*>(static_cast<char*>(a->workspace) + MLORA_WORKSPACE_HEAD_BYTES); }
size_t partials_room(const MloraAddArgs* a) {
  return a->workspace_bytes > MLORA_WORKSPACE_HEAD_BYTES ? static_cast<size_t>(a->workspace_bytes) - MLORA_WORKSPACE_HEAD_BYTES : 0;
}

// Diagnostic knobs, read from the environment once and again after mlora_reload_knobs().
struct SgmvKnobs {
  int generation = -1, ksplit, group, wgs, nt, cpl, slab, stream;
  void read() {
    generation = knob_generation();
    ksplit = env_int("MLORA_SGMV_KSPLIT", 0);
    group = env_int("MLORA_SGMV_GROUP", 0);
    wgs = env_int("MLORA_SGMV_WGS", 2048);
    nt = env_int("MLORA_SGMV_NT", 0);
    cpl = env_int("MLORA_SGMV_CPL", 8);
    stream = env_int("MLORA_SGMV_STREAM", -1);
    slab = env_int("MLORA_SLAB", 1);  // 0: never, 2: also by name and where it does not pay
  }
};
const SgmvKnobs& sgmv_knobs() {
  static SgmvKnobs k;
  if (k.generation != knob_generation()) k.read();
  return k;
}
// Column ranges of about `nt` columns (a multiple of 512: four wavefronts of 128 columns).
int fill_splits(const MloraAddArgs* a, int nt, ExpandSplit* out) {
  nt = (nt + 511) & ~511;
  if (nt < 512) nt = 512;
  int total;
  for (;;) {
    total = 0;
    for (int i = 0; i < a->num_slices; ++i) total += (a->slices[i].n + nt - 1) / nt;
    if (total <= kMaxSplits) break;
    nt *= 2;
  }
  int s = 0;
  for (int i = 0; i < a->num_slices; ++i) {
    const MloraSlice& sl = a->slices[i];
    for (int n0 = 0; n0 < sl.n; n0 += nt) {
      ExpandSplit& sp = out[s++];
      sp.b = sl.b; sp.n = sl.n; sp.y_col = sl.y_col; sp.slice = i; sp.pad = 0;
      sp.n0 = n0; sp.n1 = n0 + nt < sl.n ? n0 + nt : sl.n;
    }
  }
  return total;
}

// One fp32 partial of the intermediate: [T, slices, r].
inline size_t partial_bytes(int num_tokens, int num_slices, int r) {
  return static_cast<size_t>(num_tokens) * static_cast<size_t>(num_slices) * static_cast<size_t>(r) * sizeof(float);
}

// K parts whose sums the workspace holds (one where there is none: wide.hip needs none, the others' launches have made sure of it).
inline int parts_held(const MloraAddArgs* a) {
  const size_t room = partials_room(a), bytes = partial_bytes(a->num_tokens, a->num_slices, a->r);
  int held = 1;
  while (held < kMaxKSplit && (held + 1) * bytes <= room) ++held;
  return held;
}
// Of those, and of pieces of 64 columns, the ring's most.
inline int most_parts(const MloraAddArgs* a) {
  const int held = parts_held(a);
  return a->k / 64 < held ? a->k / 64 : held;
}

// The tiles of a call, as every launch over 64-token tiles walks them.
struct TileShape {
  bool empty;
  PlanLayout lay;
  ShrinkSlices sl;
  int tiles8;     // tiles / 8: 64-token tiles of the long segments, then the short segments
  int big_cap;    // tiles below this index are 64-token tiles
  int cols;       // columns of the outputs
};
inline TileShape tile_shape(const MloraAddArgs* a) {
  TileShape s;
  s.empty = true;
  s.lay = plan_layout(a->num_tokens, a->num_slots);
  s.big_cap = (s.lay.cap_big + 7) & ~7;
  int short_cap = a->num_slots < a->num_tokens ? a->num_slots : a->num_tokens;  // a short segment is one small tile
  if (short_cap > s.lay.cap_small) short_cap = s.lay.cap_small;
  const int cap = s.big_cap + ((short_cap + 7) & ~7);
  s.tiles8 = cap / 8;
  s.cols = 0;
  for (int i = 0; i < a->num_slices; ++i) {
    s.cols += a->slices[i].n;
    s.sl.a[i] = a->slices[i].a;
  }
  for (int i = a->num_slices; i < MLORA_MAX_SLICES; ++i) s.sl.a[i] = nullptr;
  s.empty = cap == 0 || s.cols == 0;
  return s;
}

// How a call is cut into work, shared by the two-launch form and the one with an exchange.
struct SgmvShape : TileShape {
  int ksplit;     // shrink: K parts
  int krange;     // of the one-launch form: columns of a part
  bool slab;      // shrink: the kernel of slab.hip, whose K parts need no common length
  int group;      // expand: consecutive 64-token tiles per workgroup
  int cpl;        // expand: columns per lane
  bool stream;    // expand: y with the non-temporal hint
  int nsplit;     // expand: column ranges
  int big_units;  // expand: groups of 64-token tiles
  int units;      // expand: those plus the short segments
  ExpandSplits splits;
};

// one_launch: the cut for the form whose workgroups do both products (256-column slabs and batches,
// which leave the registers the kernel needs besides; as many shrink roles per unit as it has workgroups).
inline SgmvShape sgmv_shape(const MloraAddArgs* a, const Batch& batch, bool one_launch = false) {
  const SgmvKnobs& kn = sgmv_knobs();
  SgmvShape s;
  static_cast<TileShape&>(s) = tile_shape(a);
  if (s.empty) return s;
  const int cols = s.cols;
  const int est_tiles = batch.tokens / MLORA_TILE_BIG + 1;

  // Parts that divide K, as many as powers of two until the grid has a workgroup per compute unit and parts of at most 1024 columns: of the one-launch
  // form, and what the line of slab.hip at rank 64 compares with.  (The ring's are further down.)
  const int max_parts = parts_held(a);
  auto dividing_parts = [&] {
    int unit = 512;
    while (unit > 128 && a->k % unit != 0) unit /= 2;
    int parts = kn.ksplit;
    if (parts <= 0) {
      parts = 1;
      while (parts < kMaxKSplit && a->k % (unit * parts * 2) == 0 &&
             (static_cast<long long>(est_tiles) * a->num_slices * parts < 256 || a->k / parts > 1024))
        parts *= 2;
    }
    if (parts > max_parts) parts = max_parts;
    if (parts > kMaxKSplit) parts = kMaxKSplit;
    while (parts > 1 && a->k % (unit * parts) != 0) --parts;
    return parts;
  };
  // Which shrink.  The one of sgmv.hip, whose wavefronts share a ring, except as below: where slab.hip, whose wavefronts have rings of their own, was
  // taken (up to rank 32, and by parts of its own), it takes 1.020 of that time (876 random calls; K = 8192, rank 32, 5051 tokens 42.0 / 39.4).  The best
  // of one to four parts of each, the shared ring's time over the other's, K below 1100 / 2100 / 4200 / beyond, rank 8 0.996 / 0.996 / 0.984 / 0.956, rank 16
  // 0.992 / 0.993 / 0.981 / 0.958, rank 32 0.976 / 0.980 / 0.977 / 0.972, rank 64 0.958 / 0.965 / 0.965 / 0.962 (3980 calls).
  // (MLORA_SLAB=2 takes slab.hip also by name.)
  s.slab = !one_launch && exact_rank(a->r) && slab_supported(a) && kn.slab == 2;
  // Rank 64 with one or two slices and long segments (256 tokens or more per slot with tokens) while an XCD's workgroups number no more than its 32
  // compute units and slab.hip then cuts K into more parts than divide it (with two slices into as many), none longer than 2800 columns.  The line is from when the
  // other shrink's parts had to divide K (2 slots, K = 2560, 4096 tokens 32.9 / 25.6 us, K = 3072, 3600 27.9 / 25.9, K = 5120, 4096 28.1 / 23.2).
  // In its parts of today that shrink takes 0.967 of the time on such calls (42, K 1536 to 5632, 0.87 to 1.14); tests/test_gpu_slab_rank64.py
  // holds AUTO to the line.
  int round_parts = 0;
  if (!one_launch && !s.slab && kn.slab && a->form == MLORA_FORM_AUTO && slab_supported(a) && a->r == 64 && a->num_slices <= 2 &&
      batch.tokens / batch.slots >= 4 * MLORA_TILE_BIG) {
    const int tiles = static_cast<int>((batch.tokens + 63ll * batch.slots) / MLORA_TILE_BIG);  // at most: every slot's last tile has one token
    const int most = a->num_slices == 1 ? kMaxKSplit : 2;
    int parts = 32 / ((tiles + 7) / 8 * a->num_slices);
    if (parts > most) parts = most;
    if (parts > a->k / 1024) parts = a->k / 1024;
    if (parts > max_parts) parts = max_parts;
    if (a->k <= 2800 * parts && tiles * a->num_slices * parts >= 128 && parts >= dividing_parts() + (a->num_slices == 1)) {
      round_parts = parts;
      s.slab = true;
    }
  }
  if (one_launch) {
    s.ksplit = dividing_parts();
    s.krange = a->k / s.ksplit;
  } else {
    if (kn.ksplit > 0) s.ksplit = kn.ksplit < most_parts(a) ? kn.ksplit : most_parts(a);
    else s.ksplit = round_parts > 0 ? round_parts : ring_cut(a, batch, most_parts(a)).count;
  }

  // expand: consecutive tiles per workgroup (they share their B rows when they share their
  // slot), then column ranges so that the grid has about 2048 workgroups
  int group = kn.group;
  // wide projections only: narrow ones need the workgroups.  Two tiles per workgroup, not four: on
  // the prefill batch (8 adapters) gate_up takes 72.2 against 73.2 us per call, on the mixed batch
  // (126 adapters, many of them with fewer than four tiles) 105.8 against 110.4
  if (group != 1 && group != 2 && group != 4) group = (cols >= 4096 && est_tiles >= 64) ? 2 : 1;
  if (one_launch && group == 2) group = 4;  // the one-launch kernel exists for one tile and for four
  const int target = kn.wgs;
  int nt = kn.nt;
  if (nt <= 0) {
    const long long want = static_cast<long long>(cols) * (est_tiles / group + 1) / (target > 0 ? target : 1);
    nt = want > 8192 ? 8192 : static_cast<int>(want);
  }
  s.group = group;
  s.nsplit = fill_splits(a, nt, s.splits.split);
  s.cpl = kn.cpl == 4 ? 4 : 8;
  s.stream = s.cpl == 8 && group <= 2 && (kn.stream < 0 ? static_cast<long long>(a->num_tokens) * cols * 2 >= kStreamBytes : kn.stream != 0);
  if (one_launch && a->k % 256 == 0) {
    // the unit's workgroups (one per column range) share out its shrink roles (tile, slice, K part):
    // about one role each
    if (group * a->num_slices > s.nsplit) s.group = group = 1;  // every slice has a column range: one role each at least
    int parts = kn.ksplit;
    if (parts <= 0) {
      parts = 1;
      while (parts < kMaxKSplit && group * a->num_slices * parts * 2 <= s.nsplit && a->k % (256 * parts * 2) == 0) parts *= 2;
    }
    if (parts > max_parts) parts = max_parts;
    if (parts > kMaxKSplit) parts = kMaxKSplit;
    while (parts > 1 && (a->k % (256 * parts) != 0 || group * a->num_slices * parts > s.nsplit)) --parts;
    s.ksplit = parts;
    s.krange = a->k / parts;
  }
  s.big_units = s.big_cap / group;  // big_cap is a multiple of 32: a multiple of 8 again
  s.units = s.big_units + (s.tiles8 * 8 - s.big_cap);
  return s;
}

}  // namespace

}  // namespace mlora
