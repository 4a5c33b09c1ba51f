// The apply in two launches, shrink then expand, with every weight and x row passing through LDS by
// direct loads.  Computes what the reference computes with a shrink launch, a temporary
// [slices, T, r] tensor and one or two expand launches (nanovllm_voxcpm/lora.py:291-381,
// lora_ops/triton_ops/lora_shrink_op.py:16-173, lora_expand_op.py:11-91).
//
// What it is for.  The one-launch forms over small tiles let every column range of a tile fetch the
// tile's x rows and all of A[slot] again; with a large A[slot] (rank x K) that repeated intake is
// most of a call.  Here a workgroup of the first launch takes one (tile, slice, K part), so every
// A line is fetched once per tile, and leaves its block of partial sums in the
// workspace; a workgroup of the second takes one (tile, column range), adds the parts up and expands.
//
// How operands travel.  The matrix cores want sixteen different rows in sixteen consecutive lanes.
// 128-bit loads laid out like that bring 9.4 TB/s out of the L2 into 256 compute units, loads along rows
// (128 bytes of eight rows each) 27.5, the same straight to LDS 33.0; from HBM all three bring 6.0.  A tile's
// x rows and its slot's A rows are asked for by several workgroups of an XCD, so most of a workgroup's
// intake does come out of the L2.  Direct-to-LDS loads (16 bytes per lane, lane i to byte 16 i behind a base)
// walk along rows, need no registers for what is on its way, and put the chunks where the operand reads want them: chunk p of a row goes to place p ^ (row & 7) of the row's eight, so
// that the sixteen rows of an operand read fall on different banks.  The loads are inline assembly,
// which the compiler does not count among the loads in flight: every wait for them is written here,
// and counts the younger requests of this file's own.
//
// A slot's only tile (its segment has fewer than sixteen tokens) is the only one to ask for the slot's A and B lines, so
// those carry the non-temporal hint where the call's weights are 8 MB or more (kOnceBytes): 201 tokens over 48 slots of mixed rank, K = 2048, us per call without / with: qkv
// 17.5 / 16.8, gate_up 31.0 / 29.2, down 16.9 / 15.9.  Tiles of one slot do find lines of each other in the caches:
// hinted as well, 900 tokens of 3 slots, rank 64, take 21.3 instead of 15.4 (qkv) and 18.2 instead of 13.0 (down).
#include "common.h"
#include "launch.h"
#include "dma.h"
#include "lds.h"
#include "sgmv_body.h"

namespace mlora {

namespace {

constexpr int kPairWaves = 4;
constexpr int kPairThreads = kPairWaves * kWave;
constexpr int kChunk = 128;     // bytes of a row that a step of the shrink takes
constexpr int kMaxParts = 8;    // most K parts of a launch
constexpr int kPartsAhead = 4;  // of which the expand requests this many together
// Below, a step's weights (about a hundred such calls) may still lie in the 256 MB of the memory-side cache when the next step comes, and
// the hint gives that up: 5 tokens of 5 slots, rank 64, K = 1024, weights at hand, q|k|v 7.2 us per call without, 7.7 with, o 6.5 / 7.6; one token, K =
// 2048, gate_up 8.6 / 9.1.  The kernels count the weights by the plan's header: a graph over 48 slot ids serves batches of few adapters too (us per
// call, counted by the ids / by the header: 64 tokens of 8 slots, rank 48, K = 2048, q|k|v 9.3 / 8.5, down 11.4 / 9.6; 32 of 3, rank 64, 9.8 / 8.8 and
// 10.2 / 9.1; 201 of 48, rank 64, 19.6 / 19.7, gate_up 28.5 / 28.6).
constexpr long long kOnceBytes = 8ll << 20;

// ---- shrink -------------------------------------------------------------------------------------
// A wavefront's own share of a (tile, slice, K part): chunks [c0, c1) of 128 bytes of every row, through
// a private ring of NST stages in LDS, so that no barrier stands between request and product.
// The share is two eighths of the part, [c0, cm) and [cm, c1), whose sums stay apart (first, acc): the
// eight sums of a part are then added in order, which are the sums the split form (split.hip) takes
// over its eight wavefronts and in its order, so that at the same K parts both leave the same bits.
// NA8: groups of eight ranks.  acc[rb]: lane holds ranks 16 rb + 4 (lane / 16) .. + 3 of token lane % 16.
template <int NA8> struct ShrinkShape {
  static constexpr int RB = (NA8 + 1) / 2;
  static constexpr int ND = NA8 + 2;                 // direct loads per stage
  static constexpr int NST = ND <= 6 ? 4 : 2;        // stages of a wavefront's ring: 48-96 KB per workgroup on their way
  static constexpr int BYTES = NST * ND * 1024;      // of LDS per wavefront
};

// A wavefront's walk over chunks [c0, c1) of the rows.  XG: groups of eight token rows, one where the tile has no more tokens.  step(c): before chunk c is multiplied; multiply(rb, ks, a, x).
template <int NA8, int XG, bool ONCE, typename S, typename Step, typename Multiply>
__device__ __forceinline__ void walk_chunks(char* ring, const char* abase, uint32_t arow, int rbuf, const char* xbase, const uint32_t (&xoff)[2],
                                            int c0, int c1, Step step, Multiply multiply) {
  constexpr int RB = S::RB, ND = S::ND, NST = S::NST;
  const int lane = threadIdx.x & (kWave - 1), lr = lane & 15, lg = lane >> 4;
  const uint32_t swz = static_cast<uint32_t>((lane & 7) ^ (lane >> 3)) * 16;
  uint32_t aoff[NA8];
#pragma unroll
  for (int g = 0; g < NA8; ++g) {
    const int row = g * 8 + (lane >> 3);
    aoff[g] = static_cast<uint32_t>(row < rbuf ? row : rbuf - 1) * arow + swz;
  }
  const uint32_t lds = __builtin_amdgcn_readfirstlane(lds_address(ring));
  auto issue = [&](int c, int stage) {
    const char* a = abase + static_cast<int64_t>(c) * kChunk;
    const char* x = xbase + static_cast<int64_t>(c) * kChunk;
    const uint32_t to = lds + stage * (ND * 1024);
#pragma unroll
    for (int g = 0; g < NA8; ++g) {
      if constexpr (ONCE) dma16_once(a, aoff[g], to + g * 1024);
      else dma16(a, aoff[g], to + g * 1024);
    }
#pragma unroll
    for (int i = 0; i < XG; ++i) dma16(x, xoff[i] + swz, to + (NA8 + i) * 1024);
  };
  const int n = c1 - c0;
#pragma unroll
  for (int s = 0; s < NST - 1; ++s)
    if (s < n) issue(c0 + s, s);
  MLORA_STAMP(2);  // shrink: first stages requested
  int stage = 0, into = NST - 1;
  for (int c = 0; c < n; ++c) {
    if (c + NST - 1 < n) {
      wait_lds();  // the operand reads of the step before, from the stage that is filled next, are through
      issue(c0 + c + NST - 1, into);
    }
    const int younger = n - 1 - c < NST - 1 ? n - 1 - c : NST - 1;  // stages requested behind this one
    if (NST >= 4 && younger >= 3) wait_loads<(NST >= 4 ? 3 : 0) * ND>();
    else if (NST >= 3 && younger >= 2) wait_loads<(NST >= 3 ? 2 : 0) * ND>();
    else if (younger >= 1) wait_loads<ND>();
    else wait_loads<0>();
    step(c0 + c);
    const char* st = ring + stage * (ND * 1024) + lr * 128 + ((lg ^ (lr & 7)) * 16);
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      const char* at = st + (ks == 0 ? 0 : (lg ^ (lr & 7)) & 4 ? -64 : 64);  // chunk lg, then chunk lg + 4, of the swizzled row
      Pack8 xa;
      xa.raw = *reinterpret_cast<const i32x4*>(at + NA8 * 1024 - (XG == 1 ? (lr & 8) * 128 : 0));
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) {
        Pack8 aw;
        aw.raw = *reinterpret_cast<const i32x4*>(at + rb * 2048);
        multiply(rb, ks, aw, xa);
      }
    }
    stage = stage + 1 == NST ? 0 : stage + 1;
    into = into + 1 == NST ? 0 : into + 1;
  }
  MLORA_STAMP(3);  // shrink: multiplied
}

// fp32 products of a wavefront in eight chains per block of ranks, added up as a tree: the 16x16x4 products of a chunk do not wait for
// each other, and short chains come closer to the sum than a long one.
template <int RB> struct Chains {
  f32x4 v[RB][2][4];
  __device__ __forceinline__ void clear() {
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int j = 0; j < 4; ++j) v[rb][ks][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  __device__ __forceinline__ void add(int rb, int ks, const Pack8& aw, const Pack8& xa) {
    f32x4 a, x;
    __builtin_memcpy(&a, &aw, 16);
    __builtin_memcpy(&x, &xa, 16);
#pragma unroll
    for (int j = 0; j < 4; ++j) v[rb][ks][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[j], x[j], v[rb][ks][j], 0, 0, 0);
  }
  __device__ __forceinline__ void collect(f32x4 (&to)[RB]) {
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
      mfma_settle(v[rb][0]);
      mfma_settle(v[rb][1]);
#pragma unroll
      for (int i = 0; i < 4; ++i)
        to[rb][i] = ((v[rb][0][0][i] + v[rb][0][1][i]) + (v[rb][0][2][i] + v[rb][0][3][i])) +
                    ((v[rb][1][0][i] + v[rb][1][1][i]) + (v[rb][1][2][i] + v[rb][1][3][i]));
    }
  }
};

// CHAINS (fp32): eight chains per block of ranks instead of one, one per element of a piece and half of a chunk, for buffers of the ranks
// whose calls one workgroup per token used to take, so that their error is no larger than that kernel's (rank 48, K = 1024, 2048
// tokens: 2.2e-7 of the update, with one chain 2.4e-7); 0.2 us per call.
template <typename T, int NA8, bool CHAINS, bool ONCE>
__device__ __forceinline__ void shrink_chunks(char* ring, const char* abase, uint32_t arow, int rbuf, const char* xbase, const uint32_t (&xoff)[2],
                                              int c0, int cm, int c1, f32x4 (&first)[ShrinkShape<NA8>::RB], f32x4 (&acc)[ShrinkShape<NA8>::RB]) {
  constexpr int RB = ShrinkShape<NA8>::RB;
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) first[rb] = acc[rb] = f32x4{0.f, 0.f, 0.f, 0.f};
  if constexpr (CHAINS) {
    Chains<RB> chains;
    chains.clear();
    walk_chunks<NA8, 2, ONCE, ShrinkShape<NA8>>(
        ring, abase, arow, rbuf, xbase, xoff, c0, c1,
        [&](int c) {
          if (c == cm) {  // the first of the wavefront's two shares is complete
            chains.collect(first);
            chains.clear();
          }
        },
        [&](int rb, int ks, const Pack8& aw, const Pack8& xa) { chains.add(rb, ks, aw, xa); });
    chains.collect(acc);
  } else {
    walk_chunks<NA8, 2, ONCE, ShrinkShape<NA8>>(
        ring, abase, arow, rbuf, xbase, xoff, c0, c1,
        [&](int c) {
          if (c == cm) {  // the first of the wavefront's two shares is complete
#pragma unroll
            for (int rb = 0; rb < RB; ++rb) {
              first[rb] = acc[rb];
              acc[rb] = f32x4{0.f, 0.f, 0.f, 0.f};
            }
          }
        },
        [&](int rb, int, const Pack8& aw, const Pack8& xa) { acc[rb] = Mma<T>::run(aw, xa, acc[rb]); });
    mfma_settle(acc);  // (the last product and the reads of the sums lie on two sides of the loop's exit)
  }
}

// dst: this tile's block of partial sums, sixteen rows of rp floats.
template <typename T, int NA8, bool CHAINS, bool ONCE>
__device__ __forceinline__ void shrink_tile(char* lds, const char* abase, uint32_t arow, int rbuf, const char* xbase, const uint32_t (&xoff)[2], int c0,
                                            int cm, int c1, float* __restrict__ dst, int rp, int m) {
  typedef ShrinkShape<NA8> S;
  constexpr int RB = S::RB;
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  char* ring = lds + wave * S::BYTES;
  f32x4 first[RB], acc[RB];
  shrink_chunks<T, NA8, CHAINS, ONCE>(ring, abase, arow, rbuf, xbase, xoff, c0, cm, c1, first, acc);
  // sum over the eighths of the part, the first one first, through the rings' memory
  static_assert(2 * RB * 1024 <= S::BYTES, "the ring holds the wavefront's sums");
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
    *reinterpret_cast<f32x4*>(ring + (rb * kWave + lane) * 16) = first[rb];
    *reinterpret_cast<f32x4*>(ring + ((RB + rb) * kWave + lane) * 16) = acc[rb];
  }
  __syncthreads();
  MLORA_STAMP(4);  // shrink: every wavefront's sums in LDS
  if (wave < RB) {
    f32x4 s = *reinterpret_cast<const f32x4*>(lds + tid * 16);
#pragma unroll
    for (int w = 1; w < 2 * kPairWaves; ++w) {
      const f32x4 v = *reinterpret_cast<const f32x4*>(lds + (w >> 1) * S::BYTES + (w & 1) * (RB * 1024) + tid * 16);
#pragma unroll
      for (int i = 0; i < 4; ++i) s[i] += v[i];
    }
    const int tok = lane & 15;
    if (tok < m) *reinterpret_cast<f32x4*>(dst + tok * rp + wave * 16 + 4 * (lane >> 4)) = s;
  }
}

// A tile's record, with the plan header's verdict on it.
struct PairTile {
  int slot, m, ok, plan_ok;
  int once;  // its A and B lines with the hint: the slot has no other tile (short segments come first in the list), and the batch uses `once_from` slots
};
__device__ __forceinline__ PairTile pair_tile(const i32x4 r0, const int32_t* __restrict__ plan, int tile, int T_, int num_slots, int once_from) {
  const i32x4 h0 = *reinterpret_cast<const i32x4*>(plan), h1 = *reinterpret_cast<const i32x4*>(plan + 4), h2 = *reinterpret_cast<const i32x4*>(plan + 8);
  PairTile t;
  t.slot = r0[0];
  t.m = r0[1];
  t.once = int(tile < h1[MLORA_PLAN_TILES_SHORT - 4]) & int(h1[MLORA_PLAN_NUM_ACTIVE - 4] >= once_from);
  t.plan_ok = int(h0[MLORA_PLAN_MAGIC] == MLORA_PLAN_MAGIC_VALUE) & int(h0[MLORA_PLAN_NUM_TOKENS] == T_) & int(h0[MLORA_PLAN_MAX_SLOTS] == num_slots);
  t.ok = t.plan_ok & int(tile < h1[MLORA_PLAN_TILES_SHORT - 4] + h2[MLORA_PLAN_TILES_LONG_SMALL - 8]) & int(t.m > 0) & int(t.slot >= 0) &
         int(t.slot < num_slots);
  return t;
}

// grid (8, slices * K parts, tiles / 8): blockIdx.x is the XCD, so that the workgroups of a tile share an L2.
template <typename T, bool CHAINS, bool ONCE>
__global__ __launch_bounds__(kPairThreads) void pair_shrink_kernel(const int32_t* __restrict__ plan, const void* __restrict__ xv, float* __restrict__ hws,
                                                                   int small_off, int T_, int num_slots, int kchunks, uint32_t xrow, int rbuf,
                                                                   int parts_log2, int slices_once, const int32_t* __restrict__ eff_rank, ShrinkSlices sl) {
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int num_slices = ONCE ? slices_once & 255 : slices_once, once_from = slices_once >> 8;
  // ---- one trip: tile record, plan header, the tile's token rows, the slots' ranks ------------------
  MLORA_STAMP(0);  // shrink: first instruction
  const int tile = blockIdx.z * 8 + blockIdx.x;
  const int32_t* rec = plan + small_off + tile * MLORA_SMALL_TILE_WORDS;
  const i32x4 r0 = *reinterpret_cast<const i32x4*>(rec);
  int row[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) row[i] = rec[MLORA_SMALL_TILE_ROWS + i * 8 + (lane >> 3)];
  const PairTile t = pair_tile(r0, plan, tile, T_, num_slots, once_from);
  const RankPrefetch ranks = rank_prefetch(eff_rank, num_slots, lane);
  __builtin_amdgcn_sched_barrier(0);
  if (!t.ok) {
    count_rejected_plan(plan, t.plan_ok);
    return;
  }
  MLORA_STAMP(1);  // shrink: record here
  const int slot = __builtin_amdgcn_readfirstlane(t.slot), m = __builtin_amdgcn_readfirstlane(t.m);
  const int eff = rank_pick(ranks, eff_rank, num_slots, slot, rbuf);
  if (eff == 0) return;
  const int slice = blockIdx.y >> parts_log2, part = blockIdx.y - (slice << parts_log2);
  const int p0 = (part * kchunks) >> parts_log2, p1 = ((part + 1) * kchunks) >> parts_log2;
  const int c0 = p0 + wave * (p1 - p0) / kPairWaves, c1 = p0 + (wave + 1) * (p1 - p0) / kPairWaves;
  const int cm = p0 + (2 * wave + 1) * (p1 - p0) / (2 * kPairWaves);
  const uint32_t arow = static_cast<uint32_t>(kchunks) * kChunk;
  const char* abase = uniform(static_cast<const char*>(sl.a[slice]) + static_cast<int64_t>(slot) * rbuf * arow);
  const char* xbase = static_cast<const char*>(xv);
  uint32_t xoff[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) xoff[i] = static_cast<uint32_t>(row[i]) * xrow;
  const int rp = (rbuf + 15) & ~15;
  float* dst = hws + (static_cast<int64_t>(part * num_slices + slice) * (gridDim.z * 8) + tile) * (MLORA_TILE_SMALL * rp);
  const int groups = (eff + 7) >> 3;
  auto tile_of = [&](auto once) __attribute__((always_inline)) {
    constexpr bool O = decltype(once)::value;
    if (groups <= 1) shrink_tile<T, 1, CHAINS, O>(lds, abase, arow, rbuf, xbase, xoff, c0, cm, c1, dst, rp, m);
    else if (groups == 2) shrink_tile<T, 2, CHAINS, O>(lds, abase, arow, rbuf, xbase, xoff, c0, cm, c1, dst, rp, m);
    else if (groups <= 4) shrink_tile<T, 4, CHAINS, O>(lds, abase, arow, rbuf, xbase, xoff, c0, cm, c1, dst, rp, m);
    else if (groups <= 6) shrink_tile<T, 6, CHAINS, O>(lds, abase, arow, rbuf, xbase, xoff, c0, cm, c1, dst, rp, m);
    else shrink_tile<T, 8, CHAINS, O>(lds, abase, arow, rbuf, xbase, xoff, c0, cm, c1, dst, rp, m);
  };
  if (ONCE && __builtin_amdgcn_readfirstlane(t.once)) tile_of(std::true_type{});
  else tile_of(std::false_type{});
#ifdef MLORA_TRACE
  MLORA_STAMP(5);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  MLORA_STAMP(6);  // shrink: sums acknowledged
#endif
}

// An adapter of few ranks may have a deeper ring than one that fills the buffers: the most of all.
int shrink_lds(int rbuf) {
  const int groups = (rbuf + 7) / 8;
  int most = ShrinkShape<1>::BYTES;
  auto with = [&](int b) { most = b > most ? b : most; };
  if (groups > 1) with(ShrinkShape<2>::BYTES);
  if (groups > 2) with(ShrinkShape<4>::BYTES);
  if (groups > 4) with(ShrinkShape<6>::BYTES);
  if (groups > 6) with(ShrinkShape<8>::BYTES);
  return most * kPairWaves;
}

// ---- expand -------------------------------------------------------------------------------------
// A wavefront takes SP spans of 64 columns.  C: 16-byte pieces of a B row (rank x element size / 16).
template <typename T> struct PieceOf { static constexpr int E = 16 / sizeof(T); };

// Zero the elements of a piece that hold ranks at or above `eff`; `first` is the rank of its element 0.
template <typename T> __device__ __forceinline__ void mask_piece(Pack8& p, int first, int eff) {
  if constexpr (sizeof(T) == 2) {
    mask_ranks(p, first, eff);
  } else {
#pragma unroll
    for (int d = 0; d < 4; ++d) p.u[d] = first + d < eff ? p.u[d] : 0u;
  }
}

// The values of y of a span: four columns of a token.
template <typename T> using YSpan = typename std::conditional<sizeof(T) == 2, uint2, uint4>::type;
template <int C> struct ExpandShape {
  static constexpr int KSTEPS = (C + 3) / 4;     // operand steps of the contraction (four pieces each)
  static constexpr int HROW = KSTEPS * 64 + 16;  // bytes of an LDS row of the intermediate (one part)
  static constexpr int SH = C * 4 >= 64 ? 6 : C * 4 >= 32 ? 5 : C * 4 >= 16 ? 4 : 3;  // the swizzle of the B pieces: lanes' rows lie 4 C pieces apart
};

// A wavefront's B rows [c0, c0 + 64 SP), up to column n1, to its LDS.
template <typename T, int C, int SP>
__device__ __forceinline__ void request_b(char* s_b, const char* bbase, int c0, int n1, int eff, bool once) {
  constexpr int E = PieceOf<T>::E, SH = ExpandShape<C>::SH;
  constexpr int NB = SP * C;  // direct loads of a wavefront's B rows
  const int lane = threadIdx.x & (kWave - 1);
  const uint32_t to = __builtin_amdgcn_readfirstlane(lds_address(s_b));
  const char* src = bbase + static_cast<int64_t>(c0) * (C * 16);
  const uint32_t last = static_cast<uint32_t>(n1 - c0) * C - 1;  // last piece of the range
  auto request = [&](auto once) {
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      const uint32_t u = i * 64 + lane;
      uint32_t s = u ^ ((u >> SH) & 7);
      const uint32_t kc = s % C;
      s = s < last ? s : last;
      if (kc * E < static_cast<uint32_t>(eff)) {  // (piece 0 of a row is always fetched: some lane takes part)
        if constexpr (decltype(once)::value) dma16_once(src, s * 16, to + i * 1024);
        else dma16(src, s * 16, to + i * 1024);
      }
    }
  };
  if (once) request(std::true_type{});
  else request(std::false_type{});
}

// A tile's tokens spread over the lane groups: row 4 * lg + i of the products is token lg + 4 * i, so that those of a tile of up to four or
// eight are the rows i = 0 or i < 2 (XI rows).  The one launch has a text per XI and leaves out what the others would request (64 tokens
// of 32 slots, rank 16, K = 1024, o 6.1 -> 5.8 us; of 4, q|k|v 6.0 -> 5.8); in the pair those texts gain no more than they lose (two of the shrink, three
// of the expand: -2 to +2 % over 54 shapes), but the order by itself stays: a tile of up to four tokens stores one row per lane group
// instead of four of one group (row 4 * lg + i for token 4 * lg + i / this order, us per call: 16 tokens of 4 slots, rank 64, K = 2048, q|k|v 8.17 / 7.85, o
// 7.85 / 7.51; 201 of 48 gate_up 30.2 / 28.5, rank 48 26.2 / 24.2; full tiles alike: 591 of 12, rank 24, 13.2 / 13.2 and 10.6 / 10.6).
__device__ __forceinline__ int row_of_token(int t) { return 4 * (t & 3) + (t >> 2); }
__device__ __forceinline__ i32x4 spread_rows(const int32_t* __restrict__ rec, int lg) {
  i32x4 rows;
#pragma unroll
  for (int i = 0; i < 4; ++i) rows[i] = rec[MLORA_SMALL_TILE_ROWS + 4 * i + lg];
  return rows;
}

template <typename T, int SP, int XI>
__device__ __forceinline__ void request_y(YSpan<T> (&yq)[SP][4], const T* ybase, const int64_t ys, const i32x4 rows, int c0, int n1) {
  const int lr = threadIdx.x & 15;
#pragma unroll
  for (int s = 0; s < SP; ++s) {
    int c = c0 + s * 64 + 4 * lr;
    c = c < n1 ? c : n1 - 4;
#pragma unroll
    for (int i = 0; i < XI; ++i) yq[s][i] = *reinterpret_cast<const YSpan<T>*>(ybase + static_cast<int64_t>(rows[i]) * ys + c);
  }
}

// Products and stores of a wavefront's spans, once the intermediate is in LDS.
template <typename T, int C, int SP, int XI>
__device__ __forceinline__ void finish_spans(const char* s_h, const char* s_b, const YSpan<T> (&yq)[SP][4], T* __restrict__ ybase, const int64_t ys,
                                             const i32x4 rows, int c0, int n1, int m, int eff) {
  constexpr int E = PieceOf<T>::E, KSTEPS = ExpandShape<C>::KSTEPS, HROW = ExpandShape<C>::HROW, SH = ExpandShape<C>::SH;
  constexpr bool SPLIT = sizeof(T) == 2;  // 16-bit operands: the intermediate as leading part and remainder
  const int lane = threadIdx.x & (kWave - 1), lr = lane & 15, lg = lane >> 4;
  Pack8 hop[KSTEPS], hlo[SPLIT ? KSTEPS : 1];
#pragma unroll
  for (int ks = 0; ks < KSTEPS; ++ks) {
    hop[ks].raw = *reinterpret_cast<const i32x4*>(s_h + lr * HROW + (ks * 4 + lg) * 16);
    if constexpr (SPLIT) hlo[ks].raw = *reinterpret_cast<const i32x4*>(s_h + (16 + lr) * HROW + (ks * 4 + lg) * 16);
  }
  wait_loads<0>();
  MLORA_STAMP(12);  // expand: B rows and y here
  const bool mask = eff < KSTEPS * 4 * E;
#pragma unroll
  for (int s = 0; s < SP; ++s) {
    const int c = c0 + s * 64 + 4 * lr;
    f32x4 out[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      out[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < KSTEPS; ++ks) {
        int kc = ks * 4 + lg;
        if (C % 4) kc = kc < C ? kc : C - 1;
        const uint32_t u = (s * 64 + 4 * lr + j) * C + kc;
        Pack8 bo;
        bo.raw = *reinterpret_cast<const i32x4*>(s_b + (u ^ ((u >> SH) & 7)) * 16);
        if (mask) mask_piece<T>(bo, (ks * 4 + lg) * E, eff);
        if constexpr (SPLIT) out[j] = Mma<T>::run(hlo[ks], bo, out[j]);
        out[j] = Mma<T>::run(hop[ks], bo, out[j]);
      }
    }
    // (Rows that hold no token stay the products' own to the end: handed out again, their registers would be written by the masking between
    // the products, on whose branches the compiler does not always keep the distance an MFMA's result needs.)
#pragma unroll
    for (int j = 0; j < 4; ++j) asm volatile("" : "+v"(out[j]));
    if (c < n1) {
#pragma unroll
      for (int i = 0; i < XI; ++i) {
        if (lg + 4 * i < m) {
          union { YSpan<T> raw; T e[4]; } v;
          v.raw = yq[s][i];
#pragma unroll
          for (int j = 0; j < 4; ++j) v.e[j] = from_f32<T>(to_f32(v.e[j]) + out[j][i]);
          *reinterpret_cast<YSpan<T>*>(ybase + static_cast<int64_t>(rows[i]) * ys + c) = v.raw;
        }
      }
    }
  }
}

template <typename T, int C, int SP>
__device__ __forceinline__ void expand_tile(char* lds, const float* __restrict__ hsrc, int64_t part_stride, int kparts, const f32x4 (&hv)[kPartsAhead], const char* bbase,
                                            T* __restrict__ ybase, const int64_t ys, const i32x4 rows, int n0, int n1, int m, int eff,
                                            bool once, float scaling) {
  constexpr int E = PieceOf<T>::E;          // elements per piece
  constexpr int R = C * E;                  // rank of the buffers
  constexpr int KSTEPS = ExpandShape<C>::KSTEPS, HROW = ExpandShape<C>::HROW;
  constexpr int RP = (R + 15) & ~15;
  constexpr bool SPLIT = sizeof(T) == 2;    // 16-bit operands: the intermediate as leading part and remainder
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  char* s_h = lds;                                                   // [2][16] rows
  char* s_b = lds + 2 * 16 * HROW + wave * (SP * 64 * C * 16);  // this wavefront's B rows

  // the first K parts of the intermediate, B rows, y
  const int tok = tid / 16, q4 = tid & 15;  // sixteen threads per token, four ranks (RP = 64: all of them busy) each
  const int c0 = n0 + wave * (SP * 64);
  const bool mine = c0 < n1;
  YSpan<T> yq[SP][4];
  if (mine) request_b<T, C, SP>(s_b, bbase, c0, n1, eff, once);
  request_y<T, SP, 4>(yq, ybase, ys, rows, c0, n1);
  MLORA_STAMP(10);  // expand: B rows and y requested
  // the intermediate: parts summed in order, scaled, split, to LDS in operand rows (its first
  // kPartsAhead parts were requested with the record)
  f32x4 sum = hv[0];
#pragma unroll
  for (int kp = 1; kp < kPartsAhead; ++kp) {
    if (kp < kparts) {
#pragma unroll
      for (int j = 0; j < 4; ++j) sum[j] += hv[kp][j];
    }
  }
  const float* p = hsrc + tok * RP + (q4 * 4 < RP ? q4 * 4 : 0);
  for (int kp = kPartsAhead; kp < kparts; kp += kPartsAhead) {
    f32x4 v[kPartsAhead];
#pragma unroll
    for (int k = 0; k < kPartsAhead; ++k) v[k] = *reinterpret_cast<const f32x4*>(p + (kp + k < kparts ? kp + k : 0) * part_stride);
#pragma unroll
    for (int k = 0; k < kPartsAhead; ++k) {
      if (kp + k < kparts) {
#pragma unroll
        for (int j = 0; j < 4; ++j) sum[j] += v[k][j];
      }
    }
  }
  if (q4 * 4 < KSTEPS * 4 * E) {
    T hi[4], lo[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float v = (tok < m && q4 * 4 + j < eff) ? sum[j] * scaling : 0.f;
      hi[j] = from_f32<T>(v);
      lo[j] = from_f32<T>(v - to_f32(hi[j]));
    }
    __builtin_memcpy(__builtin_assume_aligned(s_h + row_of_token(tok) * HROW + q4 * 4 * sizeof(T), 8), hi, sizeof(hi));
    if constexpr (SPLIT) __builtin_memcpy(__builtin_assume_aligned(s_h + (16 + row_of_token(tok)) * HROW + q4 * 4 * sizeof(T), 8), lo, sizeof(lo));
  }
  __syncthreads();
  MLORA_STAMP(11);  // expand: intermediate in LDS
  if (!mine) return;
  finish_spans<T, C, SP, 4>(s_h, s_b, yq, ybase, ys, rows, c0, n1, m, eff);
}

#ifdef MLORA_TRACE
#define MLORA_STAMP_END(i) do { MLORA_STAMP(i); asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); MLORA_STAMP(i + 1); } while (0)
#else
#define MLORA_STAMP_END(i) do { } while (0)
#endif
// grid (8, column ranges, tiles / 8)
template <typename T, int C, int SP, bool ONCE>
__global__ __launch_bounds__(kPairThreads) void pair_expand_kernel(const int32_t* __restrict__ plan, const float* __restrict__ hws, void* __restrict__ yv_,
                                                                   int64_t ys, int small_off, int T_, int num_slots, int kparts, int slices_once,
                                                                   float scaling, const int32_t* __restrict__ eff_rank, ExpandSplits splits) {
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  constexpr int R = C * PieceOf<T>::E, RP = (R + 15) & ~15;
  const int lane = threadIdx.x & (kWave - 1), lg = lane >> 4;
  const int num_slices = ONCE ? slices_once & 255 : slices_once, once_from = slices_once >> 8;
  MLORA_STAMP(8);  // expand: first instruction
  const ExpandSplit sp = splits.split[blockIdx.y];
  const int tile = blockIdx.z * 8 + blockIdx.x;
  const int32_t* rec = plan + small_off + tile * MLORA_SMALL_TILE_WORDS;
  const i32x4 r0 = *reinterpret_cast<const i32x4*>(rec);
  const i32x4 rows = spread_rows(rec, lg);
  const PairTile t = pair_tile(r0, plan, tile, T_, num_slots, once_from);
  const RankPrefetch ranks = rank_prefetch(eff_rank, num_slots, lane);
  // the intermediate's partial sums lie where the tile's place says: requested with the record
  const int64_t stride = static_cast<int64_t>(num_slices) * (gridDim.z * 8) * (MLORA_TILE_SMALL * RP);  // from K part to K part
  const float* hsrc = hws + (static_cast<int64_t>(sp.slice) * (gridDim.z * 8) + tile) * (MLORA_TILE_SMALL * RP);
  f32x4 hv[kPartsAhead];
  {
    const int tok = threadIdx.x / 16, q4 = threadIdx.x & 15;
#pragma unroll
    for (int kp = 0; kp < kPartsAhead; ++kp)
      hv[kp] = *reinterpret_cast<const f32x4*>(hsrc + (kp < kparts ? kp : 0) * stride + tok * RP + (q4 * 4 < RP ? q4 * 4 : 0));
  }
  __builtin_amdgcn_sched_barrier(0);
  if (!t.ok) return;
  MLORA_STAMP(9);  // expand: record here
  const int slot = __builtin_amdgcn_readfirstlane(t.slot), m = __builtin_amdgcn_readfirstlane(t.m);
  const int eff = rank_pick(ranks, eff_rank, num_slots, slot, R);
  if (eff == 0) return;
  const char* bbase = uniform(static_cast<const char*>(sp.b) + static_cast<int64_t>(slot) * sp.n * (C * 16));
  expand_tile<T, C, SP>(lds, hsrc, stride, kparts, hv, bbase, static_cast<T*>(yv_) + sp.y_col, ys, rows, sp.n0, sp.n1, m, eff,
                        ONCE && __builtin_amdgcn_readfirstlane(t.once) != 0, scaling);
  MLORA_STAMP_END(13);  // expand: stores issued, acknowledged
}

// ---- both in one launch, fp32 ------------------------------------------------------------------------
// A workgroup takes a (tile, column range) and multiplies all of K itself, an eighth per wavefront through the same rings,
// its B rows and y requested ahead of them; nothing passes between workgroups.  What bounds it is what a compute unit takes
// in, x and A whole for every range (128 KB at rank 16, K = 1024, in about 3 us); what it saves is the second launch with its
// record, sums and drain.  Figures: solo_columns.
constexpr int kSoloWaves = 8;
constexpr int kSoloThreads = kSoloWaves * kWave;
template <int NA8, int XG = 2> struct SoloShape {
  static constexpr int RB = (NA8 + 1) / 2;
  static constexpr int ND = NA8 + XG;
  static constexpr int NST = ND <= 4 ? 3 : 2;
  static constexpr int BYTES = NST * ND * 1024;
};

template <typename T, int NA8, int R, int XG>
__device__ __forceinline__ void solo_shrink(char* rings, char* s_h, int hrow_bytes, const char* abase, uint32_t arow, const char* xbase,
                                            const uint32_t (&xoff)[2], int kchunks, int m, int eff, float scaling) {
  typedef SoloShape<NA8, XG> S;
  constexpr int RB = S::RB;
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int c0 = wave * kchunks / kSoloWaves, c1 = (wave + 1) * kchunks / kSoloWaves;
  char* ring = rings + wave * S::BYTES;
  Chains<RB> chains;
  chains.clear();
  walk_chunks<NA8, XG, false, S>(ring, abase, arow, R, xbase, xoff, c0, c1, [](int) {},
                      [&](int rb, int ks, const Pack8& aw, const Pack8& xa) { chains.add(rb, ks, aw, xa); });
  static_assert(RB * 1024 <= S::BYTES, "the ring holds the wavefront's sums");
  f32x4 acc[RB];
  chains.collect(acc);
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) *reinterpret_cast<f32x4*>(ring + (rb * kWave + lane) * 16) = acc[rb];
  __syncthreads();
  MLORA_STAMP(4);  // every wavefront's sums in LDS
  // the eighths, scaled, to the operand rows of the expand: lane holds ranks 16 rb + 4 (lane / 16) .. + 3 of token lane % 16
  constexpr int BLOCKS = (R + 15) / 16;
  if (wave < BLOCKS) {
    f32x4 s = {0.f, 0.f, 0.f, 0.f};
    if (wave < RB) {
      f32x4 v[kSoloWaves];
#pragma unroll
      for (int w = 0; w < kSoloWaves; ++w) v[w] = *reinterpret_cast<const f32x4*>(rings + w * S::BYTES + tid * 16);
#pragma unroll
      for (int i = 0; i < 4; ++i) s[i] = ((v[0][i] + v[1][i]) + (v[2][i] + v[3][i])) + ((v[4][i] + v[5][i]) + (v[6][i] + v[7][i]));
    }
    const int tok = lane & 15, r0 = wave * 16 + 4 * (lane >> 4);
#pragma unroll
    for (int i = 0; i < 4; ++i) s[i] = (tok < m && r0 + i < eff) ? s[i] * scaling : 0.f;
    *reinterpret_cast<f32x4*>(s_h + row_of_token(tok) * hrow_bytes + r0 * 4) = s;
  }
}

// grid (8, column ranges, tiles / 8).  C: 16-byte pieces of a B row.
template <int C>
__global__ __launch_bounds__(kSoloThreads) void solo_kernel(const int32_t* __restrict__ plan, const void* __restrict__ xv, void* __restrict__ yv_,
                                                            int64_t ys, int small_off, int T_, int num_slots, int kchunks, uint32_t xrow, float scaling,
                                                            int ring_bytes, const int32_t* __restrict__ eff_rank, ShrinkSlices sl, ExpandSplits splits) {
  typedef float T;
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  constexpr int R = C * PieceOf<T>::E, HROW = ExpandShape<C>::HROW;
  const int tid = threadIdx.x, lane = tid & (kWave - 1), lg = lane >> 4, wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  MLORA_STAMP(0);
  const ExpandSplit sp = splits.split[blockIdx.y];
  const int tile = blockIdx.z * 8 + blockIdx.x;
  const int32_t* rec = plan + small_off + tile * MLORA_SMALL_TILE_WORDS;
  const i32x4 r0 = *reinterpret_cast<const i32x4*>(rec);
  const i32x4 rows = spread_rows(rec, lg);
  int row[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) row[i] = rec[MLORA_SMALL_TILE_ROWS + i * 8 + (lane >> 3)];
  const PairTile t = pair_tile(r0, plan, tile, T_, num_slots, 0);
  const RankPrefetch ranks = rank_prefetch(eff_rank, num_slots, lane);
  __builtin_amdgcn_sched_barrier(0);
  if (!t.ok) {
    count_rejected_plan(plan, t.plan_ok);
    return;
  }
  MLORA_STAMP(1);  // record here
  const int slot = __builtin_amdgcn_readfirstlane(t.slot), m = __builtin_amdgcn_readfirstlane(t.m);
  const int eff = rank_pick(ranks, eff_rank, num_slots, slot, R);
  if (eff == 0) return;
  const uint32_t arow = static_cast<uint32_t>(kchunks) * kChunk;
  const char* abase = uniform(static_cast<const char*>(sl.a[sp.slice]) + static_cast<int64_t>(slot) * R * arow);
  const char* bbase = uniform(static_cast<const char*>(sp.b) + static_cast<int64_t>(slot) * sp.n * (C * 16));
  uint32_t xoff[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) xoff[i] = static_cast<uint32_t>(row[i]) * xrow;
  char* s_h = lds + ring_bytes;
  char* s_b = s_h + 16 * HROW + wave * (64 * C * 16);  // (of wavefronts with columns only)
  T* const ybase = static_cast<T*>(yv_) + sp.y_col;
  const int c0 = sp.n0 + wave * 64;
  const bool mine = c0 < sp.n1;
  const int groups = (eff + 7) >> 3;
  auto rest = [&](auto xi, auto xg) __attribute__((always_inline)) {
    constexpr int XI = decltype(xi)::value, XG = decltype(xg)::value;
    YSpan<T> yq[1][4];
    if (mine) request_b<T, C, 1>(s_b, bbase, c0, sp.n1, eff, false);
    request_y<T, 1, XI>(yq, ybase, ys, rows, c0, sp.n1);
    const char* xb = static_cast<const char*>(xv);
    if (R <= 8 || groups <= 1) solo_shrink<T, 1, R, XG>(lds, s_h, HROW, abase, arow, xb, xoff, kchunks, m, eff, scaling);
    else if (R <= 16 || groups <= 2) solo_shrink<T, 2, R, XG>(lds, s_h, HROW, abase, arow, xb, xoff, kchunks, m, eff, scaling);
    else solo_shrink<T, 4, R, XG>(lds, s_h, HROW, abase, arow, xb, xoff, kchunks, m, eff, scaling);
    __syncthreads();
    MLORA_STAMP(5);  // intermediate in LDS
    if (mine) finish_spans<T, C, 1, XI>(s_h, s_b, yq, ybase, ys, rows, c0, sp.n1, m, eff);
  };
  if (m <= 4) rest(std::integral_constant<int, 1>{}, std::integral_constant<int, 1>{});
  else if (m <= 8) rest(std::integral_constant<int, 2>{}, std::integral_constant<int, 1>{});
  else rest(std::integral_constant<int, 4>{}, std::integral_constant<int, 2>{});
}

int solo_ring(int r) {
  int most = SoloShape<1>::BYTES;
  if (r > 8 && SoloShape<2>::BYTES > most) most = SoloShape<2>::BYTES;
  if (r > 16 && SoloShape<4>::BYTES > most) most = SoloShape<4>::BYTES;
  return most * kSoloWaves;
}

int expand_lds(int c, int sp) {
  const int ksteps = (c + 3) / 4, hrow = ksteps * 64 + 16;
  return 2 * 16 * hrow + kPairWaves * sp * 64 * c * 16;
}

// Diagnostic knobs, read from the environment once and again after mlora_reload_knobs().
struct PairKnobs {
  int generation = -1, kparts, sp, wgs, solo, solo_cols, once;
  void read() {
    generation = knob_generation();
    kparts = env_int("MLORA_PAIR_KPARTS", 0);
    sp = env_int("MLORA_PAIR_SP", 0);
    wgs = env_int("MLORA_PAIR_WGS", 192);
    once = env_int("MLORA_PAIR_ONCE", -1);
    solo = env_int("MLORA_SOLO", 1);  // 0: never in one launch, 2: wherever it can be
    solo_cols = env_int("MLORA_SOLO_COLS", 0) / 64 % 9 * 64;  // at most 512
  }
};
const PairKnobs& pair_knobs() {
  static PairKnobs k;
  if (k.generation != knob_generation()) k.read();
  return k;
}

int element_bytes(int dtype) { return dtype == MLORA_DTYPE_F32 ? 4 : 2; }
// One K part's partial sums: sixteen rows of the padded rank per place of the tile list and slice.
size_t part_bytes(const MloraAddArgs* a, const PlanLayout& lay) {
  return static_cast<size_t>(lay.cap_small) * MLORA_TILE_SMALL * a->num_slices * ((a->r + 15) & ~15) * sizeof(float);
}

struct PairLaunch {
  const MloraAddArgs* a;
  PlanLayout lay;
  int parts_log2, sp;
  bool once;      // instances that can request A and B of a slot's only tile with the non-temporal hint
  int slices_once;  // number of slices, and for those instances above its eight bits from how many slots with tokens on they do (a word of its own
                    // would lie behind the sixteen that arrive preloaded: 201 streams, 1760 us a step instead of 1754)
};

template <typename T, bool CHAINS, bool ONCE> void launch_pair_shrink_one(const PairLaunch& l) {
  const MloraAddArgs* a = l.a;
  ShrinkSlices sl;
  for (int i = 0; i < MLORA_MAX_SLICES; ++i) sl.a[i] = i < a->num_slices ? a->slices[i].a : nullptr;
  allow_lds<pair_shrink_kernel<T, CHAINS, ONCE>>(shrink_lds(a->r));
  hipLaunchKernelGGL((pair_shrink_kernel<T, CHAINS, ONCE>), dim3(8, static_cast<unsigned>(a->num_slices << l.parts_log2), static_cast<unsigned>(l.lay.cap_small / 8)),
                     dim3(kPairThreads), shrink_lds(a->r), static_cast<hipStream_t>(a->stream), a->plan, a->x, partials_of(a), l.lay.small_off,
                     a->num_tokens, a->num_slots, static_cast<int>(a->k * sizeof(T) / kChunk), static_cast<uint32_t>(a->x_stride * sizeof(T)), a->r,
                     l.parts_log2, l.slices_once, a->effective_rank, sl);
}

template <typename T, bool CHAINS> void launch_pair_shrink(const PairLaunch& l) {
  if (l.once) launch_pair_shrink_one<T, CHAINS, true>(l);
  else launch_pair_shrink_one<T, CHAINS, false>(l);
}

template <typename T, int C, int SP, bool ONCE> void launch_pair_expand_one(const PairLaunch& l, const ExpandSplits& splits, int total) {
  const MloraAddArgs* a = l.a;
  allow_lds<pair_expand_kernel<T, C, SP, ONCE>>(expand_lds(C, SP));
  hipLaunchKernelGGL((pair_expand_kernel<T, C, SP, ONCE>), dim3(8, static_cast<unsigned>(total), static_cast<unsigned>(l.lay.cap_small / 8)), dim3(kPairThreads),
                     expand_lds(C, SP), static_cast<hipStream_t>(a->stream), a->plan, partials_of(a), a->y, a->y_stride, l.lay.small_off, a->num_tokens,
                     a->num_slots, 1 << l.parts_log2, l.slices_once, a->scaling, a->effective_rank, splits);
}

template <typename T, int C> bool launch_pair_expand(const PairLaunch& l, const ExpandSplits& splits, int total) {
  if (l.sp == 1) {
    if (l.once) launch_pair_expand_one<T, C, 1, true>(l, splits, total);
    else launch_pair_expand_one<T, C, 1, false>(l, splits, total);
  } else {
    if (l.once) launch_pair_expand_one<T, C, 2, true>(l, splits, total);
    else launch_pair_expand_one<T, C, 2, false>(l, splits, total);
  }
  return true;
}

template <typename T> bool launch_pair_type(const PairLaunch& l, const ExpandSplits& splits, int total) {
  if constexpr (sizeof(T) == 4) {
    if (exact_rank(l.a->r)) launch_pair_shrink<T, false>(l);
    else launch_pair_shrink<T, true>(l);
  } else {
    launch_pair_shrink<T, false>(l);
  }
  constexpr int E8 = sizeof(T) / 2;  // 16-byte pieces of eight ranks
  switch (l.a->r / 8) {
    case 1: return launch_pair_expand<T, 1 * E8>(l, splits, total);
    case 2: return launch_pair_expand<T, 2 * E8>(l, splits, total);
    case 3: return launch_pair_expand<T, 3 * E8>(l, splits, total);
    case 4: return launch_pair_expand<T, 4 * E8>(l, splits, total);
    case 5: return launch_pair_expand<T, 5 * E8>(l, splits, total);
    case 6: return launch_pair_expand<T, 6 * E8>(l, splits, total);
    case 7: return launch_pair_expand<T, 7 * E8>(l, splits, total);
    case 8: return launch_pair_expand<T, 8 * E8>(l, splits, total);
  }
  return false;
}

}  // namespace

void pair_trace_set(void* buf) {
#ifdef MLORA_TRACE
  (void)hipMemcpyToSymbol(HIP_SYMBOL(trace_buf), &buf, sizeof(buf));
#else
  (void)buf;
#endif
}

bool pair_supported(const MloraAddArgs* a) {
  const int64_t e = element_bytes(a->dtype);
  if (a->k <= 0 || (a->k * e) % kChunk || !a->plan) return false;
  if (!padded_rank(a->r) || (e == 4 && a->form != MLORA_FORM_AUTO && !exact_rank(a->r))) return false;  // (by name fp32 has the instances' ranks only)
  // 32-bit offsets of the x rows, A rows and B pieces; 16-byte loads of x and B, four columns of y at a time
  if (a->num_tokens * (a->x_stride * e) >= (1ll << 32) || a->r * (a->k * e) >= (1ll << 32)) return false;
  if ((a->x_stride * e) % 16 || a->y_stride % 4 || !a->workspace || (reinterpret_cast<uintptr_t>(a->workspace) & 255)) return false;
  if ((reinterpret_cast<uintptr_t>(a->x) & 15) || (reinterpret_cast<uintptr_t>(a->y) & (4 * e - 1))) return false;
  for (int i = 0; i < a->num_slices; ++i) {
    const MloraSlice& s = a->slices[i];
    if (s.n <= 0 || s.n % 4 || s.y_col % 4 || (reinterpret_cast<uintptr_t>(s.a) & 15) || (reinterpret_cast<uintptr_t>(s.b) & 15)) return false;
    if (s.n * (a->r * e) >= (1ll << 32)) return false;
  }
  int total = 0;
  for (int i = 0; i < a->num_slices; ++i) total += (a->slices[i].n + 511) / 512;
  return total <= kMaxSplits && partials_room(a) >= part_bytes(a, plan_layout(a->num_tokens, a->num_slots));
}

namespace {
int columns_total(const MloraAddArgs* a, int nt) {
  int total = 0;
  for (int i = 0; i < a->num_slices; ++i) total += (a->slices[i].n + nt - 1) / nt;
  return total;
}
}  // namespace

// Columns of a range of the one launch where it beats the pair, else 0: fp32, x and A of a tile no more than rank 16's at K = 2048,
// and every workgroup resident at once (tile t runs on XCD t % 8, which has 32 compute units; a second round repeats the
// shrink).  us per call, the pair / one launch in ranges of 256 / 512 columns, q|k|v, o and gate_up:
//   rank 16, K = 1024:  1 token of 4 slots 6.2 / 5.3 / 5.9, 6.1 / 5.2 / 5.9, 7.1 / 5.9 / 6.6; 64 of 4 7.3 / 6.0 / 6.8, 7.2 / 5.8 / 6.5, 8.5 / 7.4 / 8.1; 64 of 32
//   8.3 / 6.3 / 7.1, 7.6 / 6.1 / 6.7, 10.5 / 18.8 / 13.2 (104 and 52 workgroups an XCD); 256 of 64 10.6 / 10.8 / 8.7 (48 and 32), 8.1 / 7.2 / 7.5.
//   rank 8, K = 1024:   64 of 4 7.1 / 5.7 / 6.1, 6.9 / 5.7 / 6.1, 8.1 / 6.8 / 7.3; 256 of 8 7.8 / 6.2 / 6.9, 7.3 / 6.0 / 6.6, 11.1 / 15.6 / 12.9.
//   rank 16, K = 2048:  64 of 4 8.0 / 7.8 / 8.6, 7.6 / 7.4 / 8.2; 64 of 32 10.2 / 12.9 / 8.9 (48 and 24), 8.1 / 8.0 / 8.5; 256 of 64 14.5 / 21.9 / 18.4.
//   rank 32, K = 1024 (256 columns: B rows of 512 do not fit the LDS):  64 of 4 8.3 / 7.6, 7.8 / 7.0, 9.7 / 9.5; 8 of 8 gate_up 8.6 / 9.0 (32); 64 of
//   32 9.8 / 8.0, 8.9 / 7.7; 256 of 64 o 10.1 / 9.3 (32), q|k|v 14.2 / 16.6 (48).  At K = 2048 it loses throughout (64 of 4 9.2 / 10.0).
//   K = 4096 loses at every rank (rank 8, 1 token: 7.1 / 8.9).
static int solo_columns(const MloraAddArgs* a, const Batch& batch) {
  if (a->dtype != MLORA_DTYPE_F32 || a->form != MLORA_FORM_AUTO || !(a->r == 8 || a->r == 16 || a->r == 32)) return 0;
  if (pair_knobs().solo != 1) {
    if (pair_knobs().solo != 2) return 0;
    return pair_knobs().solo_cols > 0 && columns_total(a, pair_knobs().solo_cols) <= kMaxSplits && a->r * pair_knobs().solo_cols <= 8192
               ? pair_knobs().solo_cols
               : columns_total(a, 256) <= kMaxSplits ? 256 : 0;
  }
  if (a->k > 2048 || static_cast<long long>(a->r) * a->k > 32768) return 0;
  const int layers = (small_tiles_about(batch) + 7) / 8;  // tiles of an XCD
  for (int nt = 256; nt <= (a->r <= 16 ? 512 : 256); nt *= 2) {
    const int total = columns_total(a, nt);
    if (total <= kMaxSplits && layers * total <= (a->r <= 16 ? 32 : 24)) return nt;
  }
  return 0;
}

namespace {
template <int C> void launch_solo_rank(const MloraAddArgs* a, const PlanLayout& lay, int total, int lds, const ShrinkSlices& sl, const ExpandSplits& splits) {
  allow_lds<solo_kernel<C>>(lds);
  hipLaunchKernelGGL((solo_kernel<C>), dim3(8, static_cast<unsigned>(total), static_cast<unsigned>(lay.cap_small / 8)), dim3(kSoloThreads), lds,
                     static_cast<hipStream_t>(a->stream), a->plan, a->x, a->y, a->y_stride, lay.small_off, a->num_tokens, a->num_slots,
                     static_cast<int>(a->k * sizeof(float) / kChunk), static_cast<uint32_t>(a->x_stride * sizeof(float)), a->scaling, solo_ring(a->r),
                     a->effective_rank, sl, splits);
}
}  // namespace

static int launch_solo(const MloraAddArgs* a, int nt) {
  const PlanLayout lay = plan_layout(a->num_tokens, a->num_slots);
  if (lay.cap_small == 0) return 0;
  ExpandSplits splits;
  const int total = columns_total(a, nt);
  int s = 0;
  for (int i = 0; i < a->num_slices; ++i)
    for (int n0 = 0; n0 < a->slices[i].n; n0 += nt) {
      ExpandSplit& d = splits.split[s++];
      d.b = a->slices[i].b; d.n = a->slices[i].n; d.y_col = a->slices[i].y_col; d.slice = i; d.pad = 0;
      d.n0 = n0; d.n1 = n0 + nt < a->slices[i].n ? n0 + nt : a->slices[i].n;
    }
  ShrinkSlices sl;
  for (int i = 0; i < MLORA_MAX_SLICES; ++i) sl.a[i] = i < a->num_slices ? a->slices[i].a : nullptr;
  const int c = a->r / 4, lds = solo_ring(a->r) + 16 * (((c + 3) / 4) * 64 + 16) + nt * c * 16;
  switch (a->r) {
    case 8: launch_solo_rank<2>(a, lay, total, lds, sl, splits); break;
    case 16: launch_solo_rank<4>(a, lay, total, lds, sl, splits); break;
    case 32: launch_solo_rank<8>(a, lay, total, lds, sl, splits); break;
    default: set_error("mlora_add_lora(pair): unsupported rank %d", a->r); return MLORA_E_UNSUPPORTED;
  }
  return check_launch("mlora_add_lora(fp32, one launch over small tiles)");
}

int launch_pair(const MloraAddArgs* a, const Batch& batch) {
  if (const int nt = solo_columns(a, batch)) return launch_solo(a, nt);
  PairLaunch l;
  l.a = a;
  l.lay = plan_layout(a->num_tokens, a->num_slots);
  const int segs = a->num_slots < a->num_tokens ? a->num_slots : a->num_tokens;
  const int by_tokens = (a->num_tokens + MLORA_TILE_SMALL - 1) / MLORA_TILE_SMALL;
  const int tiles = segs > by_tokens ? segs : by_tokens;  // about the number of tiles in use
  const int kchunks = static_cast<int>(static_cast<int64_t>(a->k) * element_bytes(a->dtype) / kChunk);
  const size_t room = partials_room(a) / part_bytes(a, l.lay);
  long long cols = 0;
  for (int i = 0; i < a->num_slices; ++i) cols += a->slices[i].n;
  // (how many slots have tokens is in the plan's header, which the kernels read: behind a capture the host knows only how many may)
  const long long per_slot = static_cast<long long>(a->r) * (static_cast<long long>(a->num_slices) * a->k + cols) * element_bytes(a->dtype);
  const long long need = (kOnceBytes + per_slot - 1) / per_slot;  // slots whose weights are that much
  const int once_from = pair_knobs().once > 0 ? 0 : need <= MLORA_MAX_SLOTS ? static_cast<int>(need) : MLORA_MAX_SLOTS + 1;
  l.once = pair_knobs().once < 0 ? batch.slots >= once_from : pair_knobs().once != 0;
  static_assert(MLORA_MAX_SLICES < 256 && MLORA_MAX_SLOTS + 1 < 1 << 23, "one word");
  l.slices_once = l.once ? a->num_slices | once_from << 8 : a->num_slices;
  // K parts: workgroups for most compute units, no more (every column range of the second launch
  // takes in every part's sums), and a chunk per wavefront at least
  int want = pair_knobs().kparts;
  l.parts_log2 = 0;
  while ((2u << l.parts_log2) <= room && (2 << l.parts_log2) <= kMaxParts && (2 << l.parts_log2) * kPairWaves <= kchunks &&
         (want > 0 ? (2 << l.parts_log2) <= want : (tiles * a->num_slices << l.parts_log2) < pair_knobs().wgs))
    ++l.parts_log2;
  l.sp = pair_knobs().sp > 0 ? pair_knobs().sp : 1;
  ExpandSplits splits;
  int nt, total;
  for (;; l.sp = 2) {
    nt = l.sp * 64 * kPairWaves;
    total = 0;
    for (int i = 0; i < a->num_slices; ++i) total += (a->slices[i].n + nt - 1) / nt;
    if (total <= kMaxSplits || l.sp == 2) break;
  }
  int s = 0;
  for (int i = 0; i < a->num_slices; ++i)
    for (int n0 = 0; n0 < a->slices[i].n; n0 += nt) {
      ExpandSplit& d = splits.split[s++];
      d.b = a->slices[i].b; d.n = a->slices[i].n; d.y_col = a->slices[i].y_col; d.slice = i; d.pad = 0;
      d.n0 = n0; d.n1 = n0 + nt < a->slices[i].n ? n0 + nt : a->slices[i].n;
    }
  if (l.lay.cap_small == 0) return 0;
  bool ok;
  if (a->dtype == MLORA_DTYPE_BF16) ok = launch_pair_type<__bf16>(l, splits, total);
  else if (a->dtype == MLORA_DTYPE_F16) ok = launch_pair_type<_Float16>(l, splits, total);
  else ok = launch_pair_type<float>(l, splits, total);
  if (!ok) { set_error("mlora_add_lora(pair): unsupported rank %d", a->r); return MLORA_E_UNSUPPORTED; }
  return check_launch("mlora_add_lora(shrink and expand launches)");
}

}  // namespace mlora
