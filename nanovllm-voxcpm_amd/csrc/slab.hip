// Shrink launch of the two-launch form over 64-token tiles (sgmv.hip): H^T = A[slot] . X_tile^T for a (tile, slice,
// K part), fp32 partial sums to the workspace.  Computes what the reference computes with its segment-grouped
// shrink kernel (nanovllm_voxcpm/lora_ops/triton_ops/lora_shrink_op.py:16-101).
//
// What bounds it is the bytes a compute unit takes in and how few instructions ask for them.  128-bit loads in the matrix
// cores' operand layout (sixteen rows in sixteen consecutive lanes) bring 9.4 TB/s out of the L2 into 256 compute units,
// loads along rows straight to LDS 33.0 (from HBM both bring 6.0), and operands that wait in registers limit
// what can be on its way.
// Here both operands go to LDS by direct loads of whole row pieces (128 bytes of eight rows per load), into a
// ring of two to four stages that each wavefront has to itself: the two wavefronts of a workgroup
// cut K between them, each multiplies all tokens and ranks of the tile over its share, so nothing but
// the sums at the end passes between them and no barrier stands between request and product.
// Two wavefronts, not four: their rings (64 KB at rank 64) keep a compute unit's 64 KB of requests on their way, and two
// workgroups fit a compute unit, so that one starts while the other sums up.  Rings of 48 KB, three
// stages at rank 64 with one workgroup per compute unit, are 1 % slower (494 calls of one or two slices, in the same K parts).
// Against x through registers it gained (rank 32, 5000 tokens, K = 4096, with the expand 21.0 -> 18.5 us per call); the ring that the wavefronts of
// sgmv.hip share takes 0.96 to 0.99 of its time (sgmv_shape), so AUTO takes this kernel for some calls of rank 64 only.
#include "common.h"
#include "dma.h"
#include "launch.h"
#include "lds.h"
#include "sgmv_body.h"

namespace mlora {

namespace {

constexpr int kSlabWaves = 2;
constexpr int kSlabThreads = kSlabWaves * kWave;
constexpr int kPiece = 128;  // bytes of a row per stage

// NA8: groups of eight ranks, TB: blocks of sixteen tokens; both operands in groups of eight rows, 1 KB each.
template <int NA8, int TB> struct SlabShape {
  static constexpr int RB = (NA8 + 1) / 2;
  static constexpr int ND = NA8 + 2 * TB;                          // direct loads per stage
  static constexpr int NST = ND > 6 ? 2 : ND > 4 ? 3 : 4;  // stages of a wavefront's ring
  static constexpr int BYTES = NST * ND * 1024;
  static_assert(RB * TB <= NST * ND, "the ring holds the wavefront's sums");
};

template <typename T, int NA8, int TB>
__device__ __forceinline__ void slab_tile(char* lds, const char* abase, uint32_t arow, int rbuf, const char* xbase, const uint32_t (&xoff)[2 * TB], int c0,
                                          int c1, float* __restrict__ dst, int64_t hrow, int m) {
  typedef SlabShape<NA8, TB> S;
  constexpr int RB = S::RB, ND = S::ND, NST = S::NST;
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int lr = lane & 15, lg = lane >> 4;
  // chunk p of a row goes to place p ^ (row & 7): the sixteen rows of an operand read fall on different banks
  const uint32_t swz = static_cast<uint32_t>((lane & 7) ^ (lane >> 3)) * 16;
  uint32_t aoff[NA8];
#pragma unroll
  for (int g = 0; g < NA8; ++g) {
    const int row = g * 8 + (lane >> 3);
    aoff[g] = static_cast<uint32_t>(row < rbuf ? row : rbuf - 1) * arow + swz;
  }
  char* ring = lds + wave * S::BYTES;
  const uint32_t to0 = __builtin_amdgcn_readfirstlane(lds_address(ring));
  auto issue = [&](int c, int stage) {
    const char* a = abase + static_cast<int64_t>(c) * kPiece;
    const char* x = xbase + static_cast<int64_t>(c) * kPiece;
    const uint32_t to = to0 + stage * (ND * 1024);
#pragma unroll
    for (int g = 0; g < 2 * TB; ++g) dma16(x, xoff[g] + swz, to + (NA8 + g) * 1024);
#pragma unroll
    for (int g = 0; g < NA8; ++g) dma16(a, aoff[g], to + g * 1024);
  };
  f32x4 acc[RB][TB];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb)
#pragma unroll
    for (int tb = 0; tb < TB; ++tb) acc[rb][tb] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int n = c1 - c0;
#pragma unroll
  for (int s = 0; s < NST - 1; ++s)
    if (s < n) issue(c0 + s, s);
  int stage = 0, into = NST - 1;
  for (int c = 0; c < n; ++c) {
    if (c + NST - 1 < n) {
      wait_lds();  // the operand reads of the step before, from the stage that is filled next, are through
      issue(c0 + c + NST - 1, into);
    }
    const int younger = n - 1 - c < NST - 1 ? n - 1 - c : NST - 1;  // stages requested behind this one
    if (NST >= 4 && younger == 3) wait_loads<(NST >= 4 ? 3 : 0) * ND>();
    else if (NST >= 3 && younger == 2) wait_loads<(NST >= 3 ? 2 : 0) * ND>();
    else if (younger == 1) wait_loads<ND>();
    else wait_loads<0>();
    const char* st = ring + stage * (ND * 1024) + lr * 128 + ((lg ^ (lr & 7)) * 16);
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      const char* at = st + (ks == 0 ? 0 : (lg ^ (lr & 7)) & 4 ? -64 : 64);  // chunk lg, then chunk lg + 4, of the swizzled row
      Pack8 xa[TB], aw[RB];
#pragma unroll
      for (int tb = 0; tb < TB; ++tb) xa[tb].raw = *reinterpret_cast<const i32x4*>(at + (NA8 + 2 * tb) * 1024);
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) aw[rb].raw = *reinterpret_cast<const i32x4*>(at + rb * 2048);
#pragma unroll
      for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int tb = 0; tb < TB; ++tb) acc[rb][tb] = Mma<T>::run(aw[rb], xa[tb], acc[rb][tb]);
    }
    stage = stage + 1 == NST ? 0 : stage + 1;
    into = into + 1 == NST ? 0 : into + 1;
  }
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) mfma_settle(acc[rb]);
  // the wavefronts' sums, the first one's first, through the rings' memory.  acc[rb][tb]: lane holds ranks 16 rb + 4 lg .. + 3
  // of token 16 tb + lr
#pragma unroll
  for (int rb = 0; rb < RB; ++rb)
#pragma unroll
    for (int tb = 0; tb < TB; ++tb) *reinterpret_cast<f32x4*>(ring + ((rb * TB + tb) * kWave + lane) * 16) = acc[rb][tb];
  __syncthreads();
#pragma unroll
  for (int q = 0; q < (RB * TB + kSlabWaves - 1) / kSlabWaves; ++q) {
    const int b = q * kSlabWaves + wave, rb = b / TB, tb = b % TB;
    if (RB * TB % kSlabWaves == 0 || b < RB * TB) {
      f32x4 v[kSlabWaves];
#pragma unroll
      for (int w = 0; w < kSlabWaves; ++w) v[w] = *reinterpret_cast<const f32x4*>(lds + w * S::BYTES + (b * kWave + lane) * 16);
#pragma unroll
      for (int w = 1; w < kSlabWaves; ++w)
#pragma unroll
        for (int i = 0; i < 4; ++i) v[0][i] += v[w][i];
      const int tok = tb * 16 + lr, r = rb * 16 + 4 * lg;
      if (tok < m && r < rbuf) *reinterpret_cast<f32x4*>(dst + tok * hrow + r) = v[0];
    }
  }
}

template <typename T, int TB>
__device__ __forceinline__ void slab_ranks(int groups, char* lds, const char* abase, uint32_t arow, int rbuf, const char* xbase,
                                           const uint32_t (&xrows)[8], int c0, int c1, float* __restrict__ dst, int64_t hrow, int m) {
  uint32_t xoff[2 * TB];
#pragma unroll
  for (int g = 0; g < 2 * TB; ++g) xoff[g] = xrows[g];
  if (groups <= 1) slab_tile<T, 1, TB>(lds, abase, arow, rbuf, xbase, xoff, c0, c1, dst, hrow, m);
  else if (groups == 2) slab_tile<T, 2, TB>(lds, abase, arow, rbuf, xbase, xoff, c0, c1, dst, hrow, m);
  else if (groups <= 4) slab_tile<T, 4, TB>(lds, abase, arow, rbuf, xbase, xoff, c0, c1, dst, hrow, m);
  else slab_tile<T, 8, TB>(lds, abase, arow, rbuf, xbase, xoff, c0, c1, dst, hrow, m);
}

// grid (8, slices * K parts, tiles / 8): blockIdx.x is the XCD
template <typename T>
__global__ __launch_bounds__(kSlabThreads) void slab_shrink_kernel(const int32_t* __restrict__ plan, const void* __restrict__ xv, float* __restrict__ hws,
                                                                   int big_off, int small_off, int big_cap, int bigrows_off, int T_, int num_slots,
                                                                   int kchunks, uint32_t xrow, int rbuf, int parts, int num_slices,
                                                                   const int32_t* __restrict__ eff_rank, ShrinkSlices sl) {
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int tile = tile_position(big_cap);
  int row[8];
#pragma unroll
  for (int g = 0; g < 8; ++g) row[g] = tile_row(plan, bigrows_off, small_off, big_cap, tile, g * 8 + (lane >> 3));
  const TileRef tr = fetch_tile(plan, big_off, small_off, big_cap, tile, T_, num_slots);
  const RankPrefetch ranks = rank_prefetch(eff_rank, num_slots, lane);
  __builtin_amdgcn_sched_barrier(0);
  if (!tr.ok) {
    count_rejected_plan(plan, tr.plan_ok);
    return;
  }
  const int slot = __builtin_amdgcn_readfirstlane(tr.slot), m = __builtin_amdgcn_readfirstlane(tr.m), start = __builtin_amdgcn_readfirstlane(tr.start);
  const int eff = rank_pick(ranks, eff_rank, num_slots, slot, rbuf);
  if (eff == 0) return;
  const int slice = blockIdx.y / parts, part = blockIdx.y - slice * parts;
  const int p0 = part * kchunks / parts, p1 = (part + 1) * kchunks / parts;
  const int c0 = p0 + wave * (p1 - p0) / kSlabWaves, c1 = p0 + (wave + 1) * (p1 - p0) / kSlabWaves;
  const uint32_t arow = static_cast<uint32_t>(kchunks) * kPiece;
  const char* abase = uniform(static_cast<const char*>(sl.a[slice]) + static_cast<int64_t>(slot) * rbuf * arow);
  const char* xbase = static_cast<const char*>(xv);
  uint32_t xoff[8];
#pragma unroll
  for (int g = 0; g < 8; ++g) xoff[g] = static_cast<uint32_t>(row[g]) * xrow;
  const int64_t hrow = static_cast<int64_t>(num_slices) * rbuf;
  float* dst = hws + static_cast<int64_t>(part) * T_ * hrow + static_cast<int64_t>(start) * hrow + slice * rbuf;
  const int groups = (eff + 7) >> 3;
  if (m <= 16) slab_ranks<T, 1>(groups, lds, abase, arow, rbuf, xbase, xoff, c0, c1, dst, hrow, m);
  else if (m <= 32) slab_ranks<T, 2>(groups, lds, abase, arow, rbuf, xbase, xoff, c0, c1, dst, hrow, m);
  else slab_ranks<T, 4>(groups, lds, abase, arow, rbuf, xbase, xoff, c0, c1, dst, hrow, m);
}

// The most LDS any adapter and tile of buffers of this rank may need.
template <int NA8> int slab_bytes_of() {
  int most = SlabShape<NA8, 1>::BYTES;
  most = SlabShape<NA8, 2>::BYTES > most ? SlabShape<NA8, 2>::BYTES : most;
  return SlabShape<NA8, 4>::BYTES > most ? SlabShape<NA8, 4>::BYTES : most;
}
int slab_lds(int r) {
  int most = slab_bytes_of<1>();
  auto with = [&](int b) { most = b > most ? b : most; };
  if (r > 8) with(slab_bytes_of<2>());
  if (r > 16) with(slab_bytes_of<4>());
  if (r > 32) with(slab_bytes_of<8>());
  return most * kSlabWaves;
}

template <typename T> void launch_slab_type(const MloraAddArgs* a, const PlanLayout& lay, int big_cap, int tiles8, int parts, const ShrinkSlices& sl) {
  allow_lds<slab_shrink_kernel<T>>(slab_lds(a->r));
  hipLaunchKernelGGL((slab_shrink_kernel<T>), dim3(8, static_cast<unsigned>(a->num_slices * parts), static_cast<unsigned>(tiles8)), dim3(kSlabThreads),
                     slab_lds(a->r), static_cast<hipStream_t>(a->stream), a->plan, a->x, partials_of(a), lay.big_off, lay.small_off, big_cap,
                     lay.bigrows_off, a->num_tokens, a->num_slots, static_cast<int>(a->k * sizeof(T) / kPiece),
                     static_cast<uint32_t>(a->x_stride * sizeof(T)), a->r, parts, a->num_slices, a->effective_rank, sl);
}

}  // namespace

// 32-bit offsets of x rows and A rows.
bool slab_supported(const MloraAddArgs* a) {
  return a->k % 64 == 0 && a->num_tokens * (a->x_stride * 2) < (1ll << 32) && static_cast<int64_t>(a->r) * a->k * 2 < (1ll << 32);
}

void launch_slab_shrink(const MloraAddArgs* a, const PlanLayout& lay, int big_cap, int tiles8, int parts, const void* const* slices) {
  ShrinkSlices sl;
  for (int i = 0; i < MLORA_MAX_SLICES; ++i) sl.a[i] = slices[i];
  if (a->dtype == MLORA_DTYPE_BF16) launch_slab_type<__bf16>(a, lay, big_cap, tiles8, parts, sl);
  else launch_slab_type<_Float16>(a, lay, big_cap, tiles8, parts, sl);
}

}  // namespace mlora
