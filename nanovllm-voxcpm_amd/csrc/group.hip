// The low-level shrink and expand over tiles of up to sixteen tokens of a slot, both products on the matrix cores.  Reference
// semantics as in token.hip: lora_shrink (zero-filled output, scaling in the shrink: lora_ops/triton_ops/lora_shrink_op.py:257-341),
// lora_expand (offset_start, add_inputs, product rounded to B's type first: lora_expand_op.py:94-170).
//
// The ops are given a slot id per token and nothing a kernel could trust to be sorted, so the one-workgroup-per-token
// kernels (token.hip) let every token fetch A[slot] and B[slot] again and add 64 lanes up per rank.  Here a workgroup serves a
// tile of a slot: it requests the slot vector and, from its own index or its token's id, the slot's weights, finds
// its tokens among the ids as they arrive, and fetches each weight once for all of them.
//
// What bounds it: two trips to memory (ids, then the rows they name) and a compute unit's intake of weights in the second one;
// hence ranks in blocks of eight or sixteen and tokens in tiles of four to sixteen, as many workgroups as the chip takes.
#include "common.h"
#include "group_layout.h"
#include "launch.h"

namespace mlora {

namespace {

struct Places : GroupPlaces {
  const int32_t* tts;
};

__device__ __forceinline__ int known_slot(const Places& p, int id) { return id >= 0 && id < p.num_slots ? id : p.num_slots; }

// Lists the tokens of a tile in ascending order; returns their number and, through `rows`, where in s_rows they stand.  By token: the
// tile that starts at token `from` of `slot`; 0 when the tokens of the slot before it do not fill whole tiles.  By slot: the tile-th
// tile of the slot, whose width follows from the slot's number of tokens; until that is known, both widths are listed.
// s_rows: MLORA_TILE_SMALL words (by slot: twice as many), s_wave: two words per wavefront.
template <int THREADS, int GRID>
__device__ __forceinline__ int list_tile(const Places& p, int first_id, int slot, int from, int tile, int* __restrict__ s_rows,
                                         int* __restrict__ s_wave, const int*& rows) {
  constexpr int W = THREADS / kWave;
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
  int late = 0, early = 0, id = first_id, half = 0, width = p.width;
  for (int base = 0; base < p.T; base += THREADS) {
    const int t = base + tid;
    if (base > 0) id = p.tts[t < p.T ? t : p.T - 1];
    const bool match = t < p.T && known_slot(p, id) == slot;
    const uint64_t set = __builtin_amdgcn_ballot_w64(match && t >= from), before = __builtin_amdgcn_ballot_w64(match && t < from);
    if (lane == 0) s_wave[half * W + wave] = __popcll(set) | (__popcll(before) << 16);
    __syncthreads();
    const int c = s_wave[half * W + (lane < W ? lane : 0)];
    int pos = late;
#pragma unroll
    for (int w = 0; w < W; ++w) {
      const int n = __builtin_amdgcn_readlane(c, w);
      if (w < wave) pos += n & 0xffff;
      late += n & 0xffff;
      early += n >> 16;
    }
    pos += __popcll(set & ((1ull << lane) - 1ull));
    if constexpr (GRID == kBySlot) width = tile_width(p, late);
    const unsigned at = pos - tile * width, wide = pos - tile * MLORA_TILE_SMALL;
    if (match && t >= from && at < static_cast<unsigned>(width)) s_rows[(width != p.width ? MLORA_TILE_SMALL : 0) + at] = t;
    if (GRID == kBySlot && base + THREADS < p.T && width == p.width) {  // (ids to come may make the slot's tiles wide ones)
      if (match && t >= from && wide < static_cast<unsigned>(MLORA_TILE_SMALL)) s_rows[MLORA_TILE_SMALL + wide] = t;
    }
    half ^= 1;
  }
  __syncthreads();
  rows = s_rows + (width != p.width ? MLORA_TILE_SMALL : 0);
  const int n = late - tile * width;
  return early % width != 0 || n <= 0 ? 0 : n < width ? n : width;
}

// By slot, behind the tiles with a place of their own: the slot and, of that, the tile that the q-th further place stands for, or slot -1.
template <int THREADS>
__device__ __forceinline__ void find_tile(const Places& p, int first_id, int q, int* __restrict__ s_hist, int* __restrict__ s_found) {
  const int tid = threadIdx.x, lane = tid & (kWave - 1);
  for (int s = tid; s < p.num_slots; s += THREADS) s_hist[s] = 0;
  if (tid == 0) s_found[0] = -1;
  __syncthreads();
  for (int base = 0; base < p.T; base += THREADS) {
    const int t = base + tid, s = t < p.T ? known_slot(p, base == 0 ? first_id : p.tts[t]) : p.num_slots;
    // (the first token's slot in one addition: one adapter's tokens, each with an addition of its own to the same word, are a queue
    // of 512 at the LDS unit)
    const uint64_t any = __builtin_amdgcn_ballot_w64(s < p.num_slots);
    if (any != 0) {
      const int one = __builtin_amdgcn_readlane(s, __builtin_ctzll(any));
      const uint64_t same = __builtin_amdgcn_ballot_w64(s == one);
      if (lane == 0) atomicAdd(&s_hist[one], __popcll(same));
      if (s < p.num_slots && s != one) atomicAdd(&s_hist[s], 1);
    }
  }
  __syncthreads();
  if (tid < kWave) {
    int run = 0;
    for (int base = 0; base < p.num_slots; base += kWave) {
      const int s = base + lane, mine = s < p.num_slots ? tiles_beyond(p, s_hist[s]) : 0;
      int sum = mine;
#pragma unroll
      for (int d = 1; d < kWave; d *= 2) {
        const int up = __shfl_up(sum, d, kWave);
        if (lane >= d) sum += up;
      }
      const int at = q - (run + sum - mine);
      if (at >= 0 && at < mine) {
        s_found[0] = s;
        s_found[1] = p.tiles + at;
      }
      run += __builtin_amdgcn_readlane(sum, kWave - 1);
    }
  }
  __syncthreads();
}

// ---- shrink -------------------------------------------------------------------------------------
constexpr int kShrinkWaves = 8;  // a wavefront takes an eighth of K, in rounds of 128 columns
constexpr int kShrinkThreads = kShrinkWaves * kWave;
constexpr int kRound = 128 * kShrinkWaves;

struct GroupShrinkParams {
  void* out;
  int64_t xs;
  int out_dtype;
  float scaling;
  const void* a[MLORA_MAX_SLICES];
};

__device__ __forceinline__ void store_as(void* out, int64_t at, float v, int dtype) {
  if (dtype == MLORA_DTYPE_F32) static_cast<float*>(out)[at] = v;
  else if (dtype == MLORA_DTYPE_F16) static_cast<_Float16*>(out)[at] = from_f32<_Float16>(v);
  else static_cast<__bf16*>(out)[at] = from_f32<__bf16>(v);
}

// out[slice, t, :] = scaling * x[t] . A[s]^T, zero for rows without a slot; grid (8, slices * blocks, places / 8), blockIdx.x the XCD
// (a slot's workgroups share one).  RW: ranks of a workgroup (8 or 16); CH: rounds whose operands are on their way together.
template <typename T, int RW, int CH, int GRID>
__global__ __launch_bounds__(kShrinkThreads) void group_shrink_kernel(const int32_t* __restrict__ tts, int T_, int num_slots, int width, int slots8,
                                                                      int tiles, int blocks, int K, int r, const void* __restrict__ x,
                                                                      GroupShrinkParams p) {
  const Places pl{{T_, num_slots, width, slots8, tiles}, tts};
  constexpr int kStageRow = 17;  // 16 chunks of 16 bytes + one of padding: operand reads hit every bank once
  constexpr int AI = RW / 4;     // loads of a round's A rows, four rows each
  __shared__ __attribute__((aligned(16))) i32x4 s_stage[kShrinkWaves * 2 * 16 * kStageRow];
  __shared__ __attribute__((aligned(16))) float s_red[kShrinkWaves * 64 * 4];
  __shared__ int s_rows[(GRID == kBySlot ? 2 : 1) * MLORA_TILE_SMALL], s_wave[2 * kShrinkWaves], s_found[2];
  static_assert(sizeof(s_stage) >= MLORA_MAX_SLOTS * sizeof(int), "the histogram takes the staging area");
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int lr = lane & 15, lg = lane >> 4;
  const int place = blockIdx.z * 8 + blockIdx.x;
  const int first_id = tts[tid < T_ ? tid : T_ - 1];
  const int place_id = GRID == kByToken ? tts[place < T_ ? place : T_ - 1] : 0;
  const int slice = blockIdx.y / blocks, r0 = (blockIdx.y - slice * blocks) * RW;
  const int rounds = K / kRound;
  const int64_t out0 = static_cast<int64_t>(slice) * T_ * r;
  int slot, from = 0, tile = 0;
  if constexpr (GRID == kByToken) {
    if (place >= T_) return;
    slot = known_slot(pl, __builtin_amdgcn_readfirstlane(place_id));
    from = place;
    if (slot == num_slots) {
      if (tid < RW && r0 + tid < r) store_as(p.out, out0 + static_cast<int64_t>(place) * r + r0 + tid, 0.f, p.out_dtype);
      return;
    }
  } else {
    tile = place / slots8;
    slot = place - tile * slots8;
    if (tile >= tiles) {
      find_tile<kShrinkThreads>(pl, first_id, place - tiles * slots8, reinterpret_cast<int*>(s_stage), s_found);
      slot = __builtin_amdgcn_readfirstlane(s_found[0]);
      if (slot < 0) return;
      tile = __builtin_amdgcn_readfirstlane(s_found[1]);
    } else if (slot >= num_slots) {
      if (slot == num_slots && tile == 0) {  // the tokens without a slot
        for (int e = tid; e < T_ * RW; e += kShrinkThreads) {
          const int t = e / RW, rank = r0 + e % RW;
          if (rank < r && known_slot(pl, tts[t]) == num_slots) store_as(p.out, out0 + static_cast<int64_t>(t) * r + rank, 0.f, p.out_dtype);
        }
      }
      return;
    }
  }
  i32x4 ast[AI * CH];
  const T* A = static_cast<const T*>(p.a[slice]) + static_cast<int64_t>(slot) * r * K + wave * (rounds * 128) + lr * 8;
  auto request_a = [&](const int from_round) {
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const int k = (from_round + c < rounds ? from_round + c : rounds - 1) * 128;
#pragma unroll
      for (int i = 0; i < AI; ++i) {
        const int row = r0 + 4 * i + lg;
        ast[AI * c + i] = load128(A + static_cast<int64_t>(row < r ? row : r - 1) * K + k);
      }
    }
  };
  request_a(0);
  __builtin_amdgcn_sched_barrier(0);
  const int* rows;
  const int left = list_tile<kShrinkThreads, GRID>(pl, first_id, slot, from, tile, s_rows, s_wave, rows);
  if (left == 0) {
    // (named as used here too, or the compiler sinks the requests behind the listing of the tokens)
#pragma unroll
    for (int j = 0; j < AI * CH; ++j) asm volatile("" ::"v"(ast[j]));
    return;
  }
  i32x4* stage = s_stage + wave * 2 * 16 * kStageRow;
  const T* xrow[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int at = 4 * i + lg < left ? 4 * i + lg : left - 1;
    xrow[i] = static_cast<const T*>(x) + static_cast<int64_t>(rows[at]) * p.xs + wave * (rounds * 128) + lr * 8;
  }
  f32x4 acc[1] = {f32x4{0.f, 0.f, 0.f, 0.f}};
  for (int now = 0; now < rounds; now += CH) {
    i32x4 xst[4 * CH];
    if (now > 0) request_a(now);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (i == 0 || 4 * i < left) {  // (rows of absent tokens are products nobody stores: any value will do)
#pragma unroll
        for (int c = 0; c < CH; ++c) xst[4 * c + i] = load128(xrow[i] + (now + c < rounds ? now + c : rounds - 1) * 128);
      } else {
#pragma unroll
        for (int c = 0; c < CH; ++c) xst[4 * c + i] = i32x4{0, 0, 0, 0};
      }
    }
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      if (now + c >= rounds) break;
      Pack8 xa[4], aw[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) stage[(4 * i + lg) * kStageRow + lr] = xst[4 * c + i];
#pragma unroll
      for (int i = 0; i < AI; ++i) stage[(16 + 4 * i + lg) * kStageRow + lr] = ast[AI * c + i];
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        xa[i].raw = stage[lr * kStageRow + 4 * i + lg];
        aw[i].raw = stage[(16 + (lr & (RW - 1))) * kStageRow + 4 * i + lg];
      }
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[0] = Mma<T>::run(xa[i], aw[i], acc[0]);
    }
  }
  mfma_settle(acc);  // (the rounds end behind a branch)
  // sum of the wavefronts' shares: a lane holds H[token 4 * lg + i][rank r0 + lr]
  *reinterpret_cast<f32x4*>(&s_red[(wave * 64 + lane) * 4]) = acc[0];
  __syncthreads();
  const int tok = tid / RW, rank = tid % RW;
  if (tok < left && r0 + rank < r) {
    float sum = 0.f;
#pragma unroll
    for (int w = 0; w < kShrinkWaves; ++w) sum += s_red[(w * 64 + (tok >> 2) * 16 + rank) * 4 + (tok & 3)];
    store_as(p.out, out0 + static_cast<int64_t>(rows[tok]) * r + r0 + rank, sum * p.scaling, p.out_dtype);
  }
}

// ---- expand -------------------------------------------------------------------------------------
constexpr int kExpandWaves = 4;
constexpr int kExpandThreads = kExpandWaves * kWave;

struct GroupExpandParams {
  const void* h; void* y;
  int64_t ys;
  int add_inputs, num_slices;
  int first[MLORA_MAX_SLICES];  // first column range of a slice
  const void* b[MLORA_MAX_SLICES];
  int n[MLORA_MAX_SLICES];
  int col[MLORA_MAX_SLICES];
};

// Eight ranks of the intermediate at the weight's precision, as the reference's kernel casts it.
template <typename T, typename H> __device__ __forceinline__ Pack8 load_h(const H* p) {
  Pack8 v;
  if constexpr (std::is_same<H, T>::value) {
    v.raw = load128(p);
  } else {
    float f[8];
    if constexpr (sizeof(H) == 4) {
      const f32x4 lo = *reinterpret_cast<const f32x4*>(p), hi = *reinterpret_cast<const f32x4*>(p + 4);
#pragma unroll
      for (int e = 0; e < 4; ++e) { f[e] = lo[e]; f[4 + e] = hi[e]; }
    } else {
      Pack8 q;
      q.raw = load128(p);
      unpack8<H>(q, f);
    }
    pack8<T>(f, v);
  }
  return v;
}

// y[t, col_i + n] (+)= round_T(h[i, t] . B_i[s]^T); grid (8, column ranges, places / 8).  A wavefront takes SP spans of 64 columns.
template <typename T, typename H, int KSTEPS, int SP, int GRID>
__global__ __launch_bounds__(kExpandThreads) void group_expand_kernel(const int32_t* __restrict__ tts, int T_, int num_slots, int width, int slots8,
                                                                      int tiles, int r, GroupExpandParams p) {
  const Places pl{{T_, num_slots, width, slots8, tiles}, tts};
  __shared__ int s_hist[GRID == kBySlot ? MLORA_MAX_SLOTS : 1], s_rows[(GRID == kBySlot ? 2 : 1) * MLORA_TILE_SMALL], s_wave[2 * kExpandWaves],
      s_found[2];
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int lr = lane & 15, lg = lane >> 4;
  const int place = blockIdx.z * 8 + blockIdx.x;
  const int first_id = tts[tid < T_ ? tid : T_ - 1];
  const int place_id = GRID == kByToken ? tts[place < T_ ? place : T_ - 1] : 0;
  int slice = 0;
  while (slice + 1 < p.num_slices && static_cast<int>(blockIdx.y) >= p.first[slice + 1]) ++slice;
  const int n = p.n[slice], c0 = ((static_cast<int>(blockIdx.y) - p.first[slice]) * kExpandWaves + wave) * (SP * 64);
  int slot, from = 0, tile = 0;
  if constexpr (GRID == kByToken) {
    if (place >= T_) return;
    slot = known_slot(pl, __builtin_amdgcn_readfirstlane(place_id));
    from = place;
  } else {
    tile = place / slots8;
    slot = place - tile * slots8;
    if (tile >= tiles) {
      find_tile<kExpandThreads>(pl, first_id, place - tiles * slots8, s_hist, s_found);
      slot = __builtin_amdgcn_readfirstlane(s_found[0]);
      if (slot < 0) return;
      tile = __builtin_amdgcn_readfirstlane(s_found[1]);
    }
  }
  if (slot >= num_slots) return;
  // (requested whether a span exists or not, clamped into the slice)
  Pack8 bop[SP][4][KSTEPS];
  const T* B = static_cast<const T*>(p.b[slice]) + static_cast<int64_t>(slot) * n * r;
#pragma unroll
  for (int s = 0; s < SP; ++s)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int col = c0 + s * 64 + 4 * lr + j;
#pragma unroll
      for (int ks = 0; ks < KSTEPS; ++ks) {
        const int piece = lg + 4 * ks;
        bop[s][j][ks].raw = load128(B + static_cast<int64_t>(col < n ? col : n - 1) * r + (piece * 8 < r ? piece * 8 : 0));
      }
    }
  __builtin_amdgcn_sched_barrier(0);
  const int* rows;
  const int left = list_tile<kExpandThreads, GRID>(pl, first_id, slot, from, tile, s_rows, s_wave, rows);
  if (left == 0 || c0 >= n) {
    // (named as used here too, or the compiler sinks the requests behind the listing of the tokens)
#pragma unroll
    for (int s = 0; s < SP; ++s)
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int ks = 0; ks < KSTEPS; ++ks) asm volatile("" ::"v"(bop[s][j][ks].raw));
    return;
  }
  const H* hin = static_cast<const H*>(p.h) + static_cast<int64_t>(slice) * T_ * r;
  T* const y = static_cast<T*>(p.y) + p.col[slice];
  // token j of a tile is row 4 * (j % 4) + j / 4 of the product: a lane then holds tokens lg, 4 + lg, 8 + lg, 12 + lg, and a
  // tile of four tokens is one request for y and one store
  Pack8 hop[KSTEPS];
  {
    const int tok = 4 * (lr & 3) + (lr >> 2);
    const H* row = hin + static_cast<int64_t>(rows[tok < left ? tok : left - 1]) * r;
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ++ks) {
      const int piece = lg + 4 * ks;
      hop[ks] = load_h<T, H>(row + (piece * 8 < r ? piece * 8 : 0));
    }
  }
  int row[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) row[i] = rows[4 * i + lg < left ? 4 * i + lg : left - 1];
  uint2 yq[SP][4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (p.add_inputs && 4 * i < left) {
#pragma unroll
      for (int s = 0; s < SP; ++s) {
        const int c = c0 + s * 64 + 4 * lr;
        yq[s][i] = *reinterpret_cast<const uint2*>(y + static_cast<int64_t>(row[i]) * p.ys + (c < n ? c : n - 4));
      }
    } else {
#pragma unroll
      for (int s = 0; s < SP; ++s) yq[s][i] = uint2{0, 0};
    }
  }
#pragma unroll
  for (int s = 0; s < SP; ++s) {
    f32x4 out[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      out[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < KSTEPS; ++ks) {
        Pack8 hv = hop[ks], bv = bop[s][j][ks];
        if ((lg + 4 * ks) * 8 >= r) hv.raw = bv.raw = i32x4{0, 0, 0, 0};  // (pieces beyond the rank)
        out[j] = Mma<T>::run(hv, bv, out[j]);
      }
    }
    const int c = c0 + s * 64 + 4 * lr;
    if (c < n) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (4 * i + lg < left) {
          union { uint2 raw; T e[4]; } v;
          v.raw = yq[s][i];
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const T d = from_f32<T>(out[j][i]);
            v.e[j] = p.add_inputs ? from_f32<T>(to_f32(v.e[j]) + to_f32(d)) : d;
          }
          *reinterpret_cast<uint2*>(y + static_cast<int64_t>(row[i]) * p.ys + c) = v.raw;
        }
      }
    }
  }
}

bool aligned(const void* p, int to) { return reinterpret_cast<uintptr_t>(p) % to == 0; }

// Diagnostic knob, read from the environment once and again after mlora_reload_knobs().
struct GroupKnobs {
  int generation = -1, use;
  void read() {
    generation = knob_generation();
    use = env_int("MLORA_GROUP", 1);  // 0: never, 2: also where one workgroup per token is the faster one
  }
};
const GroupKnobs& group_knobs() {
  static GroupKnobs k;
  if (k.generation != knob_generation()) k.read();
  return k;
}

constexpr int kMostTokens = 4096;  // of a call (every workgroup reads the slot vector)

struct ShrinkLaunch {
  const MloraShrinkArgs* a;
  Places at;
  int over, blocks;
  dim3 grid;
  GroupShrinkParams p;
};
template <typename T, int RW, int CH> void shrink_grid(const ShrinkLaunch& l) {
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, l.grid, dim3(kShrinkThreads), 0, static_cast<hipStream_t>(l.a->stream), l.at.tts, l.at.T, l.at.num_slots, l.at.width,
                       l.at.slots8, l.at.tiles, l.blocks, l.a->k, l.a->r, l.a->x, l.p);
  };
  if (l.over == kBySlot) launch(group_shrink_kernel<T, RW, CH, kBySlot>);
  else launch(group_shrink_kernel<T, RW, CH, kByToken>);
}
template <typename T, int RW> void shrink_rounds(const ShrinkLaunch& l) {
  const int rounds = l.a->k / kRound;
  if (rounds == 1) shrink_grid<T, RW, 1>(l);
  else if (rounds == 2) shrink_grid<T, RW, 2>(l);
  else shrink_grid<T, RW, 4>(l);
}
template <typename T> void shrink_type(const ShrinkLaunch& l, int rw) {
  if (rw == 8) shrink_rounds<T, 8>(l);
  else shrink_rounds<T, 16>(l);
}

struct ExpandLaunch {
  const MloraExpandArgs* a;
  Places at;
  int over, spans;
  dim3 grid;
  GroupExpandParams p;
};
template <typename T, typename H, int KSTEPS, int SP> void expand_grid(const ExpandLaunch& l) {
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, l.grid, dim3(kExpandThreads), 0, static_cast<hipStream_t>(l.a->stream), l.at.tts, l.at.T, l.at.num_slots, l.at.width,
                       l.at.slots8, l.at.tiles, l.a->r, l.p);
  };
  if (l.over == kBySlot) launch(group_expand_kernel<T, H, KSTEPS, SP, kBySlot>);
  else launch(group_expand_kernel<T, H, KSTEPS, SP, kByToken>);
}
template <typename T, typename H> void expand_ranks(const ExpandLaunch& l) {
  if (l.a->r <= 32) l.spans == 1 ? expand_grid<T, H, 1, 1>(l) : expand_grid<T, H, 1, 2>(l);
  else l.spans == 1 ? expand_grid<T, H, 2, 1>(l) : expand_grid<T, H, 2, 2>(l);
}
template <typename T> void expand_type(const ExpandLaunch& l) {
  if (l.a->h_dtype == MLORA_DTYPE_F32) expand_ranks<T, float>(l);
  else if (l.a->h_dtype == MLORA_DTYPE_F16) expand_ranks<T, _Float16>(l);
  else expand_ranks<T, __bf16>(l);
}

}  // namespace

// Where tiles of a slot beat one workgroup per token.  What a token's workgroup costs grows with the A rows it takes in; what a tile's
// costs is finding its tokens (0.5 us), and rounds once places x slices are more workgroups than the chip takes together or, with few
// slot ids, than their XCDs take (a slot's workgroups share one).  Replayed graphs, slots at random, us per call, per token / tiles:
//  - above rank 16, over the tokens: rank 32, K = 1024, one slice 64 tokens 5.5 / 4.9, 128 5.7 / 5.4, 256 6.3 / 6.9; three slices 32 tokens
//    5.6 / 5.1, 64 5.9 / 6.5 (rank 64 10.7 / 9.5);
//  - over the slots: 131 tokens of 128 ids 5.7 / 4.7, three slices 7.5 / 8.9, 259 of 256 11.0 / 13.9, but 512 of 256 16.4 / 15.5, 384 of 192
//    13.4 / 12.6; K = 4096 195 of 192 14.7 / 17.6; 403 of 400, one slice 0.73-0.87 of the per-token rate;
//  - few ids: one 48 tokens 4.52 / 4.51, 64 4.6 / 4.8, three slices 64 4.7 / 10.2 (rank 64, 512 tokens 12 / 39); two 48 tokens of three slices
//    5.6 / 6.3; four, rank 64, 512 tokens of three slices 12.5 / 14.6; eight 7.8 / 6.7;
//  - beyond 512 tokens every workgroup reads the slot vector in several steps (1000 tokens over 4 slots, rank 64, three slices: 19 / 26);
//  - up to rank 16, K = 1024: one slice 512 tokens of 8 ids 4.2 / 4.8, of 16 4.4 / 4.2; three slices 256 of 8 4.55 / 4.9, of 16 4.9 / 4.4, of
//    128 6.2 / 5.9, 192 of 128 5.75 / 5.96, 256 of 256 6.6 / 9.5 (rank 8 as from twice the tokens);
//  - K = 4096: 64 tokens of 64 ids 6.3 / 6.6, 192 of 8 6.5 / 5.75, 256 of 8 6.6 / 9.2, 48 of 2 5.3 / 5.6, 64 of one 4.7 / 6.7; K = 8192: 64 of 64
//    9.1 / 8.8, 128 of 128 12.75 / 11.7.
// The slots of a batch are not known here: with all tokens on one slot of 16 the tiles lose (rank 32, K = 1024, 384 tokens 5.0 / 6.0; at
// random 6.0 / 4.9; rank 16, three slices, 256 tokens 4.2 / 5.7 and 4.9 / 4.4).
static bool shrink_tiles_pay(int T, int L, int S, int r, int k) {
  if (T > 512) return false;
  const int spread = S * (T <= L ? T : L);
  if (r > 16) return T <= L ? spread <= 128 : (spread <= 128 || T >= 2 * L) && (L >= 8 || T * S <= 48 * L);
  if (static_cast<double>(T) * S * r * k < (k >= 4096 ? 1.2e6 : 9.0e6)) return false;
  if (T <= L) return k >= 8192 && spread <= 128;
  return (spread <= 64 || T >= 2 * L) && (L >= 16 || (k >= 4096 && L >= 3 && T <= 24 * L));
}

bool group_shrink_supported(const MloraShrinkArgs* a) {
  if (group_knobs().use == 0 || a->dtype == MLORA_DTYPE_F32 || a->num_slots < 1 || a->num_slots > MLORA_MAX_SLOTS || a->num_tokens > kMostTokens) return false;
  if (a->r < 1 || a->r > 64 || a->k < kRound || a->k % kRound || a->x_stride % 8 || !aligned(a->x, 16)) return false;
  for (int i = 0; i < a->num_slices; ++i)
    if (!aligned(a->a[i], 16)) return false;
  if (group_knobs().use == 2) return true;
  return shrink_tiles_pay(a->num_tokens, a->num_slots, a->num_slices, a->r, a->k);
}

int launch_group_shrink(const MloraShrinkArgs* a) {
  ShrinkLaunch l = {};
  l.a = a;
  l.at.tts = a->token_to_slot; l.at.T = a->num_tokens; l.at.num_slots = a->num_slots;
  l.p.out = a->out; l.p.xs = a->x_stride; l.p.out_dtype = a->out_dtype; l.p.scaling = a->scaling;
  for (int i = 0; i < a->num_slices; ++i) l.p.a[i] = a->a[i];
  // ranks in blocks of eight where blocks of sixteen would leave half of the compute units without a workgroup
  const int rw = a->r <= 8 || static_cast<long long>(groups_about(l.at.T, l.at.num_slots)) * a->num_slices * ((a->r + 15) / 16) < 128 ? 8 : 16;
  l.blocks = (a->r + rw - 1) / rw;
  const int places = lay_out(l.at, &l.over, static_cast<long long>(a->num_slices) * l.blocks, 1);
  l.grid = dim3(8, static_cast<unsigned>(a->num_slices * l.blocks), static_cast<unsigned>((places + 7) / 8));
  if (a->dtype == MLORA_DTYPE_BF16) shrink_type<__bf16>(l, rw);
  else shrink_type<_Float16>(l, rw);
  return check_launch("mlora_shrink");
}

// Measured as above, per token / tiles; columns: of all slices.
//  - rank 8: 8192 columns 256 tokens of 8 ids 6.6 / 5.1, of 128 9.0 / 9.2, 512 of 128 14.6 / 12.8; 1536 columns 512 of 32 4.80 / 4.82; fewer
//    tokens or columns lose 2 to 15 %;
//  - rank 16: 256 columns never (256 tokens of 64 3.2 / 3.4).  Over the tokens: 1024 columns 64 tokens 3.65 / 3.42, 128 4.1 / 4.2, 256 4.7 / 5.3; 8192
//    columns 64 5.9 / 7.5.  One id: 1024 columns 32 tokens 3.4 / 3.3, 64 3.44 / 3.78; 8192 64 4.6 / 7.4; three, 2048 columns 96 0.87 of
//    the per-token rate.  Four: 1024 columns 128 tokens 3.50 / 3.55, 256 3.6 / 3.7; 8192 512 14.0 / 13.1.  1024 of 128 ids at 1024 columns
//    0.90 of the per-token rate, 512 of 256 at 8192 24.4 / 25.6, 1024 of 256 39.4 / 33.6;
//  - above, over the tokens: rank 24 256 of 256 ids 256 columns 3.9 / 3.65, 512 of 512 4.6 / 5.1 (1024 columns 8.1 / 7.8; 1024 tokens 14.5 / 15.6);
//  - one id, rank 32: 1024 columns 64 tokens 4.2 / 3.9, 192 4.7 / 6.5; rank 24 to 48, of the per-token rate, 1536 columns 32 tokens 1.05-1.14, 48
//    0.94-1.01, 3072 columns 48 tokens 0.78-0.82, 4096 columns 16 1.03-1.17, 32 0.86; rank 24 8192 columns 4096 tokens 170 / 510.  Rank 56 1.05 to 2.1
//    from 1536 columns on; rank 64 256 columns 512 tokens 6.3 / 7.6, 1024 18.5 / 10.4, 8192 4096 tokens 990 / 750;
//  - more ids: rank 32 1024 columns 2048 tokens of 2 19.4 / 20.4, 1024 of 2 11.6 / 9.3; rank 24 256 columns 512 of 2 3.85 / 4.3, 4096 of 16
//    11.4 / 14.4, of 64 11.8 / 10.5; 8192 columns 4096 of 4 185 / 164; rank 64, 4096 of 64, 1800 / 119.
// All tokens on one slot of many: rank 24, 1024 columns, 512 tokens of 64 5.2 / 5.9, 8192 columns 21.9 / 13.8.
static bool expand_tiles_pay(int T, int L, int r, long long cols) {
  if (r <= 8) return cols >= 4096 && L >= 8 && L <= 128 && T >= 256 && T >= 4 * L && T <= 1024;
  if (r <= 16) {
    if (cols < 1024) return false;
    if (T <= L) return T * cols <= 65536;
    if (L < 4) return T * cols <= 32768;
    return T <= 1024 && T <= L * (cols >= 4096 ? 128 : 32) && (L <= 64 || (cols > 1024 && T >= 4 * L));
  }
  if (T <= L) return r > 32 || T <= (cols >= 1024 ? 512 : 256);
  if (L == 1) return r > 48 ? T <= 64 || cols >= 1024 : T <= 64 && T * cols <= 65536;
  return T <= 64 * L || r > 56 || (T <= 1024 * L && r * cols >= 32768);
}

bool group_expand_supported(const MloraExpandArgs* a) {
  if (group_knobs().use == 0 || a->dtype == MLORA_DTYPE_F32 || a->num_slots < 1 || a->num_slots > MLORA_MAX_SLOTS || a->num_tokens > kMostTokens) return false;
  if (a->r < 8 || a->r > 64 || a->r % 8 || a->y_stride % 4 || a->offset_start % 4 || !aligned(a->y, 8) || !aligned(a->h, 16)) return false;
  long long cols = 0;
  for (int i = 0; i < a->num_slices; ++i) {
    if (a->n[i] % 4 || !aligned(a->b[i], 16)) return false;
    cols += a->n[i];
  }
  if (cols > 1 << 23) return false;  // (column ranges of the grid)
  if (group_knobs().use == 2) return true;
  return expand_tiles_pay(a->num_tokens, a->num_slots, a->r, cols);
}

int launch_group_expand(const MloraExpandArgs* a) {
  ExpandLaunch l = {};
  l.a = a;
  l.at.tts = a->token_to_slot; l.at.T = a->num_tokens; l.at.num_slots = a->num_slots;
  l.p.h = a->h; l.p.y = a->y; l.p.ys = a->y_stride; l.p.add_inputs = a->add_inputs ? 1 : 0; l.p.num_slices = a->num_slices;
  long long cols = 0;
  for (int i = 0; i < a->num_slices; ++i) cols += a->n[i];
  l.spans = cols * groups_about(l.at.T, l.at.num_slots) >= 131072 ? 2 : 1;
  const int nt = l.spans * 64 * kExpandWaves;
  int col = a->offset_start, total = 0;
  for (int i = 0; i < a->num_slices; ++i) {
    l.p.first[i] = total;
    l.p.b[i] = a->b[i]; l.p.n[i] = a->n[i]; l.p.col[i] = col;
    col += a->n[i];
    total += (a->n[i] + nt - 1) / nt;
  }
  const int places = lay_out(l.at, &l.over, total, 0);
  l.grid = dim3(8, static_cast<unsigned>(total), static_cast<unsigned>((places + 7) / 8));
  if (a->dtype == MLORA_DTYPE_BF16) expand_type<__bf16>(l);
  else expand_type<_Float16>(l);
  return check_launch("mlora_expand");
}

}  // namespace mlora
