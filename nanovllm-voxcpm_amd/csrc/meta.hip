// On-device segment metadata: a stable counting sort of the tokens by slot id, run by one
// workgroup for every 512 tokens, that emits (a) the plan workspace the apply kernels walk and (b) any of the
// three index layouts the reference builds on the host: the engine's (slots ascending, -1
// left out: nanovllm_voxcpm/engine/lora_manager.py:77-91, utils/context.py:77-116), the kernel
// metadata's (-1 bucket first: lora_ops/triton_ops/lora_kernel_metadata.py:46-68) and the graph
// buffers' (fixed ids -1 .. L-1, counts scattered: engine/model_runner.py:727-797).
#include "common.h"

namespace mlora {

namespace {

constexpr int kMetaThreads = 512;
constexpr int kMetaWaves = kMetaThreads / kWave;

struct MetaParams {
  int L, no_lora_bucket;
  int32_t* plan;
  int32_t* sorted_idx;
  int32_t* compact_ids;
  int32_t* compact_counts;
  int32_t* compact_offsets;
  int compact_capacity;
  int32_t* dense_counts;
  int32_t* dense_offsets;
  int32_t* padded_tts;
  int padded_len;
  int32_t* scalars;
};

// Inclusive scan over the wavefront with DPP moves (within rows of sixteen, then row to row): six steps
// of a few cycles where shuffles through the LDS unit take over a hundred each.
template <typename F> __device__ __forceinline__ int wave_incl(int v, F&& op) {
  v = op(v, __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false));  // row_shr:1
  v = op(v, __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false));  // row_shr:2
  v = op(v, __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false));  // row_shr:4
  v = op(v, __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false));  // row_shr:8
  v = op(v, __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false));  // row_bcast:15 into rows 1 and 3
  v = op(v, __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false));  // row_bcast:31 into rows 2 and 3
  return v;
}
__device__ __forceinline__ int wave_incl_scan(int v) { return wave_incl(v, [](int a, int b) { return a + b; }); }
__device__ __forceinline__ int wave_max_of_nonnegative(int v) {
  return __builtin_amdgcn_readlane(wave_incl(v, [](int a, int b) { return a > b ? a : b; }), kWave - 1);
}

__host__ __device__ inline int parts_of(int T) { return T > kMetaThreads ? (T + kMetaThreads - 1) / kMetaThreads : 1; }

// A barrier for what passes through LDS: it does not wait for the global stores on their way, as
// __syncthreads does (a store's acknowledgement is most of a microsecond away).
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// Several batches share a launch: each has a workgroup of its own.
struct MetaTable { MetaParams p[MLORA_META_BATCH]; };

// The batch's slot ids by value: one per token, or runs of tokens (the slot of each and where it ends).  They
// come with the launch, so that no pinned buffer has to be filled and no copy has to run before it.
struct RunTable {
  int runs, singles;  // singles: every run is one token
  union {
    int16_t slot_of_token[MLORA_META_SINGLES];
    struct { int32_t end[MLORA_META_RUNS]; int16_t slot[MLORA_META_RUNS]; } run;
  };
};
static_assert(sizeof(RunTable) + sizeof(MetaTable) <= 4096, "both are kernel arguments");

// Where the workgroup keeps what it knows of every bucket (bucket b holds slot b - 1; bucket 0 is "no LoRA").
struct Buckets {
  int NB;
  int* rest;      // [NB] tokens of the bucket outside `before`
  int* before;    // [NB] tokens of the bucket ahead of this workgroup's own
  int* off;       // [NB + 1] first position of bucket b among LoRA tokens
  int* cidx;      // [NB + 1] compact index of bucket b
  int* ts_short;  // [NB + 1] first small tile of a short segment
  int* ts_long;   // [NB + 1] first small tile of a long segment
  int* ts_big;    // [NB + 1] first big tile of a long segment
  int* ts_over;   // [NB + 1] first of the small tiles behind a slot's first one
  uint8_t* step;  // [NB][waves] tokens of the bucket in the 64 tokens of each of the workgroup's wavefronts
};
constexpr int kBucketBytes = 2 * 4 + 6 * 4 + kMetaWaves;
constexpr int kClearedWords = 4;  // of a bucket: step, rest and before, which lie together
static_assert(kMetaWaves == 8, "the counts of a bucket are one 64-bit word");

__device__ __forceinline__ Buckets lay_out(int L, int* lds) {
  Buckets k;
  k.NB = L + 1;
  k.step = reinterpret_cast<uint8_t*>(lds);  // (8 bytes a bucket, 8-byte aligned)
  k.rest = lds + 2 * k.NB;
  k.before = k.rest + k.NB;
  k.off = k.before + k.NB;
  k.cidx = k.off + k.NB + 1;
  k.ts_short = k.cidx + k.NB + 1;
  k.ts_long = k.ts_short + k.NB + 1;
  k.ts_big = k.ts_long + k.NB + 1;
  k.ts_over = k.ts_big + k.NB + 1;
  return k;
}

__device__ __forceinline__ int sum_of_bytes(uint64_t v) {
  return static_cast<int>(__builtin_amdgcn_sad_u8(static_cast<uint32_t>(v), 0u, __builtin_amdgcn_sad_u8(static_cast<uint32_t>(v >> 32), 0u, 0u)));
}

// Sums over all buckets, the same in every thread.
struct Sums { int lora, none, compact, small_short, small_long, big, over, longest, nlong; };

struct Place { int slot, key, r; Sums n; int bad; };  // of this thread's token; sums and flag are the batch's

// The exclusive scans over the buckets, by every wavefront for itself: they store the same values to the same
// places, and each reads only what it has stored, so nobody waits for anybody.
template <typename F> __device__ __forceinline__ Sums scan_buckets(const Buckets& k, bool no_lora_bucket, F&& tokens_of) {
  const int lane = threadIdx.x & (kWave - 1), NB = k.NB;
  const int b0 = no_lora_bucket ? 0 : 1;  // first bucket of the compact arrays
  Sums r = {};
  for (int base = 0; base < NB; base += kWave) {
    const int b = base + lane;
    const int c_all = b < NB ? tokens_of(b) : 0;
    const int c = b >= 1 ? c_all : 0;  // LoRA tokens only
    const bool is_short = c < MLORA_SEGMENT_THRESHOLD;
    const int nsmall = (c + MLORA_TILE_SMALL - 1) / MLORA_TILE_SMALL;
    const int v1 = (b >= b0 && c_all > 0) ? 1 : 0, v2 = is_short ? nsmall : 0, v3 = is_short ? 0 : nsmall;
    const int v4 = is_short ? 0 : (c + MLORA_TILE_BIG - 1) / MLORA_TILE_BIG, v5 = nsmall > 1 ? nsmall - 1 : 0;
    const int i0 = wave_incl_scan(c), i1 = wave_incl_scan(v1), i2 = wave_incl_scan(v2);
    const int i3 = wave_incl_scan(v3), i4 = wave_incl_scan(v4), i5 = wave_incl_scan(v5);
    if (b < NB) {
      k.off[b] = r.lora + i0 - c;
      k.cidx[b] = r.compact + i1 - v1;
      k.ts_short[b] = r.small_short + i2 - v2;
      k.ts_long[b] = r.small_long + i3 - v3;
      k.ts_big[b] = r.big + i4 - v4;
      k.ts_over[b] = r.over + i5 - v5;
    }
    if (base == 0) r.none = __builtin_amdgcn_readlane(c_all, 0);
    r.lora += __builtin_amdgcn_readlane(i0, kWave - 1);
    r.compact += __builtin_amdgcn_readlane(i1, kWave - 1);
    r.small_short += __builtin_amdgcn_readlane(i2, kWave - 1);
    r.small_long += __builtin_amdgcn_readlane(i3, kWave - 1);
    r.big += __builtin_amdgcn_readlane(i4, kWave - 1);
    r.over += __builtin_amdgcn_readlane(i5, kWave - 1);
    r.nlong += __popcll(__ballot(b < NB && !is_short));
    const int m = wave_max_of_nonnegative(c);
    r.longest = m > r.longest ? m : r.longest;
  }
  if (lane == 0) k.off[NB] = r.lora;
  __builtin_amdgcn_wave_barrier();
  return r;
}

// Everything that is stored, by the workgroups of a batch together: what belongs to token t (when below T),
// and of what belongs to no token thread `gid` of `threads` (at least four wavefronts) takes its share.  No word is stored to twice,
// so nothing here waits for a store.
__device__ __forceinline__ void put_out(const MetaParams& p, const Buckets& k, int T, const Place& me, int gid, int threads, int t) {
  const int L = p.L, NB = k.NB, key = me.key, r = me.r;
  const Sums& n = me.n;
  // With the "no LoRA" bucket requested and no LoRA token at all, the reference's builder returns
  // early and leaves its buffers in the reset state (ids -1, counts 0, offsets 0, sort untouched).
  const bool reset_only = p.no_lora_bucket && n.lora == 0;
  const int n_neg = (p.no_lora_bucket && !reset_only) ? n.none : 0;  // tokens sorted ahead of every slot
  const int n_compact = reset_only ? 0 : n.compact;
  const PlanLayout lay = plan_layout(T, L);
  constexpr int kRecord = MLORA_SMALL_TILE_WORDS / 4;                                  // a small-tile record in 128-bit words
  constexpr int kRecordTail = (MLORA_SMALL_TILE_ROWS + MLORA_TILE_SMALL) / 4;          // those of its header and rows
  const int check = static_cast<int>(MLORA_PLAN_CHECK(T, L));
  // place of big tile q (in slot order) in the list: runs of `run` consecutive tiles go to the blocks (XCDs) in turn
  const int run = big_tile_run(n.big, n.nlong);

  // The token.  The first token of a tile stores the tile's header; a tile of n < 16 tokens lists them
  // cyclically in its sixteen entries, so that a kernel which fetches all sixteen rows touches no memory
  // beyond the rows of the tile itself.
  if (t < T) {
    if (key >= 1) {
      if (p.sorted_idx) p.sorted_idx[n_neg + k.off[key] + r] = t;
      if (p.plan) {
        const int first = k.off[key], c = k.off[key + 1] - first;
        p.plan[lay.sorted_off + first + r] = t;
        const bool is_short = c < MLORA_SEGMENT_THRESHOLD;
        const int tile = r / MLORA_TILE_SMALL, at = r % MLORA_TILE_SMALL, left = c - tile * MLORA_TILE_SMALL;
        const int rows = left < MLORA_TILE_SMALL ? left : MLORA_TILE_SMALL;
        // its record in the list of tiles and the same once more in the list by slot
        int32_t* rec = p.plan + lay.small_off + ((is_short ? k.ts_short[key] : n.small_short + k.ts_long[key]) + tile) * MLORA_SMALL_TILE_WORDS;
        int32_t* rec2 = p.plan + lay.slotrec_off + (tile == 0 ? key - 1 : lay.cap_slotrec + k.ts_over[key] + tile - 1) * MLORA_SMALL_TILE_WORDS;
        i32x4 *w = reinterpret_cast<i32x4*>(rec), *w2 = reinterpret_cast<i32x4*>(rec2);
        if (rows == 1) {
#pragma unroll
          for (int i = MLORA_SMALL_TILE_ROWS / 4; i < kRecordTail; ++i) w[i] = w2[i] = i32x4{t, t, t, t};
        } else {
          for (int pos = at; pos < MLORA_TILE_SMALL; pos += rows) {
            rec[MLORA_SMALL_TILE_ROWS + pos] = t;
            rec2[MLORA_SMALL_TILE_ROWS + pos] = t;
          }
        }
        if (at == 0) {
          w[0] = i32x4{key - 1, rows, first + r, 0};
          w2[0] = i32x4{key - 1, rows, first + r, check};
#pragma unroll
          for (int i = kRecordTail; i < kRecord; ++i) w[i] = w2[i] = i32x4{0, 0, 0, 0};
        }
        // its entry in the row list of the segment's 64-token tile, 0 (a valid row) in those past the tile's
        // count, which only the last tile of a segment has: its tokens share them out
        if (!is_short) {
          const int big = r / MLORA_TILE_BIG, bat = r % MLORA_TILE_BIG, bleft = c - big * MLORA_TILE_BIG;
          const int brows = bleft < MLORA_TILE_BIG ? bleft : MLORA_TILE_BIG;
          const int place = big_tile_place(k.ts_big[key] + big, run, lay.cap_big);
          int32_t* list = p.plan + lay.bigrows_off + place * MLORA_TILE_BIG;
          list[bat] = t;
          for (int pos = bat + brows; pos < MLORA_TILE_BIG; pos += brows) list[pos] = 0;
          if (bat == 0) reinterpret_cast<i32x4*>(p.plan + lay.big_off)[place] = i32x4{key - 1, first + r, brows, 0};
        }
      }
    } else if (p.sorted_idx && p.no_lora_bucket && !reset_only) {
      p.sorted_idx[r] = t;
    }
  }
  if (p.padded_tts) {
    for (int i = gid; i < p.padded_len; i += threads) p.padded_tts[i] = i < T ? me.slot : -1;  // (below T: i is t)
  }

  // The rest by other wavefronts than the tokens' while there are any: the header, what is stored per bucket and what no token
  // stores by one of the last four each (up to 64 tokens of 32 slots 3.3 us per launch, 4.3 with all of it behind
  // wavefront 0's tokens; in the last workgroup of several, 0.1 to 0.6 us more).
  auto share_of = [&](int waves) {
    if (T > kMetaThreads - 4 * kWave) return gid;
    const int i = threads - 1 - waves * kWave - gid;
    return i < 0 ? i + threads : i;
  };
  if (share_of(1) == 0) {
    if (p.plan) {
      int32_t* h = p.plan;
      h[MLORA_PLAN_MAGIC] = MLORA_PLAN_MAGIC_VALUE;
      h[MLORA_PLAN_NUM_TOKENS] = T;
      h[MLORA_PLAN_MAX_SLOTS] = L;
      h[MLORA_PLAN_NUM_LORA_TOKENS] = n.lora;
      h[MLORA_PLAN_NUM_ACTIVE] = n.compact - ((p.no_lora_bucket && n.none > 0) ? 1 : 0);
      h[MLORA_PLAN_NO_LORA] = n.lora == 0;
      h[MLORA_PLAN_BAD_SLOT] = me.bad;
      h[MLORA_PLAN_TILES_SHORT] = n.small_short;
      h[MLORA_PLAN_TILES_LONG_SMALL] = n.small_long;
      h[MLORA_PLAN_TILES_LONG_BIG] = n.big;
      h[MLORA_PLAN_MAX_SEGMENT] = n.longest;
      h[MLORA_PLAN_TILES_OVER] = n.over;
      for (int i = MLORA_PLAN_TILES_OVER + 1; i < MLORA_PLAN_HEADER_WORDS; ++i) h[i] = 0;  // (MLORA_PLAN_REJECTED among them)
    }
    if (p.scalars) {
      p.scalars[0] = n_compact;
      p.scalars[1] = n.lora + n_neg;
      p.scalars[2] = n.lora == 0;
      p.scalars[3] = me.bad;
    }
    if (p.dense_offsets) p.dense_offsets[0] = 0;
    if (p.compact_offsets) p.compact_offsets[n_compact] = n.lora + n_neg;
    if (p.plan) p.plan[lay.offsets_off] = 0;
  }

  // Per-bucket outputs.
  for (int b = share_of(2); b < NB; b += threads) {
    const int c = b >= 1 ? k.off[b + 1] - k.off[b] : 0;
    if (p.dense_counts) p.dense_counts[b] = c;
    if (p.dense_offsets) p.dense_offsets[b + 1] = k.off[b + 1];
    if (p.plan) {
      p.plan[lay.counts_off + b] = c;
      p.plan[lay.offsets_off + b + 1] = k.off[b + 1];
    }
    const int c_all = b >= 1 ? c : n.none;
    if (!reset_only && (b >= 1 || p.no_lora_bucket) && c_all > 0) {
      const int i = k.cidx[b];
      if (p.compact_ids) p.compact_ids[i] = b - 1;
      if (p.compact_counts) p.compact_counts[i] = c_all;
      if (p.compact_offsets) p.compact_offsets[i] = b == 0 ? 0 : n_neg + k.off[b];
    }
  }
  for (int i = n_compact + share_of(3); i < p.compact_capacity; i += threads) {
    if (p.compact_ids) p.compact_ids[i] = -1;
    if (p.compact_counts) p.compact_counts[i] = 0;
    if (p.compact_offsets) p.compact_offsets[i + 1] = 0;
  }

  // What no token stores: the places of the list of big tiles that hold none, and in the list by slot the records
  // of slots without tokens (and of the ids that round it up to a multiple of eight) and those behind the last
  // further tile.
  if (p.plan) {
    i32x4* big = reinterpret_cast<i32x4*>(p.plan + lay.big_off);
    const int block = lay.cap_big >> 3;
    for (int q = share_of(3); q < lay.cap_big; q += threads) {
      if (n.big == 0) {
        big[q] = i32x4{-1, 0, 0, 0};
        continue;
      }
      const int x = q / block, w = q - x * block, i = w / run;  // (big_tile_place the other way round)
      if ((i * 8 + x) * run + (w - i * run) >= n.big) big[q] = i32x4{-1, 0, 0, 0};
    }
    i32x4* byslot = reinterpret_cast<i32x4*>(p.plan + lay.slotrec_off);
    for (int q = share_of(0); q < lay.cap_slotrec + lay.cap_over; q += threads) {
      i32x4 head = i32x4{-1, 0, 0, check};
      if (q < L) {
        if (k.off[q + 2] != k.off[q + 1]) continue;
        head = i32x4{q, 0, k.off[q + 1], check};
      } else if (q >= lay.cap_slotrec && q - lay.cap_slotrec < n.over) {
        continue;
      }
      byslot[q * kRecord] = head;
#pragma unroll
      for (int w = 1; w < kRecord; ++w) byslot[q * kRecord + w] = i32x4{0, 0, 0, 0};
    }
  }
}

// What bounds it: the latency of one workgroup's chain - slot ids from memory, counts, scans, stores - and
// the 1.6 us of being a launch at all.  A decode step runs it for the batch's context, for the graph
// buffers of every domain and for the plan, a prefill pass for its context.  So a thread has one token and
// a batch as many workgroups as it has 512 tokens: each counts all tokens into two bins a slot (those ahead
// of its own, the rest) instead of waiting for another workgroup to tell it, which at 8192 tokens is sixteen
// ids and LDS atomics a thread.  A token's place among the equal ids of its 64 is found with ballots, that
// among the wavefronts with one 64-bit word of byte counts.  Two barriers, none of which waits for memory.
// Measured in a replayed graph against one workgroup that walked the batch twice (us per launch, plan of random
// ids / of sorted ids / three domains): 64 tokens and 32 slots 5.8 / 5.9 / 4.1 before, 3.3 / 3.4 / 3.2 now;
// 512 and 64 6.0 / 5.9 / 4.5, 4.8 / 4.6 / 3.6; 3001 and 16 11.3 / 13.1 / 7.8, 5.5 / 5.3 / 4.3; 8192 and 128
// 31.0 / 32.5 / 18.2, 10.1 / 12.7 / 6.7.  A pass of 48 calls on one token takes 181.2 us instead of 185.3, one
// of 96 on 9392 tokens 3287 instead of 3323.
// `s`: slot id of token t, -1 from T on (requested by the caller ahead of everything else)
template <typename F>
__device__ __forceinline__ Place place_by_counting(const Buckets& k, int T, int L, bool no_lora_bucket, int part, int s, F&& slot_of) {
  __shared__ int s_bad[kMetaWaves];
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
  const int parts = parts_of(T), first = part * kMetaThreads, t = first + tid;
  auto key_of = [&](int v) { return v >= 0 && v < L ? v + 1 : 0; };
  const int key = key_of(s);
  int beyond = s >= L;
  if (parts > 1) {
    constexpr int kAhead = 8;
    for (int i = tid; i < T; i += kAhead * kMetaThreads) {
      int q[kAhead];
#pragma unroll
      for (int j = 0; j < kAhead; ++j) q[j] = slot_of(i + j * kMetaThreads < T ? i + j * kMetaThreads : T - 1);
#pragma unroll
      for (int j = 0; j < kAhead; ++j) {
        // (a wavefront's 64 tokens lie on one side; where they are all of one slot one lane counts them, as
        // LDS takes atomics to one address in turn)
        const int at = i + j * kMetaThreads, kj = key_of(q[j]);
        beyond |= q[j] >= L;
        int count = at < T;
        const int have = __popcll(__ballot(count));
        if (__ballot(kj != __builtin_amdgcn_readfirstlane(kj)) == 0) count = lane == 0 ? have : 0;
        if (count) atomicAdd((at < first ? k.before : k.rest) + kj, count);
      }
    }
  }
  // Rank of this token among the equal keys of its wavefront, and the size of that group: the set of
  // lanes holding the same key is narrowed down one key bit at a time with ballots (a fixed handful of
  // steps, however many distinct keys there are).
  uint64_t peers = __ballot(t < T);
  const int key_bits = 32 - __builtin_clz(k.NB);  // keys are 0 .. NB - 1
  for (int bit = 0; bit < key_bits; ++bit) {
    const uint64_t set = __ballot((key >> bit) & 1);
    peers &= ((key >> bit) & 1) ? set : ~set;
  }
  const int ahead = __popcll(peers & ((1ull << lane) - 1));
  if (t < T && ahead == 0) k.step[key * kMetaWaves + wave] = static_cast<uint8_t>(__popcll(peers));
  const bool any_beyond = __ballot(beyond) != 0;
  if (lane == 0) s_bad[wave] = any_beyond;
  lds_barrier();

  Place me;
  const uint64_t* step = reinterpret_cast<const uint64_t*>(k.step);
  me.n = scan_buckets(k, no_lora_bucket, [&](int b) { return parts > 1 ? k.before[b] + k.rest[b] : sum_of_bytes(step[b]); });
  me.slot = s;
  me.key = key;
  me.r = k.before[key] + sum_of_bytes(step[key] & ((1ull << (8 * wave)) - 1)) + ahead;
  me.bad = 0;
#pragma unroll
  for (int w = 0; w < kMetaWaves; ++w) me.bad |= s_bad[w];
  return me;
}

// (slot vectors and sizes of the batches are leading arguments, which arrive in scalar registers: the ids are
// requested with the rest of the arguments and not behind them)
static_assert(MLORA_META_BATCH == 4, "leading arguments");
__global__ __launch_bounds__(kMetaThreads) void meta_kernel(const int32_t* tts0, const int32_t* tts1, const int32_t* tts2, const int32_t* tts3,
                                                            int T0, int T1, int T2, int T3, MetaTable table) {
  extern __shared__ __attribute__((aligned(16))) int lds[];
  const int y = blockIdx.y, part = blockIdx.x, t = part * kMetaThreads + threadIdx.x;
  const int T = y == 0 ? T0 : y == 1 ? T1 : y == 2 ? T2 : T3;
  const int32_t* tts = y == 0 ? tts0 : y == 1 ? tts1 : y == 2 ? tts2 : tts3;
  const int s = t < T ? tts[t] : -1;
  const MetaParams p = table.p[y];
  if (part >= parts_of(T)) return;
  const Buckets k = lay_out(p.L, lds);
  for (int i = threadIdx.x; i < kClearedWords * k.NB; i += kMetaThreads) lds[i] = 0;
  lds_barrier();
  const Place me = place_by_counting(k, T, p.L, p.no_lora_bucket, part, s, [&](int i) { return tts[i]; });
  put_out(p, k, T, me, t, parts_of(T) * kMetaThreads, t);
}

// The slot ids come as arguments: one per token, counted as above, or runs of tokens.  A token's place follows
// from its run, so a workgroup counts the runs and not the tokens.
__global__ __launch_bounds__(kMetaThreads) void meta_runs_kernel(int runs, int singles, int T, MetaTable table, RunTable given) {
  extern __shared__ __attribute__((aligned(16))) int lds[];
  __shared__ int s_end[MLORA_META_RUNS], s_slot[MLORA_META_RUNS], s_key[MLORA_META_RUNS], s_rank[MLORA_META_RUNS];
  __shared__ int s_over[kMetaWaves];
  static_assert(MLORA_META_RUNS <= kMetaThreads, "a thread per run");
  const int tid = threadIdx.x, part = blockIdx.x, t = part * kMetaThreads + tid;  // (all batches of the launch have T tokens)
  int s = -1, begin = 0, end = 0;
  const bool has = !singles && tid < runs;
  if (singles) {
    if (t < T) s = given.slot_of_token[t];
  } else if (has) {
    begin = tid > 0 ? given.run.end[tid - 1] : 0;
    end = given.run.end[tid];
    s = given.run.slot[tid];
  }
  const MetaParams p = table.p[blockIdx.y];
  const int L = p.L;
  const Buckets k = lay_out(L, lds);
  for (int i = tid; i < kClearedWords * k.NB; i += kMetaThreads) lds[i] = 0;
  Place me;
  if (singles) {
    lds_barrier();
    me = place_by_counting(k, T, L, p.no_lora_bucket, part, s, [&](int i) { return static_cast<int>(given.slot_of_token[i]); });
  } else {
    const int key = s >= 0 && s < L ? s + 1 : 0;
    if (has) {
      s_end[tid] = end;
      s_slot[tid] = s;
      s_key[tid] = key;
    }
    const bool any_beyond = __ballot(end > begin && s >= L) != 0;
    if ((tid & (kWave - 1)) == 0) s_over[tid / kWave] = any_beyond;
    lds_barrier();
    if (has) {
      atomicAdd(k.rest + key, end - begin);
      int rank = 0, from = 0;  // tokens of the same bucket in earlier runs
#pragma unroll 4
      for (int j = 0; j < tid; ++j) {
        const int to = s_end[j];
        rank += s_key[j] == key ? to - from : 0;
        from = to;
      }
      s_rank[tid] = rank - begin;
    }
    lds_barrier();
    me.n = scan_buckets(k, p.no_lora_bucket, [&](int b) { return k.rest[b]; });
    int lo = 0, hi = t < T ? runs - 1 : 0;  // the first run that ends behind t
    while (lo < hi) {
      const int mid = (lo + hi) >> 1;
      if (s_end[mid] > t) hi = mid; else lo = mid + 1;
    }
    me.slot = s_slot[lo];
    me.key = s_key[lo];
    me.r = s_rank[lo] + t;
    me.bad = 0;
#pragma unroll
    for (int w = 0; w < kMetaWaves; ++w) me.bad |= s_over[w];
  }
  put_out(p, k, T, me, t, parts_of(T) * kMetaThreads, t);
}

}  // namespace

}  // namespace mlora

using namespace mlora;

extern "C" size_t mlora_plan_workspace_bytes(int32_t num_tokens, int32_t max_slots) {
  if (num_tokens < 0 || max_slots < 0) return 0;
  return static_cast<size_t>(plan_layout(num_tokens, max_slots).total_words) * sizeof(int32_t);
}

namespace {

int check_meta(const MloraMetaArgs* a, bool by_value) {
  if (a->num_tokens < 0 || a->max_slots < 0 || a->compact_capacity < 0 || a->padded_len < 0) {
    set_error("mlora_meta_build: negative size"); return MLORA_E_INVALID;
  }
  if (a->max_slots > MLORA_MAX_SLOTS) {
    set_error("mlora_meta_build: max_slots=%d exceeds %d", a->max_slots, MLORA_MAX_SLOTS); return MLORA_E_TOO_LARGE;
  }
  if (a->num_tokens > 0 && !a->token_to_slot && !by_value) { set_error("mlora_meta_build: NULL token_to_slot"); return MLORA_E_INVALID; }
  if (reinterpret_cast<uintptr_t>(a->plan) & 15) { set_error("mlora_meta_build: plan must be 16-byte aligned"); return MLORA_E_INVALID; }
  if (a->padded_token_to_slot && a->padded_len < a->num_tokens) {
    set_error("mlora_meta_build: padded_len=%d is shorter than num_tokens=%d", a->padded_len, a->num_tokens);
    return MLORA_E_INVALID;
  }
  if (a->compact_ids || a->compact_counts || a->compact_offsets) {
    const int t = a->num_tokens, l = a->max_slots + (a->no_lora_bucket ? 1 : 0);
    const int need = t < l ? t : l;
    if (a->compact_capacity < need) {
      set_error("mlora_meta_build: compact_capacity=%d cannot hold %d buckets", a->compact_capacity, need);
      return MLORA_E_INVALID;
    }
  }
  return 0;
}

}  // namespace

namespace {

int build_many(const MloraMetaArgs* list, int32_t count, const RunTable* given) {
  if (count < 0 || (count > 0 && !list)) { set_error("mlora_meta_build: NULL args"); return MLORA_E_INVALID; }
  for (int i = 0; i < count; ++i) {
    if (int rc = check_meta(list + i, given != nullptr)) return rc;
  }
  for (int first = 0; first < count; first += MLORA_META_BATCH) {
    const int n = count - first < MLORA_META_BATCH ? count - first : MLORA_META_BATCH;
    MetaTable table;
    const int32_t* tts[MLORA_META_BATCH] = {};
    int T[MLORA_META_BATCH] = {}, parts = 1;
    size_t lds = 0;
    for (int i = 0; i < n; ++i) {
      const MloraMetaArgs* a = list + first + i;
      MetaParams& p = table.p[i];
      tts[i] = a->token_to_slot; T[i] = a->num_tokens; p.L = a->max_slots; p.no_lora_bucket = a->no_lora_bucket ? 1 : 0;
      p.plan = a->plan; p.sorted_idx = a->sorted_idx;
      p.compact_ids = a->compact_ids; p.compact_counts = a->compact_counts; p.compact_offsets = a->compact_offsets;
      p.compact_capacity = a->compact_ids || a->compact_counts || a->compact_offsets ? a->compact_capacity : 0;
      p.dense_counts = a->dense_counts; p.dense_offsets = a->dense_offsets;
      p.padded_tts = a->padded_token_to_slot; p.padded_len = a->padded_len;
      p.scalars = a->scalars;
      const size_t need = static_cast<size_t>(kBucketBytes) * (p.L + 2);
      lds = need > lds ? need : lds;
      parts = parts_of(T[i]) > parts ? parts_of(T[i]) : parts;
    }
    for (int i = n; i < MLORA_META_BATCH; ++i) table.p[i] = table.p[0];  // (not in the grid)
    hipStream_t st = static_cast<hipStream_t>(list[0].stream);
    if (given) hipLaunchKernelGGL(meta_runs_kernel, dim3(parts, n), dim3(kMetaThreads), lds, st, given->runs, given->singles, T[0], table, *given);
    else hipLaunchKernelGGL(meta_kernel, dim3(parts, n), dim3(kMetaThreads), lds, st, tts[0], tts[1], tts[2], tts[3], T[0], T[1], T[2], T[3], table);
    if (int rc = check_launch("mlora_meta_build")) return rc;
  }
  return 0;
}

}  // namespace

extern "C" int mlora_meta_build_many(const MloraMetaArgs* list, int32_t count) { return build_many(list, count, nullptr); }

extern "C" int mlora_meta_build_runs(const MloraMetaArgs* list, int32_t count, const int32_t* run_slots, const int32_t* run_counts, int32_t runs) {
  if (count < 0 || runs < 0 || (count > 0 && !list) || (runs > 0 && (!run_slots || !run_counts))) {
    set_error("mlora_meta_build_runs: NULL args"); return MLORA_E_INVALID;
  }
  RunTable t;
  t.runs = runs;
  t.singles = 1;
  int64_t total = 0;
  for (int i = 0; i < runs; ++i) {
    if (run_counts[i] < 0) { set_error("mlora_meta_build_runs: run %d has a negative count", i); return MLORA_E_INVALID; }
    t.singles &= run_counts[i] == 1;
    total += run_counts[i];
  }
  for (int i = 0; i < count; ++i) {
    if (list[i].num_tokens != total) {
      set_error("mlora_meta_build_runs: the runs hold %lld tokens, batch %d has %d", static_cast<long long>(total), i, list[i].num_tokens);
      return MLORA_E_INVALID;
    }
  }
  if (runs > (t.singles ? MLORA_META_SINGLES : MLORA_META_RUNS)) { set_error("mlora_meta_build_runs: %d runs", runs); return MLORA_E_TOO_LARGE; }
  int end = 0;
  for (int i = 0; i < runs; ++i) {
    const int slot = run_slots[i] < -1 ? -1 : run_slots[i] > 0x7fff ? 0x7fff : run_slots[i];  // (no slot; beyond every slot)
    end += run_counts[i];
    if (t.singles) {
      t.slot_of_token[i] = static_cast<int16_t>(slot);
    } else {
      t.run.end[i] = end;
      t.run.slot[i] = static_cast<int16_t>(slot);
    }
  }
  return build_many(list, count, &t);
}

extern "C" int mlora_meta_build(const MloraMetaArgs* a) {
  if (!a) { set_error("mlora_meta_build: NULL args"); return MLORA_E_INVALID; }
  return mlora_meta_build_many(a, 1);
}
