// An index in any order -> the entries in order of their rows: perm (entry numbers) and row pointers, the input of
// the segmented reductions (csr_reduce.h with rows through perm). Two levels: entries are binned by bucket of R
// consecutive rows, then every bucket is sorted by row in LDS.
//   count : at most 256 workgroups with equal shares of the index, each a histogram over the buckets in LDS that it adds
//           to the bucket totals; also: is the index in order and inside [0, N)? The workgroup that arrives last turns
//           the totals into bucket starts (a launch of its own for that took 10-15 us of a single CU's latencies).
//   place : a workgroup per tile: the tile sorted by bucket in LDS, one atomic per bucket that occurs reserves the
//           tile's run, (row in bucket, entry) words leave in runs. An index found in order gets its row pointers and
//           the identity from this launch instead, and the passes behind it return at once. Words of 32 bits where both
//           fit (10 M entries onto 100 k rows: 24 + 6 bits), else of 64: place and sort move 8 or 12 bytes an entry less.
//   sort  : a workgroup per bucket of up to 8192 or 16384 entries: counting sort by row in LDS, row pointers and perm out. A
//           bucket with more entries (hubs, few rows) is taken in chunks: each goes back in order of its rows, the row
//           counts meet in memory, the chunk that arrives last turns them into row pointers,
//   place chunks : ... and the chunks' entries then go from there to their places, each behind the row's entries of the
//           chunks that were counted before.
// Entries of a row come in no particular order (a reader that needs the first of equal values compares positions).
// Entries outside [0, N) are left out.
// What it costs: 16 bytes of index, 4 or 8 written and read per entry for the words, 4 for perm; what bounds the passes is the
// chain of each workgroup (load, rank, reserve, store), so every lane has all its loads on the way before it needs one. us for
// clear / count / place / sort / place chunks: 2.3 M entries onto 268 k rows 5 / 16 / 15 / 9 / 5, 10 M even onto 100 k rows
// 5 / 26 / 50 / 26 / 5, 10 M under a Zipf(1.2) index onto 100 k rows 5 / 26 / 46 / 36 / 18 (two thirds of them in one bucket;
// with loads one after the other, words of 64 bits and the chunks ranked a second time 5 / 53 / 59 / 44 / 47, the scatter sum
// of 32 floats 432 us against 358 now and 367 with the tables below). In front of a segmented reduction this replaced tables of
// output rows in LDS per bucket (one LDS atomic per element, bank conflicts, slabs or atomics to put chunks together):
// 2.3 M x 128 bf16, sum 660 -> 205 us; 10 M x 64 floats onto 1 M rows, sum / max 965 / 946 -> 719 / 843 us.
#pragma once

#include "device_utils.h"

namespace ts {

constexpr int kRsBlock = 1024;        // count, place
constexpr int kRsPer = 8;             // entries per lane of place
constexpr int kRsTile = kRsPer * kRsBlock;
// entries that one sorting workgroup holds in LDS (in registers before: 16 per lane): 512 lanes below kRsLarge entries
// (more, shorter workgroups: 2.3 M entries 10.7 against 16.8 us), 1024 above, where fewer buckets save more in count
// and place (10 M entries onto 1 M rows: 138 against 147 us for the three passes)
constexpr int kRsSortPer = 16;
constexpr int64_t kRsLarge = (int64_t)1 << 22;
constexpr int kRsMaxBuckets = 4096;   // histogram of count and place
constexpr int kRsMaxShift = 13;       // rows per bucket (log2): histogram of the sorting workgroup
constexpr int kRsCountPer = 8;
constexpr int kRsCountGroups = 256;   // (512: twice the additions to the totals)

struct RowSortArgs {
  const int64_t *index;
  int64_t sb, se;        // element strides of the index over batches and entries
  int64_t B, E, N;
  int64_t n, rows;       // B * E entries, B * N rows
  int identity;          // an index in order: write the identity to perm (a reader that looks at state[0] does without)
  int flat;              // one batch, unit stride: entry e is index[e] (no 64-bit multiplications per entry)
  int rshift, nb;        // rows per bucket (log2), buckets
  int cap;               // entries that one sorting workgroup takes
  int max_big;           // buckets above that: at most this many ...
  int max_chunks;        // ... in at most this many chunks
  uint32_t *totals;      // [nb] entries per bucket, cleared by the call
  uint32_t *sync;        // [0] ticket of the count pass, [1 ...] of every large bucket: cleared with totals
  int32_t *state;        // [0] 0: the index is in order, 1: it is not; [1] chunks of large buckets; [2] large buckets
  uint32_t *starts;      // [nb + 1]
  uint32_t *cursor;      // [nb]
  int32_t *chunk_info;   // [3][max_chunks]: bucket, first chunk of the bucket, number of the large bucket
  uint32_t *row_cnt;     // [max_big << rshift]
  uint32_t *chunk_off;   // [max_chunks << rshift] offset of a chunk's entries inside every row
  int eshift;            // words of the binned entries: (row in bucket << eshift) | entry; below 32: words of 32 bits
  void *binned;          // [n] words of 32 or 64 bits
  int32_t *perm;         // [n] out
  int64_t *ptr;          // [rows + 1] out
};

struct RowSortPlan {
  bool ok;
  RowSortArgs p;
  size_t bytes;
};

inline RowSortPlan row_sort_plan(int64_t B, int64_t E, int64_t N, void *ws, size_t ws_bytes) {
  RowSortPlan r;
  r.ok = false;
  r.bytes = 0;
  RowSortArgs &p = r.p;
  if (B < 1 || E < 1 || N < 1 || B > 0x7FFFFFFFll / E || B > 0x7FFFFFFFll / N) return r;
  p.B = B;
  p.E = E;
  p.N = N;
  p.n = B * E;
  p.rows = B * N;
  if (p.n > 0x7FFFF000ll || p.rows >= 0x7FFFF000ll) return r;
  // Buckets: about 1024 (the tiles of place then write runs of 8 entries, 64 bytes), fewer for small inputs, more so
  // that a bucket of average size stays below the capacity of a sorting workgroup.
  p.cap = kRsSortPer * (p.n < kRsLarge ? 512 : 1024);
  int64_t want = p.n / (p.cap / 4);
  if (want > 1024) want = 1024;
  if (want < 16) want = 16;
  auto buckets = [&](int s) { return (p.rows + ((int64_t)1 << s) - 1) >> s; };
  int rs = 0;
  while (buckets(rs) > want) ++rs;
  while (rs > 0 && buckets(rs - 1) <= kRsMaxBuckets && p.n / buckets(rs) > p.cap * 3 / 4) --rs;
  if (rs > kRsMaxShift) {
    rs = kRsMaxShift;
    if (buckets(rs) > kRsMaxBuckets) return r;  // above 33.5 M rows
  }
  p.rshift = rs;
  p.nb = (int)buckets(rs);
  p.eshift = 1;
  while (((int64_t)1 << p.eshift) < p.n) ++p.eshift;
  if (p.eshift + rs > 32) p.eshift = 32;
  p.max_big = (int)(p.n / p.cap);
  p.max_chunks = 2 * p.max_big;
  auto up = [](size_t x) { return (x + 255) & ~(size_t)255; };
  size_t off = 0;
  auto take = [&](size_t bytes) { const size_t o = off; off += up(bytes); return o; };
  const size_t o_tot = take((size_t)p.nb * 4 + (size_t)(p.max_big + 1) * 4);  // totals, then the tickets
  const size_t o_state = take(16);
  const size_t o_st = take((size_t)(p.nb + 1) * 4), o_cur = take((size_t)p.nb * 4);
  const size_t o_ci = take((size_t)p.max_chunks * 12);
  const size_t o_rc = take(((size_t)p.max_big << rs) * 4), o_co = take(((size_t)p.max_chunks << rs) * 4);
  const size_t o_bin = take((size_t)p.n * (p.eshift < 32 ? 4 : 8)), o_perm = take((size_t)p.n * 4), o_ptr = take((size_t)(p.rows + 1) * 8);
  r.bytes = off;
  if (ws == nullptr || ws_bytes < off || (reinterpret_cast<uintptr_t>(ws) & 15) != 0) return r;
  char *base = static_cast<char *>(ws);
  p.totals = reinterpret_cast<uint32_t *>(base + o_tot);
  p.sync = p.totals + p.nb;
  p.state = reinterpret_cast<int32_t *>(base + o_state);
  p.starts = reinterpret_cast<uint32_t *>(base + o_st);
  p.cursor = reinterpret_cast<uint32_t *>(base + o_cur);
  p.chunk_info = reinterpret_cast<int32_t *>(base + o_ci);
  p.row_cnt = reinterpret_cast<uint32_t *>(base + o_rc);
  p.chunk_off = reinterpret_cast<uint32_t *>(base + o_co);
  p.binned = base + o_bin;
  p.perm = reinterpret_cast<int32_t *>(base + o_perm);
  p.ptr = reinterpret_cast<int64_t *>(base + o_ptr);
  r.ok = true;
  return r;
}

// Adds 1 to counter[bucket] for every lane with bucket >= 0 and returns the value before the lane's own
// addition. Twice over, the lanes that share the bucket of the first lane still waiting go through one atomic
// of their leader (with a heavy-tailed index nearly all lanes: the bucket of the hubs, which would otherwise
// queue up on one LDS address); whoever is left adds on its own.
__device__ __forceinline__ int32_t bin_take(int32_t *counter, int32_t bucket) {
  int32_t before = 0;
  bool waiting = bucket >= 0;
#pragma unroll
  for (int round = 0; round < 2; ++round) {
    const uint64_t todo = __ballot(waiting);
    if (todo == 0) break;
    // head and first are the same for the whole wavefront: scalar registers, v_readlane instead of a shuffle
    const int head = __builtin_ctzll((unsigned long long)todo);
    const int32_t first = __builtin_amdgcn_readlane(bucket, head);
    const bool with_head = waiting && bucket == first;
    const uint64_t same = __ballot(with_head);
    // lanes of `same` below this one (v_mbcnt): the head's is 0
    const int32_t below = (int32_t)__builtin_amdgcn_mbcnt_hi((uint32_t)(same >> 32),
                                                             __builtin_amdgcn_mbcnt_lo((uint32_t)same, 0u));
    int32_t base = 0;
    if (with_head && below == 0) base = atomicAdd(&counter[first], __popcll(same));
    base = __builtin_amdgcn_readlane(base, head);
    if (with_head) {
      before = base + below;
      waiting = false;
    }
  }
  if (waiting) before = atomicAdd(&counter[bucket], 1);
  return before;
}

// As bin_take, with a leader's round only for the bucket that many lanes met last (hot, the same for all lanes: an index in
// order, a hub): everybody else adds on its own, which costs fewer instructions.
__device__ __forceinline__ uint32_t rs_take(uint32_t *counter, int32_t bucket, int32_t &hot) {
  const uint64_t same = __ballot(bucket == hot);
  if (__popcll(same) >= 12) {
    uint32_t base = 0;
    const uint32_t below = __builtin_amdgcn_mbcnt_hi((uint32_t)(same >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)same, 0u));
    if (bucket == hot) {
      if (hot >= 0 && below == 0) base = atomicAdd(&counter[hot], (uint32_t)__popcll(same));
    } else if (bucket >= 0) {
      base = atomicAdd(&counter[bucket], 1u);
    }
    const uint32_t lead = (uint32_t)__builtin_amdgcn_readlane((int)base, __builtin_ctzll((unsigned long long)same));
    return bucket == hot ? lead + below : base;
  }
  hot = __builtin_amdgcn_readfirstlane(bucket);
  return bucket >= 0 ? atomicAdd(&counter[bucket], 1u) : 0u;
}
// Counts without the value before. A wavefront keeps the bucket that many of its lanes met last (a hub, an index in order) and
// that bucket's count in scalar registers; everybody else adds in LDS, where lanes with one address queue up.
struct RsHot {
  int32_t bucket;
  uint32_t count;
};
__device__ __forceinline__ void rs_count_flush(uint32_t *counter, const RsHot &hot) {
  if (hot.count != 0 && hot.bucket >= 0 && (threadIdx.x & (kWave - 1)) == 0) atomicAdd(&counter[hot.bucket], hot.count);
}
__device__ __forceinline__ void rs_count_one(uint32_t *counter, int32_t bucket, RsHot &hot) {
  const uint32_t c = (uint32_t)__popcll(__ballot(bucket == hot.bucket));
  if (c >= 6) {
    hot.count += c;
    if (bucket >= 0 && bucket != hot.bucket) atomicAdd(&counter[bucket], 1u);
  } else {
    rs_count_flush(counter, hot);
    hot.bucket = __builtin_amdgcn_readfirstlane(bucket);
    hot.count = 0;
    if (bucket >= 0) atomicAdd(&counter[bucket], 1u);
  }
}

// Index of entry be of the flattened [B, E], and the row it means: -1 for an index outside [0, N). FLAT: RowSortArgs::flat at
// compile time (-1: not). Apart, so that a lane has all its loads on the way before it needs the first: a load behind a
// condition is waited for on the spot (8 loads one after the other: count and place of 10 M entries 33 and 58 us, so 26 and 51).
template <int FLAT = -1> __device__ __forceinline__ int64_t rs_load(const RowSortArgs &p, int64_t be) {
  if (FLAT < 0 ? p.flat != 0 : FLAT != 0) return p.index[be];
  uint32_t b = 0, e = (uint32_t)be;
  if (p.B > 1) { b = (uint32_t)be / (uint32_t)p.E; e = (uint32_t)be - b * (uint32_t)p.E; }
  return p.index[(int64_t)b * p.sb + (int64_t)e * p.se];
}
template <int FLAT = -1> __device__ __forceinline__ int32_t rs_row(const RowSortArgs &p, int64_t be, int64_t idx) {
  int32_t row0 = 0;
  if (!(FLAT < 0 ? p.flat != 0 : FLAT != 0) && p.B > 1) row0 = (int32_t)((uint32_t)be / (uint32_t)p.E) * (int32_t)p.N;
  return (uint64_t)idx < (uint64_t)p.N ? row0 + (int32_t)idx : -1;
}
template <int FLAT = -1> __device__ __forceinline__ int32_t rs_node(const RowSortArgs &p, int64_t be) {
  return rs_row<FLAT>(p, be, rs_load<FLAT>(p, be));
}

// exclusive prefix sums of s[0 .. n), in place; every lane owns `per` neighbouring values. Returns the total.
template <int BLOCK> __device__ __forceinline__ uint32_t rs_scan_lds(uint32_t *s, int n, uint32_t *s_wave) {
  const int per = (n + BLOCK - 1) / BLOCK;
  const int i0 = threadIdx.x * per;
  int32_t mine = 0;
  for (int j = 0; j < per; ++j) mine += i0 + j < n ? (int32_t)s[i0 + j] : 0;
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  const int32_t incl = wave_inclusive_sum(mine);
  if (lane == kWave - 1) s_wave[wave] = (uint32_t)incl;
  __syncthreads();
  uint32_t run = (uint32_t)(incl - mine), total = 0;
#pragma unroll
  for (int w = 0; w < BLOCK / kWave; ++w) {
    const uint32_t x = s_wave[w];
    run += w < wave ? x : 0u;
    total += x;
  }
  for (int j = 0; j < per; ++j) {
    if (i0 + j >= n) break;
    const uint32_t h = s[i0 + j];
    s[i0 + j] = run;
    run += h;
  }
  __syncthreads();
  return total;
}

static __global__ __launch_bounds__(kBlock) void rs_clear_kernel(uint32_t *p, int n) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i < n) p[i] = 0;
}

template <int FLAT> static __global__ __launch_bounds__(kRsBlock) void rs_count_kernel(RowSortArgs p) {
  __shared__ uint32_t s_hist[kRsMaxBuckets];
  __shared__ uint32_t s_wave[3][kRsBlock / kWave];
  __shared__ int s_desc, s_last;
  for (int i = threadIdx.x; i < p.nb; i += kRsBlock) s_hist[i] = 0;
  if (threadIdx.x == 0) s_desc = 0;
  __syncthreads();
  const int64_t per = (p.n + gridDim.x - 1) / gridDim.x;
  const int64_t lo = (int64_t)blockIdx.x * per;
  const int64_t hi = lo + per < p.n ? lo + per : p.n;
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  int32_t node[kRsCountPer];
  int64_t next[kRsCountPer];
  auto load = [&](int64_t b0) {  // (past the end: the last entry again)
#pragma unroll
    for (int j = 0; j < kRsCountPer; ++j) {
      const int64_t be = b0 + threadIdx.x + (int64_t)j * kRsBlock;
      next[j] = rs_load<FLAT>(p, be < hi ? be : hi - 1);
    }
  };
  bool descent = false;
  RsHot hot = {-1, 0};
  if (lo < hi) load(lo);
  for (int64_t b0 = lo; b0 < hi; b0 += (int64_t)kRsCountPer * kRsBlock) {
#pragma unroll
    for (int j = 0; j < kRsCountPer; ++j) {
      const int64_t be = b0 + threadIdx.x + (int64_t)j * kRsBlock;
      node[j] = be < hi ? rs_row<FLAT>(p, be, next[j]) : -1;
    }
    if (b0 + (int64_t)kRsCountPer * kRsBlock < hi) load(b0 + (int64_t)kRsCountPer * kRsBlock);
    // The entry before a lane's entry is the neighbouring lane's; the first lane of a wavefront needs the entry before
    // the wavefront's first one: lane j loads it for row j (one load instruction for all rows).
    int32_t edge = -1;
    if (lane < kRsCountPer) {
      const int64_t be = b0 + (int64_t)(threadIdx.x - lane) + (int64_t)lane * kRsBlock;
      if (be > 0 && be < hi) edge = rs_node<FLAT>(p, be - 1);
    }
#pragma unroll
    for (int j = 0; j < kRsCountPer; ++j) {
      const int32_t e0 = __builtin_amdgcn_readlane(edge, j);
      const int32_t up = lane_up1(node[j]);  // by every lane: lane 0's value is what lane 1 reads
      const int32_t prev = lane == 0 ? e0 : up;
      const bool live = b0 + threadIdx.x + (int64_t)j * kRsBlock < hi;
      descent = descent || (live && node[j] < prev) || (live && node[j] < 0);
    }
#pragma unroll
    for (int j = 0; j < kRsCountPer; ++j) rs_count_one(s_hist, node[j] >> p.rshift, hot);  // (-1 stays -1)
  }
  rs_count_flush(s_hist, hot);
  if (__ballot(descent) != 0) s_desc = 1;
  __syncthreads();
  constexpr int PER = kRsMaxBuckets / kRsBlock;
  uint32_t back[PER];
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int i = threadIdx.x + k * kRsBlock;
    const uint32_t h = i < p.nb ? s_hist[i] : 0;
    back[k] = h != 0 ? atomicAdd(&p.totals[i], h) : 0;
  }
  uint32_t sink = 0;
#pragma unroll
  for (int k = 0; k < PER; ++k) sink |= back[k];
  asm volatile("" ::"v"(sink) : "memory");  // the returns are in: this workgroup's share is in the totals
  __syncthreads();
  // the ticket counts the workgroups in its low half and those that saw a descent in its high half
  if (threadIdx.x == 0) {
    const uint32_t t = atomicAdd(p.sync, 1u + (s_desc ? 0x10000u : 0u));
    s_last = (t & 0xFFFFu) == gridDim.x - 1 ? 1 : 0;
    s_desc = (s_desc != 0 || (t >> 16) != 0) ? 1 : 0;
  }
  __syncthreads();
  if (!s_last) return;
  // ---- the last workgroup: bucket starts, and the chunks of buckets above p.cap entries
  const bool unsorted = s_desc != 0;
  const int pb = (p.nb + kRsBlock - 1) / kRsBlock;
  uint32_t t[PER];
  int32_t sum_t = 0, sum_c = 0, sum_b = 0;
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int i = threadIdx.x * pb + j;
    t[j] = (j < pb && i < p.nb) ? atomicOr(&p.totals[i], 0u) : 0u;  // read where the additions were performed
  }
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    sum_t += (int32_t)t[j];
    if (t[j] > (uint32_t)p.cap) {
      sum_c += (int32_t)((t[j] + p.cap - 1) / p.cap);
      sum_b += 1;
    }
  }
  const int32_t it = wave_inclusive_sum(sum_t), ic = wave_inclusive_sum(sum_c), ib = wave_inclusive_sum(sum_b);
  if (lane == kWave - 1) {
    s_wave[0][wave] = (uint32_t)it;
    s_wave[1][wave] = (uint32_t)ic;
    s_wave[2][wave] = (uint32_t)ib;
  }
  __syncthreads();
  uint32_t run_t = (uint32_t)(it - sum_t), run_c = (uint32_t)(ic - sum_c), run_b = (uint32_t)(ib - sum_b);
  uint32_t all_t = 0, all_c = 0, all_b = 0;
#pragma unroll
  for (int w = 0; w < kRsBlock / kWave; ++w) {
    run_t += w < wave ? s_wave[0][w] : 0u;
    run_c += w < wave ? s_wave[1][w] : 0u;
    run_b += w < wave ? s_wave[2][w] : 0u;
    all_t += s_wave[0][w];
    all_c += s_wave[1][w];
    all_b += s_wave[2][w];
  }
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int i = threadIdx.x * pb + j;
    if (j >= pb || i >= p.nb) break;
    p.starts[i] = run_t;
    p.cursor[i] = run_t;
    run_t += t[j];
    if (t[j] > (uint32_t)p.cap) {
      s_hist[run_b] = run_c << 12 | (uint32_t)i;  // (chunks < 2^18, buckets <= 2^12)
      run_c += (t[j] + p.cap - 1) / p.cap;
      ++run_b;
    }
  }
  if (unsorted && all_c != 0) {
    // who is chunk c: the last large bucket whose first chunk is not behind it (one lane that lists the chunks of its bucket
    // is what the launch then waits for: 10 M entries, 409 chunks in one bucket, 13 us)
    __syncthreads();
    for (uint32_t c = threadIdx.x; c < all_c; c += kRsBlock) {
      uint32_t b = 0, n = all_b;
      while (n > 1) {
        const uint32_t half = n / 2;
        if ((s_hist[b + half] >> 12) <= c) { b += half; n -= half; } else { n = half; }
      }
      p.chunk_info[c] = (int32_t)(s_hist[b] & 0xFFFu);
      p.chunk_info[p.max_chunks + c] = (int32_t)(s_hist[b] >> 12);
      p.chunk_info[2 * p.max_chunks + c] = (int32_t)b;
    }
  }
  if (threadIdx.x == 0) {
    p.starts[p.nb] = all_t;
    p.ptr[p.rows] = (int64_t)all_t;
    p.state[0] = unsorted ? 1 : 0;
    p.state[1] = unsorted ? (int32_t)all_c : 0;
    p.state[2] = unsorted ? (int32_t)all_b : 0;
  }
}

// row pointers and identity for an index in order and inside [0, N): the tile of entries at lo
__device__ __forceinline__ void rs_identity(const RowSortArgs &p, int64_t lo, GapList &s_gaps) {
  if (threadIdx.x == 0) s_gaps.n = 0;
  __syncthreads();
  int64_t at[kRsPer], before[kRsPer];
#pragma unroll
  for (int j = 0; j < kRsPer; ++j) {
    const int64_t be = lo + threadIdx.x + (int64_t)j * kRsBlock, c = be < p.n ? be : p.n - 1;
    at[j] = rs_load(p, c);
    before[j] = rs_load(p, c > 0 ? c - 1 : 0);
  }
#pragma unroll
  for (int j = 0; j < kRsPer; ++j) {
    const int64_t be = lo + threadIdx.x + (int64_t)j * kRsBlock;
    const bool live = be < p.n;
    int64_t top = -1, bot = 0;
    if (live) {
      if (p.identity) p.perm[be] = (int32_t)be;
      top = rs_row(p, be, at[j]);
      bot = be == 0 ? 0 : (int64_t)rs_row(p, be - 1, before[j]) + 1;
    }
    gap_rows(p.ptr, bot, top, be, s_gaps);
    gap_rows(p.ptr, top + 1, live && be == p.n - 1 ? p.rows : top, p.n, s_gaps);
  }
  __syncthreads();
  gap_rows_finish(p.ptr, s_gaps);
}

// (eight wavefronts per SIMD, i.e. at most 64 vector registers: two workgroups per CU)
template <int FLAT, typename W>
static __global__ __launch_bounds__(kRsBlock) __attribute__((amdgpu_waves_per_eu(8, 8)))
void rs_place_kernel(RowSortArgs p) {
  extern __shared__ uint32_t s_rows[];
  static_assert(kRsTile * 8 + 2048 + kRsMaxBuckets * 8 <= 160 * 1024, "a workgroup's LDS: 160 KB with counts and bases");
  __shared__ uint64_t s_stage[kRsTile];
  __shared__ uint32_t s_wave[kRsBlock / kWave];
  __shared__ GapList s_gaps;
  uint32_t *s_cnt = s_rows;  // [nb] counts, then the tile's exclusive prefix
  uint32_t *s_base = s_cnt + p.nb;  // [nb] first word of the tile's run in every bucket, less the run's place in the tile
  const int64_t lo = (int64_t)blockIdx.x * kRsTile;
  if (p.state[0] == 0) {
    rs_identity(p, lo, s_gaps);
    return;
  }
  // the row counts of large buckets, for the next launch
  const int64_t n_cnt = (int64_t)p.state[2] << p.rshift;
  for (int64_t i = (int64_t)blockIdx.x * kRsBlock + threadIdx.x; i < n_cnt; i += (int64_t)gridDim.x * kRsBlock) p.row_cnt[i] = 0;
  for (int i = threadIdx.x; i < p.nb; i += kRsBlock) s_cnt[i] = 0;
  int32_t node[kRsPer];
  uint32_t rank[kRsPer];
  {
    int64_t idx[kRsPer];
#pragma unroll
    for (int j = 0; j < kRsPer; ++j) {
      const int64_t be = lo + threadIdx.x + (int64_t)j * kRsBlock;
      idx[j] = rs_load<FLAT>(p, be < p.n ? be : p.n - 1);
    }
#pragma unroll
    for (int j = 0; j < kRsPer; ++j) {
      const int64_t be = lo + threadIdx.x + (int64_t)j * kRsBlock;
      node[j] = be < p.n ? rs_row<FLAT>(p, be, idx[j]) : -1;
    }
  }
  __syncthreads();
  int32_t hot = -1;
#pragma unroll
  for (int j = 0; j < kRsPer; ++j)
    rank[j] = rs_take(s_cnt, node[j] >> p.rshift, hot);  // (-1 stays -1)
  __syncthreads();
  constexpr int PER = kRsMaxBuckets / kRsBlock;
  uint32_t first[PER];  // of buckets threadIdx.x + k * kRsBlock
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int i = threadIdx.x + k * kRsBlock;
    const uint32_t h = i < p.nb ? s_cnt[i] : 0;
    first[k] = h != 0 ? atomicAdd(&p.cursor[i], h) : 0;
  }
  __syncthreads();
  const int total = (int)rs_scan_lds<kRsBlock>(s_cnt, p.nb, s_wave);
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int i = threadIdx.x + k * kRsBlock;
    if (i < p.nb) s_base[i] = first[k] - s_cnt[i];
  }
  const uint32_t mask = (1u << p.rshift) - 1;
  constexpr int BITS = sizeof(W) == 4 ? 32 : 45;  // of a word (13 for the row in its bucket), above them its bucket
#pragma unroll
  for (int j = 0; j < kRsPer; ++j) {
    if (node[j] < 0) continue;
    const uint32_t b = (uint32_t)node[j] >> p.rshift;
    const uint32_t be = (uint32_t)(lo + threadIdx.x + (int64_t)j * kRsBlock);
    s_stage[s_cnt[b] + rank[j]] = (uint64_t)b << BITS | (W)((uint32_t)node[j] & mask) << (sizeof(W) == 4 ? p.eshift : 32) | be;
  }
  __syncthreads();
#pragma unroll
  for (int j0 = 0; j0 < kRsPer; j0 += 4) {
    uint64_t w[4];
    uint32_t to[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int pos = (int)threadIdx.x + (j0 + j) * kRsBlock;
      w[j] = s_stage[pos];
      w[j] = pos < total ? w[j] : 0;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) to[j] = s_base[(uint32_t)(w[j] >> BITS)] + threadIdx.x + (uint32_t)((j0 + j) * kRsBlock);
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if ((int)threadIdx.x + (j0 + j) * kRsBlock < total) static_cast<W *>(p.binned)[to[j]] = (W)(w[j] & (((uint64_t)1 << BITS) - 1));
  }
}

template <int BLOCK, typename W>
static __global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(BLOCK == 512 ? 6 : 8)))
void rs_sort_kernel(RowSortArgs p) {
  constexpr int CAP = kRsSortPer * BLOCK, CAP_LOG = BLOCK == 512 ? 13 : 14;
  extern __shared__ uint32_t s_rows[];
  __shared__ uint32_t s_stage[CAP];
  __shared__ uint32_t s_wave[BLOCK / kWave];
  __shared__ int s_last;
  static_assert(CAP * 4 + 1024 + (4 << kRsMaxShift) <= 160 * 1024, "a workgroup's LDS: 160 KB with the row counts");
  uint32_t *s_hist = s_rows;  // [rows per bucket]
  if (p.state[0] == 0) return;
  const int R = 1 << p.rshift;
  // (the chunks come first: each takes as long as the largest bucket)
  int bucket = (int)blockIdx.x - p.max_chunks, chunk = -1, big = 0, first = 0;
  if (bucket < 0) {
    chunk = (int)blockIdx.x;
    if (chunk >= p.state[1]) return;
    bucket = p.chunk_info[chunk];
    first = p.chunk_info[p.max_chunks + chunk];
    big = p.chunk_info[2 * p.max_chunks + chunk];
  }
  const uint32_t b_lo = p.starts[bucket], b_hi = p.starts[bucket + 1];
  uint32_t lo = b_lo, hi = b_hi;
  if (chunk < 0) {
    if (hi - lo > (uint32_t)CAP) return;
  } else {
    lo = b_lo + (uint32_t)(chunk - first) * CAP;
    hi = lo + CAP < b_hi ? lo + CAP : b_hi;
  }
  for (int i = threadIdx.x; i < R; i += BLOCK) s_hist[i] = 0;
  const int cnt = (int)(hi - lo);
  const int shift = sizeof(W) == 4 ? p.eshift : 32;
  const W *words = static_cast<const W *>(p.binned);
  W word[kRsSortPer];
  uint32_t row_rank[kRsSortPer];  // row << CAP_LOG | rank in the row
#pragma unroll
  for (int j = 0; j < kRsSortPer; ++j) {
    const int i = j * BLOCK + (int)threadIdx.x;
    word[j] = words[i < cnt ? lo + (uint32_t)i : 0];
  }
  __syncthreads();
  int32_t hot = -1;
#pragma unroll
  for (int j = 0; j < kRsSortPer; ++j) {
    if (j * BLOCK >= cnt) break;  // (the same for the workgroup)
    const int i = j * BLOCK + (int)threadIdx.x;
    const uint32_t r = (uint32_t)(word[j] >> shift);
    row_rank[j] = r << CAP_LOG | rs_take(s_hist, i < cnt ? (int32_t)r : -1, hot);
  }
  const uint32_t entry_mask = sizeof(W) == 4 ? (1u << p.eshift) - 1 : ~0u;
  __syncthreads();
  const int64_t row0 = (int64_t)bucket << p.rshift;
  const int n_rows = p.rows - row0 < R ? (int)(p.rows - row0) : R;
  if (chunk < 0) {
    rs_scan_lds<BLOCK>(s_hist, R, s_wave);
    for (int i = threadIdx.x; i < n_rows; i += BLOCK) p.ptr[row0 + i] = (int64_t)(lo + s_hist[i]);
#pragma unroll
    for (int j = 0; j < kRsSortPer; ++j) {
      const int i = j * BLOCK + (int)threadIdx.x;
      const uint32_t rr = row_rank[j];
      if (i < cnt) s_stage[s_hist[rr >> CAP_LOG] + (rr & (CAP - 1))] = (uint32_t)word[j] & entry_mask;
    }
    __syncthreads();
#pragma unroll 8
    for (int i = threadIdx.x; i < cnt; i += BLOCK) p.perm[lo + (uint32_t)i] = (int32_t)s_stage[i];
    return;
  }
  // A chunk of a large bucket: its counts to the bucket's; what they found there is the chunk's offset inside every row. The
  // chunk's words go back in order of their rows; of 64 bits as [cnt] entries of 32 and behind them [cnt] rows of 16 bits.
  rs_scan_lds<BLOCK>(s_hist, R, s_wave);
  uint32_t sink = 0;
  for (int i = threadIdx.x; i < R; i += BLOCK) {
    const uint32_t at = s_hist[i], h = (i + 1 < R ? s_hist[i + 1] : (uint32_t)cnt) - at;
    if (h == 0) continue;
    const uint32_t before = atomicAdd(&p.row_cnt[((int64_t)big << p.rshift) + i], h);
    p.chunk_off[((int64_t)chunk << p.rshift) + i] = before - at;
    sink |= before;
  }
#pragma unroll
  for (int j = 0; j < kRsSortPer; ++j) {
    const int i = j * BLOCK + (int)threadIdx.x;
    const uint32_t rr = row_rank[j];
    if (i < cnt) s_stage[s_hist[rr >> CAP_LOG] + (rr & (CAP - 1))] = (uint32_t)word[j];
  }
  __syncthreads();
  uint32_t *entries = reinterpret_cast<uint32_t *>(static_cast<W *>(p.binned) + lo);
  for (int i = threadIdx.x; i < cnt; i += BLOCK) entries[i] = s_stage[i];
  asm volatile("" ::"v"(sink) : "memory");  // the returns are in: the counts are in memory
  __syncthreads();
  if (threadIdx.x == 0) {
    const uint32_t m = (b_hi - b_lo + CAP - 1) / CAP;
    s_last = atomicAdd(&p.sync[1 + big], 1u) == m - 1 ? 1 : 0;
  }
  if constexpr (sizeof(W) == 8) {
    uint16_t *s_srow = reinterpret_cast<uint16_t *>(s_stage);
#pragma unroll
    for (int j = 0; j < kRsSortPer; ++j) {
      const uint32_t rr = row_rank[j];
      if (j * BLOCK + (int)threadIdx.x < cnt) s_srow[s_hist[rr >> CAP_LOG] + (rr & (CAP - 1))] = (uint16_t)(rr >> CAP_LOG);
    }
    __syncthreads();
    uint16_t *rows = reinterpret_cast<uint16_t *>(entries + cnt);
    for (int i = threadIdx.x; i < cnt; i += BLOCK) rows[i] = s_srow[i];
  } else {
    __syncthreads();
  }
  if (!s_last) return;
  for (int i = threadIdx.x; i < R; i += BLOCK) s_hist[i] = atomicOr(&p.row_cnt[((int64_t)big << p.rshift) + i], 0u);
  __syncthreads();
  rs_scan_lds<BLOCK>(s_hist, R, s_wave);
  for (int i = threadIdx.x; i < n_rows; i += BLOCK) p.ptr[row0 + i] = (int64_t)(b_lo + s_hist[i]);
}

// the chunks of large buckets, each in order of its rows: every entry to its place among its row's
constexpr int kRsPiece = 8;  // entries per lane; a chunk is 4 or 8 pieces
template <typename W> static __global__ __launch_bounds__(kBlock) void rs_place_chunks_kernel(RowSortArgs p) {
  const int pieces = p.cap / (kRsPiece * kBlock), n = p.state[1] * pieces;
  for (int q = (int)blockIdx.x; q < n; q += (int)gridDim.x) {
    const int chunk = q / pieces, i0 = (q - chunk * pieces) * (kRsPiece * kBlock) + (int)threadIdx.x;
    const int bucket = p.chunk_info[chunk];
    const uint32_t lo = p.starts[bucket] + (uint32_t)(chunk - p.chunk_info[p.max_chunks + chunk]) * (uint32_t)p.cap;
    const uint32_t left = p.starts[bucket + 1] - lo;
    const int cnt = left < (uint32_t)p.cap ? (int)left : p.cap;
    const int64_t *ptr = p.ptr + ((int64_t)bucket << p.rshift);
    const uint32_t *off = p.chunk_off + ((int64_t)chunk << p.rshift);
    const uint32_t *entries = reinterpret_cast<const uint32_t *>(static_cast<const W *>(p.binned) + lo);
    const uint16_t *rows = reinterpret_cast<const uint16_t *>(entries + cnt);  // (words of 64 bits)
    uint32_t e[kRsPiece], r[kRsPiece];
#pragma unroll
    for (int j = 0; j < kRsPiece; ++j) {  // (past the end: the last entry again)
      const int i = i0 + j * kBlock < cnt ? i0 + j * kBlock : cnt - 1;
      e[j] = entries[i];
      if constexpr (sizeof(W) == 8) r[j] = rows[i];
    }
    if constexpr (sizeof(W) == 4) {
#pragma unroll
      for (int j = 0; j < kRsPiece; ++j) {
        r[j] = e[j] >> p.eshift;
        e[j] &= (1u << p.eshift) - 1;
      }
    }
#pragma unroll
    for (int j = 0; j < kRsPiece; ++j) r[j] = (uint32_t)ptr[r[j]] + off[r[j]] + (uint32_t)(i0 + j * kBlock);
#pragma unroll
    for (int j = 0; j < kRsPiece; ++j)
      if (i0 + j * kBlock < cnt) p.perm[r[j]] = (int32_t)e[j];
  }
}

// entries of every row, from the row pointers
static __global__ __launch_bounds__(kBlock) void row_lengths_kernel(const int64_t *ptr, int32_t *len, int64_t rows) {
  for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < rows; i += (int64_t)gridDim.x * kBlock)
    len[i] = (int32_t)(ptr[i + 1] - ptr[i]);
}

// Backward of scatter min / max over entries sorted by row: grad_in[e, k] = grad[row, k] where arg[row, k] == e, else 0.
// Every row of grad_in is written once, in one piece, and the entries of a row read its gradient and positions from the
// vector L1. (A fill of grad_in and a scatter of single elements into it writes the buffer twice: 2.3 M x 64 floats onto
// 282 k rows 368 us, of which the scatter 260; now 220 with 55 for the sort, 3.7 TB/s in rows of 256 bytes in no order.) U: bits of an element. A workgroup takes 4 positions per worker.
template <typename U, int VEC>
static __global__ __launch_bounds__(kBlock) void rs_arg_rows_kernel(RowSortArgs p, const U *__restrict__ grad,
                                                                    const int64_t *__restrict__ arg,
                                                                    U *__restrict__ grad_in, int64_t K, int G) {
  constexpr int Q = 4;
  const int W = kBlock / G, w = threadIdx.x / G, lg = threadIdx.x - w * G;
  const int64_t col = ((int64_t)blockIdx.y * G + lg) * VEC;
  if (col >= K) return;
  const int64_t n = p.ptr[p.rows];  // entries inside [0, N)
  const int64_t base = (int64_t)blockIdx.x * W * Q + w;
  int32_t e[Q], row[Q];
#pragma unroll
  for (int q = 0; q < Q; ++q) e[q] = base + (int64_t)q * W < n ? p.perm[base + (int64_t)q * W] : -1;
#pragma unroll
  for (int q = 0; q < Q; ++q) row[q] = e[q] >= 0 ? rs_node(p, e[q]) : 0;
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    if (e[q] < 0) continue;
    const Vec<int64_t, VEC> a = load_vec<int64_t, VEC>(arg + (int64_t)row[q] * K + col);
    const Vec<U, VEC> g = load_vec<U, VEC>(grad + (int64_t)row[q] * K + col);
    const int64_t at = p.B > 1 ? (int64_t)((uint32_t)e[q] % (uint32_t)p.E) : (int64_t)e[q];  // inside its batch
    Vec<U, VEC> o;
#pragma unroll
    for (int v = 0; v < VEC; ++v) o.v[v] = a.v[v] == at ? g.v[v] : (U)0;
    store_vec_stream<U, VEC>(grad_in + (int64_t)e[q] * K + col, o);
  }
}
// ... and zeros for the entries outside [0, N), if there are any
template <typename U>
static __global__ __launch_bounds__(kBlock) void rs_zero_outside_kernel(RowSortArgs p, U *__restrict__ grad_in, int64_t K) {
  if (p.ptr[p.rows] == p.n) return;
  const int64_t waves = (int64_t)gridDim.x * (kBlock / kWave);
  for (int64_t e = (int64_t)blockIdx.x * (kBlock / kWave) + threadIdx.x / kWave; e < p.n; e += waves) {
    if (rs_node(p, e) >= 0) continue;
    for (int64_t k = threadIdx.x & (kWave - 1); k < K; k += kWave) grad_in[e * K + k] = (U)0;
  }
}
template <typename U, int VEC>
inline int launch_arg_rows(const RowSortArgs &p, const void *grad, const int64_t *arg, void *grad_in, int64_t K,
                           hipStream_t stream) {
  const int64_t lanes = (K + VEC - 1) / VEC;
  int G = 1;
  while (G < lanes && G < kWave) G <<= 1;
  const int64_t per = (int64_t)(kBlock / G) * 4, ychunks = (lanes + G - 1) / G;
  if (ychunks > 65535) return TS_ERR_UNSUPPORTED;
  hipLaunchKernelGGL((rs_arg_rows_kernel<U, VEC>), dim3((unsigned)((p.n + per - 1) / per), (unsigned)ychunks), dim3(kBlock), 0,
                     stream, p, static_cast<const U *>(grad), arg, static_cast<U *>(grad_in), K, G);
  hipLaunchKernelGGL(rs_zero_outside_kernel<U>, dim3(1024), dim3(kBlock), 0, stream, p, static_cast<U *>(grad_in), K);
  return hipGetLastError() == hipSuccess ? TS_OK : TS_ERR_LAUNCH;
}

template <typename W> inline int launch_row_sort_words(const RowSortArgs &p, hipStream_t stream) {
  const dim3 gt((unsigned)((p.n + kRsTile - 1) / kRsTile));
  if (p.flat)
    hipLaunchKernelGGL((rs_place_kernel<1, W>), gt, dim3(kRsBlock), (size_t)p.nb * 8, stream, p);
  else
    hipLaunchKernelGGL((rs_place_kernel<0, W>), gt, dim3(kRsBlock), (size_t)p.nb * 8, stream, p);
  const dim3 gs((unsigned)(p.nb + p.max_chunks));
  const size_t lds = (size_t)4 << p.rshift;
  if (p.cap == kRsSortPer * 512)
    hipLaunchKernelGGL((rs_sort_kernel<512, W>), gs, dim3(512), lds, stream, p);
  else
    hipLaunchKernelGGL((rs_sort_kernel<1024, W>), gs, dim3(1024), lds, stream, p);
  if (p.max_chunks > 0) {
    const int64_t pieces = (int64_t)p.max_chunks * (p.cap / (kRsPiece * kBlock));
    hipLaunchKernelGGL(rs_place_chunks_kernel<W>, dim3((unsigned)(pieces < 2048 ? pieces : 2048)), dim3(kBlock), 0, stream, p);
  }
  return hipGetLastError() == hipSuccess ? TS_OK : TS_ERR_LAUNCH;
}

inline int launch_row_sort(const RowSortArgs &args, const int64_t *index, int64_t sb, int64_t se, bool identity,
                           hipStream_t stream) {
  RowSortArgs p = args;
  p.identity = identity ? 1 : 0;
  p.index = index;
  p.sb = sb;
  p.se = se;
  p.flat = p.B == 1 && se == 1;
  const int n_clear = p.nb + 1 + p.max_big;
  hipLaunchKernelGGL(rs_clear_kernel, dim3((unsigned)((n_clear + kBlock - 1) / kBlock)), dim3(kBlock), 0, stream, p.totals,
                     n_clear);
  int64_t groups = (p.n + kRsCountPer * kRsBlock - 1) / (kRsCountPer * kRsBlock);
  if (groups > kRsCountGroups) groups = kRsCountGroups;
  if (p.flat)
    hipLaunchKernelGGL(rs_count_kernel<1>, dim3((unsigned)groups), dim3(kRsBlock), 0, stream, p);
  else
    hipLaunchKernelGGL(rs_count_kernel<0>, dim3((unsigned)groups), dim3(kRsBlock), 0, stream, p);
  return p.eshift < 32 ? launch_row_sort_words<uint32_t>(p, stream) : launch_row_sort_words<uint64_t>(p, stream);
}

}  // namespace ts
