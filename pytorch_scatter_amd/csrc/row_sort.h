// An index in any order -> the entries in order of their rows: perm (entry numbers) and row pointers, the input of
// the segmented reductions (csr_reduce.h with rows through perm). Two levels: entries are binned by bucket of R
// consecutive rows inside tiles of up to 8192 entries, then every bucket is sorted by row in LDS.
//   place : a workgroup per tile: the tile's entries sorted by bucket in LDS leave as 32-bit words in one piece, with the
//           offset of every bucket among them. Also: does the index descend or leave [0, N) in this tile? If no tile says
//           so the row pointers that the tiles wrote on the way stand, and the passes behind return at once.
//   sort  : a workgroup per bucket of up to 8192 or 16384 entries collects its runs from all tiles. What lies before the
//           bucket is the sum of its offsets over the tiles, so nothing has to be counted in front, nothing is cleared,
//           and nothing meets in memory. Counting sort by row in LDS, row pointers and perm out.
//   chunk : a bucket with more entries (hubs, few rows) is taken in chunks, which begin their search for runs where the sort
//           pass noted it (a round of 1024 tiles): each is left in order of its rows, the row
//           counts meet in memory, the chunk that arrives last turns them into row pointers,
//   place chunks : ... and the chunks' entries then go from there to their places, each behind the row's entries of the
//           chunks that were counted before.
// Entries of a row come in no particular order (a reader that needs the first of equal values compares positions).
// Entries outside [0, N) are left out.
// What it costs: 8 bytes of index, 4 written and read per entry for the words, 4 for perm. What bounds it: place the loads
// (10 M entries: 120 MB in 27 us), sort the instructions, about 35 an entry (with the prefix over a workgroup's wavefronts
// as a loop over their sums, a third more: 69 us at 10 M). us of place / sort / chunk / place chunks, the last two at least
// 4.6 each for launches that return at once: 1 M entries onto 66 k rows 7 / 10 / 5 / 5, 2.3 M onto 268 k 10 / 13 / 5 / 5,
// 5 M 16 / 24 / 5 / 5, 10 M onto 333 k 27 / 51 / 5 / 5, 10 M onto 100 k, a fifth of them in one row, 29 / 47 / 30 / 14.
// With a pass over the index that counted into the buckets first and place sending every run to its bucket (clear / count /
// place / sort / place chunks): 1 M 5 / 10 / 9 / 8 / 4, 2.3 M 5 / 16 / 16 / 9 / 5, 10 M even 5 / 26 / 50 / 26 / 5. Scatter sums
// and maxima of 0.3 to 10 M entries, rows of 64 to 256 bytes: 0.94 of the time in the geometric mean.
#pragma once

#include "device_utils.h"

namespace ts {

constexpr int kRsBlock = 1024;        // place
constexpr int kRsLocal = 13;          // bits of an entry's place in its tile: tiles of up to 8192 entries
// entries that one sorting workgroup holds in registers: 16 per lane, 512 lanes below kRsLarge entries (more, shorter
// workgroups), 1024 above, where fewer buckets leave longer runs in the tiles
constexpr int kRsSortPer = 16;
constexpr int64_t kRsLarge = (int64_t)1 << 22;
constexpr int kRsMaxBuckets = 4096;   // counters of place
constexpr int kRsMaxShift = 13;       // rows per bucket (log2): counters of the sorting workgroup
constexpr int kRsMaxRounds = 256;     // 2^31 entries in tiles of 8192, in rounds of 1024 tiles

struct RowSortArgs {
  const int64_t *index;
  int64_t sb, se;        // element strides of the index over batches and entries
  int64_t B, E, N;
  int64_t n, rows;       // B * E entries, B * N rows
  int identity;          // an index in order: write the identity to perm (a reader that looks at state[0] does without);
                         // perm_row is written whenever there is one
  int flat;              // one batch, unit stride: entry e is index[e] (no 64-bit multiplications per entry)
  int rshift, nb;        // rows per bucket (log2), buckets
  int per;               // entries per lane of place: a tile holds per * kRsBlock
  int tiles;
  int pitch;             // 16-bit words from one tile's offsets to the next: nb + 1, rounded up
  int cap;               // entries that one sorting workgroup takes
  int max_big;           // buckets above that: at most this many ...
  int max_chunks;        // ... in at most this many chunks
  uint32_t nonce;        // tag of the call, never 0
  const int *gate;       // reads 0: every pass returns at once (null: they run)
  int32_t *state;        // [0] 0: the index is in order, 1: it is not; [1] chunks of large buckets; [2] large buckets;
                         // [3] the nonce of the latest call that met an index that is not in order; [4] 1 if these
                         // passes ran (the caller's word for a gate)
  uint16_t *off;         // [tiles][pitch] first entry of every bucket among the tile's words; [nb]: how many there are
  int log;               // a tile's words lie at tile << log
  uint32_t *words;       // [tiles << log] a tile's entries by bucket: row in the bucket << kRsLocal | place in the tile
  uint32_t *big;         // [max_big][4] large buckets: bucket, first place in perm, entries, first chunk
  uint32_t *arrived;     // [max_big] chunks that have added their counts
  int32_t *chunk_big;    // [max_chunks] the chunk's large bucket,
  uint32_t *chunk_at;    // [max_chunks][2] where its search for its runs begins: a tile, entries of the bucket before that tile
  uint32_t *row_cnt;     // [max_big << rshift]
  uint32_t *chunk_off;   // [max_chunks << rshift] offset of a chunk's entries inside every row
  uint32_t *by_row;      // [n] entries of chunks, each chunk in order of its rows,
  uint16_t *by_row_row;  // [n] and their rows in the bucket
  int32_t *perm;         // [n] out
  int32_t *perm_row;     // [n] out, may be null: the row of every entry of perm
  int64_t *ptr;          // [rows + 1] out
};

struct RowSortPlan {
  bool ok;
  RowSortArgs p;
  size_t bytes;       // results and scratch
  size_t kept_bytes;  // the results (state, perm, perm_row, ptr) alone, which come first
};

// with_rows: perm_row as well. kept: the results lie there and the scratch alone at ws (bytes - kept_bytes); with ws null
// the plan describes the results of an earlier call.
inline RowSortPlan row_sort_plan(int64_t B, int64_t E, int64_t N, void *ws, size_t ws_bytes, bool with_rows = false,
                                 void *kept = nullptr) {
  RowSortPlan r;
  r.ok = false;
  r.bytes = r.kept_bytes = 0;
  RowSortArgs &p = r.p;
  if (B < 1 || E < 1 || N < 1 || B > 0x7FFFFFFFll / E || B > 0x7FFFFFFFll / N) return r;
  p.B = B;
  p.E = E;
  p.N = N;
  p.n = B * E;
  p.rows = B * N;
  if (p.n > 0x7FFFF000ll || p.rows >= 0x7FFFF000ll) return r;
  // Buckets: about 1024 (a tile of place then leaves runs of 8 entries), fewer for small inputs, more so that a bucket
  // of average size stays below the capacity of a sorting workgroup -- where that is within reach: from 34 to 67 M entries on
  // all of them are taken in chunks anyhow, and short runs cost the chunks a line for two entries (200 M entries onto 2 M rows, us of
  // the chunks with 3907 buckets, each chunk looking through all tiles from the first one on: 4820; with 977 and a tile to
  // begin at: 1390; the whole sort 7020 / 2890).
  p.cap = kRsSortPer * (p.n < kRsLarge ? 512 : 1024);
  int64_t want = p.n / (p.cap / 4);
  if (want > 1024) want = 1024;
  if (want < 16) want = 16;
  auto buckets = [&](int s) { return (p.rows + ((int64_t)1 << s) - 1) >> s; };
  int rs = 0;
  while (buckets(rs) > want) ++rs;
  int fine = rs;
  while (fine > 0 && buckets(fine - 1) <= kRsMaxBuckets && p.n / buckets(fine) > p.cap * 3 / 4) --fine;
  if (p.n / buckets(fine) <= p.cap) rs = fine;
  if (rs > kRsMaxShift) {
    rs = kRsMaxShift;
    if (buckets(rs) > kRsMaxBuckets) return r;  // above 33.5 M rows
  }
  p.rshift = rs;
  p.nb = (int)buckets(rs);
  // tiles: up to 8192 entries, fewer where all tiles then run at once (two workgroups per CU)
  const int64_t per = (p.n + 512 * kRsBlock - 1) / (512 * kRsBlock);
  p.per = per > 8 ? 8 : (int)per;
  p.log = 10;
  while (1 << (p.log - 10) < p.per) ++p.log;
  const int64_t tile = (int64_t)p.per * kRsBlock;
  p.tiles = (int)((p.n + tile - 1) / tile);
  p.pitch = (p.nb + 2) & ~1;
  // (entries / cap + 1 chunks at most of a bucket with more than cap)
  p.max_big = (int)(p.n / p.cap < p.nb ? p.n / p.cap : p.nb);
  p.max_chunks = (int)(p.n / p.cap) + p.max_big;
  auto up = [](size_t x) { return (x + 255) & ~(size_t)255; };
  size_t off = 0;
  auto take = [&](size_t bytes) { const size_t o = off; off += up(bytes); return o; };
  const size_t big_n = p.max_big > 0 ? (size_t)p.n : 0;
  const size_t o_state = take(32);
  const size_t o_perm = take((size_t)p.n * 4), o_prow = take(with_rows ? (size_t)p.n * 4 : 0), o_ptr = take((size_t)(p.rows + 1) * 8);
  r.kept_bytes = off;
  const size_t o_off = take((size_t)p.tiles * p.pitch * 2), o_words = take(((size_t)p.tiles << p.log) * 4);
  const size_t o_big = take((size_t)p.max_big * 16), o_arr = take((size_t)p.max_big * 4), o_cb = take((size_t)p.max_chunks * 4),
               o_at = take((size_t)p.max_chunks * 8);
  const size_t o_rc = take(((size_t)p.max_big << rs) * 4), o_co = take(((size_t)p.max_chunks << rs) * 4);
  const size_t o_br = take(big_n * 4), o_brr = take(big_n * 2);
  r.bytes = off;
  if (ws == nullptr && kept == nullptr) return r;
  if (ws != nullptr && (ws_bytes < (kept != nullptr ? off - r.kept_bytes : off) || (reinterpret_cast<uintptr_t>(ws) & 15) != 0)) return r;
  if ((reinterpret_cast<uintptr_t>(kept) & 15) != 0) return r;
  char *results = static_cast<char *>(kept != nullptr ? kept : ws);
  char *base = kept == nullptr ? results : static_cast<char *>(ws) - r.kept_bytes;
  p.state = reinterpret_cast<int32_t *>(results + o_state);
  p.off = reinterpret_cast<uint16_t *>(base + o_off);
  p.words = reinterpret_cast<uint32_t *>(base + o_words);
  p.big = reinterpret_cast<uint32_t *>(base + o_big);
  p.arrived = reinterpret_cast<uint32_t *>(base + o_arr);
  p.chunk_big = reinterpret_cast<int32_t *>(base + o_cb);
  p.chunk_at = reinterpret_cast<uint32_t *>(base + o_at);
  p.row_cnt = reinterpret_cast<uint32_t *>(base + o_rc);
  p.chunk_off = reinterpret_cast<uint32_t *>(base + o_co);
  p.by_row = reinterpret_cast<uint32_t *>(base + o_br);
  p.by_row_row = reinterpret_cast<uint16_t *>(base + o_brr);
  p.perm = reinterpret_cast<int32_t *>(results + o_perm);
  p.perm_row = with_rows ? reinterpret_cast<int32_t *>(results + o_prow) : nullptr;
  p.ptr = reinterpret_cast<int64_t *>(results + o_ptr);
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

// s_wave: a number per wavefront. Their sum over the wavefronts before this one, and over all of them: a scan in every wavefront
// (a loop over the numbers takes three instructions for each, a third of what the sorting workgroups executed).
template <int BLOCK> __device__ __forceinline__ uint32_t rs_waves_before(const uint32_t *s_wave, uint32_t &total) {
  constexpr int W = BLOCK / kWave;
  const int lane = threadIdx.x & (kWave - 1), wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x / kWave);
  const int32_t incl = wave_inclusive_sum(lane < W ? (int32_t)s_wave[lane] : 0);
  total = (uint32_t)__builtin_amdgcn_readlane(incl, W - 1);
  return wave > 0 ? (uint32_t)__builtin_amdgcn_readlane(incl, wave - 1) : 0u;
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
  uint32_t total, run = (uint32_t)(incl - mine) + rs_waves_before<BLOCK>(s_wave, total);
  for (int j = 0; j < per; ++j) {
    if (i0 + j >= n) break;
    const uint32_t h = s[i0 + j];
    s[i0 + j] = run;
    run += h;
  }
  __syncthreads();
  return total;
}

// A tile of entries by bucket. A tile whose rows do not descend writes the row pointers that its entries mark and perm_row
// as well: they stand if no tile has seen a descent, else the sorting passes write all of them again.
template <int FLAT, int PER>
static __global__ __launch_bounds__(kRsBlock) __attribute__((amdgpu_waves_per_eu(8, 8)))
void rs_place_kernel(RowSortArgs p) {
  constexpr int TILE = PER * kRsBlock;
  static_assert(TILE <= 1 << kRsLocal, "a place in the tile has kRsLocal bits");
  extern __shared__ uint32_t s_cnt[];  // [nb] counts, then the tile's exclusive prefix
  __shared__ uint32_t s_stage[TILE];
  __shared__ uint32_t s_wave[kRsBlock / kWave];
  __shared__ GapList s_gaps;
  __shared__ int s_desc;
  const int64_t lo = (int64_t)blockIdx.x * TILE;
  if (p.gate != nullptr && *p.gate == 0) return;
  const int lane = threadIdx.x & (kWave - 1);
  int32_t node[PER];
  uint32_t rank[PER];
  int64_t idx[PER];
  const uint32_t left = (uint32_t)(p.n - lo < TILE ? p.n - lo : TILE);
#pragma unroll
  for (int j = 0; j < PER; ++j) {  // (past the end: the last entry again)
    const uint32_t i = threadIdx.x + j * kRsBlock < left ? threadIdx.x + j * kRsBlock : left - 1;
    idx[j] = FLAT ? (p.index + lo)[i] : rs_load<FLAT>(p, lo + i);
  }
  // The entry before a lane's entry is the neighbouring lane's; the first lane of a wavefront needs the entry before the
  // wavefront's first one: lane j loads it for row j (one load instruction for all rows).
  int32_t edge = -1;
  if (lane < PER) {
    const int64_t be = lo + (int64_t)(threadIdx.x - lane) + (int64_t)lane * kRsBlock;
    if (be > 0 && be < p.n) edge = rs_node<FLAT>(p, be - 1);
  }
  for (int i = threadIdx.x; i < p.nb; i += kRsBlock) s_cnt[i] = 0;
  if (threadIdx.x == 0) {
    s_desc = 0;
    s_gaps.n = 0;
    if (blockIdx.x == 0) {
      p.state[1] = p.state[2] = 0;
      p.state[4] = 1;
    }
  }
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const uint32_t i = threadIdx.x + j * kRsBlock;
    node[j] = i < left ? rs_row<FLAT>(p, lo + i, idx[j]) : -1;
  }
  __syncthreads();
  bool descent = false;
  int32_t hot = -1;
  auto before = [&](int j) {
    const int32_t e0 = __builtin_amdgcn_readlane(edge, j);
    const int32_t up = lane_up1(node[j]);  // by every lane: lane 0's value is what lane 1 reads
    return lane == 0 ? e0 : up;
  };
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int32_t prev = before(j);
    descent = descent || (threadIdx.x + j * kRsBlock < left && (node[j] < prev || node[j] < 0));
    rank[j] = rs_take(s_cnt, node[j] >> p.rshift, hot);  // (-1 stays -1)
  }
  if (__ballot(descent) != 0 && lane == 0) s_desc = 1;
  __syncthreads();
  const bool in_order = s_desc == 0;
  if (!in_order && threadIdx.x == 0) p.state[3] = (int32_t)p.nonce;
  const int total = (int)rs_scan_lds<kRsBlock>(s_cnt, p.nb, s_wave);
  uint16_t *off = p.off + (size_t)blockIdx.x * p.pitch;
  for (int i = threadIdx.x; i <= p.nb; i += kRsBlock) off[i] = (uint16_t)(i < p.nb ? s_cnt[i] : (uint32_t)total);
  const uint32_t mask = (1u << p.rshift) - 1;
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    if (node[j] < 0) continue;
    const uint32_t at = threadIdx.x + (uint32_t)(j * kRsBlock);
    s_stage[s_cnt[(uint32_t)node[j] >> p.rshift] + rank[j]] = ((uint32_t)node[j] & mask) << kRsLocal | at;
  }
  __syncthreads();
  uint32_t *words = p.words + ((size_t)blockIdx.x << p.log);
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int pos = (int)threadIdx.x + j * kRsBlock;
    if (pos < total) words[pos] = s_stage[pos];
  }
  if (!in_order) return;
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int64_t be = lo + threadIdx.x + (int64_t)j * kRsBlock;
    const bool live = be < p.n;
    const int32_t prev = before(j);
    const int64_t top = live ? (int64_t)node[j] : -1, bot = live ? (be == 0 ? 0 : (int64_t)prev + 1) : 0;
    if (live && p.perm_row != nullptr) p.perm_row[be] = node[j];
    gap_rows(p.ptr, bot, top, be, s_gaps);
    if (lo + TILE >= p.n) gap_rows(p.ptr, top + 1, live && be == p.n - 1 ? p.rows : top, p.n, s_gaps);
  }
  __syncthreads();
  gap_rows_finish(p.ptr, s_gaps);
}

// Where the entries of a bucket lie: in every tile a run of its words. Places of the bucket are numbered through all tiles.
template <int BLOCK> struct RsRuns {
  uint32_t start[BLOCK];                      // of a round of BLOCK tiles, the runs that are not empty: word - place
  uint32_t bits[kRsSortPer * BLOCK / 32];     // places at which a run begins,
  uint32_t pre[kRsSortPer * BLOCK / 32];      // their number before every 32 places
  uint32_t wave[3][BLOCK / kWave];
  uint32_t first;                             // number of the first run that holds one of the places asked for
};

// the offsets of bucket `bucket` in tile t: first word, number of words
__device__ __forceinline__ void rs_run_of(const RowSortArgs &p, int bucket, int t, uint32_t &a, uint32_t &c) {
  a = c = 0;
  if (t < p.tiles) {
    uint32_t two;  // (one load, whatever its alignment: every tile's offsets lie in a line of their own)
    __builtin_memcpy(&two, p.off + (size_t)t * p.pitch + bucket, 4);
    a = two & 0xFFFFu;
    c = (two >> 16) - a;
  }
}

// at[j]: the word at place skip + j * BLOCK + threadIdx.x of the bucket, for places below skip + cnt (else 0). The tiles before
// t_first hold `done` of the bucket's entries, none of those asked for; a0, c0: rs_run_of of tile t_first + threadIdx.x. A place finds its run by counting the run starts before it (a search over the runs'
// starts takes nine dependent LDS reads an entry).
template <int BLOCK>
__device__ __forceinline__ void rs_places(const RowSortArgs &p, int bucket, uint32_t skip, int cnt, uint32_t a0, uint32_t c0,
                                          RsRuns<BLOCK> &s, uint32_t (&at)[kRsSortPer], int t_first = 0, uint32_t done = 0) {
  constexpr int WORDS = kRsSortPer * BLOCK / 32;
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
#pragma unroll
  for (int j = 0; j < kRsSortPer; ++j) at[j] = 0;
  for (int t0 = t_first; t0 < p.tiles && done < skip + (uint32_t)cnt; t0 += BLOCK) {
    uint32_t a = a0, c = c0;
    if (t0 > t_first) rs_run_of(p, bucket, t0 + tid, a, c);
    const uint32_t incl = (uint32_t)wave_inclusive_sum((int32_t)c);
    const uint64_t some = __ballot(c > 0);
    uint32_t ord = __builtin_amdgcn_mbcnt_hi((uint32_t)(some >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)some, 0u));
    if (lane == kWave - 1) {
      s.wave[0][wave] = incl;
      s.wave[1][wave] = (uint32_t)__popcll(some);
    }
    if (tid < WORDS) s.bits[tid] = 0;
    __syncthreads();
    uint32_t total, runs;
    const uint32_t before = incl - c + rs_waves_before<BLOCK>(s.wave[0], total);
    ord += rs_waves_before<BLOCK>(s.wave[1], runs);
    if (done + total > skip) {  // (the same for the workgroup)
      const int32_t from = (int32_t)(done + before - skip);  // the run's first place among those asked for
      const int32_t head = from > 0 ? from : 0, end = from + (int32_t)c < cnt ? from + (int32_t)c : cnt;
      if (c > 0 && head < end) {
        s.start[ord] = ((uint32_t)(t0 + tid) << p.log) + a - (uint32_t)from;
        atomicOr(&s.bits[head >> 5], 1u << (head & 31));
        if (from <= 0 || before == 0) s.first = ord;
      }
      __syncthreads();
      const uint32_t pc = tid < WORDS ? (uint32_t)__popc(s.bits[tid]) : 0u;
      const uint32_t pi = (uint32_t)wave_inclusive_sum((int32_t)pc);
      if (lane == kWave - 1) s.wave[2][wave] = pi;
      __syncthreads();
      const uint32_t pb = pi - pc + s.first + rs_waves_before<BLOCK>(s.wave[2], runs);
      if (tid < WORDS) s.pre[tid] = pb;
      __syncthreads();
      const int lo = (int32_t)(done - skip) > 0 ? (int32_t)(done - skip) : 0;
      const int hi = (int32_t)(done + total - skip) < cnt ? (int32_t)(done + total - skip) : cnt;
      const uint32_t upto = 0xFFFFFFFFu >> (31 - (tid & 31));
#pragma unroll
      for (int j = 0; j < kRsSortPer; ++j) {
        const int i = j * BLOCK + tid, w = j * (BLOCK / 32) + (tid >> 5);
        const uint32_t run = s.pre[w] + (uint32_t)__popc(s.bits[w] & upto) - 1;
        if (i >= lo && i < hi) at[j] = s.start[run] + (uint32_t)i;
        if ((j & 3) == 3) __builtin_amdgcn_sched_barrier(0);
      }
    }
    __syncthreads();
    done += total;
  }
}

// The words at[] on the way together, then the rank of every entry in its row: entry[j] and row << CAP_LOG | rank.
template <int BLOCK, int CAP_LOG>
__device__ __forceinline__ void rs_rank(const RowSortArgs &p, const uint32_t (&at)[kRsSortPer], int cnt, uint32_t *s_hist,
                                        uint32_t (&entry)[kRsSortPer], uint32_t (&row_rank)[kRsSortPer]) {
  const uint32_t tile = (uint32_t)(p.per * kRsBlock);
#pragma unroll
  for (int j = 0; j < kRsSortPer; ++j) {
    entry[j] = p.words[at[j]];
    if ((j & 3) == 3) __builtin_amdgcn_sched_barrier(0);  // (the addresses of all 16 at once take 32 registers)
  }
  int32_t hot = -1;
#pragma unroll
  for (int j = 0; j < kRsSortPer; ++j) {
    const uint32_t r = entry[j] >> kRsLocal;
    row_rank[j] = r << CAP_LOG;
    if (j * BLOCK < cnt)  // (the same for the workgroup)
      row_rank[j] |= rs_take(s_hist, j * BLOCK + (int)threadIdx.x < cnt ? (int32_t)r : -1, hot);
    // (from kRsLarge entries on a tile fills its 1 << kRsLocal words)
    if (BLOCK == 1024)
      entry[j] = (at[j] & ~((1u << kRsLocal) - 1)) | (entry[j] & ((1u << kRsLocal) - 1));
    else
      entry[j] = __umul24(at[j] >> p.log, tile) + (entry[j] & ((1u << kRsLocal) - 1));
    if ((j & 3) == 3) __builtin_amdgcn_sched_barrier(0);
  }
}

// row0 + the row in the bucket of every entry, in the order of s_hist, to out: through the stage, for stores in whole lines
template <int BLOCK, int CAP_LOG, typename U>
__device__ __forceinline__ void rs_store_rows(const uint32_t (&row_rank)[kRsSortPer], int cnt, const uint32_t *s_hist,
                                              uint32_t *s_stage, int32_t row0, U *out) {
  __syncthreads();
#pragma unroll
  for (int j = 0; j < kRsSortPer; ++j) {
    const uint32_t rr = row_rank[j];
    if (j * BLOCK + (int)threadIdx.x < cnt)
      s_stage[s_hist[rr >> CAP_LOG] + (rr & ((1u << CAP_LOG) - 1))] = (uint32_t)row0 + (rr >> CAP_LOG);
    if ((j & 3) == 3) __builtin_amdgcn_sched_barrier(0);
  }
  __syncthreads();
#pragma unroll 4
  for (uint32_t i = threadIdx.x; i < (uint32_t)cnt; i += BLOCK) out[i] = (U)s_stage[i];
}

template <int BLOCK>
static __global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(BLOCK == 512 ? 6 : 8)))
void rs_sort_kernel(RowSortArgs p) {
  constexpr int CAP = kRsSortPer * BLOCK, CAP_LOG = BLOCK == 512 ? 13 : 14;
  extern __shared__ uint32_t s_hist[];  // [rows per bucket]
  __shared__ uint32_t s_stage[CAP];
  __shared__ RsRuns<BLOCK> s_runs;
  __shared__ uint32_t s_wave[BLOCK / kWave];
  __shared__ uint32_t s_round[kRsMaxRounds];  // entries of the bucket in every BLOCK tiles, if there are more than that
  static_assert(CAP * 4 + sizeof(RsRuns<BLOCK>) + 4 * kRsMaxRounds + 256 + (4 << kRsMaxShift) <= 160 * 1024, "a workgroup's LDS: 160 KB");
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
  if (p.gate != nullptr && *p.gate == 0) return;
  const bool unsorted = p.state[3] == (int32_t)p.nonce;
  if (blockIdx.x == 0 && tid == 0) p.state[0] = unsorted ? 1 : 0;
  if (!unsorted) {
    if (p.identity)
      for (int64_t i = (int64_t)blockIdx.x * BLOCK + tid; i < p.n; i += (int64_t)gridDim.x * BLOCK) p.perm[i] = (int32_t)i;
    return;
  }
  // neighbouring buckets, whose runs share lines, on one of the eight dies (workgroups go to them in turn)
  const int per_die = (p.nb + 7) / 8, bucket = (int)(blockIdx.x & 7) * per_die + (int)(blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per_die || bucket >= p.nb) return;
  // The bucket's first place in perm is the number of entries in buckets before it: the sum of its offsets in all tiles.
  uint32_t a0, c0, base = 0, cnt_u = 0;
  rs_run_of(p, bucket, tid, a0, c0);
  {
    uint32_t a = a0, c = c0;
    const int rounds = (p.tiles + BLOCK - 1) / BLOCK;
    if (rounds > 1) {
      if (tid < kRsMaxRounds) s_round[tid] = 0;
      __syncthreads();
      for (int k = 0; k < rounds; ++k) {
        uint32_t at = 0, ct = c0;
        if (k > 0) rs_run_of(p, bucket, tid + k * BLOCK, at, ct);
        const uint32_t sum = (uint32_t)wave_inclusive_sum((int32_t)ct);
        if (lane == kWave - 1) atomicAdd(&s_round[k], sum);
        if (k > 0) {
          a += at;
          c += ct;
        }
      }
    }
    const int32_t ia = wave_inclusive_sum((int32_t)a), ic = wave_inclusive_sum((int32_t)c);
    if (lane == kWave - 1) {
      s_runs.wave[0][wave] = (uint32_t)ia;
      s_runs.wave[1][wave] = (uint32_t)ic;
    }
    const int R = 1 << p.rshift;
    for (int i = tid; i < R; i += BLOCK) s_hist[i] = 0;
    __syncthreads();
#pragma unroll 4
    for (int w = 0; w < BLOCK / kWave; ++w) {
      base += s_runs.wave[0][w];
      cnt_u += s_runs.wave[1][w];
    }
    __syncthreads();
  }
  if (bucket == p.nb - 1 && tid == 0) p.ptr[p.rows] = (int64_t)base + cnt_u;
  const int R = 1 << p.rshift;
  if (cnt_u > (uint32_t)CAP) {
    // for the passes behind: the bucket's chunks, its counters cleared
    const uint32_t m = (cnt_u + CAP - 1) / CAP;
    if (tid == 0) {
      const uint32_t first = (uint32_t)atomicAdd(&p.state[1], (int32_t)m), big = (uint32_t)atomicAdd(&p.state[2], 1);
      s_runs.wave[0][0] = first;
      s_runs.wave[1][0] = big;
      uint32_t *rec = p.big + 4 * (size_t)big;
      rec[0] = (uint32_t)bucket;
      rec[1] = base;
      rec[2] = cnt_u;
      rec[3] = first;
      p.arrived[big] = 0;
    }
    __syncthreads();
    const uint32_t first = s_runs.wave[0][0], big = s_runs.wave[1][0];
    for (uint32_t c = tid; c < m; c += BLOCK) {
      p.chunk_big[first + c] = (int32_t)big;
      uint32_t before = 0;
      int k = 0;
      if (p.tiles > BLOCK)
        while (before + s_round[k] <= c * CAP) before += s_round[k++];  // (their sum is more than c * CAP)
      p.chunk_at[2 * (first + c)] = (uint32_t)(k * BLOCK);
      p.chunk_at[2 * (first + c) + 1] = before;
    }
    for (int i = tid; i < R; i += BLOCK) p.row_cnt[((int64_t)big << p.rshift) + i] = 0;
    return;
  }
  const int cnt = (int)cnt_u;
  uint32_t at[kRsSortPer], entry[kRsSortPer], row_rank[kRsSortPer];
  rs_places<BLOCK>(p, bucket, 0, cnt, a0, c0, s_runs, at);
  rs_rank<BLOCK, CAP_LOG>(p, at, cnt, s_hist, entry, row_rank);
  __syncthreads();
  const int64_t row0 = (int64_t)bucket << p.rshift;
  const int n_rows = p.rows - row0 < R ? (int)(p.rows - row0) : R;
  rs_scan_lds<BLOCK>(s_hist, R, s_wave);
  for (int i = tid; i < n_rows; i += BLOCK) p.ptr[row0 + i] = (int64_t)(base + s_hist[i]);
#pragma unroll
  for (int j = 0; j < kRsSortPer; ++j) {
    const uint32_t rr = row_rank[j];
    if (j * BLOCK + tid < cnt) s_stage[s_hist[rr >> CAP_LOG] + (rr & (CAP - 1))] = entry[j];
    if ((j & 3) == 3) __builtin_amdgcn_sched_barrier(0);
  }
  __syncthreads();
  int32_t *perm = p.perm + base;
#pragma unroll 4
  for (uint32_t i = tid; i < (uint32_t)cnt; i += BLOCK) perm[i] = (int32_t)s_stage[i];
  if (p.perm_row != nullptr)
    rs_store_rows<BLOCK, CAP_LOG>(row_rank, cnt, s_hist, s_stage, (int32_t)row0, p.perm_row + base);
}

// The chunks of large buckets. A chunk's row counts go to the bucket's; what they found there is the chunk's offset inside
// every row. Its entries are left in order of their rows.
template <int BLOCK>
static __global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(BLOCK == 512 ? 6 : 8)))
void rs_chunk_kernel(RowSortArgs p) {
  constexpr int CAP = kRsSortPer * BLOCK, CAP_LOG = BLOCK == 512 ? 13 : 14;
  extern __shared__ uint32_t s_hist[];  // [rows per bucket]
  __shared__ uint32_t s_stage[CAP];
  __shared__ RsRuns<BLOCK> s_runs;
  __shared__ uint32_t s_wave[BLOCK / kWave];
  __shared__ int s_last;
  const int tid = threadIdx.x, chunk = (int)blockIdx.x;
  if (p.gate != nullptr && *p.gate == 0) return;
  if (p.state[0] == 0 || chunk >= p.state[1]) return;
  const int big = p.chunk_big[chunk];
  const uint32_t *rec = p.big + 4 * (size_t)big;
  const int bucket = (int)rec[0];
  const uint32_t base = rec[1], total = rec[2], skip = (uint32_t)(chunk - (int)rec[3]) * CAP;
  const int cnt = total - skip < (uint32_t)CAP ? (int)(total - skip) : CAP;
  const int R = 1 << p.rshift;
  for (int i = tid; i < R; i += BLOCK) s_hist[i] = 0;
  uint32_t a0, c0;
  const int t_first = (int)p.chunk_at[2 * chunk];
  rs_run_of(p, bucket, t_first + tid, a0, c0);
  uint32_t at[kRsSortPer], entry[kRsSortPer], row_rank[kRsSortPer];
  rs_places<BLOCK>(p, bucket, skip, cnt, a0, c0, s_runs, at, t_first, p.chunk_at[2 * chunk + 1]);
  rs_rank<BLOCK, CAP_LOG>(p, at, cnt, s_hist, entry, row_rank);
  __syncthreads();
  const int64_t row0 = (int64_t)bucket << p.rshift;
  const int n_rows = p.rows - row0 < R ? (int)(p.rows - row0) : R;
  rs_scan_lds<BLOCK>(s_hist, R, s_wave);
  uint32_t sink = 0;
  for (int i = tid; i < R; i += BLOCK) {
    const uint32_t from = s_hist[i], h = (i + 1 < R ? s_hist[i + 1] : (uint32_t)cnt) - from;
    if (h == 0) continue;
    const uint32_t before = atomicAdd(&p.row_cnt[((int64_t)big << p.rshift) + i], h);
    p.chunk_off[((int64_t)chunk << p.rshift) + i] = before - from;
    sink |= before;
  }
#pragma unroll
  for (int j = 0; j < kRsSortPer; ++j) {
    const uint32_t rr = row_rank[j];
    if (j * BLOCK + tid < cnt) s_stage[s_hist[rr >> CAP_LOG] + (rr & (CAP - 1))] = entry[j];
    if ((j & 3) == 3) __builtin_amdgcn_sched_barrier(0);
  }
  asm volatile("" ::"v"(sink) : "memory");  // the returns are in: the counts are in memory
  __syncthreads();
  if (tid == 0) {
    const uint32_t m = (total + CAP - 1) / CAP;
    s_last = atomicAdd(&p.arrived[big], 1u) == m - 1 ? 1 : 0;
  }
#pragma unroll 8
  for (int i = tid; i < cnt; i += BLOCK) p.by_row[base + skip + (uint32_t)i] = s_stage[i];
  rs_store_rows<BLOCK, CAP_LOG>(row_rank, cnt, s_hist, s_stage, 0, p.by_row_row + base + skip);
  __syncthreads();
  if (!s_last) return;
  // the chunk that arrives last: the bucket's row pointers
  for (int i = tid; i < R; i += BLOCK) s_hist[i] = atomicOr(&p.row_cnt[((int64_t)big << p.rshift) + i], 0u);
  __syncthreads();
  rs_scan_lds<BLOCK>(s_hist, R, s_wave);
  for (int i = tid; i < n_rows; i += BLOCK) p.ptr[row0 + i] = (int64_t)(base + s_hist[i]);
}

// the chunks of large buckets, each in order of its rows: every entry to its place among its row's
constexpr int kRsPiece = 8;  // entries per lane; a chunk is 4 or 8 pieces
static __global__ __launch_bounds__(kBlock) void rs_place_chunks_kernel(RowSortArgs p) {
  if ((p.gate != nullptr && *p.gate == 0) || p.state[0] == 0) return;
  const int pieces = p.cap / (kRsPiece * kBlock), n = p.state[1] * pieces;
  for (int q = (int)blockIdx.x; q < n; q += (int)gridDim.x) {
    const int chunk = q / pieces, i0 = (q - chunk * pieces) * (kRsPiece * kBlock) + (int)threadIdx.x;
    const uint32_t *rec = p.big + 4 * (size_t)p.chunk_big[chunk];
    const uint32_t skip = (uint32_t)(chunk - (int)rec[3]) * (uint32_t)p.cap, left = rec[2] - skip;
    const int cnt = left < (uint32_t)p.cap ? (int)left : p.cap;
    const int64_t row0 = (int64_t)rec[0] << p.rshift;
    const int64_t *ptr = p.ptr + row0;
    const uint32_t *off = p.chunk_off + ((int64_t)chunk << p.rshift);
    const uint32_t *entries = p.by_row + rec[1] + skip;
    const uint16_t *rows = p.by_row_row + rec[1] + skip;
    uint32_t e[kRsPiece], r[kRsPiece], to[kRsPiece];
#pragma unroll
    for (int j = 0; j < kRsPiece; ++j) {  // (past the end: the last entry again)
      const int i = i0 + j * kBlock < cnt ? i0 + j * kBlock : cnt - 1;
      e[j] = entries[i];
      r[j] = rows[i];
    }
#pragma unroll
    for (int j = 0; j < kRsPiece; ++j) to[j] = (uint32_t)ptr[r[j]] + off[r[j]] + (uint32_t)(i0 + j * kBlock);
#pragma unroll
    for (int j = 0; j < kRsPiece; ++j) {
      if (i0 + j * kBlock >= cnt) continue;
      p.perm[to[j]] = (int32_t)e[j];
      if (p.perm_row != nullptr) p.perm_row[to[j]] = (int32_t)row0 + (int32_t)r[j];
    }
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
// 282 k rows 368 us, of which the scatter 260; this kernel 173, 4.7 TB/s in rows of 256 bytes in no order.)
// U: bits of an element. A worker takes 4 neighbouring places.
template <typename U, int VEC>
static __global__ __launch_bounds__(kBlock) void rs_arg_rows_kernel(RowSortArgs p, const U *__restrict__ grad,
                                                                    const int64_t *__restrict__ arg,
                                                                    U *__restrict__ grad_in, int64_t K, int G) {
  constexpr int Q = 4;
  typedef int32_t i4 __attribute__((ext_vector_type(4)));
  const int W = kBlock / G, w = threadIdx.x / G, lg = threadIdx.x - w * G;
  const int64_t col = ((int64_t)blockIdx.y * G + lg) * VEC;
  const int64_t n = p.ptr[p.rows];  // entries inside [0, N)
  const int64_t p0 = ((int64_t)blockIdx.x * W + w) * Q;
  if (col >= K || p0 >= n) return;
  const int cnt = n - p0 < Q ? (int)(n - p0) : Q;
  i4 row = *reinterpret_cast<const i4 *>(p.perm_row + p0);  // (the arrays end on whole 256 bytes)
  i4 e = {(int)p0, (int)p0 + 1, (int)p0 + 2, (int)p0 + 3};
  if (p.state[0] != 0) e = *reinterpret_cast<const i4 *>(p.perm + p0);
#pragma unroll
  for (int q = 1; q < Q; ++q) row[q] = q < cnt ? row[q] : row[0];
  // neighbouring places mostly share a row or two: those of the first and the last are on the way together, a third one's behind a
  // condition (2.3 M x 64 floats onto 282 k rows 173 us; with a row's loads for every place 207: twice as much from the vector L1)
  Vec<int64_t, VEC> a[2];
  Vec<U, VEC> g[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int64_t at = (int64_t)row[i == 0 ? 0 : Q - 1] * K + col;
    a[i] = load_vec<int64_t, VEC>(arg + at);
    g[i] = load_vec<U, VEC>(grad + at);
  }
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    if (q >= cnt) continue;
    if (q > 0 && row[q] != row[0]) {
      if (row[q] == row[Q - 1]) {
        a[0] = a[1];
        g[0] = g[1];
      } else {
        a[0] = load_vec<int64_t, VEC>(arg + (int64_t)row[q] * K + col);
        g[0] = load_vec<U, VEC>(grad + (int64_t)row[q] * K + col);
      }
      row[0] = row[q];
    }
    const uint32_t pos = p.B > 1 ? (uint32_t)e[q] % (uint32_t)p.E : (uint32_t)e[q];  // inside its batch
    Vec<U, VEC> o;
#pragma unroll
    for (int v = 0; v < VEC; ++v) o.v[v] = (uint32_t)a[0].v[v] == pos ? g[0].v[v] : (U)0;  // (positions fit 31 bits)
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

template <int FLAT> inline void launch_rs_place(const RowSortArgs &p, hipStream_t stream) {
  const dim3 grid((unsigned)p.tiles);
  const size_t lds = (size_t)p.nb * 4;
  switch (p.per) {
  case 1: hipLaunchKernelGGL((rs_place_kernel<FLAT, 1>), grid, dim3(kRsBlock), lds, stream, p); break;
  case 2: hipLaunchKernelGGL((rs_place_kernel<FLAT, 2>), grid, dim3(kRsBlock), lds, stream, p); break;
  case 3: hipLaunchKernelGGL((rs_place_kernel<FLAT, 3>), grid, dim3(kRsBlock), lds, stream, p); break;
  case 4: hipLaunchKernelGGL((rs_place_kernel<FLAT, 4>), grid, dim3(kRsBlock), lds, stream, p); break;
  case 5: hipLaunchKernelGGL((rs_place_kernel<FLAT, 5>), grid, dim3(kRsBlock), lds, stream, p); break;
  case 6: hipLaunchKernelGGL((rs_place_kernel<FLAT, 6>), grid, dim3(kRsBlock), lds, stream, p); break;
  case 7: hipLaunchKernelGGL((rs_place_kernel<FLAT, 7>), grid, dim3(kRsBlock), lds, stream, p); break;
  default: hipLaunchKernelGGL((rs_place_kernel<FLAT, 8>), grid, dim3(kRsBlock), lds, stream, p); break;
  }
}
template <int BLOCK> inline void launch_rs_sort(const RowSortArgs &p, hipStream_t stream) {
  const size_t lds = (size_t)4 << p.rshift;
  hipLaunchKernelGGL(rs_sort_kernel<BLOCK>, dim3((unsigned)((p.nb + 7) / 8 * 8)), dim3(BLOCK), lds, stream, p);
  if (p.max_chunks == 0) return;
  hipLaunchKernelGGL(rs_chunk_kernel<BLOCK>, dim3((unsigned)p.max_chunks), dim3(BLOCK), lds, stream, p);
  const int64_t pieces = (int64_t)p.max_chunks * (p.cap / (kRsPiece * kBlock));
  hipLaunchKernelGGL(rs_place_chunks_kernel, dim3((unsigned)(pieces < 2048 ? pieces : 2048)), dim3(kBlock), 0, stream, p);
}

// nonce: tag of the call (any value; a repeated one only costs an index in order its short way)
inline int launch_row_sort(const RowSortArgs &args, const int64_t *index, int64_t sb, int64_t se, bool identity,
                           uint64_t nonce, hipStream_t stream, const int *gate = nullptr) {
  RowSortArgs p = args;
  p.gate = gate;
  p.identity = identity ? 1 : 0;
  p.index = index;
  p.sb = sb;
  p.se = se;
  p.flat = p.B == 1 && se == 1;
  p.nonce = (uint32_t)nonce | 1u;
  if (p.flat)
    launch_rs_place<1>(p, stream);
  else
    launch_rs_place<0>(p, stream);
  if (p.cap == kRsSortPer * 512)
    launch_rs_sort<512>(p, stream);
  else
    launch_rs_sort<1024>(p, stream);
  return hipGetLastError() == hipSuccess ? TS_OK : TS_ERR_LAUNCH;
}

}  // namespace ts
