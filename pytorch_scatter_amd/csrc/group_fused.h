// Softmax / log-softmax over groups in one pass, forward and backward, for an index that is in order
// (included by group_softmax.h).
//
// With a sorted index a group is a run of neighbouring entries. A workgroup stages a tile of entries in LDS
// (16-byte coalesced loads), finds the runs from the index, and finishes every run that lies inside the tile
// there: maximum, sum of exponentials and result all come from LDS, so src is read once and out written once
// (composite/softmax.py:8-59 makes two scatters, two gathers and four elementwise passes of it). A run that
// crosses a tile border leaves a partial per tile (maximum as a key, sum relative to that maximum); a second
// kernel puts the partials of a run together (sums rescaled by exp(m_tile - m_run)) and finishes those entries
// from src. Every tile checks the order of its part of the index; one descent anywhere sets a flag, and the
// caller's three-pass kernels, gated on that flag, then overwrite the result. No atomics on data: the result
// does not depend on scheduling.
//
// ORDERED (forward): an index in any order whose entries were sorted by group first (row_sort.h); the rows that group_rows.h, which
// holds them in registers, does not do better (16-bit elements, groups of 65 to 128 entries). The same tiles over the sorted
// entries: the rows of a tile are gathered through perm and the results go back the same way, so src is still read once
// and out written once, and no launch depends on a verdict. A tile takes the groups that begin in its window of three quarters
// of what it holds; the row pointers tell which groups are too long for that, and only those leave partials, put together once
// per group by a launch of their own. Rows wider than a tile holds are taken in column slices. Sums are held in double. What
// bounds it: the chain of a tile (row pointers, perm, rows, four passes over LDS) at four workgroups per CU; 1 M x 64 floats
// 174 us for 512 MB (2.9 TB/s).
//
//   forward   m = run maximum (entries beat lowest(), NaN never wins, no winner: 0), e = exp(src - m),
//             s = sum e;  softmax e / s,  log-softmax (src - m) - log(s + eps)
//   backward  softmax: y * (g - sum y * g);  log-softmax: g - exp(y) * sum g
#pragma once

namespace ts {

constexpr int kFusedMaxTile = 2048;   // entries per tile at most (run starts are 16-bit words with a flag bit)
constexpr int kFusedShortRun = 12;    // runs of up to this many entries inside a tile: one lane per (run, columns)
constexpr int kFusedGroup = 8;        // longer ones: eight lanes, and a wavefront from kFusedGroup * kFusedShortRun entries on
constexpr int kFusedRowBytes = 128;   // widest row the tiles are built for
constexpr int kFusedPer = kFusedMaxTile / kBlock;
constexpr int kFusedVecs = 8;          // 16-byte units of a tile (forward) or of its two tiles (backward) per lane: 32 KB
constexpr int kFusedFragBlock = 128;  // second kernel: one wavefront for the run that enters a tile, one for the run that leaves

struct FusedArgs {
  int te;            // entries per tile: kBlock * epl
  int epl;           // neighbouring entries per lane when the runs are found
  int G;             // second kernel: lanes per partial (power of two >= min(K, 64))
  int tile_vecs;     // 16-byte units of LDS per staged tile
  int short_run;     // runs of more entries than this inside a tile take eight lanes,
  int long_run;      // of more than this a wavefront
  int64_t nt;        // tiles per batch
  int32_t *meta;     // [B * nt][4]: entries of the entering run, first entry of the leaving run, entries, tile is one run that enters and leaves
  void *ckey;        // [B * nt][2][K] forward: keys of the partial maxima (entering, leaving)
  void *csum;        // [B * nt][2][K] partial sums
  int *flag;         // != 0: the index is not in order, nothing here runs (or counts)
  // ORDERED: the entries sorted by group. g describes one list: B 1, E all entries, N all groups
  const int32_t *state = nullptr;     // [0] 0: the index was in order, the order is that of memory
  const int64_t *n_sorted = nullptr;  // entries that belong to a group
  const int32_t *perm = nullptr;      // entry at every place of the order (not written when state[0] is 0)
  const int32_t *group = nullptr;     // and its group
  const int64_t *ptr = nullptr;       // [groups + 1] first place of every group
  int tw = 0;                         // window of a tile: entries from tw * tile on; te is what a tile holds
  const int64_t *index = nullptr;     // as the caller gave it, for the entries that belong to no group
  int64_t sb = 0, se = 0, E0 = 0, N0 = 0;
  int kcols = 0, slices = 1;          // columns that a workgroup takes, workgroups that share a tile of entries
  const int *gate = nullptr;          // reads 0: these launches return at once (null: they run)
  uint32_t inv_units = 0, inv_last = 0;  // 2^31 / (16-byte units of a row of a slice), rounded up; of the last slice
};

inline bool group_fused_mode(int mode) {
  return mode == GS_SOFTMAX || mode == GS_LOG_SOFTMAX || mode == GS_SOFTMAX_BWD || mode == GS_LOG_SOFTMAX_BWD;
}

// bytes of the tiles' records for a call of this shape (0: the tiles do not apply), the larger of forward and backward
inline size_t group_fused_scratch_bytes(int64_t B, int64_t E, int64_t K, int elem_bytes) {
  const int64_t row = K * elem_bytes;
  if (row > kFusedRowBytes || E < 2) return 0;
  size_t most = 0;
  for (int backward = 0; backward < 2; ++backward) {
    int64_t te = (backward ? 16384 : 32768) / row;
    int epl = 1;
    while (epl * 2 * kBlock <= te && epl * 2 <= kFusedPer) epl *= 2;
    te = (int64_t)epl * kBlock;
    const size_t tiles = (size_t)(B * ((E + te - 1) / te));
    const size_t acc = elem_bytes == 8 ? 8 : 4;
    auto up = [](size_t x) { return (x + 255) & ~(size_t)255; };
    const size_t end = up(tiles * 16) + 2 * up(tiles * 2 * K * acc);
    if (end > most) most = end;
  }
  return most;
}

// Scratch of the tiles, carved from the front of the group workspace (the three-pass kernels rewrite that
// space if they run at all); the flag sits behind the workspace of the three passes.
inline bool group_fused_plan(const GroupArgs &g, int mode, int elem_bytes, void *ws, size_t ws_three_pass,
                             bool force, FusedArgs &f) {
  if (!group_fused_mode(mode)) return false;
  const bool backward = mode == GS_SOFTMAX_BWD || mode == GS_LOG_SOFTMAX_BWD;
  const int64_t row = g.K * elem_bytes;
  if (row > kFusedRowBytes || g.E < 2) return false;
  auto al16 = [](const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
  if (!al16(g.src) || !al16(g.out) || (backward && !al16(g.grad))) return false;
  if (g.B > 1 && (g.E * row) % 16 != 0) return false;  // every batch starts on a 16-byte border
  // the launches that return at once cost more than the passes saved below these sizes (sorted index, 9 entries
  // per group, 32-byte rows: forward 31 against 34 us at 8 MB, 45 against 79 us at 32 MB; backward 63 against
  // 51 us and 52 against 58 us)
  if (!force && g.B * g.E * row < ((int64_t)(backward ? 32 : 16) << 20)) return false;
  int64_t te = (backward ? 16384 : 32768) / row;  // 32 KB of LDS per tile
  if (const char *env = getenv("TS_GROUP_TILE")) te = atoi(env);  // tuning aid
  int epl = 1;
  while (epl * 2 * kBlock <= te && epl * 2 <= kFusedPer) epl *= 2;
  te = (int64_t)epl * kBlock;
  if (te * row * (backward ? 2 : 1) > (int64_t)kFusedVecs * kBlock * 16) return false;
  f.te = (int)te;
  f.short_run = kFusedShortRun;
  f.long_run = kFusedGroup * kFusedShortRun;
  if (const char *env = getenv("TS_GROUP_SHORT_RUN")) f.short_run = atoi(env) < 4 ? 4 : atoi(env);  // tuning aids
  if (const char *env = getenv("TS_GROUP_LONG_RUN")) f.long_run = atoi(env);
  if (f.long_run < f.short_run) f.long_run = f.short_run;
  f.epl = epl;
  f.nt = (g.E + te - 1) / te;
  if (g.B * f.nt >= 0x7FFFFFFFll) return false;
  int G = 1;
  while (G < g.K && G < kWave) G *= 2;
  f.G = G;
  f.tile_vecs = (int)((te * row + 15) / 16);
  const size_t acc = elem_bytes == 8 ? 8 : 4;
  auto up = [](size_t x) { return (x + 255) & ~(size_t)255; };
  const size_t tiles = (size_t)(g.B * f.nt);
  const size_t o_key = up(tiles * 16), o_sum = o_key + up(tiles * 2 * g.K * acc);
  const size_t end = o_sum + up(tiles * 2 * g.K * acc);
  // the records of the tiles: in the caller's extra scratch when it has room, else in the front of the three passes'
  // workspace (which they rewrite if they run at all)
  // (rows of up to 64 bytes: with few, large groups every run crosses tiles, and for wider rows the three passes are then
  // ahead -- 4 M entries in 4 k groups, sorted: 8 floats 184 -> 148 us with the tiles, 64 bf16 892 -> 1058 us)
  const bool extra = g.fused_ws != nullptr && end <= g.fused_ws_bytes && row <= 64 &&
                     (reinterpret_cast<uintptr_t>(g.fused_ws) & 15) == 0;
  if (!extra && end > ws_three_pass) return false;
  char *base = extra ? static_cast<char *>(g.fused_ws) : static_cast<char *>(ws);
  f.meta = reinterpret_cast<int32_t *>(base);
  f.ckey = base + o_key;
  f.csum = base + o_sum;
  f.flag = reinterpret_cast<int *>(static_cast<char *>(ws) + ws_three_pass);  // (always behind the three passes' part)
  return true;
}

// A look at up to 1024 pairs of neighbours spread over the index: *flag = 1 (not in order, the tiles do not
// run) if at least 1/64 of them descend, else 0 (the tiles run and check every pair).
// Also clears `clear_n` 8-byte words at `clear` (the bucket totals of the passes that follow an index found out of order).
static __global__ __launch_bounds__(1024) void group_order_sample_kernel(GroupArgs g, int *flag, int force,
                                                                          unsigned long long *clear, int clear_n) {
  __shared__ int s_desc, s_pairs;
  for (int i = threadIdx.x; i < clear_n; i += 1024) clear[i] = 0;
  if (threadIdx.x == 0) { s_desc = 0; s_pairs = 0; }
  __syncthreads();
  const int64_t total = g.B * g.E;
  const int64_t step = (total - 1) / 1024 + 1;
  const int64_t be = (int64_t)threadIdx.x * step;
  if (be + 1 < total) {
    const int64_t b = be / g.E, e = be - b * g.E;
    if (e + 1 < g.E) {
      const int64_t *idx = g.index + b * g.sb;
      atomicAdd(&s_pairs, 1);
      if (idx[(e + 1) * g.se] < idx[e * g.se]) atomicAdd(&s_desc, 1);
    }
  }
  __syncthreads();
  if (threadIdx.x == 0) *flag = (!force && s_desc * 64 >= s_pairs && s_desc > 0) ? 1 : 0;
}

// the type of a run's sum
template <typename T, bool ORDERED> struct FusedSum { typedef typename Acc<T>::type type; };
template <typename T> struct FusedSum<T, true> { typedef double type; };

// combination of two partials of a run, a before b: maximum as a key, sum relative to that maximum.
// A partial in which nothing beat lowest() (key == empty) was summed relative to 0 and holds 0 or NaN: taken as is.
template <typename T, typename S>
__device__ __forceinline__ void fused_absorb(typename OrdKey<typename Acc<T>::type>::bits &ka, S &sa,
                                             typename OrdKey<typename Acc<T>::type>::bits kb, S sb) {
  typedef typename Acc<T>::type F;
  typedef typename OrdKey<F>::bits KB;
  const KB empty = group_empty_key<T>();
  if (kb > ka) {
    const F fac = ka == empty ? (F)1 : exp_acc(OrdKey<F>::dec(ka) - OrdKey<F>::dec(kb));
    sa = sa * (S)fac + sb;
    ka = kb;
  } else {
    const F fac = (kb == empty || kb == ka) ? (F)1 : exp_acc(OrdKey<F>::dec(kb) - OrdKey<F>::dec(ka));
    sa = sa + sb * (S)fac;
  }
}

__device__ __forceinline__ float fast_rcp(float v) { return __builtin_amdgcn_rcpf(v); }
__device__ __forceinline__ double fast_rcp(double v) { return 1.0 / v; }

// Which entries of the tile begin a run, and whether that run's index lies outside [0, N). The index is loaded
// coalesced (lane tid takes entries tid, tid + 256, ...: with one value per entry the index is two thirds of the
// bytes); an entry's predecessor comes from the neighbouring lane, for the first lane of a wavefront from memory.
// The flags go through LDS (a byte per entry) so that afterwards every lane holds those of its EPL neighbouring
// entries e0 .. e0 + EPL - 1 as bit masks. All index loads are issued before `between` runs (the caller's stores
// of the staged tile, which wait for the tile's loads). Ends with the workgroup in step (barrier).
template <int EPL, typename I, typename Between>
__device__ __forceinline__ void fused_find_runs(const I *idx, int64_t se, int64_t j0, int tid, int ne, int64_t E,
                                                int64_t N, uint8_t *s_flag, Between &&between, uint32_t &headmask,
                                                uint32_t &badmask, bool &descent, bool &enters, bool &leaves) {
  const int lane = tid & (kWave - 1);
  I id[EPL], edge[EPL];
#pragma unroll
  for (int q = 0; q < EPL; ++q) {
    const int e = tid + q * kBlock;
    id[q] = e < ne ? idx[(j0 + e) * se] : 0;
  }
#pragma unroll
  for (int q = 0; q < EPL; ++q) {
    const int e = tid + q * kBlock;
    edge[q] = (lane == 0 && e < ne && j0 + e > 0) ? idx[(j0 + e - 1) * se] : 0;
  }
  const int e_last = ne - 1;
  const bool owns_last = (e_last & (kBlock - 1)) == tid;
  I next = 0;
  const bool have_next = owns_last && j0 + ne < E;
  if (have_next) next = idx[(j0 + ne) * se];
  between();
#pragma unroll
  for (int q = 0; q < EPL; ++q) {
    const int e = tid + q * kBlock;
    I up;  // by every lane, lane 0 included: its value is what lane 1 reads
    if constexpr (sizeof(I) == 8)
      up = lane_up1_64(id[q]);
    else
      up = lane_up1(id[q]);
    const I prev = lane == 0 ? edge[q] : up;
    if (e < ne) {
      const bool have_prev = j0 + e > 0;
      const bool head = e == 0 || id[q] != prev;
      const bool bad = head && (id[q] < 0 || id[q] >= N);
      if (have_prev && id[q] < prev) descent = true;
      if (e == 0 && have_prev && id[q] == prev) enters = true;
      if (e == e_last && have_next && next == id[q]) leaves = true;
      s_flag[e] = (uint8_t)((head ? 1 : 0) | (bad ? 2 : 0));
    }
  }
  __syncthreads();
  const int e0 = tid * EPL;
#pragma unroll
  for (int i = 0; i < EPL; ++i) {
    if (e0 + i < ne) {
      const uint32_t fl = s_flag[e0 + i];
      headmask |= (fl & 1u) << i;
      badmask |= (fl >> 1 & 1u) << i;
    }
  }
}

// the entries from j0 on that belong to no group: zeros in columns [k_first, k_first + K)
template <typename T>
__device__ __forceinline__ void fused_zero_outside(const GroupArgs &g, const FusedArgs &f, int64_t j0, int k_first, int K) {
  for (int64_t be = j0 + threadIdx.x / kWave; be < g.E && be < j0 + f.tw; be += kBlock / kWave) {
    int64_t b, e;
    split_edge(be, g.E / f.E0, f.E0, b, e);
    const int64_t at = f.index[b * f.sb + e * f.se];
    if (at >= 0 && at < f.N0) continue;
    for (int k = threadIdx.x & (kWave - 1); k < K; k += kWave)
      static_cast<T *>(g.out)[be * g.K + k_first + k] = from_acc<T>((typename Acc<T>::type)0);
  }
}
// i / units for i < 2^15, inv = 2^31 / units rounded up
__device__ __forceinline__ int fused_unit_entry(int i, uint32_t inv) { return (int)__umulhi((uint32_t)i << 1, inv); }

// The places [a, b) of the order that tile t takes. enters / leaves: the group at a began in another tile and is too long
// for it; the group at the window's end goes on in the next tile.
struct FusedSpan {
  int64_t a, b;
  bool enters, leaves;
};
__device__ __forceinline__ FusedSpan fused_span(const FusedArgs &f, int64_t t, int64_t E) {
  const int64_t w0 = t * f.tw, w1 = w0 + f.tw < E ? w0 + f.tw : E;
  const int32_t g0 = f.group[w0], g1 = f.group[w1 - 1];
  const int64_t s0 = f.ptr[g0], e0 = f.ptr[g0 + 1], s1 = f.ptr[g1], e1 = f.ptr[g1 + 1];
  auto fits = [&](int64_t s, int64_t e) { return e <= (int64_t)((uint32_t)s / (uint32_t)f.tw) * f.tw + f.te; };
  FusedSpan r;
  r.enters = s0 < w0 && !fits(s0, e0);
  r.a = s0 < w0 && !r.enters ? e0 : w0;
  r.leaves = e1 > w1 && !fits(s1, e1);
  r.b = e1 > w1 && !r.leaves ? e1 : w1;
  return r;
}

template <typename T, int CV, int MODE, bool ORDERED = false>
__global__ __launch_bounds__(kBlock, 4) void group_fused_kernel(GroupArgs g, FusedArgs f) {
  typedef typename Acc<T>::type F;
  typedef typename FusedSum<T, ORDERED>::type S;
  typedef typename OrdKey<F>::bits KB;
  typedef uint32_t u4 __attribute__((ext_vector_type(4)));
  constexpr bool kBackward = MODE == GS_SOFTMAX_BWD || MODE == GS_LOG_SOFTMAX_BWD;
  static_assert(!ORDERED || !kBackward, "the backward pass over sorted entries: group_rows.h");
  constexpr int W = kBlock / kWave;
  // [tile of src][backward: tile of grad][run starts: te + 2 16-bit words, bit 15: index outside [0, N)]
  extern __shared__ u4 s_dyn[];
  __shared__ int s_wsum[W];
  __shared__ int s_info[6];  // run enters from the tile before, run leaves into the next tile, runs for a wavefront, descent seen,
                             // runs for eight lanes, some run belongs to no group
  __shared__ uint32_t s_bad[kFusedMaxTile / 32];  // forward: entries of runs that belong to no group
  __shared__ int32_t s_long[kFusedMaxTile / 4 + 2];  // runs for eight lanes from the front, for a wavefront from the back
  if (!ORDERED && *f.flag != 0) return;
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
  if (tid < 6) s_info[tid] = 0;
  if (!ORDERED && tid < kFusedMaxTile / 32) s_bad[tid] = 0;
  __syncthreads();
  const int KR = (int)g.K;  // columns of a row in memory; of this workgroup:
  const int k_first = ORDERED ? (int)blockIdx.y * f.kcols : 0;
  const int K = ORDERED ? (KR - k_first < f.kcols ? KR - k_first : f.kcols) : KR;
  const int64_t b = ORDERED ? 0 : blockIdx.x / f.nt, t = blockIdx.x - b * f.nt;
  const int64_t E = ORDERED ? *f.n_sorted : g.E;  // (of a call that the gate stops: anything)
  const bool through = ORDERED && f.state[0] != 0;
  const bool flat = !ORDERED || (!through && f.slices == 1);  // the tile is one range of memory
  if constexpr (ORDERED) {
    if (f.gate != nullptr && *f.gate == 0) return;
    if (E != g.E) fused_zero_outside<T>(g, f, t * f.tw, k_first, K);
    if (t * f.tw >= E) return;
  }
  FusedSpan span;
  if constexpr (ORDERED) span = fused_span(f, t, E);
  const int64_t j0 = ORDERED ? span.a : t * f.te;
  const int ne = ORDERED ? (int)(span.b - j0) : (int)(E - j0 < f.te ? E - j0 : f.te);
  if (ORDERED && ne <= 0) {  // (a group that the tile before has taken ends with the window)
    if (tid < 4 && blockIdx.y == 0) f.meta[t * 4 + tid] = 0;
    return;
  }
  T *s_src = reinterpret_cast<T *>(s_dyn);
  T *s_grad = reinterpret_cast<T *>(s_dyn + f.tile_vecs);
  uint16_t *s_start = reinterpret_cast<uint16_t *>(s_dyn + (kBackward ? 2 : 1) * f.tile_vecs);

  // ---- the tile of src (and grad): whole 16-byte units (the unit behind the last entry stays inside its page),
  // every load of the tile and of the index in flight before the first one is waited for
  const int nvec = (int)(((size_t)ne * K * sizeof(T) + 15) / 16);
  const int nstage = kBackward ? 2 * f.tile_vecs : f.tile_vecs;  // unit v of the staged space: tile v / tile_vecs
  constexpr int kPer = 16 / (int)sizeof(T);
  const uint32_t inv = ORDERED ? (blockIdx.y == gridDim.y - 1 ? f.inv_last : f.inv_units) : 0;
  // ORDERED, not flat: a lane's unit q of a tile is unit tid + q * kBlock, of the row at place[q]
  constexpr int Q = kFusedVecs;
  int32_t place[ORDERED ? Q : 1];
  auto unit_at = [&](int q) {
    const int v = tid + q * kBlock, u = v < nvec ? v : nvec - 1;
    return (int64_t)place[q] * KR + k_first + (u - fused_unit_entry(u, inv) * (K / CV)) * CV;
  };
  u4 stage[kFusedVecs];
  if (flat) {
    const u4 *p0 = reinterpret_cast<const u4 *>(static_cast<const T *>(g.src) + (b * g.E + j0) * K);
    const u4 *p1 = kBackward ? reinterpret_cast<const u4 *>(static_cast<const T *>(g.grad) + (b * g.E + j0) * K) : p0;
#pragma unroll
    for (int q = 0; q < kFusedVecs; ++q) {
      const int v = tid + q * kBlock;
      const bool second = kBackward && v >= f.tile_vecs;
      const int vv = second ? v - f.tile_vecs : v;
      if (v < nstage && vv < nvec) stage[q] = __builtin_nontemporal_load((second ? p1 : p0) + vv);
    }
  } else if constexpr (ORDERED) {
    const T *p0 = static_cast<const T *>(g.src);
    static_assert(!ORDERED || CV * sizeof(T) == 16, "rows of whole 16-byte units");
    // No load behind a condition of its own (past the end: the last unit again), else the lane waits for each load of perm on
    // the spot (1 M x 64 floats in groups of three: 255 us, 174 like this; 2.3 M x 8 floats 111 / 95).
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const int v = tid + q * kBlock;
      place[q] = (int32_t)j0 + fused_unit_entry(v < nvec ? v : nvec - 1, inv);
    }
    if (through) {
#pragma unroll
      for (int q = 0; q < Q; ++q) place[q] = f.perm[place[q]];
    }
#pragma unroll
    for (int q = 0; q < Q; ++q) stage[q] = *reinterpret_cast<const u4 *>(p0 + unit_at(q));
  }

  // ---- runs: a lane looks at epl neighbouring entries
  const int64_t *idx = g.index + b * g.sb;
  const int e0 = tid * f.epl;
  uint8_t *s_flag = reinterpret_cast<uint8_t *>(s_start);  // read by all lanes before the run starts are written
  uint32_t headmask = 0, badmask = 0;
  bool descent = false, lane_enters = false, lane_leaves = false;
  auto stage_to_lds = [&]() {
    if (!flat) {
#pragma unroll
      for (int q = 0; q < Q; ++q) {
        const int v = tid + q * kBlock;
        if (v >= nvec) continue;
        s_dyn[v] = stage[q];
      }
      return;
    }
#pragma unroll
    for (int q = 0; q < kFusedVecs; ++q) {
      const int v = tid + q * kBlock;
      const int vv = (kBackward && v >= f.tile_vecs) ? v - f.tile_vecs : v;
      if (v < nstage && vv < nvec) s_dyn[v] = stage[q];
    }
  };
  auto find_runs = [&](const auto *id, int64_t se) {
    switch (f.epl) {
    case 1: fused_find_runs<1>(id, se, j0, tid, ne, E, g.N, s_flag, stage_to_lds, headmask, badmask, descent, lane_enters, lane_leaves); break;
    case 2: fused_find_runs<2>(id, se, j0, tid, ne, E, g.N, s_flag, stage_to_lds, headmask, badmask, descent, lane_enters, lane_leaves); break;
    case 4: fused_find_runs<4>(id, se, j0, tid, ne, E, g.N, s_flag, stage_to_lds, headmask, badmask, descent, lane_enters, lane_leaves); break;
    default: fused_find_runs<8>(id, se, j0, tid, ne, E, g.N, s_flag, stage_to_lds, headmask, badmask, descent, lane_enters, lane_leaves); break;
    }
  };
  if constexpr (ORDERED)
    find_runs(f.group, 1);
  else
    find_runs(idx, g.se);
  if (lane_enters) s_info[0] = 1;
  if (lane_leaves) s_info[1] = 1;
  if (badmask != 0) s_info[5] = 1;
  const int heads = __popc(headmask);
  const int incl = wave_inclusive_sum(heads);
  if (lane == kWave - 1) s_wsum[wave] = incl;
  if (__ballot(descent) != 0 && lane == 0) s_info[3] = 1;
  __syncthreads();
  int base = incl - heads, nruns = 0;
#pragma unroll
  for (int w = 0; w < W; ++w) {
    if (w < wave) base += s_wsum[w];
    nruns += s_wsum[w];
  }
#pragma unroll
  for (int i = 0; i < kFusedPer; ++i) {
    if (headmask & (1u << i)) s_start[base++] = (uint16_t)((e0 + i) | ((badmask >> i & 1u) << 15));
  }
  if (tid == 0) s_start[nruns] = (uint16_t)ne;
  __syncthreads();
  if (!ORDERED && s_info[3] != 0) {
    // not in order: whatever this launch writes is overwritten by the gated passes that follow
    if (tid == 0 && __hip_atomic_load(f.flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0) atomicOr(f.flag, 1);
    return;
  }
  const bool enters = ORDERED ? span.enters : s_info[0] != 0, leaves = ORDERED ? span.leaves : s_info[1] != 0;

  const int64_t tile = b * f.nt + t;
  KB *ckey = static_cast<KB *>(f.ckey) + tile * 2 * KR + k_first;
  S *csum = static_cast<S *>(f.csum) + tile * 2 * KR + k_first;
  const F eps = (F)g.eps;

  // The runs of the tile, CV columns at a time: one lane per (run, columns) for short runs, eight lanes or a
  // wavefront for longer ones. fn(run, first column, first entry of this lane, step): the lanes that share a run
  // meet in butterflies, so every one of them holds the run's result. `classify` sorts the longer runs into
  // the two lists first (a later pass over the same tile reuses them).
  const int kc = K / CV;
  const int kc_shift = (kc & (kc - 1)) == 0 ? __ffs(kc) - 1 : -1;  // a division per unit otherwise
  auto for_runs = [&](auto &&fn, bool classify) {
    for (int u = tid; u < nruns * kc; u += kBlock) {
      const int r = kc_shift >= 0 ? u >> kc_shift : u / kc, c = u - r * kc;
      const int len = (s_start[r + 1] & 0x7FFF) - (s_start[r] & 0x7FFF);
      if (len > f.short_run) {
        if (classify && c == 0) {
          if (len > f.long_run)
            s_long[kFusedMaxTile / 4 + 1 - atomicAdd(&s_info[2], 1)] = r;
          else
            s_long[atomicAdd(&s_info[4], 1)] = r;
        }
        continue;
      }
      fn(r, c * CV, 0, 1);
    }
    if (classify) __syncthreads();
    const int nmed = s_info[4], nlong = s_info[2];
    for (int u = tid / kFusedGroup; u < nmed * kc; u += kBlock / kFusedGroup) {
      const int q = kc_shift >= 0 ? u >> kc_shift : u / kc;
      fn(s_long[q], (u - q * kc) * CV, tid & (kFusedGroup - 1), kFusedGroup);
    }
    for (int u = wave; u < nlong * kc; u += W) {
      const int q = kc_shift >= 0 ? u >> kc_shift : u / kc;
      fn(s_long[kFusedMaxTile / 4 + 1 - q], (u - q * kc) * CV, lane, kWave);
    }
  };
  // the entries of a run that this launch finishes: all of them unless the run enters or leaves the tile
  const int w_lo = enters ? (s_start[1] & 0x7FFF) : 0;  // nruns == 1: s_start[1] == ne
  const int w_hi = leaves ? (s_start[nruns - 1] & 0x7FFF) : ne;
  T *out_t = static_cast<T *>(g.out) + (b * g.E + j0) * K;
  const int el_lo = w_lo * K, el_hi = w_hi * K;
  // ORDERED, not flat: the lane's unit q of the tile to its row
  auto store_unit = [&](int q, const u4 &unit) {
    if constexpr (ORDERED) {
      const int v = tid + q * kBlock;
      if (v * kPer >= el_lo && v * kPer < el_hi) *reinterpret_cast<u4 *>(static_cast<T *>(g.out) + unit_at(q)) = unit;
    }
  };

  if constexpr (!kBackward) {
    // Forward. The tile's values stay in the registers they were loaded into; LDS holds, element by element,
    // first the values, then the run's maximum, then exp(value - maximum), then the run's divisor (or logarithm):
    // the passes over the runs only reduce and spread (cheap, one lane per run), exp and the division run one
    // lane per element.
    const KB empty = group_empty_key<T>();
    constexpr bool kSameType = sizeof(T) == sizeof(F);
    // maximum over the entries that are no NaN (maxnum returns the other operand); a winner has to beat lowest()
    const F lowest = to_acc<T>(ElemLim<T>::lowest());
    auto run_max = [&](int r, int c0, int first, int step) {
      const int lo = s_start[r] & 0x7FFF, hi = s_start[r + 1] & 0x7FFF;
      F top[CV];
#pragma unroll
      for (int v = 0; v < CV; ++v) top[v] = -INFINITY;
      for (int e = lo + first; e < hi; e += step) {
        const Vec<T, CV> x = load_vec<T, CV>(s_src + e * K + c0);
#pragma unroll
        for (int v = 0; v < CV; ++v) top[v] = max_acc(top[v], to_acc<T>(x.v[v]));
      }
#pragma unroll
      for (int v = 0; v < CV; ++v) top[v] = group_butterfly(top[v], step, [](F p, F q) { return max_acc(p, q); });
      const bool frag_in = r == 0 && enters, frag_out = r == nruns - 1 && leaves;
      if ((frag_in || frag_out) && first == 0) {
#pragma unroll
        for (int v = 0; v < CV; ++v) ckey[(frag_in ? 0 : 1) * KR + c0 + v] = top[v] > lowest ? OrdKey<F>::enc(top[v]) : empty;
      }
      Vec<T, CV> m;
#pragma unroll
      for (int v = 0; v < CV; ++v) m.v[v] = from_acc<T>(top[v] > lowest ? top[v] : (F)0);
      for (int e = lo + first; e < hi; e += step) store_vec<T, CV>(s_src + e * K + c0, m);
    };
    auto run_sum = [&](int r, int c0, int first, int step) {
      const int lo = s_start[r] & 0x7FFF, hi = s_start[r + 1] & 0x7FFF;
      S s[CV];
#pragma unroll
      for (int v = 0; v < CV; ++v) s[v] = (S)0;
      for (int e = lo + first; e < hi; e += step) {
        const Vec<T, CV> x = load_vec<T, CV>(s_src + e * K + c0);
#pragma unroll
        for (int v = 0; v < CV; ++v) s[v] += (S)to_acc<T>(x.v[v]);
      }
#pragma unroll
      for (int v = 0; v < CV; ++v) s[v] = group_butterfly(s[v], step, [](S p, S q) { return p + q; });
      const bool frag_in = r == 0 && enters, frag_out = r == nruns - 1 && leaves;
      if (frag_in || frag_out) {
        if (first == 0) {
#pragma unroll
          for (int v = 0; v < CV; ++v) csum[(frag_in ? 0 : 1) * KR + c0 + v] = s[v];
        }
        return;
      }
      Vec<T, CV> d;
#pragma unroll
      for (int v = 0; v < CV; ++v) {
        if (MODE == GS_SOFTMAX)  // fp32 / fp64: the reciprocal, one division per run instead of one per entry
          d.v[v] = kSameType && !ORDERED ? from_acc<T>((F)1 / (F)s[v]) : from_acc<T>((F)s[v]);
        else
          d.v[v] = from_acc<T>(log_acc(round_elem<T>(round_elem<T>((F)s[v]) + eps)));
      }
      for (int e = lo + first; e < hi; e += step) store_vec<T, CV>(s_src + e * K + c0, d);
      if (!ORDERED && (s_start[r] >> 15) != 0 && c0 == 0) {  // a run that belongs to no group: its entries yield 0
        for (int e = lo + first; e < hi; e += step) atomicOr(&s_bad[e >> 5], 1u << (e & 31));
      }
    };

    for_runs(run_max, true);
    __syncthreads();
#pragma unroll
    for (int q = 0; q < kFusedVecs; ++q) {
      const int v = tid + q * kBlock;
      if (v < nvec) {
        Vec<T, kPer> x, m;
        __builtin_memcpy(&x, &stage[q], 16);
        __builtin_memcpy(&m, &s_dyn[v], 16);
#pragma unroll
        for (int i = 0; i < kPer; ++i) {
          const F z = round_elem<T>(to_acc<T>(x.v[i]) - to_acc<T>(m.v[i]));
          m.v[i] = from_acc<T>(exp_acc(z));
          x.v[i] = MODE == GS_SOFTMAX ? m.v[i] : from_acc<T>(z);
        }
        __builtin_memcpy(&s_dyn[v], &m, 16);
        __builtin_memcpy(&stage[q], &x, 16);
      }
    }
    __syncthreads();
    for_runs(run_sum, false);
    __syncthreads();
    const bool any_bad = !ORDERED && s_info[5] != 0;
#pragma unroll
    for (int q = 0; q < kFusedVecs; ++q) {
      const int v = tid + q * kBlock;
      if (v < nvec && (v + 1) * kPer > el_lo && v * kPer < el_hi) {
        Vec<T, kPer> x, d;
        __builtin_memcpy(&x, &stage[q], 16);
        __builtin_memcpy(&d, &s_dyn[v], 16);
#pragma unroll
        for (int i = 0; i < kPer; ++i) {
          F res;
          if (MODE == GS_SOFTMAX) {
            // 16-bit floats: e and the rounded sum are exact in fp32 and the quotient is rounded to 8 or 11 bits,
            // so the hardware reciprocal (1 ulp of fp32) stands in for the division
            if (ORDERED)
              res = to_acc<T>(x.v[i]) / to_acc<T>(d.v[i]);
            else
              res = to_acc<T>(x.v[i]) * (kSameType ? to_acc<T>(d.v[i]) : fast_rcp(to_acc<T>(d.v[i])));
          } else {
            F l = to_acc<T>(d.v[i]);
            asm volatile("" : "+v"(l));  // see group_finish_kernel
            res = to_acc<T>(x.v[i]) - l;
          }
          if (any_bad) {
            const int e = (v * kPer + i) / K;
            if (e < ne && (s_bad[e >> 5] >> (e & 31) & 1u) != 0) res = (F)0;
          }
          x.v[i] = from_acc<T>(res);
        }
        u4 r;
        __builtin_memcpy(&r, &x, 16);
        if (!flat) {
          store_unit(q, r);
        } else if (v * kPer >= el_lo && (v + 1) * kPer <= el_hi) {
          __builtin_nontemporal_store(r, reinterpret_cast<u4 *>(out_t) + v);
        } else {
#pragma unroll
          for (int i = 0; i < kPer; ++i) {
            if (v * kPer + i >= el_lo && v * kPer + i < el_hi) out_t[v * kPer + i] = x.v[i];
          }
        }
      }
    }
  } else {
    // Backward: the tiles of y and g in LDS, one pass over the runs that sums and finishes in place.
    auto run_bwd = [&](int r, int c0, int first, int step) {
      const int lo = s_start[r] & 0x7FFF, hi = s_start[r + 1] & 0x7FFF;
      const bool valid = (s_start[r] >> 15) == 0;
      const bool frag_in = r == 0 && enters, frag_out = r == nruns - 1 && leaves;
      S s[CV];
#pragma unroll
      for (int v = 0; v < CV; ++v) s[v] = (S)0;
      for (int e = lo + first; e < hi; e += step) {
        const Vec<T, CV> y = load_vec<T, CV>(s_src + e * K + c0);
        const Vec<T, CV> gr = load_vec<T, CV>(s_grad + e * K + c0);
#pragma unroll
        for (int v = 0; v < CV; ++v)
          s[v] += MODE == GS_SOFTMAX_BWD ? (S)(to_acc<T>(y.v[v]) * to_acc<T>(gr.v[v])) : (S)to_acc<T>(gr.v[v]);
      }
#pragma unroll
      for (int v = 0; v < CV; ++v) s[v] = group_butterfly(s[v], step, [](S p, S q) { return p + q; });
      if (frag_in || frag_out) {
        if (first == 0) {
#pragma unroll
          for (int v = 0; v < CV; ++v) csum[(frag_in ? 0 : 1) * KR + c0 + v] = s[v];
        }
        return;
      }
      for (int e = lo + first; e < hi; e += step) {
        Vec<T, CV> y = load_vec<T, CV>(s_src + e * K + c0);
        const Vec<T, CV> gr = load_vec<T, CV>(s_grad + e * K + c0);
#pragma unroll
        for (int v = 0; v < CV; ++v) {
          const F yv = to_acc<T>(y.v[v]), gv = to_acc<T>(gr.v[v]);
          const F sum = (F)s[v];
          const F res = MODE == GS_SOFTMAX_BWD ? yv * (gv - sum) : gv - exp_acc(yv) * sum;
          y.v[v] = from_acc<T>(valid ? res : (F)0);
        }
        store_vec<T, CV>(s_src + e * K + c0, y);
      }
    };
    for_runs(run_bwd, true);
    __syncthreads();
    // the finished runs leave the tile: whole 16-byte units, single elements at the two ends
    if (w_hi > w_lo) {
      const int v_lo = (el_lo + kPer - 1) / kPer, v_hi = el_hi / kPer;
      if (v_lo >= v_hi) {
        for (int i = el_lo + tid; i < el_hi; i += kBlock) out_t[i] = s_src[i];
      } else {
        u4 *q = reinterpret_cast<u4 *>(out_t);
        for (int v = v_lo + tid; v < v_hi; v += kBlock) __builtin_nontemporal_store(s_dyn[v], q + v);
        for (int i = el_lo + tid; i < v_lo * kPer; i += kBlock) out_t[i] = s_src[i];
        for (int i = v_hi * kPer + tid; i < el_hi; i += kBlock) out_t[i] = s_src[i];
      }
    }
  }
  if (tid == 0 && blockIdx.y == 0) {
    const bool one = nruns == 1 && enters && leaves;
    int32_t *meta = f.meta + tile * 4;
    const int shift = ORDERED ? (int)(j0 - t * f.tw) : 0;  // (ORDERED: places from the window's begin on)
    meta[0] = enters ? w_lo : 0;
    meta[1] = shift + (one ? ne : (leaves ? w_hi : ne));
    meta[2] = shift + ne;
    meta[3] = one ? 1 : 0;
  }
}

// Second kernel: the run that enters a tile (wavefront 0) and the run that leaves it (wavefront 1). The partials
// of such a run are those of the tile in which it begins (its leaving run), of the tiles it fills, and of the tile
// in which it ends (its entering run). Every tile of the run combines them in the same order, so all of them use
// the same maximum and sum; then the workgroup finishes the tile's entries of the two runs from src.
template <typename T, int MODE, bool ORDERED = false>
__global__ __launch_bounds__(kFusedFragBlock) void group_fused_fragment_kernel(GroupArgs g, FusedArgs f) {
  typedef typename Acc<T>::type F;
  typedef typename FusedSum<T, ORDERED>::type S;
  typedef typename OrdKey<F>::bits KB;
  constexpr bool kBackward = MODE == GS_SOFTMAX_BWD || MODE == GS_LOG_SOFTMAX_BWD;
  extern __shared__ double s_fin_raw[];  // [2 runs][K]: maximum, sum
  F *s_fin = reinterpret_cast<F *>(s_fin_raw);
  if (!ORDERED && *f.flag != 0) return;
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
  const int KR = (int)g.K, k_first = ORDERED ? (int)blockIdx.y * f.kcols : 0;
  const int K = ORDERED ? (KR - k_first < f.kcols ? KR - k_first : f.kcols) : KR;
  const int64_t b = ORDERED ? 0 : blockIdx.x / f.nt, t = blockIdx.x - b * f.nt;
  const int64_t j0 = t * (ORDERED ? f.tw : f.te);
  const bool through = ORDERED && f.state[0] != 0;
  if constexpr (ORDERED) {
    if ((f.gate != nullptr && *f.gate == 0) || j0 >= *f.n_sorted) return;
  }
  const int32_t *meta_b = f.meta + b * f.nt * 4;
  const int head_len = meta_b[t * 4 + 0], tail_start = meta_b[t * 4 + 1], ne = meta_b[t * 4 + 2];
  const bool whole = meta_b[t * 4 + 3] != 0;
  const bool has = wave == 0 ? head_len > 0 : tail_start < ne;
  if constexpr (ORDERED) {
    if (head_len <= 0 && tail_start >= ne) return;
    if (has) {
      // the group's partials put together lie with the tile in which it begins
      const int64_t first = wave == 0 ? (int64_t)((uint32_t)f.ptr[f.group[j0]] / (uint32_t)f.tw) : t;
      const KB *key = static_cast<const KB *>(f.ckey) + (first * 2 + 1) * KR + k_first;
      const S *sum = static_cast<const S *>(f.csum) + (first * 2 + 1) * KR + k_first;
      for (int k = lane; k < K; k += kWave) {
        s_fin[(wave * K + k) * 2] = key[k] == group_empty_key<T>() ? (F)0 : OrdKey<F>::dec(key[k]);
        s_fin[(wave * K + k) * 2 + 1] = (F)sum[k];
      }
    }
  } else if (has) {
    auto filled = [&](int64_t i) { return meta_b[i * 4 + 3] != 0; };
    int64_t first = t, last = t;
    if (wave == 0) {
      // the tile in which the run begins: the nearest one before t that the run does not fill (tile 0 cannot be filled)
      first = t - 1;
      while (true) {
        const int64_t i = first - lane;
        const uint64_t stop = __ballot(i <= 0 || !filled(i));
        if (stop != 0) {
          first -= __ffsll((unsigned long long)stop) - 1;
          break;
        }
        first -= kWave;
      }
      if (first < 0) first = 0;
    }
    if (wave == 1 || whole) {
      last = t + 1;
      while (true) {
        const int64_t i = last + lane;
        const uint64_t stop = __ballot(i >= f.nt - 1 || !filled(i));
        if (stop != 0) {
          last += __ffsll((unsigned long long)stop) - 1;
          break;
        }
        last += kWave;
      }
      if (last > f.nt - 1) last = f.nt - 1;
    }
    const int G = f.G, parts = kWave / G;
    const int j = lane / G, lg = lane - j * G;
    const KB *ckey = static_cast<const KB *>(f.ckey) + b * f.nt * 2 * KR + k_first;
    const S *csum = static_cast<const S *>(f.csum) + b * f.nt * 2 * KR + k_first;
    for (int k0 = 0; k0 < K; k0 += G) {
      const int k = k0 + lg;
      const bool col_ok = k < K;
      KB key = kBackward ? (KB)0 : group_empty_key<T>();
      S sum = (S)0;
      for (int64_t i = first + j; i <= last; i += parts) {
        const int64_t p = (i * 2 + (i == first ? 1 : 0)) * KR + (col_ok ? k : 0);
        if constexpr (kBackward) {
          sum += csum[p];
        } else {
          fused_absorb<T>(key, sum, ckey[p], csum[p]);
        }
      }
      for (int off = parts / 2; off >= 1; off >>= 1) {
        const KB ok = __shfl_down(key, off * G);
        const S os = __shfl_down(sum, off * G);
        if constexpr (kBackward) {
          sum += os;
        } else {
          fused_absorb<T>(key, sum, ok, os);
        }
      }
      if (j == 0 && col_ok) {
        F m = (F)0;
        if constexpr (!kBackward) m = key == group_empty_key<T>() ? (F)0 : OrdKey<F>::dec(key);
        s_fin[(wave * K + k) * 2] = m;
        s_fin[(wave * K + k) * 2 + 1] = (F)sum;
      }
    }
  }
  __syncthreads();
  const int64_t lo_t = ORDERED ? 0 : (b * g.E + j0) * K;
  const T *src_t = static_cast<const T *>(g.src) + lo_t;
  const T *grad_t = kBackward ? static_cast<const T *>(g.grad) + lo_t : nullptr;
  T *out_t = static_cast<T *>(g.out) + lo_t;
  const int64_t *idx = g.index + b * g.sb;
  const F eps = (F)g.eps;
  for (int w = 0; w < 2; ++w) {
    const int lo = w == 0 ? 0 : tail_start, hi = w == 0 ? head_len : ne;
    if (hi <= lo) continue;
    auto finish = [&](F xv, F gv, int k) {
      const F m = s_fin[(w * K + k) * 2], s = s_fin[(w * K + k) * 2 + 1];
      if (MODE == GS_SOFTMAX) return round_elem<T>(exp_acc(round_elem<T>(xv - m))) / round_elem<T>(s);
      if (MODE == GS_LOG_SOFTMAX) {
        F l = round_elem<T>(log_acc(round_elem<T>(round_elem<T>(s) + eps)));
        asm volatile("" : "+v"(l));  // see group_finish_kernel
        return round_elem<T>(xv - m) - l;
      }
      if (MODE == GS_SOFTMAX_BWD) return xv * (gv - s);
      return gv - exp_acc(xv) * s;
    };
    if constexpr (ORDERED) {
      // 16-byte units, four on the way together: a unit's row comes from perm first
      constexpr int U = 4, C = kVecBytes / (int)sizeof(T);
      const int units = K / C;
      const uint32_t inv = blockIdx.y == gridDim.y - 1 ? f.inv_last : f.inv_units;
      for (int v0 = lo * units + tid; v0 < hi * units; v0 += U * kFusedFragBlock) {
        int64_t at[U];
        int k[U];
        Vec<T, C> x[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {  // (past the end: the last unit again)
          const int v = v0 + u * kFusedFragBlock < hi * units ? v0 + u * kFusedFragBlock : hi * units - 1;
          const int e = fused_unit_entry(v, inv);
          k[u] = (v - e * units) * C;
          at[u] = j0 + e;
        }
        if (through) {
#pragma unroll
          for (int u = 0; u < U; ++u) at[u] = f.perm[at[u]];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
          at[u] = at[u] * KR + k_first + k[u];
          x[u] = load_vec<T, C>(src_t + at[u]);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
          if (v0 + u * kFusedFragBlock >= hi * units) continue;
#pragma unroll
          for (int c = 0; c < C; ++c)
            x[u].v[c] = from_acc<T>(finish(to_acc<T>(x[u].v[c]), (F)0, k[u] + c));
          store_vec<T, C>(out_t + at[u], x[u]);
        }
      }
    } else {
      const int64_t group = idx[(j0 + (w == 0 ? 0 : ne - 1)) * g.se];
      const bool valid = group >= 0 && group < g.N;
      for (int i = lo * K + tid; i < hi * K; i += kFusedFragBlock) {
        const F res = finish(to_acc<T>(src_t[i]), kBackward ? to_acc<T>(grad_t[i]) : (F)0, i % K);
        out_t[i] = from_acc<T>(valid ? res : (F)0);
      }
    }
  }
}

template <typename T, int CV, int MODE>
int launch_group_fused(const GroupArgs &g, const FusedArgs &f, bool force, hipStream_t stream, bool sample = true) {
  constexpr bool kBackward = MODE == GS_SOFTMAX_BWD || MODE == GS_LOG_SOFTMAX_BWD;
  typedef typename Acc<T>::type F;
  if (sample) hipLaunchKernelGGL(group_order_sample_kernel, dim3(1), dim3(1024), 0, stream, g, f.flag, force ? 1 : 0,
                     g.bins != nullptr ? g.bins->totals : nullptr, g.bins != nullptr ? g.bins->nb : 0);
  const size_t lds = (size_t)f.tile_vecs * 16 * (kBackward ? 2 : 1) + ((size_t)f.te + 2) * 2;
  const unsigned tiles = (unsigned)(g.B * f.nt);
  hipLaunchKernelGGL((group_fused_kernel<T, CV, MODE>), dim3(tiles), dim3(kBlock), lds, stream, g, f);
  hipLaunchKernelGGL((group_fused_fragment_kernel<T, MODE>), dim3(tiles), dim3(kFusedFragBlock),
                     (size_t)g.K * 4 * sizeof(F), stream, g, f);
  return hipGetLastError() == hipSuccess ? TS_OK : TS_ERR_LAUNCH;
}

// ORDERED, between the two: the partials of a long group meet in the tile in which it begins (its leaving run), once for
// all tiles that it crosses (every tile for itself is quadratic in their number: 10 M entries x 32 floats, a fifth of them in
// one group, 7 ms). Bound by the longest group's chain: 10 M x 8 floats, 2 M in one group, 54 us with every partial waited
// for on the spot, 28 with eight on the way. At least 4.8 us, with or without such a group.
template <typename T>
__global__ __launch_bounds__(kBlock) void group_fused_combine_kernel(GroupArgs g, FusedArgs f) {
  typedef typename Acc<T>::type F;
  typedef typename OrdKey<F>::bits KB;
  __shared__ KB s_key[kBlock];
  __shared__ double s_sum[kBlock];
  if (f.gate != nullptr && *f.gate == 0) return;
  const int64_t t = blockIdx.x, w0 = t * f.tw, E = *f.n_sorted;
  if (w0 >= E) return;
  const int32_t *meta = f.meta + t * 4;
  if (meta[1] >= meta[2] || meta[3] != 0) return;  // no group begins here and goes on
  const int KR = (int)g.K, k_first = (int)blockIdx.y * f.kcols, K = KR - k_first < f.kcols ? KR - k_first : f.kcols;
  const int64_t last = (f.ptr[f.group[w0 + meta[2] - 1] + 1] - 1) / f.tw;
  const int G = f.G, parts = kBlock / G, j = threadIdx.x / G, lg = threadIdx.x - j * G;
  KB *ckey = static_cast<KB *>(f.ckey) + k_first;
  double *csum = static_cast<double *>(f.csum) + k_first;
  for (int k0 = 0; k0 < K; k0 += G) {
    const int k = k0 + lg < K ? k0 + lg : K - 1;
    KB key = group_empty_key<T>();
    double sum = 0.0;
    constexpr int U = 8;  // partials on the way together
    for (int64_t i0 = t + j; i0 <= last; i0 += U * parts) {
      KB ku[U];
      double su[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {  // (past the end: the last tile's again)
        const int64_t i = i0 + u * parts < last ? i0 + u * parts : last;
        const int64_t p = (i * 2 + (i == t ? 1 : 0)) * KR + k;
        ku[u] = ckey[p];
        su[u] = csum[p];
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (i0 + u * parts > last) continue;
        fused_absorb<T>(key, sum, ku[u], su[u]);
      }
    }
    s_key[threadIdx.x] = key;
    s_sum[threadIdx.x] = sum;
    __syncthreads();
    for (int half = parts / 2; half >= 1; half >>= 1) {
      if (j < half) {
        const int o = threadIdx.x + half * G;
        fused_absorb<T>(s_key[threadIdx.x], s_sum[threadIdx.x], s_key[o], s_sum[o]);
      }
      __syncthreads();
    }
    if (j == 0 && k0 + lg < K) {
      const int64_t p = (t * 2 + 1) * KR + k;
      ckey[p] = s_key[threadIdx.x];
      csum[p] = s_sum[threadIdx.x];
    }
    __syncthreads();
  }
}

// Tiles over entries that were sorted by group. K columns in slices of at most 128 bytes.
// bytes: of the tiles' records; ws null: only that.
struct FusedOrderedPlan {
  size_t bytes;
  FusedArgs f;
};
inline FusedOrderedPlan group_fused_ordered_plan(int64_t n, int64_t K, int elem_bytes, void *ws) {
  FusedOrderedPlan r;
  r.bytes = 0;
  FusedArgs &f = r.f;
  const int vec = 16 / elem_bytes;
  if (K % vec != 0) return r;
  const int64_t most = 128 / elem_bytes;
  int64_t slices = (K + most - 1) / most, kc = (K + slices - 1) / slices;
  kc = (kc + vec - 1) / vec * vec;
  slices = (K + kc - 1) / kc;
  if (slices > 65535) return r;
  const int64_t row = kc * elem_bytes;
  int64_t te = 32768 / row;
  if (const char *env = getenv("TS_GROUP_TILE")) te = te < atoi(env) ? te : atoi(env);  // tuning aid
  int epl = 1;
  while (epl * 2 * kBlock <= te && epl * 2 <= kFusedPer) epl *= 2;
  f.epl = epl;
  f.te = epl * kBlock;
  f.tw = f.te / 4 * 3;
  f.short_run = kFusedShortRun;
  f.long_run = kFusedGroup * kFusedShortRun;
  f.nt = (n + f.tw - 1) / f.tw;
  f.kcols = (int)kc;
  f.slices = (int)slices;
  int G = 1;
  while (G < kc && G < kWave) G *= 2;
  f.G = G;
  f.tile_vecs = (int)((f.te * row + 15) / 16);
  auto inverse = [&](int64_t units) { return (uint32_t)((((uint64_t)1 << 31) + units - 1) / units); };
  f.inv_units = inverse(kc / vec);
  f.inv_last = inverse((K - (slices - 1) * kc) / vec);
  auto up = [](size_t x) { return (x + 255) & ~(size_t)255; };
  const size_t o_key = up((size_t)f.nt * 16), o_sum = o_key + up((size_t)f.nt * 2 * K * (elem_bytes == 8 ? 8 : 4));
  r.bytes = o_sum + up((size_t)f.nt * 2 * K * 8);
  char *base = static_cast<char *>(ws);
  f.meta = reinterpret_cast<int32_t *>(base);
  f.ckey = base + o_key;
  f.csum = base + o_sum;
  f.flag = nullptr;
  return r;
}
template <typename T, int CV, int MODE> int launch_group_fused_ordered(const GroupArgs &g, const FusedArgs &f, hipStream_t stream) {
  typedef typename Acc<T>::type F;
  const size_t lds = (size_t)f.tile_vecs * 16 + ((size_t)f.te + 2) * 2;
  const dim3 grid((unsigned)f.nt, (unsigned)f.slices);
  hipLaunchKernelGGL((group_fused_kernel<T, CV, MODE, true>), grid, dim3(kBlock), lds, stream, g, f);
  hipLaunchKernelGGL((group_fused_combine_kernel<T>), grid, dim3(kBlock), 0, stream, g, f);
  hipLaunchKernelGGL((group_fused_fragment_kernel<T, MODE, true>), grid, dim3(kFusedFragBlock),
                     (size_t)f.kcols * 4 * sizeof(F), stream, g, f);
  return hipGetLastError() == hipSuccess ? TS_OK : TS_ERR_LAUNCH;
}

}  // namespace ts
