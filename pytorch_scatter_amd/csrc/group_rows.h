// Softmax, log-softmax (forward and backward), logsumexp, standard deviation and sums of narrow rows over entries that were sorted by group
// (row_sort.h): rows of the entries in registers, gathered once.
//
// A worker of `lanes` lanes holds four neighbouring places of the order (kRowsHeld), a lane VEC columns of each of them. It walks its
// places in the order: running maximum, then running sum, reset where a group begins; the value at a group's end is handed
// back to its places, and the results go out through perm. Only a group that crosses workers meets in LDS: the worker in
// which it begins puts the parts together. Columns never meet, so a worker is as wide as the row needs (nine lanes for 33
// floats; the last lane's columns begin early and overlap its neighbour's, whose values it computes again), and rows of any
// width and alignment take 16-byte accesses (8 bytes for 16-bit elements, to hold as many values as the others do).
// A tile (workgroup) takes the groups that begin in its window of three quarters of its places; a group that is too long
// for that leaves a partial per tile. group_rows_combine_kernel puts those together, once per group; softmax then finishes
// such places from src (group_rows_finish_kernel).
//
//   forward    m = maximum (entries beat lowest(), NaN never wins, no winner: 0), e = exp(src - m), s = sum e;
//              softmax e / s,  log-softmax (src - m) - log(s + eps)
//   backward   softmax: y * (g - sum y * g);  log-softmax: g - exp(y) * sum g
//   logsumexp  log(s + eps) + m, the maximum from -inf on;  std  sum, mean, squared deviations from it, all from registers
// Sums are held in double. Intermediates that the reference holds in the element type are rounded to it.
#pragma once

#include <type_traits>

#include "group_softmax.h"
#include "row_sort.h"

namespace ts {

constexpr int kRowsHeld = 4;          // places of the order that a worker holds
constexpr int kRowsBlock = kBlock;
constexpr int kRowsCombine = 1024;    // lanes of a workgroup that puts long groups together:
constexpr int kRowsTeam = 16;         // lanes, one column each, for a group that crosses up to
constexpr int kRowsTeamSpan = 64;     // this many tiles
constexpr int kRowsTeams = kRowsCombine / kRowsTeam;
constexpr int kRowsMaxLanes = 16;     // lanes of a worker at most: wider rows are taken in column slices

template <typename T> constexpr int group_rows_full() { return sizeof(T) == 8 ? 2 : 4; }  // columns per lane
inline int group_rows_vec(int64_t K, int elem_bytes) { return K >= (elem_bytes == 8 ? 2 : 4) ? (elem_bytes == 8 ? 2 : 4) : 1; }

struct GroupRowsArgs {
  int lanes;          // of a worker
  int workers;        // of a workgroup
  uint32_t inv;       // 2^16 / lanes, rounded up
  int te, tw;         // places of a tile, of its window
  int kcols, slices;  // columns that a workgroup takes, workgroups that share a tile
  int64_t nt;         // tiles
  int stream;         // results leave past the caches (whole 128-byte lines)
  int32_t *meta;      // [nt][4]: entries of the entering run, first place of the leaving run, places (all from the window's begin
                      // on), tile is one run that enters and leaves
  uint64_t *pa;       // [nt][2][K] partials of the entering / leaving run: key of the maximum; std: bits of the sum
  double *pb;         //            sum; std: squared deviations from the run's mean
  const int32_t *state;     // [0] 0: the index was in order, the order is that of memory
  const int64_t *ptr;       // [groups + 1] first place of every group (the last: entries that belong to a group)
  const int32_t *perm;      // entry at every place of the order (not written when state[0] is 0)
  const int32_t *group;     // and its group
  const int64_t *index;     // as the caller gave it, for the entries that belong to no group
  int64_t sb, se, E0, N0;
  const int *gate;          // reads 0: these launches return at once (null: they run)
};

struct GroupRowsPlan {
  size_t bytes;  // of the tiles' records; 0: does not apply
  GroupRowsArgs f;
};
// n entries in `groups` groups. ws null: only the bytes.
inline GroupRowsPlan group_rows_plan(int64_t n, int64_t groups, int64_t K, int elem_bytes, void *ws) {
  GroupRowsPlan r;
  r.bytes = 0;
  GroupRowsArgs &f = r.f;
  if (n < 1 || groups < 1 || K < 1) return r;
  const int vec = group_rows_vec(K, elem_bytes);
  const int64_t all = (K + vec - 1) / vec;
  // sixteen lanes; eight for rows that are whole lines, in groups that a tile of 64 places would often cut (256 floats in order, 2.4 M
  // entries in groups of 76, forward and backward: 4894 us, 3930 with eight; 100 floats, whose pieces are not lines: 900 / 1019)
  int most = K * elem_bytes % 128 == 0 && n > 12 * groups ? kRowsMaxLanes / 2 : kRowsMaxLanes;
  if (const char *env = getenv("TS_GROUP_LANES")) most = atoi(env);  // tuning aid
  const int64_t slices = (all + most - 1) / most;
  if (slices > 65535) return r;
  f.lanes = (int)((all + slices - 1) / slices);
  f.slices = (int)((all + f.lanes - 1) / f.lanes);
  f.kcols = f.lanes * vec;
  f.workers = kRowsBlock / f.lanes;
  f.inv = 65536u / (uint32_t)f.lanes + 1;
  f.te = f.workers * kRowsHeld;
  f.tw = f.te / 4 * 3 & ~(kRowsHeld - 1);
  f.nt = (n + f.tw - 1) / f.tw;
  if ((K + kRowsTeam - 1) / kRowsTeam > 65535) return r;
  f.stream = (K * elem_bytes) % 128 == 0 && f.kcols * elem_bytes % 128 == 0;
  auto up = [](size_t x) { return (x + 255) & ~(size_t)255; };
  const size_t o_pa = up((size_t)f.nt * 16), o_pb = o_pa + up((size_t)f.nt * 2 * K * 8);
  r.bytes = o_pb + up((size_t)f.nt * 2 * K * 8);
  char *base = static_cast<char *>(ws);
  f.meta = reinterpret_cast<int32_t *>(base);
  f.pa = reinterpret_cast<uint64_t *>(base + o_pa);
  f.pb = reinterpret_cast<double *>(base + o_pb);
  return r;
}

// VEC elements from an address that need not be a multiple of their size
template <typename T, int VEC> __device__ __forceinline__ Vec<T, VEC> rows_load(const T *p) {
  Vec<T, VEC> v;
  __builtin_memcpy(&v, p, sizeof(v));
  return v;
}
template <typename T, int VEC> __device__ __forceinline__ void rows_store(T *p, const Vec<T, VEC> &v, bool stream) {
  if (stream)  // (then the address is a multiple of the size)
    store_vec_stream<T, VEC>(p, v);
  else
    __builtin_memcpy(p, &v, sizeof(v));
}

// the places [a, b) that tile t takes, relative to its window's begin. enters / leaves: the group at a began in another tile
// and is too long for it; the group at the window's end goes on in the next tile.
struct RowsSpan {
  int a, b;
  bool enters, leaves;
};
__device__ __forceinline__ RowsSpan rows_span(const GroupRowsArgs &f, int64_t w0, int64_t n, int32_t g0, int32_t g1) {
  const int64_t w1 = w0 + f.tw < n ? w0 + f.tw : n;
  const int64_t s0 = f.ptr[g0], e0 = f.ptr[g0 + 1], s1 = f.ptr[g1], e1 = f.ptr[g1 + 1];
  auto fits = [&](int64_t s, int64_t e) { return e <= (int64_t)((uint32_t)s / (uint32_t)f.tw) * f.tw + f.te; };
  RowsSpan r;
  r.enters = s0 < w0 && !fits(s0, e0);
  r.a = s0 < w0 && !r.enters ? (int)(e0 - w0) : 0;
  r.leaves = e1 > w1 && !fits(s1, e1);
  r.b = (int)((e1 > w1 && !r.leaves ? e1 : w1) - w0);
  return r;
}

// the entries of a window that belong to no group: zeros in columns [k_first, k_first + K)
template <typename T>
__device__ __forceinline__ void rows_zero_outside(const GroupArgs &g, const GroupRowsArgs &f, int64_t j0, int k_first, int K) {
  for (int64_t be = j0 + threadIdx.x / kWave; be < g.E && be < j0 + f.tw; be += kRowsBlock / kWave) {
    int64_t b, e;
    split_edge(be, g.E / f.E0, f.E0, b, e);
    const int64_t at = f.index[b * f.sb + e * f.se];
    if (at >= 0 && at < f.N0) continue;
    for (int k = threadIdx.x & (kWave - 1); k < K; k += kWave)
      static_cast<T *>(g.out)[be * g.K + k_first + k] = from_acc<T>((typename Acc<T>::type)0);
  }
}

// A worker's places: which are the tile's, where groups begin and end among them.
struct RowsPlaces {
  uint32_t valid, head, end;  // one bit per place
  bool enters, leaves, whole;  // the first place goes on with the worker's before, the last with the worker's behind; both, and no
                               // group begins or ends here
};
__device__ __forceinline__ RowsPlaces rows_places_of(const int32_t (&gr)[kRowsHeld + 2], int p0, const RowsSpan &s) {
  RowsPlaces r = {0, 0, 0, false, false, false};
#pragma unroll
  for (int i = 0; i < kRowsHeld; ++i) {
    const int p = p0 + i;
    const bool in = p >= s.a && p < s.b;
    r.valid |= (in ? 1u : 0u) << i;
    r.head |= (in && (p == s.a || gr[i + 1] != gr[i]) ? 1u : 0u) << i;
    r.end |= (in && (p == s.b - 1 || gr[i + 1] != gr[i + 2]) ? 1u : 0u) << i;
  }
  r.enters = (r.valid & 1u) != 0 && (r.head & 1u) == 0;
  r.leaves = (r.valid >> (kRowsHeld - 1)) != 0 && (r.end >> (kRowsHeld - 1)) == 0;
  r.whole = r.enters && r.leaves && r.end == 0;
  return r;
}
// the groups of a worker's places (one before, one behind) and the entries there; p: the first place, a multiple of kRowsHeld.
// all: entries of the call (those behind the last that belongs to a group are anything)
__device__ __forceinline__ void rows_load_order(const GroupRowsArgs &f, int64_t p, int64_t all, int32_t (&gr)[kRowsHeld + 2],
                                                int32_t (&row)[kRowsHeld]) {
  typedef int32_t i4 __attribute__((ext_vector_type(4)));
  static_assert(kRowsHeld == 4, "");
  const int64_t last = (all - 1) & ~(int64_t)(kRowsHeld - 1), at = p < last ? p : last;  // (the arrays end on whole 256 bytes)
  const i4 q = *reinterpret_cast<const i4 *>(f.group + at), e = *reinterpret_cast<const i4 *>(f.perm + at);
  gr[0] = f.group[at > 0 ? at - 1 : 0];
  gr[kRowsHeld + 1] = f.group[at + kRowsHeld < all ? at + kRowsHeld : all - 1];
#pragma unroll
  for (int i = 0; i < kRowsHeld; ++i) {
    gr[i + 1] = q[i];
    row[i] = e[i];
  }
}
// the nearest worker behind / before `w` that is not one run from end to end (there is one)
__device__ __forceinline__ int rows_next_open(const uint32_t *s_whole, int w) {
  for (int v = w + 1;; v = (v & ~31) + 32) {
    const uint32_t open = ~s_whole[v >> 5] >> (v & 31);
    if (open != 0) return v + __builtin_ctz(open);
  }
}
__device__ __forceinline__ int rows_prev_open(const uint32_t *s_whole, int w) {
  for (int v = w - 1;; v = (v & ~31) - 1) {
    const uint32_t open = ~s_whole[v >> 5] << (31 - (v & 31));
    if (open != 0) return v - __builtin_clz(open);
  }
}

// x / s: the quotient from the reciprocal (1 ulp) and one correction by its remainder, which leaves what rounding leaves (s is
// a sum of exponentials, at least 1 or not a number; a division takes ten instructions)
__device__ __forceinline__ float rows_divide(float x, float s) {
  const float r = fast_rcp(s), q = x * r;
  return fmaf(fmaf(-q, s, x), r, q);
}
__device__ __forceinline__ double rows_divide(double x, double s) { return x / s; }

// a or b, by value: a choice between two elements of arrays is turned into one between their addresses otherwise, and the arrays
// then live in memory
template <typename A> __device__ __forceinline__ A rows_pick(bool first, A a, A b) { return first ? a : b; }

// at(i) for every bit i that a lane has in ends, the lanes' first bits together: a wavefront goes round as often as one of its
// lanes has groups that end, not once for every place
template <int S, typename At> __device__ __forceinline__ void rows_at_ends(uint32_t ends, At &&at) {
  while (ends != 0) {
    at(__builtin_ctz(ends));
    ends &= ends - 1;
  }
}
template <typename T, bool ROUND> __device__ __forceinline__ typename Acc<T>::type round_elem_if(typename Acc<T>::type v) {
  return ROUND ? round_elem<T>(v) : v;
}

// A lane's values of its worker's places, what runs over them, and how the parts of a group that crosses workers meet. An array of
// parts in LDS holds a slot per lane: what a group left in a worker that it entered, and, where it began, the whole.
template <typename A, int VEC> struct RowsAcross {
  A *in, *whole;
  const uint32_t *s_whole;
  int w, l, L;
  // Of the run that leaves the worker, own: all of it. Returns that of the run that enters.
  template <typename Join>
  __device__ __forceinline__ void meet(const RowsPlaces &at, A (&own)[VEC], A (&entered)[VEC], int &w_open, int &w_last, Join &&join) const {
    __syncthreads();
    if (at.leaves && !at.whole) {
      w_last = rows_next_open(s_whole, w);
      const A *p = in + ((w + 1) * L + l) * VEC;
      // (a hub in rows of one column: 256 workers to go through, so that reads have to be on the way together)
      constexpr int U = VEC == 1 ? 8 : 2;
      int v = w;
      for (; v + U <= w_last; v += U, p += U * L * VEC) {
        A part[U][VEC];
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
          for (int c = 0; c < VEC; ++c) part[u][c] = p[u * L * VEC + c];
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
          for (int c = 0; c < VEC; ++c) own[c] = join(own[c], part[u][c]);
      }
      for (; v < w_last; ++v, p += L * VEC) {
#pragma unroll
        for (int c = 0; c < VEC; ++c) own[c] = join(own[c], p[c]);
      }
#pragma unroll
      for (int c = 0; c < VEC; ++c) whole[(w * L + l) * VEC + c] = own[c];
    }
    __syncthreads();
    if (at.enters) {
      w_open = rows_prev_open(s_whole, w);
      const A *p = whole + (w_open * L + l) * VEC;
#pragma unroll
      for (int c = 0; c < VEC; ++c) entered[c] = p[c];
    }
    if (at.whole) {
#pragma unroll
      for (int c = 0; c < VEC; ++c) own[c] = entered[c];
    }
  }
};

template <typename T, int VEC, int MODE>
__global__ __launch_bounds__(kRowsBlock) void group_rows_kernel(GroupArgs g, GroupRowsArgs f) {
  typedef typename Acc<T>::type F;
  typedef typename OrdKey<F>::bits KB;
  typedef Vec<T, VEC> V;
  constexpr int S = kRowsHeld;
  constexpr bool kBackward = MODE == GS_SOFTMAX_BWD || MODE == GS_LOG_SOFTMAX_BWD;
  constexpr bool kEntries = kBackward || MODE == GS_SOFTMAX || MODE == GS_LOG_SOFTMAX;  // a result per entry
  constexpr bool kMax = MODE == GS_SOFTMAX || MODE == GS_LOG_SOFTMAX || MODE == GS_LSE;
  __shared__ __align__(16) F s_top[kMax ? 2 : 1][kMax ? kRowsBlock * VEC : 1];
  __shared__ __align__(16) double s_sum[2][kRowsBlock * VEC];
  __shared__ uint32_t s_whole[kRowsBlock / 32 + 1];  // workers that are one run from end to end
  __shared__ uint8_t s_end[MODE == GS_STD ? kRowsBlock : 1], s_head[MODE == GS_STD ? kRowsBlock : 1];
  // Every load that needs no other one is on the way before the first is waited for: what the tile has to know (a gate, the
  // entries, whether the order is that of memory, the groups at the window's ends) and every worker's part of the order.
  const int tid = threadIdx.x, K = (int)g.K, L = f.lanes;
  const int w = (int)(((uint32_t)tid * f.inv) >> 16), l = tid - w * L;
  const int64_t t = blockIdx.x, w0 = t * f.tw;
  const int gate = f.gate != nullptr ? *f.gate : 1;
  const bool through = f.state[0] != 0;
  const int64_t n = f.ptr[g.N];
  const int32_t g0 = f.group[w0];
  int32_t g1 = f.group[w0 + f.tw < g.E ? w0 + f.tw - 1 : g.E - 1];
  int32_t gr[S + 2], row[S];
  rows_load_order(f, w0 + w * S, g.E, gr, row);
  if (gate == 0) return;
  const int k_first = (int)blockIdx.y * f.kcols, k_end = K - k_first < f.kcols ? K : k_first + f.kcols;
  if (kEntries && n != g.E) rows_zero_outside<T>(g, f, w0, k_first, k_end - k_first);
  if (w0 >= n) return;
  if (n < w0 + f.tw) g1 = f.group[n - 1];
  if (tid <= kRowsBlock / 32) s_whole[tid] = 0;
  const int first = k_first + l * VEC;
  const bool lane_on = w < f.workers && first < k_end;
  const int col = !lane_on ? 0 : first + VEC <= K ? first : K - VEC;  // the last lane: columns that its neighbour has as well
  V x[S], y[kBackward ? S : 1];
  // The rows of a place outside the tile's are not needed, but may be read: inside the window, where few are, before the row
  // pointers say so; behind it, only if the tile's last group goes on there. What such a place leaves ends where a group
  // begins, in front of the tile's places, or is not looked at, behind them.
  const RowsSpan span = rows_span(f, w0, n, g0, g1);
  auto load_rows = [&](int lo, int hi) {
#pragma unroll
    for (int i = 0; i < S; ++i) {
      const int p = w * S + i;
      row[i] = p >= lo && p < hi && w0 + p < n && lane_on ? (through ? row[i] : (int32_t)(w0 + p)) : 0;
      const int64_t o = (int64_t)row[i] * K + col;
      x[i] = rows_load<T, VEC>(static_cast<const T *>(g.src) + o);
      if constexpr (kBackward) y[i] = rows_load<T, VEC>(static_cast<const T *>(g.grad) + o);
    }
  };
  load_rows(span.a, span.b);
  if (span.b <= span.a) {  // (a group that the tile before has taken ends with the window)
    if (tid < 4 && blockIdx.y == 0) f.meta[t * 4 + tid] = 0;
    return;
  }
  RowsPlaces at = rows_places_of(gr, w * S, span);
  if (!lane_on) at = {0, 0, 0, false, false, false};
  const int32_t g_first = f.group[w0 + span.a], g_last = f.group[w0 + span.b - 1];
  uint32_t inside = 0;  // places whose group the tile holds as a whole
#pragma unroll
  for (int i = 0; i < S; ++i)
    inside |= (!(span.enters && gr[i + 1] == g_first) && !(span.leaves && gr[i + 1] == g_last) ? 1u : 0u) << i;
  inside &= at.valid;
  // this worker holds the begin of the run that enters the tile, the end of the one that leaves (the window ends with a worker)
  const bool at_first = span.enters && at.valid != 0 && w == 0, at_last = span.leaves && at.valid != 0 && w * S + S == span.b;
  const bool none = at.head == 0;  // the last place's run entered the worker
  const int fe = __builtin_ctz(at.end | 1u << (S - 1));  // the first end (or the last place)
  uint64_t *const pa = f.pa + t * 2 * K + col;
  double *const pb = f.pb + t * 2 * K + col;
  int w_open = w, w_last = w;  // the workers in which a run that crosses workers begins and ends
  __syncthreads();
  if (l == 0 && at.whole) atomicOr(&s_whole[w >> 5], 1u << (w & 31));
  if constexpr (MODE == GS_STD) {
    if (l == 0 && w < f.workers) {
      s_end[w] = (uint8_t)fe;
      s_head[w] = (uint8_t)(31 - __builtin_clz(at.head | 1u));
    }
  }
  const RowsAcross<F, VEC> tops = {s_top[0], s_top[kMax ? 1 : 0], s_whole, w, l, L};
  const RowsAcross<double, VEC> adds = {s_sum[0], s_sum[1], s_whole, w, l, L};

  // ---- maxima: m[i] of the run of place i
  F m[S][VEC];
  if constexpr (kMax) {
    const F lowest = to_acc<T>(ElemLim<T>::lowest());
    F run[VEC], in[VEC];
#pragma unroll
    for (int i = 0; i < S; ++i) {
      const bool head = i == 0 || (at.head >> i & 1u) != 0;
#pragma unroll
      for (int c = 0; c < VEC; ++c) m[i][c] = run[c] = max_acc(rows_pick(head, (F)-INFINITY, run[c]), to_acc<T>(x[i].v[c]));
      if (at.enters && i == fe) {
#pragma unroll
        for (int c = 0; c < VEC; ++c) tops.in[tid * VEC + c] = run[c];
      }
    }
    tops.meet(at, run, in, w_open, w_last, [](F p, F q) { return max_acc(p, q); });
    if (at_last) {
#pragma unroll
      for (int c = 0; c < VEC; ++c) {
        const F top = rows_pick(none, in[c], run[c]);
        pa[K + c] = MODE == GS_LSE || top > lowest ? OrdKey<F>::enc(top) : group_empty_key<T>();
      }
    }
#pragma unroll
    for (int i = S - 1; i >= 0; --i) {
      const bool end = (at.end >> i & 1u) != 0, back = at.enters && i <= fe;
#pragma unroll
      for (int c = 0; c < VEC; ++c) {
        run[c] = rows_pick(end, m[i][c], run[c]);
        m[i][c] = rows_pick(back, in[c], run[c]);
      }
    }
    if (at_first) {
#pragma unroll
      for (int c = 0; c < VEC; ++c)
        pa[c] = MODE == GS_LSE || m[0][c] > lowest ? OrdKey<F>::enc(m[0][c]) : group_empty_key<T>();
    }
    // what is added up, for the results in x: softmax and logsumexp e, log-softmax z
#pragma unroll
    for (int i = 0; i < S; ++i) {
#pragma unroll
      for (int c = 0; c < VEC; ++c) {
        const F top = MODE == GS_LSE || m[i][c] > lowest ? m[i][c] : (F)0;
        F z = round_elem<T>(to_acc<T>(x[i].v[c]) - top);
        if (MODE == GS_LSE && z != z) z = -INFINITY;  // NaN entries and -inf - -inf drop out (logsumexp.py:41)
        x[i].v[c] = from_acc<T>(MODE == GS_LOG_SOFTMAX ? z : exp_acc(z));
      }
    }
  }
  const F eps = (F)g.eps;
  // ---- sums of term(i, c) over the run of every place: sum[i] at its end, as a float; run / in: of the runs that leave / enter
  F sum[S][VEC];
  double run[VEC], in[VEC] = {};
  auto sums = [&](auto &&term) {
#pragma unroll
    for (int i = 0; i < S; ++i) {
      const bool head = i == 0 || (at.head >> i & 1u) != 0;
#pragma unroll
      for (int c = 0; c < VEC; ++c) {
        run[c] = rows_pick(head, 0.0, run[c]) + (double)term(i, c);
        sum[i][c] = (F)run[c];
      }
      if ((at.enters || at_first) && i == fe) {
#pragma unroll
        for (int c = 0; c < VEC; ++c) {
          adds.in[tid * VEC + c] = run[c];
          in[c] = rows_pick(at_first, run[c], in[c]);  // (the run that enters the tile, if it ends in its first worker)
        }
      }
    }
    adds.meet(at, run, in, w_open, w_last, [](double p, double q) { return p + q; });
  };
  // records of the runs that enter and leave the tile: their sums
  auto keep_sums = [&]() {
    if (at_first) {
#pragma unroll
      for (int c = 0; c < VEC; ++c) pb[c] = rows_pick(at.end != 0, in[c], run[c]);
    }
    if (at_last) {
#pragma unroll
      for (int c = 0; c < VEC; ++c) pb[K + c] = rows_pick(none, in[c], run[c]);
    }
  };
  if constexpr (kEntries) {
    if constexpr (MODE == GS_SOFTMAX)
      sums([&](int i, int c) { return to_acc<T>(x[i].v[c]); });
    else if constexpr (MODE == GS_LOG_SOFTMAX)
      sums([&](int i, int c) { return round_elem<T>(exp_acc(to_acc<T>(x[i].v[c]))); });
    else if constexpr (MODE == GS_SOFTMAX_BWD)
      sums([&](int i, int c) { return to_acc<T>(x[i].v[c]) * to_acc<T>(y[i].v[c]); });
    else
      sums([&](int i, int c) { return to_acc<T>(y[i].v[c]); });
    keep_sums();
    if constexpr (MODE == GS_LOG_SOFTMAX) {
      // the logarithm once for a group, not at every place where some lane of the wavefront has an end
      rows_at_ends<S>(at.end | (at.leaves ? 1u << S : 0u), [&](int i) {
        const bool back = at.enters && i == fe;
#pragma unroll
        for (int c = 0; c < VEC; ++c) {
          F s = i == S ? (F)run[c] : (F)in[c];
#pragma unroll
          for (int j = 0; j < S; ++j) s = rows_pick(i == j && !back, sum[j][c], s);
          s = round_elem<T>(log_acc(round_elem<T>(round_elem<T>(s) + eps)));
#pragma unroll
          for (int j = 0; j < S; ++j) sum[j][c] = rows_pick(i == j, s, sum[j][c]);
          m[0][c] = rows_pick(i == S, s, m[0][c]);
        }
      });
    }
    F cur[VEC];  // of the run of the place: sum, log-softmax its logarithm
#pragma unroll
    for (int c = 0; c < VEC; ++c) cur[c] = MODE == GS_LOG_SOFTMAX ? m[0][c] : (F)run[c];
#pragma unroll
    for (int i = S - 1; i >= 0; --i) {
      const bool end = (at.end >> i & 1u) != 0, back = MODE != GS_LOG_SOFTMAX && at.enters && i <= fe;
#pragma unroll
      for (int c = 0; c < VEC; ++c) {
        cur[c] = rows_pick(end, sum[i][c], cur[c]);
        sum[i][c] = round_elem_if<T, !kBackward>(rows_pick(back, (F)in[c], cur[c]));
      }
      if ((inside >> i & 1u) == 0) continue;
      V r;
#pragma unroll
      for (int c = 0; c < VEC; ++c) {
        const F xv = to_acc<T>(x[i].v[c]);
        F res, s = sum[i][c];
        if (MODE == GS_SOFTMAX) {
          res = rows_divide(xv, s);
        } else if (MODE == GS_LOG_SOFTMAX) {
          asm volatile("" : "+v"(s));  // see group_finish_kernel
          res = xv - s;
        } else if (MODE == GS_SOFTMAX_BWD) {
          res = xv * (to_acc<T>(y[kBackward ? i : 0].v[c]) - s);
        } else {
          res = to_acc<T>(y[kBackward ? i : 0].v[c]) - exp_acc(xv) * s;
        }
        r.v[c] = from_acc<T>(res);
      }
      rows_store<T, VEC>(static_cast<T *>(g.out) + (int64_t)row[i] * K + col, r, f.stream != 0);
    }
  } else if constexpr (MODE == GS_SUM) {
    sums([&](int i, int c) { return to_acc<T>(x[i].v[c]); });
    keep_sums();
    rows_at_ends<S>(at.end & inside, [&](int i) {
      const bool back = at.enters && i == fe;
      int32_t group = gr[1];
#pragma unroll
      for (int j = 1; j < S; ++j) group = rows_pick(i == j, gr[j + 1], group);
      V r;
#pragma unroll
      for (int c = 0; c < VEC; ++c) {
        F s = (F)in[c];
#pragma unroll
        for (int j = 0; j < S; ++j) s = rows_pick(i == j && !back, sum[j][c], s);
        r.v[c] = from_acc<T>(s);
      }
      rows_store<T, VEC>(static_cast<T *>(g.out) + (int64_t)group * K + col, r, false);
    });
  } else if constexpr (MODE == GS_LSE) {
    sums([&](int i, int c) { return round_elem<T>(to_acc<T>(x[i].v[c])); });
    keep_sums();
    rows_at_ends<S>(at.end & inside, [&](int i) {
      const bool back = at.enters && i == fe;
      int32_t group = gr[1];
#pragma unroll
      for (int j = 1; j < S; ++j) group = rows_pick(i == j, gr[j + 1], group);
      V r;
#pragma unroll
      for (int c = 0; c < VEC; ++c) {
        F s = (F)in[c], top = m[0][c];
#pragma unroll
        for (int j = 0; j < S; ++j) {
          s = rows_pick(i == j && !back, sum[j][c], s);
          top = rows_pick(i == j, m[j][c], top);
        }
        r.v[c] = group_lse_of<T>(top, s, eps);
      }
      rows_store<T, VEC>(static_cast<T *>(g.out) + (int64_t)group * K + col, r, false);
    });
  } else {
    // ---- std: sums, means (in m), sums of squared deviations
    sums([&](int i, int c) { return to_acc<T>(x[i].v[c]); });
    // entries of the run that enters, that ends at place i, that leaves
    const int start = at.enters ? w_open * S + (int)s_head[w_open] : 0;
    auto count_at = [&](int i) {
      const uint32_t before = at.head & ((2u << i) - 1u);
      return before != 0 ? i + 1 - (31 - __builtin_clz(before)) : w * S + i + 1 - start;
    };
    int32_t cnt_out = 0;
    if (at.leaves) {
      const int from = at.whole ? start : w * S + (int)s_head[w], v = at.whole ? rows_next_open(s_whole, w) : w_last;
      cnt_out = v * S + (int)s_end[v] + 1 - from;
    }
    double total_first[VEC], total_last[VEC];
#pragma unroll
    for (int c = 0; c < VEC; ++c) {
      total_first[c] = rows_pick(at.end != 0, in[c], run[c]);
      total_last[c] = rows_pick(none, in[c], run[c]);
    }
    // at the ends (and for the run that leaves): total and mean
    F mean_out[VEC] = {};
    rows_at_ends<S>(at.end | (at.leaves ? 1u << S : 0u), [&](int i) {
      const bool back = at.enters && i == fe;
      const int32_t cnt = i == S ? cnt_out : count_at(i);
      int32_t group = gr[1];
#pragma unroll
      for (int j = 1; j < S; ++j) group = rows_pick(i == j, gr[j + 1], group);
      V tot;
#pragma unroll
      for (int c = 0; c < VEC; ++c) {
        F s = rows_pick(i == S, (F)run[c], (F)in[c]);
#pragma unroll
        for (int j = 0; j < S; ++j) s = rows_pick(i == j && !back, sum[j][c], s);
        tot.v[c] = from_acc<T>(s);
        const F mean = group_mean<T>(tot.v[c], cnt);
#pragma unroll
        for (int j = 0; j < S; ++j) sum[j][c] = rows_pick(i == j, mean, sum[j][c]);
        mean_out[c] = rows_pick(i == S, mean, mean_out[c]);
      }
      if ((inside >> i & 1u) != 0) rows_store<T, VEC>(static_cast<T *>(g.total_w) + (int64_t)group * K + col, tot, false);
    });
#pragma unroll
    for (int i = S - 1; i >= 0; --i) {
#pragma unroll
      for (int c = 0; c < VEC; ++c) m[i][c] = mean_out[c] = rows_pick((at.end >> i & 1u) != 0, sum[i][c], mean_out[c]);
    }
    sums([&](int i, int c) {
      const F d = round_elem<T>(to_acc<T>(x[i].v[c]) - m[i][c]);
      return round_elem<T>(d * d);
    });
    // a run that crosses tiles: its sum, and the squared deviations from the mean of its part here, taken to that mean itself
    auto part = [&](int64_t o, double total, double dev, F mean, int32_t entries) {
      const double d = total / entries - (double)mean, m2 = dev - entries * d * d;
      pa[o] = (uint64_t)__double_as_longlong(total);
      pb[o] = m2 < 0.0 ? 0.0 : m2;
    };
    if (at_first) {
      const int32_t entries = at.end != 0 ? fe + 1 : cnt_out;  // (the run begins with the worker)
#pragma unroll
      for (int c = 0; c < VEC; ++c) part(c, total_first[c], rows_pick(at.end != 0, in[c], run[c]), m[0][c], entries);
    }
    if (at_last) {
#pragma unroll
      for (int c = 0; c < VEC; ++c) part(K + c, total_last[c], rows_pick(none, in[c], run[c]), m[S - 1][c], count_at(S - 1));
    }
    rows_at_ends<S>(at.end & inside, [&](int i) {
      const bool back = at.enters && i == fe;
      const F div = group_divisor<T>(count_at(i), g.unbiased);
      int32_t group = gr[1];
#pragma unroll
      for (int j = 1; j < S; ++j) group = rows_pick(i == j, gr[j + 1], group);
      V r;
#pragma unroll
      for (int c = 0; c < VEC; ++c) {
        F s = (F)in[c];
#pragma unroll
        for (int j = 0; j < S; ++j) s = rows_pick(i == j && !back, sum[j][c], s);
        r.v[c] = from_acc<T>(sqrt_acc(round_elem<T>(round_elem<T>(s) / div)));
      }
      rows_store<T, VEC>(static_cast<T *>(g.out) + (int64_t)group * K + col, r, false);
    });
  }
  if (tid == 0 && blockIdx.y == 0) {
    int32_t *meta = f.meta + t * 4;
    const int64_t e0 = f.ptr[g_first + 1] - w0, s1 = f.ptr[g_last] - w0;
    const bool one = span.enters && span.leaves && g_first == g_last;
    meta[0] = span.enters ? (e0 < span.b ? (int32_t)e0 : span.b) : 0;
    meta[1] = one || !span.leaves ? span.b : (int32_t)s1;
    meta[2] = span.b;
    meta[3] = one ? 1 : 0;
  }
}

// The partials of a group that crosses tiles meet in the tile in which it begins (its leaving run), once for all tiles that it
// crosses (every tile for itself is quadratic in their number). Softmax leaves the result there; logsumexp and std write the
// group's result, and the workgroups together the groups without entries (std: and all counts). A team of sixteen lanes takes
// sixteen columns of such a group, the workgroup those that cross more than 64 tiles: 64 partials by eight on the way together.
template <typename T, int MODE>
__global__ __launch_bounds__(kRowsCombine) void group_rows_combine_kernel(GroupArgs g, GroupRowsArgs f) {
  constexpr bool kBackward = MODE == GS_SOFTMAX_BWD || MODE == GS_LOG_SOFTMAX_BWD || MODE == GS_SUM;  // (a sum alone)
  constexpr bool kReduce = MODE == GS_LSE || MODE == GS_STD || MODE == GS_SUM;
  // the kind of partial: log-softmax as softmax, the backward passes carry a sum alone
  typedef GroupBinPart<T, MODE == GS_STD ? GS_STD : MODE == GS_LSE ? GS_LSE : GS_SOFTMAX> Part;
  __shared__ Part s_part[kRowsCombine];
  __shared__ int32_t s_long[kRowsTeams];
  __shared__ int s_n;
  if (f.gate != nullptr && *f.gate == 0) return;
  const int tid = threadIdx.x;
  if constexpr (kReduce) {
    T *out = static_cast<T *>(g.out), *total = static_cast<T *>(g.total_w);
    const int64_t step = (int64_t)gridDim.x * kRowsCombine;
    if (blockIdx.y == 0) {
      for (int64_t i = (int64_t)blockIdx.x * kRowsCombine + tid; i < (g.N + kWave - 1) / kWave * kWave; i += step) {
        const int64_t len = i < g.N ? f.ptr[i + 1] - f.ptr[i] : 1;
        if (MODE == GS_STD && i < g.N) g.count_w[i] = (int32_t)len;
        if (g.K <= 16) {  // few columns: a lane its own
          for (int64_t k = len == 0 ? 0 : g.K; k < g.K; ++k) {
            out[i * g.K + k] = from_acc<T>((typename Acc<T>::type)0);
            if (MODE == GS_STD) total[i * g.K + k] = from_acc<T>((typename Acc<T>::type)0);
          }
          continue;
        }
        uint64_t empty = __ballot(len == 0);
        const int64_t base = i - (tid & (kWave - 1));
        while (empty != 0) {  // the wavefront's empty groups, one after the other
          const int64_t row = (base + __builtin_ctzll(empty)) * g.K;
          empty &= empty - 1;
          for (int64_t k = tid & (kWave - 1); k < g.K; k += kWave) {
            out[row + k] = from_acc<T>((typename Acc<T>::type)0);
            if (MODE == GS_STD) total[row + k] = from_acc<T>((typename Acc<T>::type)0);
          }
        }
      }
    }
  }
  const int64_t n = f.ptr[g.N], tiles = (n + f.tw - 1) / f.tw, t0 = (int64_t)blockIdx.x * kRowsTeams;
  if (t0 >= tiles) return;
  const int K = (int)g.K, team = tid / kRowsTeam, k = (int)blockIdx.y * kRowsTeam + (tid & (kRowsTeam - 1));
  const bool col_on = k < K;
  // partials i0, i0 + step, ... of the run that begins in tile t: U on the way together (past the end: the last tile's again)
  auto add_up = [&](auto u_const, int64_t t, int32_t first_n, int64_t i0, int step, int64_t last) {
    constexpr int U = decltype(u_const)::value;
    Part sum = Part::identity();
    if (kBackward) sum.a = 0;
    for (; i0 <= last; i0 += U * step) {
      Part p[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int64_t i = i0 + u * step < last ? i0 + u * step : last;
        const int64_t at = (i * 2 + (i == t ? 1 : 0)) * K + (col_on ? k : 0);
        p[u].a = kBackward ? 0 : f.pa[at];
        p[u].b = f.pb[at];
        p[u].n = MODE == GS_STD ? (i == t ? first_n : f.meta[i * 4]) : 0;
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (i0 + u * step > last) continue;
        if constexpr (kBackward)
          sum.b += p[u].b;
        else
          sum.absorb(p[u]);
      }
    }
    return sum;
  };
  auto leave = [&](int64_t t, int32_t group, const Part &r) {
    if (!col_on) return;
    if constexpr (MODE == GS_SUM) {
      static_cast<T *>(g.out)[(int64_t)group * K + k] = from_acc<T>((typename Acc<T>::type)r.b);
    } else if constexpr (MODE == GS_STD || MODE == GS_LSE) {
      group_bin_emit<T, MODE>(g, (int64_t)group * K + k, group, k, r);
    } else {
      const int64_t at = (t * 2 + 1) * K + k;
      if (!kBackward) f.pa[at] = r.a;
      f.pb[at] = r.b;
    }
  };
  if (tid == 0) s_n = 0;
  __syncthreads();
  const int64_t t_own = t0 + team;
  if (t_own < tiles) {
    const int32_t begin = f.meta[t_own * 4 + 1], end = f.meta[t_own * 4 + 2];
    if (begin < end && f.meta[t_own * 4 + 3] == 0) {  // a group begins here and goes on
      const int32_t group = f.group[t_own * f.tw + end - 1];
      const int64_t last = (f.ptr[group + 1] - 1) / f.tw;
      if (last - t_own <= kRowsTeamSpan)
        leave(t_own, group, add_up(std::integral_constant<int, 4>(), t_own, end - begin, t_own, 1, last));
      else if ((tid & (kRowsTeam - 1)) == 0)
        s_long[atomicAdd(&s_n, 1)] = team;
    }
  }
  __syncthreads();
  const int found = s_n;
  for (int q = 0; q < found; ++q) {
    const int64_t t = t0 + s_long[q];
    const int32_t begin = f.meta[t * 4 + 1], end = f.meta[t * 4 + 2], group = f.group[t * f.tw + end - 1];
    s_part[tid] = add_up(std::integral_constant<int, 8>(), t, end - begin, t + team, kRowsTeams, (f.ptr[group + 1] - 1) / f.tw);
    __syncthreads();
    for (int half = kRowsTeams / 2; half >= 1; half >>= 1) {
      if (team < half) {
        if constexpr (kBackward)
          s_part[tid].b += s_part[tid + half * kRowsTeam].b;
        else
          s_part[tid].absorb(s_part[tid + half * kRowsTeam]);
      }
      __syncthreads();
    }
    if (team == 0) leave(t, group, s_part[tid]);
    __syncthreads();
  }
}

// softmax, the places of a tile that belong to a group put together from several tiles: from src, as in group_rows_kernel
template <typename T, int VEC, int MODE>
__global__ __launch_bounds__(kRowsBlock) void group_rows_finish_kernel(GroupArgs g, GroupRowsArgs f) {
  typedef typename Acc<T>::type F;
  typedef typename OrdKey<F>::bits KB;
  typedef Vec<T, VEC> V;
  constexpr int S = kRowsHeld;
  constexpr bool kBackward = MODE == GS_SOFTMAX_BWD || MODE == GS_LOG_SOFTMAX_BWD;
  if (f.gate != nullptr && *f.gate == 0) return;
  const int64_t n = f.ptr[g.N], t = blockIdx.x, w0 = t * f.tw;
  if (w0 >= n) return;
  const int head_len = f.meta[t * 4], tail_start = f.meta[t * 4 + 1], ne = f.meta[t * 4 + 2];
  if (head_len <= 0 && tail_start >= ne) return;
  const int tid = threadIdx.x, K = (int)g.K, L = f.lanes;
  const int w = (int)(((uint32_t)tid * f.inv) >> 16), l = tid - w * L;
  const int k_first = (int)blockIdx.y * f.kcols, k_end = K - k_first < f.kcols ? K : k_first + f.kcols;
  const int first = k_first + l * VEC, p0 = w * S;
  if (w >= f.workers || first >= k_end || p0 >= ne || (p0 >= head_len && p0 + S <= tail_start)) return;
  const int col = first + VEC <= K ? first : K - VEC;
  const bool through = f.state[0] != 0;
  int32_t gr[S + 2], row[S];
  rows_load_order(f, w0 + p0, g.E, gr, row);
  V x[S], y[kBackward ? S : 1];
  bool on[S];
#pragma unroll
  for (int i = 0; i < S; ++i) {
    const int p = p0 + i;
    on[i] = p < head_len || (p >= tail_start && p < ne);
    row[i] = on[i] ? (through ? row[i] : (int32_t)(w0 + p)) : 0;
    const int64_t o = (int64_t)row[i] * K + col;
    x[i] = rows_load<T, VEC>(static_cast<const T *>(g.src) + o);
    if constexpr (kBackward) y[i] = rows_load<T, VEC>(static_cast<const T *>(g.grad) + o);
  }
  // the entering run's values lie with the tile in which it begins, the leaving run's here or, if it fills the tile, there as well
  const F eps = (F)g.eps;
  F top[2][VEC], sum[2][VEC];
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    if (r == 0 ? head_len <= 0 : tail_start >= ne) {
#pragma unroll
      for (int c = 0; c < VEC; ++c) top[r][c] = sum[r][c] = (F)0;
      continue;
    }
    const int64_t begin = r == 0 ? (int64_t)((uint32_t)f.ptr[f.group[w0]] / (uint32_t)f.tw) : t;
#pragma unroll
    for (int c = 0; c < VEC; ++c) {
      const int64_t at = (begin * 2 + 1) * K + col + c;
      const F s = (F)f.pb[at];
      if constexpr (kBackward) {
        top[r][c] = (F)0;
        sum[r][c] = s;
      } else {
        const KB key = (KB)f.pa[at];
        top[r][c] = key == group_empty_key<T>() ? (F)0 : OrdKey<F>::dec(key);
        sum[r][c] = MODE == GS_SOFTMAX ? round_elem<T>(s) : round_elem<T>(log_acc(round_elem<T>(round_elem<T>(s) + eps)));
      }
    }
  }
#pragma unroll
  for (int i = 0; i < S; ++i) {
    if (!on[i]) continue;
    const int r = p0 + i < head_len ? 0 : 1;
    V o;
#pragma unroll
    for (int c = 0; c < VEC; ++c) {
      const F xv = to_acc<T>(x[i].v[c]), m = r == 0 ? top[0][c] : top[1][c];
      F res, s = r == 0 ? sum[0][c] : sum[1][c];
      if (MODE == GS_SOFTMAX) {
        res = round_elem<T>(exp_acc(round_elem<T>(xv - m))) / s;
      } else if (MODE == GS_LOG_SOFTMAX) {
        asm volatile("" : "+v"(s));  // see group_finish_kernel
        res = round_elem<T>(xv - m) - s;
      } else if (MODE == GS_SOFTMAX_BWD) {
        res = xv * (to_acc<T>(y[kBackward ? i : 0].v[c]) - s);
      } else {
        res = to_acc<T>(y[kBackward ? i : 0].v[c]) - exp_acc(xv) * s;
      }
      o.v[c] = from_acc<T>(res);
    }
    rows_store<T, VEC>(static_cast<T *>(g.out) + (int64_t)row[i] * K + col, o, f.stream != 0);
  }
}

// Backward of std and logsumexp over the order of the forward pass: a place's row of src is gathered and its gradient goes
// out; what it needs of its group (std: sum, count, result, gradient; logsumexp: result, gradient) is read by neighbouring
// places together. (In the order of memory every entry fetches two lines of its group from anywhere.)
constexpr int kRowsMapHeld = 4;  // places of a worker
template <typename T, int VEC, int MODE>
__global__ __launch_bounds__(kRowsBlock) void group_rows_map_kernel(GroupArgs g, GroupRowsArgs f) {
  typedef typename Acc<T>::type F;
  typedef Vec<T, VEC> V;
  constexpr int S = kRowsMapHeld;
  const int tid = threadIdx.x, K = (int)g.K, L = f.lanes;
  const int w = (int)(((uint32_t)tid * f.inv) >> 16), l = tid - w * L;
  // (an index in order that other tiles took: no order, the groups come from the index)
  const bool here = f.state[4] == 0;
  const int64_t n = here ? g.E : f.ptr[g.N], w0 = (int64_t)blockIdx.x * (f.workers * S);
  const int k_first = (int)blockIdx.y * f.kcols, k_end = K - k_first < f.kcols ? K : k_first + f.kcols;
  if (n != g.E) {  // zeros for the entries that belong to no group
    for (int64_t be = w0 + tid / kWave; be < g.E && be < w0 + f.workers * S; be += kRowsBlock / kWave) {
      int64_t b, e;
      split_edge(be, g.E / f.E0, f.E0, b, e);
      const int64_t at = f.index[b * f.sb + e * f.se];
      if (at >= 0 && at < f.N0) continue;
      for (int k = k_first + (tid & (kWave - 1)); k < k_end; k += kWave)
        static_cast<T *>(g.out)[be * K + k] = from_acc<T>((F)0);
    }
  }
  const int first = k_first + l * VEC;
  const int64_t p0 = w0 + w * S;
  if (w >= f.workers || first >= k_end || p0 >= n) return;
  const int col = first + VEC <= K ? first : K - VEC;
  int32_t gr[S], row[S];
  bool none[S];
#pragma unroll
  for (int i = 0; i < S; ++i) none[i] = false;
  if (here) {
#pragma unroll
    for (int i = 0; i < S; ++i) {
      const int64_t p = p0 + i < n ? p0 + i : n - 1;
      int64_t b, e;
      split_edge(p, g.E / f.E0, f.E0, b, e);
      const int64_t at = f.index[b * f.sb + e * f.se];
      none[i] = at < 0 || at >= f.N0;
      gr[i] = none[i] ? 0 : (int32_t)(b * f.N0 + at);
      row[i] = (int32_t)p;
    }
  } else {
    const bool through = f.state[0] != 0;
#pragma unroll
    for (int i = 0; i < S; ++i) gr[i] = f.group[p0 + i < n ? p0 + i : n - 1];
#pragma unroll
    for (int i = 0; i < S; ++i) {
      const int64_t p = p0 + i < n ? p0 + i : n - 1;
      row[i] = through ? f.perm[p] : (int32_t)p;
    }
  }
  V x[S], res[S], go[S], tot[MODE == GS_STD_BWD ? S : 1];
  int32_t cnt[MODE == GS_STD_BWD ? S : 1];
#pragma unroll
  for (int i = 0; i < S; ++i) {
    const int64_t at = (int64_t)gr[i] * K + col;
    x[i] = rows_load<T, VEC>(static_cast<const T *>(g.src) + (int64_t)row[i] * K + col);
    res[i] = rows_load<T, VEC>(static_cast<const T *>(g.node_out) + at);
    go[i] = rows_load<T, VEC>(static_cast<const T *>(g.node_grad) + at);
    if constexpr (MODE == GS_STD_BWD) {
      tot[i] = rows_load<T, VEC>(static_cast<const T *>(g.total) + at);
      cnt[i] = g.count[gr[i]];
    }
  }
#pragma unroll
  for (int i = 0; i < S; ++i) {
    if (p0 + i >= n) continue;
    V o;
#pragma unroll
    for (int c = 0; c < VEC; ++c) {
      const F xv = to_acc<T>(x[i].v[c]), ov = to_acc<T>(res[i].v[c]), gv = to_acc<T>(go[i].v[c]);
      if constexpr (MODE == GS_STD_BWD) {
        // a group whose std is 0 gets 0 / 0 = NaN, as autograd gives for the reference's sqrt at 0
        const F wt = gv / (ov * group_divisor<T>(cnt[i], g.unbiased));
        o.v[c] = from_acc<T>(none[i] ? (F)0 : wt * (xv - group_mean<T>(tot[i].v[c], cnt[i])));
      } else {
        const F e = exp_acc(xv - ov);
        o.v[c] = from_acc<T>(none[i] || xv != xv || e != e ? (F)0 : gv * e);
      }
    }
    rows_store<T, VEC>(static_cast<T *>(g.out) + (int64_t)row[i] * K + col, o, f.stream != 0);
  }
}

// Backward of a scatter sum or mean over the order of its forward pass: every entry's gradient is its row's (divided by the row's
// entries). Places of a row read it together, and only the entries' rows are written in no order, in whole pieces: 2.3 M x 128 bf16
// onto 268 k rows, 115 us (5.7 TB/s) against 165 for a gather in the order of memory, which fetches every row from anywhere.
struct RowsSpreadArgs {
  const void *grad;  // [rows, K]
  void *grad_in;     // [n, K]
  int64_t K;
  int lanes, workers;
  uint32_t inv;
  int kcols, stream;
};
template <typename T, int VEC, bool DIV>
__global__ __launch_bounds__(kBlock) void rows_spread_kernel(RowSortArgs p, RowsSpreadArgs a) {
  typedef Vec<T, VEC> V;
  constexpr int Q = 4;
  typedef int32_t i4 __attribute__((ext_vector_type(4)));
  const int tid = threadIdx.x, K = (int)a.K, L = a.lanes;
  const int w = (int)(((uint32_t)tid * a.inv) >> 16), l = tid - w * L;
  const int64_t n = p.ptr[p.rows], w0 = (int64_t)blockIdx.x * (a.workers * Q);
  const int k_first = (int)blockIdx.y * a.kcols, k_end = K - k_first < a.kcols ? K : k_first + a.kcols;
  T *out = static_cast<T *>(a.grad_in);
  if (n != p.n) {  // zeros for the entries outside [0, N)
    for (int64_t e = w0 + tid / kWave; e < p.n && e < w0 + a.workers * Q; e += kBlock / kWave) {
      if (rs_node(p, e) >= 0) continue;
      for (int k = k_first + (tid & (kWave - 1)); k < k_end; k += kWave) out[e * K + k] = zero_elem<T>();
    }
  }
  const int first = k_first + l * VEC;
  const int64_t p0 = w0 + w * Q;
  if (w >= a.workers || first >= k_end || p0 >= n) return;
  const int col = first + VEC <= K ? first : K - VEC;  // (the last lane: columns that its neighbour has as well)
  const i4 row = *reinterpret_cast<const i4 *>(p.perm_row + p0);  // (the arrays end on whole 256 bytes)
  i4 entry = {(int)p0, (int)p0 + 1, (int)p0 + 2, (int)p0 + 3};
  if (p.state[0] != 0) entry = *reinterpret_cast<const i4 *>(p.perm + p0);
  V g[Q];
  int64_t len[DIV ? Q : 1];
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    const int64_t r = p0 + q < n ? row[q] : row[0];
    g[q] = rows_load<T, VEC>(static_cast<const T *>(a.grad) + r * K + col);
    if constexpr (DIV) len[q] = p.ptr[r + 1] - p.ptr[r];
  }
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    if (p0 + q >= n) continue;
    if constexpr (DIV) {
#pragma unroll
      for (int v = 0; v < VEC; ++v) g[q].v[v] = div_elem<T>(g[q].v[v], count_as<T>(len[q]));
    }
    rows_store<T, VEC>(out + (int64_t)entry[q] * K + col, g[q], a.stream != 0);
  }
}
template <typename T> int launch_rows_spread(const RowSortArgs &p, const void *grad, void *grad_in, int64_t K, bool mean, hipStream_t stream);
template <typename T> int launch_rows_spread_t(const RowSortArgs &p, const void *grad, void *grad_in, int64_t K, bool mean, hipStream_t stream) {
  constexpr int VEC = kVecBytes / (int)sizeof(T);
  RowsSpreadArgs a;
  a.grad = grad;
  a.grad_in = grad_in;
  a.K = K;
  const int64_t all = (K + VEC - 1) / VEC, slices = (all + kWave - 1) / kWave;
  if (K < VEC || slices > 65535 || K > 0x7FFFFFFFll) return TS_ERR_UNSUPPORTED;
  a.lanes = (int)((all + slices - 1) / slices);
  a.workers = kBlock / a.lanes;
  a.inv = 65536u / (uint32_t)a.lanes + 1;
  a.kcols = a.lanes * VEC;
  a.stream = K * (int64_t)sizeof(T) % 128 == 0 && (reinterpret_cast<uintptr_t>(grad_in) & 127) == 0;
  const int64_t per = (int64_t)a.workers * 4;
  const dim3 grid((unsigned)((p.n + per - 1) / per), (unsigned)((all + a.lanes - 1) / a.lanes));
  if (mean)
    hipLaunchKernelGGL((rows_spread_kernel<T, VEC, true>), grid, dim3(kBlock), 0, stream, p, a);
  else
    hipLaunchKernelGGL((rows_spread_kernel<T, VEC, false>), grid, dim3(kBlock), 0, stream, p, a);
  return hipGetLastError() == hipSuccess ? TS_OK : TS_ERR_LAUNCH;
}

template <typename T, int VEC, int MODE> int launch_group_rows_m(const GroupArgs &g, const GroupRowsArgs &f, hipStream_t stream) {
  constexpr bool kReduce = MODE == GS_LSE || MODE == GS_STD || MODE == GS_SUM;
  if constexpr (MODE == GS_STD_BWD || MODE == GS_LSE_BWD) {
    const int64_t per = (int64_t)f.workers * kRowsMapHeld;
    hipLaunchKernelGGL((group_rows_map_kernel<T, VEC, MODE>), dim3((unsigned)((g.E + per - 1) / per), (unsigned)f.slices),
                       dim3(kRowsBlock), 0, stream, g, f);
  } else {
    const dim3 grid((unsigned)f.nt, (unsigned)f.slices);
    hipLaunchKernelGGL((group_rows_kernel<T, VEC, MODE>), grid, dim3(kRowsBlock), 0, stream, g, f);
    int64_t shares = (f.nt + kRowsTeams - 1) / kRowsTeams;
    if (kReduce) {  // (and a workgroup for 1024 groups, which may be empty: 450 k single values onto 266 k rows, ten workgroups 347 us)
      const int64_t want = (g.N + kRowsCombine - 1) / kRowsCombine;
      shares = shares < want ? (want < 2048 ? want : 2048 < shares ? shares : 2048) : shares;
    }
    hipLaunchKernelGGL((group_rows_combine_kernel<T, MODE>), dim3((unsigned)shares, (unsigned)((g.K + kRowsTeam - 1) / kRowsTeam)),
                       dim3(kRowsCombine), 0, stream, g, f);
    if constexpr (!kReduce) hipLaunchKernelGGL((group_rows_finish_kernel<T, VEC, MODE>), grid, dim3(kRowsBlock), 0, stream, g, f);
  }
  return hipGetLastError() == hipSuccess ? TS_OK : TS_ERR_LAUNCH;
}
template <typename T, int VEC> int launch_group_rows_v(const GroupArgs &g, const GroupRowsArgs &f, int mode, hipStream_t stream) {
  switch (mode) {
  case GS_SOFTMAX: return launch_group_rows_m<T, VEC, GS_SOFTMAX>(g, f, stream);
  case GS_LOG_SOFTMAX: return launch_group_rows_m<T, VEC, GS_LOG_SOFTMAX>(g, f, stream);
  case GS_SOFTMAX_BWD: return launch_group_rows_m<T, VEC, GS_SOFTMAX_BWD>(g, f, stream);
  case GS_LOG_SOFTMAX_BWD: return launch_group_rows_m<T, VEC, GS_LOG_SOFTMAX_BWD>(g, f, stream);
  case GS_LSE: return launch_group_rows_m<T, VEC, GS_LSE>(g, f, stream);
  case GS_LSE_BWD: return launch_group_rows_m<T, VEC, GS_LSE_BWD>(g, f, stream);
  case GS_STD: return launch_group_rows_m<T, VEC, GS_STD>(g, f, stream);
  case GS_STD_BWD: return launch_group_rows_m<T, VEC, GS_STD_BWD>(g, f, stream);
  case GS_SUM: return launch_group_rows_m<T, VEC, GS_SUM>(g, f, stream);
  default: return TS_ERR_BAD_ARG;
  }
}
template <typename T> int launch_group_rows(const GroupArgs &g, const GroupRowsArgs &f, int mode, hipStream_t stream);

#define TS_INSTANTIATE_GROUP_ROWS(T)                                                                              \
  template <> int launch_group_rows<T>(const GroupArgs &g, const GroupRowsArgs &f, int mode, hipStream_t stream) { \
    if (g.K >= group_rows_full<T>()) return launch_group_rows_v<T, group_rows_full<T>()>(g, f, mode, stream);     \
    return launch_group_rows_v<T, 1>(g, f, mode, stream);                                                         \
  }                                                                                                               \
  template <> int launch_rows_spread<T>(const RowSortArgs &p, const void *grad, void *grad_in, int64_t K, bool mean, \
                                        hipStream_t stream) {                                                     \
    return launch_rows_spread_t<T>(p, grad, grad_in, K, mean, stream);                                            \
  }

}  // namespace ts
