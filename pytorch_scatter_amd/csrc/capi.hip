// The C ABI declared in include/ts_hip.h: argument checks, kernel plans and
// dispatch on the element type. Nothing here allocates or synchronises.
#include <hip/hip_runtime.h>
#include <hip/hip_version.h>
#include <stdlib.h>

#include <atomic>
#include <chrono>
#include <type_traits>

#include "csr_reduce.h"
#include "csr_gather.h"
#include "coo_gather.h"
#include "scatter.h"
#include "elementwise.h"
#include "group_softmax.h"
#include "group_rows.h"
#include "index_format.h"
#include "row_sort.h"
#include "scatter_small.h"

using namespace ts;

namespace {

const int kElemBytes[9] = {4, 8, 2, 2, 4, 8, 2, 1, 1};
const int kAccBytes[9] = {4, 8, 4, 4, 4, 8, 2, 1, 1};

inline bool valid_dtype(int d) { return d >= 0 && d < 9; }
inline bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }
inline bool is_float_dtype(int d) { return d == TS_F32 || d == TS_F64 || d == TS_F16 || d == TS_BF16; }

#define TS_DISPATCH(dtype, EXPR)                      \
  switch (dtype) {                                    \
  case TS_F32: { typedef float T; return EXPR; }      \
  case TS_F64: { typedef double T; return EXPR; }     \
  case TS_F16: { typedef f16_t T; return EXPR; }      \
  case TS_BF16: { typedef bf16_t T; return EXPR; }    \
  case TS_I32: { typedef int32_t T; return EXPR; }    \
  case TS_I64: { typedef int64_t T; return EXPR; }    \
  case TS_I16: { typedef int16_t T; return EXPR; }    \
  case TS_I8: { typedef int8_t T; return EXPR; }      \
  case TS_U8: { typedef uint8_t T; return EXPR; }     \
  default: return TS_ERR_BAD_ARG;                     \
  }

int dispatch_csr_reduce(int dtype, const CsrReduceArgs &a, const CsrPlan &p, int64_t B, int reduce,
                        hipStream_t s) {
  TS_DISPATCH(dtype, launch_csr_reduce<T>(a, p, B, reduce, s))
}
int dispatch_csr_gather(int dtype, const CsrGatherArgs &a, const CsrPlan &p, int64_t B, bool divide,
                        hipStream_t s) {
  TS_DISPATCH(dtype, launch_csr_gather<T>(a, p, B, divide, s))
}
int dispatch_coo_gather(int dtype, const CooGatherArgs &a, const CooGatherPlan &p, int64_t B,
                        bool divide, hipStream_t s) {
  TS_DISPATCH(dtype, launch_coo_gather<T>(a, p, B, divide, s))
}
int dispatch_scatter(int dtype, const ScatterArgs &a, int reduce, int vec, hipStream_t s) {
  TS_DISPATCH(dtype, launch_scatter<T>(a, reduce, vec, s))
}
int dispatch_divide(int dtype, void *out, const int32_t *count, int64_t rows, int64_t K, hipStream_t s) {
  TS_DISPATCH(dtype, launch_divide_by_count<T>(out, count, rows, K, s))
}
int dispatch_sorted_args(int dtype, void *out, int64_t *arg, const int32_t *perm, int64_t B, int64_t per_batch,
                         int64_t E, int64_t perm_batch_stride, bool is_max, hipStream_t s) {
  TS_DISPATCH(dtype, launch_sorted_args<T>(out, arg, perm, B, per_batch, E, perm_batch_stride, is_max, s))
}
int dispatch_arg_backward(int dtype, const void *g, const int64_t *arg, void *gi, int64_t B, int64_t N,
                          int64_t E, int64_t K, hipStream_t s) {
  TS_DISPATCH(dtype, launch_arg_backward<T>(g, arg, gi, B, N, E, K, s))
}

int dispatch_group_softmax(int dtype, const GroupArgs &g, int mode, int vec, hipStream_t s) {
  switch (dtype) {
  case TS_F32: return launch_group_softmax<float>(g, mode, vec, s);
  case TS_F64: return launch_group_softmax<double>(g, mode, vec, s);
  case TS_F16: return launch_group_softmax<f16_t>(g, mode, vec, s);
  case TS_BF16: return launch_group_softmax<bf16_t>(g, mode, vec, s);
  default: return TS_ERR_UNSUPPORTED;
  }
}

int dispatch_group_rows(int dtype, const GroupArgs &g, const GroupRowsArgs &f, int mode, hipStream_t s) {
  switch (dtype) {
  case TS_F32: return launch_group_rows<float>(g, f, mode, s);
  case TS_F64: return launch_group_rows<double>(g, f, mode, s);
  case TS_F16: return launch_group_rows<f16_t>(g, f, mode, s);
  case TS_BF16: return launch_group_rows<bf16_t>(g, f, mode, s);
  default: return TS_ERR_UNSUPPORTED;
  }
}

// The reductions keep edge positions in 32 bits inside a tile. B is only bounded by the 64-bit element
// offsets: kernels that put the batch into a grid dimension are launched in slices (for_batch_slices).
inline bool sizes_ok(int64_t B, int64_t N, int64_t E, int64_t K) {
  return B >= 0 && N >= 0 && E >= 0 && K >= 0 && E < 0x7FFFFFFFll && N < 0x7FFFFFFFll &&
         B < 0x7FFFFFFFll && K < ((int64_t)1 << 40);
}

// grid.y / grid.z hold at most 65535 workgroups: batches beyond that take further launches on the
// same stream. fn(first batch, number of batches) -> status.
constexpr int64_t kMaxGridBatches = 65535;
template <typename F> int for_batch_slices(int64_t B, F fn) {
  for (int64_t b0 = 0; b0 < B; b0 += kMaxGridBatches) {
    const int rc = fn(b0, B - b0 < kMaxGridBatches ? B - b0 : kMaxGridBatches);
    if (rc != TS_OK) return rc;
  }
  return TS_OK;
}
template <typename P> inline P *offset_bytes(P *p, int64_t bytes) {
  typedef typename std::conditional<std::is_const<P>::value, const char, char>::type C;
  return p == nullptr ? nullptr : reinterpret_cast<P *>(reinterpret_cast<C *>(p) + bytes);
}

int env_int(const char *name, int fallback) {
  const char *v = getenv(name);
  return v ? atoi(v) : fallback;
}

// Tag of one call's carry flags: a process-wide counter that starts at the clock, 1 .. 2^61.
uint64_t next_nonce() {
  static std::atomic<uint64_t> counter{(uint64_t)std::chrono::steady_clock::now().time_since_epoch().count()};
  return (counter.fetch_add(1, std::memory_order_relaxed) & ((1ull << 61) - 1)) + 1;
}

struct CsrWs {
  size_t total, off_args, off_meta;
};

CsrWs csr_workspace(const CsrPlan &p, int64_t B, int64_t K, int dtype, int reduce) {
  CsrWs w;
  w.total = csr_ws_bytes(p, B, K, kAccBytes[dtype], reduce == TS_MIN || reduce == TS_MAX, &w.off_args,
                         &w.off_meta);
  return w;
}

// Workspace for either plan: buffers that are not 16-byte aligned take one element per lane,
// which changes the tile size and with it the number of partial results.
// The last kStatusBytes of what the *_workspace_bytes functions report hold the call's status word.
constexpr size_t kStatusBytes = 256;
size_t csr_workspace_max(int64_t B, int64_t N, int64_t E, int64_t K, int dtype, int reduce, bool allow_small = true) {
  const bool wa = reduce == TS_MIN || reduce == TS_MAX;
  const size_t w1 = csr_workspace(csr_plan(N, E, K, kElemBytes[dtype], true, false, wa, allow_small), B, K, dtype, reduce).total;
  const size_t w0 = csr_workspace(csr_plan(N, E, K, kElemBytes[dtype], false, false, wa, allow_small), B, K, dtype, reduce).total;
  return (w1 > w0 ? w1 : w0) + kStatusBytes;
}
inline unsigned long long *status_word(void *ws, size_t reported_bytes) {
  return reinterpret_cast<unsigned long long *>(static_cast<char *>(ws) + reported_bytes - kStatusBytes);
}

int run_csr_reduce_slice(const void *src, const int64_t *indptr, void *out, int64_t *arg_out, void *count_out,
                         int64_t B, int64_t N, int64_t E, int64_t K, int64_t indptr_batch_stride, int dtype,
                         int reduce, int accumulate, void *ws, size_t ws_bytes, hipStream_t stream,
                         const int32_t *perm, int64_t perm_batch_stride, bool want_perm_args, bool *perm_args_done,
                         unsigned long long *status, bool status_reset, uint64_t status_nonce) {
  const bool al = aligned16(src) && aligned16(out);
  // permuted rows always take the wide kernel (the narrow one stages consecutive entries)
  const CsrPlan p = csr_plan(N, E, K, kElemBytes[dtype], al, false, reduce == TS_MIN || reduce == TS_MAX,
                             perm == nullptr);
  const CsrWs w = csr_workspace(p, B, K, dtype, reduce);
  if (ws == nullptr || ws_bytes < w.total) return TS_ERR_WORKSPACE;
  CsrReduceArgs a;
  a.src = src;
  a.indptr = indptr;
  a.out = out;
  a.arg_out = arg_out;
  a.count_out = count_out;
  a.N = N;
  a.E = E;
  a.K = K;
  a.indptr_batch_stride = indptr_batch_stride;
  a.accumulate = accumulate;
  a.G = p.G;
  a.BI = p.BI;
  a.ipw = p.ipw;
  a.nblk = p.nblk;
  a.ws_vals = ws;
  a.ws_args = reinterpret_cast<int32_t *>(static_cast<char *>(ws) + w.off_args);
  a.ws_meta = reinterpret_cast<int64_t *>(static_cast<char *>(ws) + w.off_meta);
  // rows that cross tiles are finished inside the kernel when the carries fit 32- / 64-bit atomics and the
  // four words of workspace per tile give every column chunk its flag; else by the second kernel
  a.lookback = !p.small && kAccBytes[dtype] >= 4 && p.ychunks <= 4 && p.nblk > 1 && env_int("TS_CSR_LOOKBACK", 1);
  a.nonce = next_nonce();
  a.status = status;
  a.status_reset = status_reset ? 1 : 0;
  a.status_nonce = status_nonce;
  a.carry_spin = env_int("TS_CSR_SPIN", kCarrySpin);  // test aid: -1 makes every look-back give up at once
  a.perm = perm;
  a.perm_batch_stride = perm_batch_stride;
  // every row is finished inside the first kernel unless the second one runs: then the positions can leave it
  // in src's order right away;
  // when the output is large: the lookup at every row end makes the wavefront wait, a pass over [N, K]
  // afterwards moves 20 bytes per element (C4, 3.2 M elements: 13 us as a pass, +17 us fused; 68 M: 334 vs 150 us)
  a.perm_args = perm != nullptr && (a.lookback || p.nblk <= 1) && want_perm_args;
  if (perm_args_done) *perm_args_done = a.perm_args != 0;
  if (p.ychunks > kMaxGridBatches) return TS_ERR_UNSUPPORTED;
  return dispatch_csr_reduce(dtype, a, p, B, reduce, stream);
}

int run_csr_reduce(const void *src, const int64_t *indptr, void *out, int64_t *arg_out, void *count_out,
                   int64_t B, int64_t N, int64_t E, int64_t K, int64_t indptr_batch_stride, int dtype,
                   int reduce, int accumulate, void *ws, size_t ws_bytes, unsigned long long *status,
                   hipStream_t stream, const int32_t *perm = nullptr, int64_t perm_batch_stride = 0,
                   bool *perm_args_done = nullptr) {
  const int64_t s = kElemBytes[dtype];
  const bool want_perm_args = B * N * K >= ((int64_t)8 << 20);
  const uint64_t status_nonce = next_nonce();  // one for all slices: the status words describe the whole call
  // every slice reuses the workspace: the launches follow each other on one stream
  return for_batch_slices(B, [&](int64_t b0, int64_t nb) {
    return run_csr_reduce_slice(offset_bytes(src, b0 * E * K * s), indptr + b0 * indptr_batch_stride,
                                offset_bytes(out, b0 * N * K * s), arg_out ? arg_out + b0 * N * K : nullptr,
                                offset_bytes(count_out, b0 * N * s), nb, N, E, K, indptr_batch_stride, dtype, reduce,
                                accumulate, ws, ws_bytes, stream, perm ? perm + b0 * perm_batch_stride : nullptr,
                                perm_batch_stride, want_perm_args, perm_args_done, status, b0 == 0, status_nonce);
  });
}

// ---- scatter of wide rows: the index is sorted by row (row_sort.h), then a segmented reduction over permuted rows.
// No atomics on out, no table misses, whatever the index; an index found in order skips the sorting passes.
// RowsRoute: does a call take this route, and its workspace: row sort, carries of the reduction, status words (the
// last kStatusBytes: a row that crosses tiles is finished by a bounded wait, as in the segment operators).
struct RowsRoute {
  bool ok;
  size_t sort_bytes, csr_bytes;
  size_t total() const { return sort_bytes + csr_bytes + kStatusBytes; }
};
inline int rows_acc_bytes(int dtype, int reduce) {
  const bool sum = reduce == TS_SUM || reduce == TS_MEAN;
  return kElemBytes[dtype] == 8 || (sum && is_float_dtype(dtype)) ? 8 : 4;
}
CsrPlan rows_csr_plan(int64_t rows, int64_t n, int64_t K, int dtype, bool al, int reduce) {
  CsrPlan p = csr_plan(rows, n, K, kElemBytes[dtype], al, false, reduce == TS_MIN || reduce == TS_MAX, false);
  if (getenv("TS_CSR_IPW")) return p;  // tuning aid
  // Items per worker: about 1024 workgroups, 24 ... 72 items each, up to 192 where a worker takes single columns (144: the
  // workgroups of 1 M entries just miss running all at once, sum / max of 1 M x 33 floats 59 / 67 against 50 / 62 us; 384:
  // 59 / 77). A hub row is put together from the carries of all its tiles, so short tiles cost there what they gain
  // elsewhere (1 M x 33 floats, a fifth of them in one row, sum / max: 24 items 90 / 116 us, 72 56 / 68, 192 50 / 64; 300 k x
  // 32 floats, max: 24 items 38 us, 40 42, 64 50, even index 24 / 31 / 41).
  const int64_t items = rows + n;
  const int W = kCsrBlock / p.G;
  // (min / max of bytes, sixteen columns to a lane, and of rows of 16 lanes and more: 40 at least; 1 M x 64 bytes 153 us, 216 at
  // 24, 600 k x 128 bf16 80 / 94)
  const bool minmax = reduce == TS_MIN || reduce == TS_MAX;
  const int most = p.vec == 1 ? 192 : (items >= ((int64_t)32 << 20) ? 64 : 72);
  const int least = minmax && (kElemBytes[dtype] == 1 || p.G >= 16) ? 40 : 24;
  int64_t want = items / ((int64_t)W * 1024);
  want = want > most ? most : (want < least ? least : want);
  const int cap = kCsrMaxItems / W;
  p.ipw = want > cap ? cap : (int)want;
  p.BI = W * p.ipw;
  p.nblk = (items + p.BI - 1) / p.BI;
  return p;
}
inline int rows_meta_stride(const CsrPlan &p) { return p.ychunks > 4 ? p.ychunks : 4; }
RowsRoute rows_route(int64_t B, int64_t E, int64_t K, int64_t N, int dtype, int reduce) {
  RowsRoute r = {false, 0, 0};
  const int mode = env_int("TS_SCATTER_BINNED", 1);  // tuning aid: 0 never, 2 at any size
  const int64_t row_bytes = K * kElemBytes[dtype], n = B * E, rows = B * N;
  if (mode == 0 || B < 1 || E < 1 || N < 1 || row_bytes < 64 || row_bytes > 0xFFFFFFFFll || !env_int("TS_CSR_LOOKBACK", 1)) return r;
  const bool minmax = reduce == TS_MIN || reduce == TS_MAX;
  if (!minmax && reduce != TS_SUM && reduce != TS_MEAN) return r;
  if (!minmax && kAccBytes[dtype] < 4) return r;
  // From where the five launches of the sort and the reduction (27-31 us on the smallest inputs) cost less than the kernels
  // without them. The host knows sizes only; a line lies where an even and a Zipf(1.2) index, each shuffled and in order,
  // gain together (us of these four, without / with; the lines were drawn from 0.1 to 10 M entries, 0.3 to 30000 a row, when the sort
  // took a third longer, and could lie lower in places: the first two calls are below theirs):
  //   sums, 4 bytes: 300 k x 64, 3 a row 80 94 41 60 / 46 65 40 42; 300 k x 32, 10 a row 45 62 26 51 / 32 54 26 31
  //   fewer entries than rows (out is what moves): int64 1 M x 16 135 113 128 187 / 123 196 118 158, float 4.6 M x 16 424 317
  //   410 286 / 426 447 367 381, bf16 600 k x 64 102 629 92 101 / 141 208 132 172
  //   bf16, 1000 a row: 100 k x 64 25 22 16 16 / 30 46 25 24; doubles the same 30 26 15 15 / 29 47 23 24
  //   rows of 64 bytes, 30000 entries a row: float 4.6 M x 16 140 139 108 130 / 165 169 100 101, double x 8 83 82 106 117 /
  //   164 168 98 99
  //   min / max, 4 bytes: 600 k x 16, 10 a row 73 99 46 62 / 45 106 36 78; 300 k x 32, 10 a row 61 83 41 96 / 38 79 30 51
  //   1000 entries a row (a key table in LDS takes most): 600 k x 16 59 73 21 22 / 59 90 49 63, 300 k x 32 58 62 21 23 / 45 68
  //   35 42, double 300 k x 8 63 58 26 28 / 44 70 35 44
  //   30000 a row: 10 M x 16 270 300 151 157 / 362 359 214 212, 1 M x 32 60 60 37 40 / 87 95 60 62, bf16 300 k x 64 52 51 38 38
  //   / 88 94 64 63
  const int es = kElemBytes[dtype];
  const int64_t MB = 1000000, kNever = INT64_MAX;
  int64_t min_bytes;
  if (minmax) {
    // (without the sort they fill and walk a table of 8-byte keys as large as out: from 256 MB of keys the sort wins anyhow)
    min_bytes = rows * K * 8 >= 256 * MB ? MB : (es == 4 ? 28 * MB : es == 8 ? 16 * MB : 20 * MB);
    // rows that meet hundreds of entries: a key table in LDS takes most of them
    if (n >= 512 * rows && es >= 4 && row_bytes <= 128) min_bytes = es == 8 ? 30 * MB : 70 * MB;
    if (n >= 8192 * rows) {
      const int64_t least = es == 8 ? (row_bytes < 128 ? 60 * MB : 0) : es == 4 ? (row_bytes < 128 ? kNever : 140 * MB)
                                                                                : (row_bytes <= 128 ? 140 * MB : 30 * MB);
      if (min_bytes < least) min_bytes = least;
    }
  } else {
    min_bytes = es >= 4 ? 40 * MB : (n >= 32 * rows ? 6 * MB : 32 * MB);
    if (row_bytes < 128) min_bytes *= 2;
    if (n < 2 * rows) min_bytes *= 2;
    // rows that the kernels without the sort add in whole words (the others element by element, which loses anywhere)
    const bool words = es == 2 ? row_bytes % 4 == 0 : row_bytes % kVecBytes == 0;
    if (reduce == TS_SUM && words) {  // (TS_MEAN: the deviation, whose other kernels cost more)
      int64_t least = 0;
      if (n < rows && row_bytes <= 512) least = row_bytes < 128 || (es == 8 && row_bytes <= 128) ? 320 * MB : 140 * MB;
      if (es == 2 && n >= 512 * rows) least = 16 * MB;
      if (es == 8 && n >= 64 * rows) least = 60 * MB;
      if (es >= 4 && row_bytes == 64 && n >= 8192 * rows) least = kNever;
      if (min_bytes < least) min_bytes = least;
    }
  }
  if (mode != 2 && n * row_bytes < min_bytes) return r;
  const RowSortPlan sp = row_sort_plan(B, E, N, nullptr, 0);
  if (sp.bytes == 0) return r;
  for (int al = 0; al < 2; ++al) {
    const CsrPlan p = rows_csr_plan(rows, n, K, dtype, al != 0, reduce);
    if (p.ychunks > kMaxGridBatches) return r;
    const size_t b = csr_ws_bytes(p, 1, K, rows_acc_bytes(dtype, reduce), minmax, nullptr, nullptr, rows_meta_stride(p));
    if (b > r.csr_bytes) r.csr_bytes = b;
  }
  r.sort_bytes = sp.bytes;
  r.ok = true;
  return r;
}
// sorted: as launch_row_sort leaves it (without the identity); ws: RowsRoute::csr_bytes and behind them the status words.
// status_nonce: one for all reductions of a call; the first of them (status_reset) writes it into word 0.
int rows_reduce_args(CsrReduceArgs &a, const CsrPlan &p, const void *src, const RowSortArgs &sorted, void *out,
                     int64_t *arg_out, int64_t B, int64_t E, int64_t K, int64_t N, int dtype, int reduce, int out_given,
                     void *ws, size_t ws_bytes, uint64_t status_nonce, bool status_reset) {
  const int64_t n = B * E, rows = B * N;
  size_t off_args = 0, off_meta = 0;
  a.meta_stride = rows_meta_stride(p);
  if (csr_ws_bytes(p, 1, K, rows_acc_bytes(dtype, reduce), reduce == TS_MIN || reduce == TS_MAX, &off_args, &off_meta,
                   a.meta_stride) > ws_bytes)
    return TS_ERR_WORKSPACE;
  a.src = src;
  a.indptr = sorted.ptr;
  a.out = out;
  a.arg_out = arg_out;
  a.count_out = nullptr;
  a.N = rows;
  a.E = n;
  a.K = K;
  a.indptr_batch_stride = 0;
  a.accumulate = out_given ? 1 : 0;
  a.G = p.G;
  a.BI = p.BI;
  a.ipw = p.ipw;
  a.nblk = p.nblk;
  a.ws_vals = ws;
  a.ws_args = reinterpret_cast<int32_t *>(static_cast<char *>(ws) + off_args);
  a.ws_meta = reinterpret_cast<int64_t *>(static_cast<char *>(ws) + off_meta);
  a.lookback = p.nblk > 1;
  a.nonce = next_nonce();
  a.perm = sorted.perm;
  a.unsorted = sorted.state;
  a.perm_batch_stride = 0;
  a.perm_args = 0;
  a.any_order = 1;
  a.arg_E = E;
  a.status = status_word(ws, ws_bytes + kStatusBytes);
  a.status_reset = status_reset ? 1 : 0;
  a.status_nonce = status_nonce;
  a.carry_spin = env_int("TS_CSR_SPIN", kCarrySpin);  // test aid: -1 makes every look-back give up at once
  return TS_OK;
}
int run_rows_reduce(const void *src, const RowSortArgs &sorted, void *out, int64_t *arg_out, int64_t B,
                    int64_t E, int64_t K, int64_t N, int dtype, int reduce, int out_given, void *ws, size_t ws_bytes,
                    uint64_t status_nonce, hipStream_t s) {
  const CsrPlan p = rows_csr_plan(B * N, B * E, K, dtype, aligned16(src) && aligned16(out), reduce);
  CsrReduceArgs a;
  const int rc = rows_reduce_args(a, p, src, sorted, out, arg_out, B, E, K, N, dtype, reduce, out_given, ws, ws_bytes,
                                  status_nonce, true);
  return rc != TS_OK ? rc : dispatch_csr_reduce(dtype, a, p, 1, reduce, s);
}

int run_csr_gather(int dtype, const CsrGatherArgs &args, const CsrPlan &p, int64_t B, bool divide, hipStream_t s) {
  if (p.ychunks > kMaxGridBatches) return TS_ERR_UNSUPPORTED;
  const int64_t sz = kElemBytes[dtype];
  return for_batch_slices(B, [&](int64_t b0, int64_t nb) {
    CsrGatherArgs a = args;
    a.src = offset_bytes(args.src, b0 * args.N * args.K * sz);
    a.indptr = args.indptr + b0 * args.indptr_batch_stride;
    a.out = offset_bytes(args.out, b0 * args.E * args.K * sz);
    return dispatch_csr_gather(dtype, a, p, nb, divide, s);
  });
}

int run_coo_gather(int dtype, const CooGatherArgs &args, const CooGatherPlan &p, int64_t B, bool divide,
                   hipStream_t s) {
  if (p.ychunks > kMaxGridBatches) return TS_ERR_UNSUPPORTED;
  const int64_t sz = kElemBytes[dtype];
  return for_batch_slices(B, [&](int64_t b0, int64_t nb) {
    CooGatherArgs a = args;
    a.src = offset_bytes(args.src, b0 * args.N * args.K * sz);
    a.index = args.index + b0 * args.index_batch_stride;
    a.count = offset_bytes(args.count, b0 * args.N * sz);
    a.out = offset_bytes(args.out, b0 * args.E * args.K * sz);
    return dispatch_coo_gather(dtype, a, p, nb, divide, s);
  });
}

// sorted index [B, E] -> row pointers [B, N + 1] (contiguous)
int run_coo_to_indptr(const int64_t *index, int64_t *ptr, int64_t B, int64_t E, int64_t N, int64_t index_batch_stride,
                      hipStream_t s) {
  const int per = E < ((int64_t)1 << 20) ? 1 : kCooPtrPerThread;
  const int64_t per_block = (int64_t)kBlock * per;
  return for_batch_slices(B, [&](int64_t b0, int64_t nb) {
    dim3 grid((unsigned)((E + 1 + per_block - 1) / per_block), (unsigned)nb);
    if (per == 1)
      hipLaunchKernelGGL(coo_to_indptr_kernel<1>, grid, dim3(kBlock), 0, s, index + b0 * index_batch_stride,
                         ptr + b0 * (N + 1), N, E, index_batch_stride);
    else
      hipLaunchKernelGGL(coo_to_indptr_kernel<kCooPtrPerThread>, grid, dim3(kBlock), 0, s,
                         index + b0 * index_batch_stride, ptr + b0 * (N + 1), N, E, index_batch_stride);
    return hipGetLastError() == hipSuccess ? (int)TS_OK : (int)TS_ERR_LAUNCH;
  });
}

}  // namespace

extern "C" {

namespace {
thread_local int g_scatter_route = TS_ROUTE_NONE;
}
void ts_note_scatter_route(int route) { g_scatter_route = route; }
int ts_scatter_last_route(void) { return g_scatter_route; }
const char *ts_scatter_route_name(int route) {
  static const char *const names[] = {
      "none", "sum: atomic", "sum: runs", "sum: table", "sum: table or runs (sample)", "sum: buckets or runs (sample)",
      "sum: buckets or segmented reduction (index checked)", "mul: atomic", "mul: table", "min/max: atomic",
      "min/max: runs", "min/max: runs or table (sample)", "min/max: table", "min/max: table, one value per entry",
      "min/max: slabs, one value per entry", "min/max: buckets", "min/max: buckets or segmented reduction (index checked)",
      "min/max: 64-bit elements, two passes", "sum: single values in buckets, table or runs (sample)",
      "sum: runs, entries per row counted by the same launch", "sum: single values, tables in slabs",
      "sum, mean, min or max of a small input: one launch", "sum: narrow rows, entries sorted by row"};
  return route >= 0 && route < (int)(sizeof(names) / sizeof(names[0])) ? names[route] : "unknown";
}

namespace {
// every fixed-pattern cross-lane helper of dpp.h applied to x = 3 * lane + 1, one row of 64 results each
__global__ __launch_bounds__(kWave) void lane_ops_selftest_kernel(int32_t *out) {
  const int lane = threadIdx.x;
  const int x = 3 * lane + 1;
  int row = 0;
  out[64 * row++ + lane] = lane_up1(x);
  out[64 * row++ + lane] = lane_xor<1>(x);
  out[64 * row++ + lane] = lane_xor<2>(x);
  out[64 * row++ + lane] = lane_xor<4>(x);
  out[64 * row++ + lane] = lane_xor<8>(x);
  out[64 * row++ + lane] = lane_xor<16>(x);
  out[64 * row++ + lane] = lane_xor<32>(x);
  out[64 * row++ + lane] = lane_down<1>(x);
  out[64 * row++ + lane] = lane_down<2>(x);
  out[64 * row++ + lane] = lane_down<4>(x);
  out[64 * row++ + lane] = lane_down<8>(x);
  out[64 * row++ + lane] = lane_down<16>(x);
  out[64 * row++ + lane] = lane_down<32>(x);
  out[64 * row++ + lane] = wave_inclusive_sum(x);
  out[64 * row++ + lane] = (int)lane_up1_64(((int64_t)x << 32) | (uint32_t)(x + 7));
  out[64 * row++ + lane] = (int)(lane_up1_64(((int64_t)x << 32) | (uint32_t)(x + 7)) >> 32);
  float f = (float)x * 0.5f;
  out[64 * row++ + lane] = (int)(lane_xor<16>(f) * 2.0f);
}
}  // namespace

int ts_selftest_lane_ops(int32_t *out, ts_stream_t stream) {
  if (!out) return TS_ERR_BAD_ARG;
  hipLaunchKernelGGL(lane_ops_selftest_kernel, dim3(1), dim3(kWave), 0, static_cast<hipStream_t>(stream), out);
  return hipGetLastError() == hipSuccess ? TS_OK : TS_ERR_LAUNCH;
}

int ts_status_gave_up(const unsigned long long *words) {
  return words != nullptr && words[0] != 0 && words[1] == words[0];
}

const char *ts_error_string(int status) {
  switch (status) {
  case TS_OK: return "ok";
  case TS_ERR_BAD_ARG: return "bad argument (null pointer, negative size or unknown dtype/reduce code)";
  case TS_ERR_UNSUPPORTED: return "unsupported combination of dtype / reduce / size";
  case TS_ERR_WORKSPACE: return "workspace missing or too small";
  case TS_ERR_LAUNCH: return "HIP kernel launch failed";
  default: return "unknown status";
  }
}

int64_t ts_hip_version(void) { return HIP_VERSION; }


size_t ts_segment_csr_workspace_bytes(int64_t B, int64_t N, int64_t E, int64_t K, int dtype, int reduce) {
  if (!valid_dtype(dtype) || !sizes_ok(B, N, E, K)) return 0;
  // the plan may fall back to one element per lane for unaligned buffers; the
  // tile count does not depend on that choice
  return csr_workspace_max(B, N, E, K, dtype, reduce);
}

int ts_segment_csr(const void *src, const int64_t *indptr, void *out, int64_t *arg_out, int64_t B,
                   int64_t N, int64_t E, int64_t K, int64_t indptr_batch_stride, int dtype, int reduce,
                   void *workspace, size_t workspace_bytes, ts_stream_t stream) {
  if (!valid_dtype(dtype) || !sizes_ok(B, N, E, K)) return TS_ERR_BAD_ARG;
  if (reduce != TS_SUM && reduce != TS_MEAN && reduce != TS_MIN && reduce != TS_MAX) return TS_ERR_UNSUPPORTED;
  if (B * N * K == 0) return TS_OK;
  if (!indptr || !out || (E * K > 0 && !src)) return TS_ERR_BAD_ARG;
  if ((reduce == TS_MIN || reduce == TS_MAX) && !arg_out) return TS_ERR_BAD_ARG;
  const size_t need = csr_workspace_max(B, N, E, K, dtype, reduce);
  if (!workspace || workspace_bytes < need) return TS_ERR_WORKSPACE;
  return run_csr_reduce(src, indptr, out, arg_out, nullptr, B, N, E, K, indptr_batch_stride, dtype, reduce, 0,
                        workspace, need - kStatusBytes, status_word(workspace, need), static_cast<hipStream_t>(stream));
}

int ts_gather_csr(const void *src, const int64_t *indptr, void *out, int64_t B, int64_t N, int64_t E,
                  int64_t K, int64_t indptr_batch_stride, int dtype, ts_stream_t stream) {
  if (!valid_dtype(dtype) || !sizes_ok(B, N, E, K)) return TS_ERR_BAD_ARG;
  if (B * E * K == 0 || N == 0) return TS_OK;
  if (!src || !indptr || !out) return TS_ERR_BAD_ARG;
  const CsrPlan p = csr_plan(N, E, K, kElemBytes[dtype], aligned16(src) && aligned16(out), true);
  CsrGatherArgs a;
  a.src = src;
  a.indptr = indptr;
  a.out = out;
  a.N = N;
  a.E = E;
  a.K = K;
  a.indptr_batch_stride = indptr_batch_stride;
  a.G = p.G;
  a.BI = p.BI;
  a.ipw = p.ipw;
  a.nblk = p.nblk;
  return run_csr_gather(dtype, a, p, B, false, static_cast<hipStream_t>(stream));
}

int ts_segment_mean_csr_backward(const void *grad_out, const int64_t *indptr, void *grad_in, int64_t B,
                                 int64_t N, int64_t E, int64_t K, int64_t indptr_batch_stride, int dtype,
                                 ts_stream_t stream) {
  if (!valid_dtype(dtype) || !sizes_ok(B, N, E, K)) return TS_ERR_BAD_ARG;
  if (!is_float_dtype(dtype)) return TS_ERR_UNSUPPORTED;
  if (B * E * K == 0 || N == 0) return TS_OK;
  if (!grad_out || !indptr || !grad_in) return TS_ERR_BAD_ARG;
  const CsrPlan p = csr_plan(N, E, K, kElemBytes[dtype], aligned16(grad_out) && aligned16(grad_in), true, true);
  CsrGatherArgs a;
  a.src = grad_out;
  a.indptr = indptr;
  a.out = grad_in;
  a.N = N;
  a.E = E;
  a.K = K;
  a.indptr_batch_stride = indptr_batch_stride;
  a.G = p.G;
  a.BI = p.BI;
  a.ipw = p.ipw;
  a.nblk = p.nblk;
  return run_csr_gather(dtype, a, p, B, true, static_cast<hipStream_t>(stream));
}

// ---- ts_segment_csr for callers that cannot allocate: the partial results of rows that cross tiles
// live in a file-scope device array instead of a caller's workspace. Every GPU holds its own copy
// of the array at its own address; the address is looked up once per device, with that device current.
constexpr size_t kStaticScratchBytes = (size_t)TS_STATIC_SCRATCH_BYTES;
constexpr int kStaticScratchDevices = 64;
static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];
static std::atomic<void *> g_scratch_ptr[kStaticScratchDevices];

static int static_scratch_ptr(void **out) {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kStaticScratchDevices) return TS_ERR_LAUNCH;
  void *p = g_scratch_ptr[dev].load(std::memory_order_acquire);
  if (p == nullptr) {
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || p == nullptr) return TS_ERR_LAUNCH;
    g_scratch_ptr[dev].store(p, std::memory_order_release);
  }
  *out = p;
  return TS_OK;
}

int ts_segment_csr_static(const void *src, const int64_t *indptr, void *out, int64_t *arg_out, int64_t B,
                          int64_t N, int64_t E, int64_t K, int64_t indptr_batch_stride, int dtype, int reduce,
                          ts_stream_t stream) {
  if (!valid_dtype(dtype) || !sizes_ok(B, N, E, K)) return TS_ERR_BAD_ARG;
  if (reduce != TS_SUM && reduce != TS_MEAN && reduce != TS_MIN && reduce != TS_MAX) return TS_ERR_UNSUPPORTED;
  if (B * N * K == 0) return TS_OK;
  if (!indptr || !out || (E * K > 0 && !src)) return TS_ERR_BAD_ARG;
  if ((reduce == TS_MIN || reduce == TS_MAX) && !arg_out) return TS_ERR_BAD_ARG;
  // the array is fixed in size: larger inputs must bring a workspace (ts_segment_csr)
  const size_t need = csr_workspace_max(B, N, E, K, dtype, reduce);
  if (need > kStaticScratchBytes) return TS_ERR_WORKSPACE;
  void *ws = nullptr;
  const int rc = static_scratch_ptr(&ws);
  if (rc != TS_OK) return rc;
  // Nothing in the array has to start at zero: the carry flags of a call hold that call's nonce, and
  // the second kernel only reads what the first one wrote in the same call.
  return run_csr_reduce(src, indptr, out, arg_out, nullptr, B, N, E, K, indptr_batch_stride, dtype, reduce, 0, ws,
                        need - kStatusBytes, status_word(ws, need), static_cast<hipStream_t>(stream));
}

size_t ts_segment_csr_permuted_workspace_bytes(int64_t B, int64_t N, int64_t E, int64_t K, int dtype, int reduce) {
  if (!valid_dtype(dtype) || !sizes_ok(B, N, E, K)) return 0;
  return csr_workspace_max(B, N, E, K, dtype, reduce, false);
}

int ts_segment_csr_permuted(const void *src, const int32_t *perm, const int64_t *indptr, void *out,
                            int64_t *arg_out, int64_t B, int64_t N, int64_t E, int64_t K,
                            int64_t perm_batch_stride, int64_t indptr_batch_stride, int dtype, int reduce,
                            void *workspace, size_t workspace_bytes, ts_stream_t stream) {
  if (!valid_dtype(dtype) || !sizes_ok(B, N, E, K)) return TS_ERR_BAD_ARG;
  if (reduce != TS_SUM && reduce != TS_MEAN && reduce != TS_MIN && reduce != TS_MAX) return TS_ERR_UNSUPPORTED;
  if (E >= 0x7FFFFFFFll) return TS_ERR_UNSUPPORTED;  // 32-bit row numbers
  if (B * N * K == 0) return TS_OK;
  if (!indptr || !out || (E * K > 0 && (!src || !perm))) return TS_ERR_BAD_ARG;
  if ((reduce == TS_MIN || reduce == TS_MAX) && !arg_out) return TS_ERR_BAD_ARG;
  hipStream_t s = static_cast<hipStream_t>(stream);
  bool args_done = false;
  const size_t need = csr_workspace_max(B, N, E, K, dtype, reduce, false);
  if (!workspace || workspace_bytes < need) return TS_ERR_WORKSPACE;
  const int rc = run_csr_reduce(src, indptr, out, arg_out, nullptr, B, N, E, K, indptr_batch_stride, dtype, reduce,
                                0, workspace, need - kStatusBytes, status_word(workspace, need), s, perm,
                                perm_batch_stride, &args_done);
  if (rc != TS_OK || (reduce != TS_MIN && reduce != TS_MAX) || args_done) return rc;
  return dispatch_sorted_args(dtype, out, arg_out, perm, B, N * K, E, perm_batch_stride, reduce == TS_MAX, s);
}

size_t ts_segment_coo_workspace_bytes(int64_t B, int64_t N, int64_t E, int64_t K, int dtype, int reduce) {
  if (!valid_dtype(dtype) || !sizes_ok(B, N, E, K)) return 0;
  const size_t ptr_bytes = ((size_t)B * (N + 1) * 8 + 255) & ~(size_t)255;
  return ptr_bytes + csr_workspace_max(B, N, E, K, dtype, reduce);
}

int ts_segment_coo(const void *src, const int64_t *index, void *out, void *arg_out, void *count_out,
                   int64_t B, int64_t N, int64_t E, int64_t K, int64_t index_batch_stride, int dtype,
                   int reduce, int out_given, void *workspace, size_t workspace_bytes, ts_stream_t stream) {
  if (!valid_dtype(dtype) || !sizes_ok(B, N, E, K)) return TS_ERR_BAD_ARG;
  if (reduce != TS_SUM && reduce != TS_MEAN && reduce != TS_MIN && reduce != TS_MAX) return TS_ERR_UNSUPPORTED;
  if (B * N * K == 0) return TS_OK;
  if (!out || (E > 0 && (!index || (K > 0 && !src)))) return TS_ERR_BAD_ARG;
  if ((reduce == TS_MIN || reduce == TS_MAX) && !arg_out) return TS_ERR_BAD_ARG;
  const size_t ptr_bytes = ((size_t)B * (N + 1) * 8 + 255) & ~(size_t)255;
  const size_t need = ptr_bytes + csr_workspace_max(B, N, E, K, dtype, reduce);
  if (!workspace || workspace_bytes < need) return TS_ERR_WORKSPACE;
  hipStream_t s = static_cast<hipStream_t>(stream);
  int64_t *ptr = static_cast<int64_t *>(workspace);
  const int rc = run_coo_to_indptr(index, ptr, B, E, N, index_batch_stride, s);
  if (rc != TS_OK) return rc;
  return run_csr_reduce(src, ptr, out, static_cast<int64_t *>(arg_out), count_out, B, N, E, K, N + 1, dtype,
                        reduce, out_given ? 1 : 0, static_cast<char *>(workspace) + ptr_bytes,
                        need - ptr_bytes - kStatusBytes, status_word(workspace, need), s);
}

int ts_gather_coo(const void *src, const int64_t *index, void *out, int64_t B, int64_t N, int64_t E,
                  int64_t K, int64_t index_batch_stride, int dtype, ts_stream_t stream) {
  if (!valid_dtype(dtype) || !sizes_ok(B, N, E, K)) return TS_ERR_BAD_ARG;
  if (B * E * K == 0 || N == 0) return TS_OK;
  if (!src || !index || !out) return TS_ERR_BAD_ARG;
  const CooGatherPlan p = coo_gather_plan(E, K, kElemBytes[dtype], aligned16(src) && aligned16(out));
  CooGatherArgs a;
  a.src = src;
  a.index = index;
  a.count = nullptr;
  a.out = out;
  a.N = N;
  a.E = E;
  a.K = K;
  a.index_batch_stride = index_batch_stride;
  a.G = p.G;
  a.epw = p.epw;
  return run_coo_gather(dtype, a, p, B, false, static_cast<hipStream_t>(stream));
}

int ts_segment_mean_coo_backward(const void *grad_out, const int64_t *index, const void *count,
                                 void *grad_in, int64_t B, int64_t N, int64_t E, int64_t K,
                                 int64_t index_batch_stride, int dtype, ts_stream_t stream) {
  if (!valid_dtype(dtype) || !sizes_ok(B, N, E, K)) return TS_ERR_BAD_ARG;
  if (!is_float_dtype(dtype)) return TS_ERR_UNSUPPORTED;
  if (B * E * K == 0 || N == 0) return TS_OK;
  if (!grad_out || !index || !count || !grad_in) return TS_ERR_BAD_ARG;
  const CooGatherPlan p = coo_gather_plan(E, K, kElemBytes[dtype], aligned16(grad_out) && aligned16(grad_in));
  CooGatherArgs a;
  a.src = grad_out;
  a.index = index;
  a.count = count;
  a.out = grad_in;
  a.N = N;
  a.E = E;
  a.K = K;
  a.index_batch_stride = index_batch_stride;
  a.G = p.G;
  a.epw = p.epw;
  return run_coo_gather(dtype, a, p, B, true, static_cast<hipStream_t>(stream));
}

}  // extern "C"
namespace {
// Sums of rows below 64 bytes over sorted entries (group_rows.h), where adding in memory is slowest: 16-bit elements (packed pairs, or
// one by one in rows of odd width), floats of nine columns and more, from where they outgrow what the launches of the sort cost. us
// without / with, ten entries a row unless said, in random order | in order | a power law's hubs (p ~ i^-1.2, the sort's worst, memory's
// best: its hot rows are added up in LDS):
//   16 bits  10 M x 24  3943 / 448 | 479 / 371 | 3351 / 603      10 M x 8  1393 / 289 | 164 / 166 | 574 / 359
//            10 M x 5   1317 / 291 | 334 / 162 | 648 / 342       10 M x 3  1012 / 283 | 205 / 152 | 422 / 323
//            2 M x 16    486 / 81  |  67 / 68  | 276 / 117       2 M x 6    304 / 72  |  57 / 50  | 152 / 97
//            9.7 M x 24, four a row 4097 / 581; 2.4 M x 16, 14 a row, with the backward pass 671 / 146; 629 k x 15 in order 81 / 35
//     left   10 M x 4    928 / 279 | 128 / 114 | 291 / 321       2 M x 4    177 / 66  |  39 / 41  |  76 / 99
//            10 M x 2    922 / 266 |  77 / 120 | 258 / 297       700 k x 6   92 / 40  |  21 / 31  |  57 / 66
//            and, with fewer than two entries a row, 654 k x 8 83 / 108
//   floats   10 M x 15  1021 / 403 | 477 / 265 | 615 / 556       10 M x 9   799 / 331 | 453 / 213 | 467 / 439
//            10 M x 12   787 / 344 | 266 / 217 | 452 / 472       5.8 M x 13, nine a row 624 / 236
//     left   10 M x 8    502 / 290 | 171 / 164 | 231 / 382       10 M x 5   638 / 307 | 282 / 162 | 291 / 377
//            2 M x 13    200 / 88  | 120 / 66  | 111 / 127
// Rows of whole 16-byte units gain least in order, so their lines lie higher: 16 bits 12 M elements in place of 8 M (700 k x 16 165 / 43 |
// 41 / 38 | 99 / 76; calls below it keep their 256 bytes of scratch), floats 100 M in place of 40 M.
// The sums are held in double (the packed adds round to 16 bits every time). TS_SCATTER_NARROW (tuning aid): 0 never, 2 at any size.
bool scatter_narrow_rule(int64_t B, int64_t E, int64_t K, int64_t N, int dtype) {
  const int es = kElemBytes[dtype];
  const int64_t row_bytes = K * es, n = B * E, M = 1000000;
  if (!is_float_dtype(dtype) || row_bytes >= 64 || n < 1 || B * N < 1) return false;
  const int mode = env_int("TS_SCATTER_NARROW", 1);
  if (mode == 0) return false;
  if (mode == 2) return true;
  if (E < 2 * N) return false;
  if (es == 2) return K >= 3 && K != 4 && n * K >= (row_bytes % kVecBytes == 0 ? 12 * M : 8 * M);
  return es == 4 && K >= 9 && n * K >= (row_bytes % kVecBytes == 0 ? 100 * M : 40 * M);
}
size_t scatter_narrow_records(int64_t B, int64_t E, int64_t K, int64_t N, int dtype) {
  return group_rows_plan(B * E, B * N, K, kElemBytes[dtype], nullptr).bytes;
}
size_t scatter_narrow_bytes(int64_t B, int64_t E, int64_t K, int64_t N, int dtype) {
  if (!scatter_narrow_rule(B, E, K, N, dtype)) return 0;
  const size_t sort = row_sort_plan(B, E, N, nullptr, 0, true).bytes, records = scatter_narrow_records(B, E, K, N, dtype);
  return sort == 0 || records == 0 ? 0 : sort + records;
}
int run_scatter_narrow(const void *src, const int64_t *index, void *out, int64_t B, int64_t E, int64_t K, int64_t N, int64_t sb,
                       int64_t se, int dtype, void *ws, size_t ws_bytes, int32_t *count_out, hipStream_t s) {
  const size_t records = scatter_narrow_records(B, E, K, N, dtype);
  const RowSortPlan sp = row_sort_plan(B, E, N, static_cast<char *>(ws) + records, ws_bytes - records, true);
  if (!sp.ok) return TS_ERR_WORKSPACE;
  int rc = launch_row_sort(sp.p, index, sb, se, false, next_nonce(), s);
  if (rc != TS_OK) return rc;
  GroupRowsPlan p = group_rows_plan(B * E, B * N, K, kElemBytes[dtype], ws);
  GroupArgs g = {};
  g.src = src;
  g.out = out;
  g.B = 1;
  g.E = B * E;
  g.K = K;
  g.N = B * N;
  p.f.state = sp.p.state;
  p.f.ptr = sp.p.ptr;
  p.f.perm = sp.p.perm;
  p.f.group = sp.p.perm_row;
  p.f.gate = nullptr;
  p.f.index = index;
  p.f.sb = sb;
  p.f.se = se;
  p.f.E0 = E;
  p.f.N0 = N;
  rc = dispatch_group_rows(dtype, g, p.f, GS_SUM, s);
  if (rc != TS_OK || count_out == nullptr) return rc;
  hipLaunchKernelGGL(row_lengths_kernel, dim3(grid_for(B * N)), dim3(kBlock), 0, s, sp.p.ptr, count_out, B * N);
  return hipGetLastError() == hipSuccess ? TS_OK : TS_ERR_LAUNCH;
}
}  // namespace
extern "C" {

size_t ts_scatter_workspace_bytes(int64_t B, int64_t E, int64_t K, int64_t N, int dtype, int reduce) {
  if (!valid_dtype(dtype) || !sizes_ok(B, N, E, K)) return 0;
  const bool any_size = env_int("TS_SCATTER_BINNED", 1) == 2;
  const RowsRoute rr = reduce == TS_MEAN ? RowsRoute{false, 0, 0} : rows_route(B, E, K, N, dtype, reduce);
  if (reduce == TS_MIN || reduce == TS_MAX) {
    if (rr.ok) return rr.total();
    if (kElemBytes[dtype] > 4) return 0;  // 64-bit elements do not use packed keys
    if (env_int("TS_SCATTER_LDS_K1", 1) && env_int("TS_SCATTER_LDS", 1)) {
      const size_t k1 = k1_plan(B, E, K, N, kElemBytes[dtype], nullptr, 0, env_int("TS_SCATTER_LDS", 1) == 2).bytes;
      if (k1 != 0) return k1;
    }
    // one flag for the sample of the index that picks the kernel when few entries meet in an output row
    const int probe = env_int("TS_SCATTER_SKEW", 1);
    return probe && skew_probe_shape(B, E, K, N, kElemBytes[dtype], probe == 2) ? 256 : 0;
  }
  if (reduce == TS_SUM && kAccBytes[dtype] >= 4) {  // table slots: int32 for int32, 8 bytes for the other types
    if (rr.ok) return rr.total();
    const size_t narrow = scatter_narrow_bytes(B, E, K, N, dtype);
    if (narrow != 0) return narrow;
    if (env_int("TS_SCATTER_LDS", 1)) {
      // one 4-byte value per entry: (row in bucket, value) words, 8 bytes of scratch per entry
      const size_t payload = bin_plan_payload(B, E, K, N, kElemBytes[dtype], nullptr, 0, any_size).bytes;
      if (payload != 0) return payload;
      // single 4-byte values from 2^19 entries: a table per workgroup, handed over in slabs (with room for the counts
      // of scatter mean)
      if ((dtype == TS_F32 || dtype == TS_I32) && env_int("TS_SCATTER_LDS", 1) == 1 && env_int("TS_SCATTER_SLABS", 1)) {
        const size_t slabs =
            s1_plan(B, E, K, N, kElemBytes[dtype], nullptr, 0, true, env_int("TS_SCATTER_SLABS", 1) == 2).bytes;
        if (slabs != 0) return slabs;
      }
    }
    // one word for the sample of the index that keeps a sorted one away from the table kernel
    const bool table = (is_float_dtype(dtype) || dtype == TS_I32 || dtype == TS_I64) &&
                       env_int("TS_SCATTER_LDS", 1) == 1 && sum_table_by_size(B, E, K, N, kElemBytes[dtype]);
    return table ? 256 : 0;
  }
  return 0;
}

size_t ts_scatter_workspace_zero_bytes(int64_t B, int64_t E, int64_t K, int64_t N, int dtype, int reduce) {
  if (!valid_dtype(dtype) || !sizes_ok(B, N, E, K)) return 0;
  if ((reduce != TS_MIN && reduce != TS_MAX) || kElemBytes[dtype] > 4) return 0;
  if (!env_int("TS_SCATTER_LDS_K1", 1) || !env_int("TS_SCATTER_LDS", 1)) return 0;
  return k1_plan(B, E, K, N, kElemBytes[dtype], nullptr, 0, env_int("TS_SCATTER_LDS", 1) == 2).zero_bytes;
}

int ts_scatter(const void *src, const int64_t *index, void *out, int64_t *arg_out, int64_t B, int64_t E,
               int64_t K, int64_t N, int64_t index_stride_b, int64_t index_stride_e, int64_t index_stride_k,
               int dtype, int reduce, int out_given, ts_stream_t stream) {
  return ts_scatter_with_workspace(src, index, out, arg_out, B, E, K, N, index_stride_b, index_stride_e,
                                   index_stride_k, dtype, reduce, out_given, nullptr, 0, stream);
}

}  // extern "C"
namespace {
// ts_scatter_with_workspace; count_out / count_flag: see ScatterArgs (a sum through the buckets that counts as well)
int scatter_ws_impl(const void *src, const int64_t *index, void *out, int64_t *arg_out, int64_t B,
                    int64_t E, int64_t K, int64_t N, int64_t index_stride_b, int64_t index_stride_e,
                    int64_t index_stride_k, int dtype, int reduce, int out_given, void *workspace,
                    size_t workspace_bytes, ts_stream_t stream, int32_t *count_out, const int **count_flag,
                    int *count_done = nullptr) {
  if (!valid_dtype(dtype) || !sizes_ok(B, N, E, K)) return TS_ERR_BAD_ARG;
  if (reduce != TS_SUM && reduce != TS_MUL && reduce != TS_MIN && reduce != TS_MAX) return TS_ERR_UNSUPPORTED;
  ts_note_scatter_route(TS_ROUTE_NONE);
  if (B * N * K == 0) return TS_OK;
  if (!out || (B * E * K > 0 && (!src || !index))) return TS_ERR_BAD_ARG;
  if ((reduce == TS_MIN || reduce == TS_MAX) && !arg_out) return TS_ERR_BAD_ARG;
  ScatterArgs a;
  a.src = src;
  a.index = index;
  a.out = out;
  a.arg_out = arg_out;
  a.B = B;
  a.E = E;
  a.K = K;
  a.N = N;
  a.sb = index_stride_b;
  a.se = index_stride_e;
  a.sk = index_stride_k;
  a.out_given = out_given ? 1 : 0;
  a.count_out = count_out;
  a.count_flag = count_flag;
  a.count_done = count_done;
  a.precheck = env_int("TS_SCATTER_PRECHECK", 1);   // tuning aids
  a.lds_cache = env_int("TS_SCATTER_LDS", 1);
  a.lds_epb = env_int("TS_SCATTER_EPB", 0);
  a.run_reduce = env_int("TS_SCATTER_RUNS", 1);
  a.lds_k1 = env_int("TS_SCATTER_LDS_K1", 1);
  a.skew_probe = env_int("TS_SCATTER_SKEW", 1);  // tuning aid: 0 never, 2 at any size
  if (const int binned = env_int("TS_SCATTER_BINNED", 1)) {  // tuning aid: 0 never, 2 at any size
    a.bin_ws = workspace;
    a.bin_ws_bytes = workspace_bytes;
    a.bin_any_size = binned == 2;
  }
  const int full = kVecBytes / kElemBytes[dtype];
  const int vec = (full > 1 && K % full == 0 && aligned16(src)) ? full : 1;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (a.bin_ws != nullptr && index_stride_k == 0 && B * E * K > 0 && aligned16(workspace)) {
    const RowsRoute rr = rows_route(B, E, K, N, dtype, reduce);
    if (rr.ok && workspace_bytes >= rr.total()) {
      RowSortPlan sp = row_sort_plan(B, E, N, workspace, rr.sort_bytes);
      if (!sp.ok) return TS_ERR_WORKSPACE;
      ts_note_scatter_route(reduce == TS_SUM ? TS_ROUTE_SUM_BUCKETS_OR_SEGMENTED : TS_ROUTE_MINMAX_BUCKETS_OR_SEGMENTED);
      int rc = launch_row_sort(sp.p, index, index_stride_b, index_stride_e, false, next_nonce(), s);
      if (rc != TS_OK) return rc;
      rc = run_rows_reduce(src, sp.p, out, arg_out, B, E, K, N, dtype, reduce, out_given,
                           static_cast<char *>(workspace) + rr.sort_bytes, rr.csr_bytes, next_nonce(), s);
      if (rc != TS_OK || count_out == nullptr) return rc;
      hipLaunchKernelGGL(row_lengths_kernel, dim3(grid_for(B * N)), dim3(kBlock), 0, s, sp.p.ptr, count_out, B * N);
      if (count_done != nullptr) *count_done = 1;
      return hipGetLastError() == hipSuccess ? TS_OK : TS_ERR_LAUNCH;
    }
  }
  if (reduce == TS_SUM && !out_given && a.bin_ws != nullptr && index_stride_k == 0 && B * E * K > 0 && aligned16(workspace)) {
    const size_t need = scatter_narrow_bytes(B, E, K, N, dtype);
    if (need != 0 && workspace_bytes >= need) {
      ts_note_scatter_route(TS_ROUTE_SUM_NARROW_SORTED);
      const int rc = run_scatter_narrow(src, index, out, B, E, K, N, index_stride_b, index_stride_e, dtype, workspace,
                                        workspace_bytes, count_out, s);
      if (rc == TS_OK && count_out != nullptr && count_done != nullptr) *count_done = 1;
      return rc;
    }
  }
  if (reduce == TS_SUM && workspace != nullptr && workspace_bytes >= 256 && aligned16(workspace) &&
      !(env_int("TS_SCATTER_LDS", 1) &&
        bin_plan_payload(B, E, K, N, kElemBytes[dtype], nullptr, 0, a.bin_any_size != 0).bytes != 0))
    a.order_ws = static_cast<int *>(workspace);
  return dispatch_scatter(dtype, a, reduce, vec, s);
}
}  // namespace
namespace {
// Scatter with wide rows whose order stays for the backward pass. us forward and backward, without / with the order:
//   sums   the gradients' rows in whole lines, from 32 MB of them: 2.3 M x 128 bf16 onto 268 k rows 361 / 304, 603 k x 128 floats
//          onto 176 k 194 / 163, 1.9 M x 32 floats onto 1.05 M 201 / 186. What the L2 holds is gathered faster than entries' rows are
//          written in no order: 9.7 M x 16 floats onto 65 k 386 / 541; so are rows that are not whole lines, 742 k x 100 doubles 290 / 357
//   min / max   from 366 MB of entries, beyond the memory-side cache: 2.3 M x 64 floats onto 282 k rows 454 / 381, 678 k x 256 floats
//          onto 19 k 511 / 304, 678 k x 128 doubles onto 1.4 k 336 / 300; with up to eight entries a row from 32 MB: 3.2 M x 32 floats
//          onto 1.1 M 618 / 430, 3.4 M x 8 doubles onto 429 k 234 / 210. Else a fill and a scatter of single elements: 525 k x 128
//          floats onto 2.4 k 147 / 160; 240 k x 100 floats under a hub 112 / 128 (rows that are not whole 64 bytes)
// TS_SCATTER_ORDER (tuning aid): 0 never, 2 wherever the entries are sorted.
bool scatter_order_ok(int64_t B, int64_t E, int64_t K, int64_t N, int dtype, int reduce, RowsRoute &rr) {
  if (!valid_dtype(dtype) || !is_float_dtype(dtype) || !sizes_ok(B, N, E, K) || B * E * K == 0 || N == 0) return false;
  if (reduce != TS_SUM && reduce != TS_MIN && reduce != TS_MAX) return false;
  const int mode = env_int("TS_SCATTER_ORDER", 1);
  const int64_t row_bytes = K * kElemBytes[dtype], MB = (int64_t)1 << 20;
  if (mode == 0 || (reduce != TS_SUM && row_bytes % kVecBytes != 0)) return false;
  if (mode != 2) {
    if (reduce == TS_SUM && (row_bytes % 128 != 0 || B * N * row_bytes < 32 * MB)) return false;
    if (reduce != TS_SUM && (row_bytes % 64 != 0 || B * E * row_bytes < (E > 8 * N ? 366 * MB : 32 * MB))) return false;
  }
  rr = rows_route(B, E, K, N, dtype, reduce);
  return rr.ok;
}
}  // namespace
extern "C" {

size_t ts_scatter_order_bytes(int64_t B, int64_t E, int64_t K, int64_t N, int dtype, int reduce) {
  RowsRoute rr;
  return scatter_order_ok(B, E, K, N, dtype, reduce, rr) ? row_sort_plan(B, E, N, nullptr, 0, true).kept_bytes : 0;
}

size_t ts_scatter_order_workspace_bytes(int64_t B, int64_t E, int64_t K, int64_t N, int dtype, int reduce) {
  RowsRoute rr;
  if (!scatter_order_ok(B, E, K, N, dtype, reduce, rr)) return 0;
  const RowSortPlan sp = row_sort_plan(B, E, N, nullptr, 0, true);
  return sp.bytes - sp.kept_bytes + rr.csr_bytes + kStatusBytes;
}

int ts_scatter_ordered(const void *src, const int64_t *index, void *out, int64_t *arg_out, int32_t *count, int64_t B, int64_t E,
                       int64_t K, int64_t N, int64_t index_stride_b, int64_t index_stride_e, int dtype, int reduce, int out_given,
                       void *order, size_t order_bytes, void *workspace, size_t workspace_bytes, ts_stream_t stream) {
  RowsRoute rr;
  if (!scatter_order_ok(B, E, K, N, dtype, reduce, rr)) return TS_ERR_UNSUPPORTED;
  ts_note_scatter_route(TS_ROUTE_NONE);
  if (!src || !index || !out || (reduce != TS_SUM && !arg_out)) return TS_ERR_BAD_ARG;
  if (!order || !aligned16(order) || !workspace || !aligned16(workspace)) return TS_ERR_WORKSPACE;
  const size_t kept = row_sort_plan(B, E, N, nullptr, 0, true).kept_bytes;
  const size_t sort = row_sort_plan(B, E, N, nullptr, 0, true).bytes - kept;
  if (order_bytes < kept || workspace_bytes < sort + rr.csr_bytes + kStatusBytes) return TS_ERR_WORKSPACE;
  const RowSortPlan sp = row_sort_plan(B, E, N, workspace, sort, true, order);
  if (!sp.ok) return TS_ERR_WORKSPACE;
  hipStream_t s = static_cast<hipStream_t>(stream);
  ts_note_scatter_route(reduce == TS_SUM ? TS_ROUTE_SUM_BUCKETS_OR_SEGMENTED : TS_ROUTE_MINMAX_BUCKETS_OR_SEGMENTED);
  int rc = launch_row_sort(sp.p, index, index_stride_b, index_stride_e, false, next_nonce(), s);
  if (rc != TS_OK) return rc;
  rc = run_rows_reduce(src, sp.p, out, arg_out, B, E, K, N, dtype, reduce, out_given,
                       static_cast<char *>(workspace) + sort, rr.csr_bytes, next_nonce(), s);
  if (rc != TS_OK || count == nullptr) return rc;
  hipLaunchKernelGGL(row_lengths_kernel, dim3(grid_for(B * N)), dim3(kBlock), 0, s, sp.p.ptr, count, B * N);
  return hipGetLastError() == hipSuccess ? TS_OK : TS_ERR_LAUNCH;
}

int ts_scatter_ordered_backward(const void *grad_out, const int64_t *arg, const int64_t *index, void *grad_in, int64_t B,
                                int64_t E, int64_t K, int64_t N, int64_t index_stride_b, int64_t index_stride_e, int dtype,
                                int mean, const void *order, size_t order_bytes, ts_stream_t stream) {
  RowsRoute rr;
  // (minimum and maximum take their order at the same sizes)
  if (!scatter_order_ok(B, E, K, N, dtype, arg != nullptr ? TS_MAX : TS_SUM, rr)) return TS_ERR_UNSUPPORTED;
  if (!grad_out || !index || !grad_in) return TS_ERR_BAD_ARG;
  RowSortPlan sp = row_sort_plan(B, E, N, nullptr, 0, true, const_cast<void *>(order));
  if (!order || !aligned16(order) || order_bytes < sp.kept_bytes || !sp.ok) return TS_ERR_WORKSPACE;
  RowSortArgs p = sp.p;
  p.index = index;
  p.sb = index_stride_b;
  p.se = index_stride_e;
  p.flat = B == 1 && index_stride_e == 1;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (arg != nullptr) {
    if (!aligned16(grad_out) || !aligned16(arg) || !aligned16(grad_in)) return TS_ERR_UNSUPPORTED;
    switch (kElemBytes[dtype]) {
    case 2: return launch_arg_rows<uint16_t, 8>(p, grad_out, arg, grad_in, K, s);
    case 4: return launch_arg_rows<uint32_t, 4>(p, grad_out, arg, grad_in, K, s);
    default: return launch_arg_rows<uint64_t, 2>(p, grad_out, arg, grad_in, K, s);
    }
  }
  switch (dtype) {
  case TS_F32: return launch_rows_spread<float>(p, grad_out, grad_in, K, mean != 0, s);
  case TS_F64: return launch_rows_spread<double>(p, grad_out, grad_in, K, mean != 0, s);
  case TS_F16: return launch_rows_spread<f16_t>(p, grad_out, grad_in, K, mean != 0, s);
  default: return launch_rows_spread<bf16_t>(p, grad_out, grad_in, K, mean != 0, s);
  }
}

int ts_scatter_with_workspace(const void *src, const int64_t *index, void *out, int64_t *arg_out, int64_t B,
                              int64_t E, int64_t K, int64_t N, int64_t index_stride_b, int64_t index_stride_e,
                              int64_t index_stride_k, int dtype, int reduce, int out_given, void *workspace,
                              size_t workspace_bytes, ts_stream_t stream) {
  return scatter_ws_impl(src, index, out, arg_out, B, E, K, N, index_stride_b, index_stride_e, index_stride_k, dtype, reduce,
                         out_given, workspace, workspace_bytes, stream, nullptr, nullptr);
}

}  // extern "C"
namespace {
SmallPlan scatter_small_plan(int64_t B, int64_t E, int64_t K, int64_t N, int dtype, int reduce, bool aligned, bool any_size) {
  const int es = kElemBytes[dtype], full = kVecBytes / es;
  return small_plan(B, E, K, N, es, K % full == 0 && aligned ? full : 1, reduce, any_size);
}
template <typename T> int run_scatter_small(const SmallArgs &a, const SmallPlan &p, bool aligned, int reduce, hipStream_t s) {
  constexpr int kFull = kVecBytes / (int)sizeof(T);
  if (reduce == TS_MEAN) reduce = TS_SUM;
  return a.K % kFull == 0 && aligned ? launch_scatter_small<T, kFull>(a, p, reduce, s) : launch_scatter_small<T, 1>(a, p, reduce, s);
}
}  // namespace
extern "C" {

int ts_scatter_small_applies(int64_t B, int64_t E, int64_t K, int64_t N, int dtype, int reduce) {
  // (most calls end here: nothing is read from the environment)
  if (E > kSmallPer * kSmallBlock || !valid_dtype(dtype) || !is_float_dtype(dtype) || !sizes_ok(B, N, E, K) ||
      (reduce != TS_SUM && reduce != TS_MEAN && reduce != TS_MIN && reduce != TS_MAX))
    return 0;
  auto both = [&](bool any_size) {
    return scatter_small_plan(B, E, K, N, dtype, reduce, true, any_size).ok &&
           scatter_small_plan(B, E, K, N, dtype, reduce, false, any_size).ok;
  };
  if (!both(true)) return 0;
  const int mode = env_int("TS_SCATTER_SMALL", 1);  // (tuning aid) 0 never, 2 at any size that the kernel holds
  return mode == 2 || (mode != 0 && both(false)) ? 1 : 0;
}

int ts_scatter_small(const void *src, const int64_t *index, void *out, void *count, int64_t *arg_out, int64_t B, int64_t E,
                     int64_t K, int64_t N, int64_t index_stride_b, int64_t index_stride_e, int dtype, int reduce, int out_given,
                     ts_stream_t stream) {
  ts_note_scatter_route(TS_ROUTE_NONE);
  if (!ts_scatter_small_applies(B, E, K, N, dtype, reduce)) return TS_ERR_UNSUPPORTED;
  if (!src || !index || !out || ((reduce == TS_MIN || reduce == TS_MAX) && !arg_out)) return TS_ERR_BAD_ARG;
  const bool al = aligned16(src);
  const SmallPlan p = scatter_small_plan(B, E, K, N, dtype, reduce, al, true);
  ts_note_scatter_route(TS_ROUTE_SMALL);
  SmallArgs a = {};
  a.src = src;
  a.index = index;
  a.out = out;
  a.count = count;
  a.arg_out = arg_out;
  a.sb = index_stride_b;
  a.se = index_stride_e;
  a.B = B;
  a.E = E;
  a.K = K;
  a.N = N;
  a.mean = reduce == TS_MEAN ? 1 : 0;
  a.out_given = out_given ? 1 : 0;
  hipStream_t s = static_cast<hipStream_t>(stream);
  switch (dtype) {
  case TS_F32: return run_scatter_small<float>(a, p, al, reduce, s);
  case TS_F64: return run_scatter_small<double>(a, p, al, reduce, s);
  case TS_F16: return run_scatter_small<f16_t>(a, p, al, reduce, s);
  default: return run_scatter_small<bf16_t>(a, p, al, reduce, s);
  }
}

size_t ts_scatter_count_workspace_bytes(int64_t B, int64_t E, int64_t N) {
  if (B < 0 || E < 0 || N < 0 || !env_int("TS_SCATTER_LDS", 1) || !env_int("TS_SCATTER_BINNED", 1)) return 0;
  return bin_plan_payload(B, E, 1, N, 4, nullptr, 0, env_int("TS_SCATTER_BINNED", 1) == 2).bytes;
}

int ts_scatter_count(const int64_t *index, int32_t *count, int64_t B, int64_t E, int64_t N,
                     int64_t index_stride_b, int64_t index_stride_e, ts_stream_t stream) {
  return ts_scatter_count_with_workspace(index, count, B, E, N, index_stride_b, index_stride_e, nullptr, 0, stream);
}

int ts_scatter_count_with_workspace(const int64_t *index, int32_t *count, int64_t B, int64_t E, int64_t N,
                                    int64_t index_stride_b, int64_t index_stride_e, void *workspace,
                                    size_t workspace_bytes, ts_stream_t stream) {
  if (B < 0 || E < 0 || N < 0) return TS_ERR_BAD_ARG;
  if (B * N == 0) return TS_OK;
  if (!count || (B * E > 0 && !index)) return TS_ERR_BAD_ARG;
  hipStream_t s = static_cast<hipStream_t>(stream);
  hipLaunchKernelGGL(fill_kernel<int32_t>, dim3(grid_for(B * N)), dim3(kBlock), 0, s, count, B * N, (int32_t)0);
  if (B * E > 0) {
    // a sum of ones with K = 1: same kernels as scatter sum (src == nullptr adds 1.0 per entry)
    ScatterArgs a;
    a.src = nullptr;
    a.index = index;
    a.out = count;
    a.arg_out = nullptr;
    a.B = B;
    a.E = E;
    a.K = 1;
    a.N = N;
    a.sb = index_stride_b;
    a.se = index_stride_e;
    a.sk = 0;
    a.out_given = 1;
    a.precheck = 1;
    a.lds_cache = env_int("TS_SCATTER_LDS", 1);
    a.lds_epb = env_int("TS_SCATTER_EPB", 0);
    bool binned = false, three_way = false, table_launched = false;
    // A large count under an unsorted index, given scratch: the entries are binned by bucket of output rows like a sum
    // of one value per entry (bin_plan_payload; the "value" of an entry is 1) instead of one device atomic per entry
    // that misses the table. A sample of the index decides; the kernels below then run only for an index that looks sorted.
    if (workspace != nullptr && a.lds_cache && env_int("TS_SCATTER_BINNED", 1) && env_int("TS_SCATTER_RUNS", 1) &&
        B * N < 0x7FFFFFFFll) {  // (the kernels behind it that can be told to stand back)
      const BinPlan bp = bin_plan_payload(B, E, 1, N, 4, workspace, workspace_bytes, env_int("TS_SCATTER_BINNED", 1) == 2);
      if (bp.ok) {
        // the sample of the index gives one of three answers: sorted (the run kernel below), skewed (the table
        // kernel below), even (the buckets); without the table kernel or the sample only the first and the last
        three_way = a.lds_cache == 1 && sum_table_by_size(B, E, 1, N, 4) && B * E >= 2 * kBinBlock &&
                    !getenv("TS_BIN_NO_SAMPLE");
        TableCall table;
        if (three_way && value_tiles_take(bp.p, B * E)) {
          table.tn_mask = kLdsAccRows - 1;
          table.epb = per_cu_chunk_edges(a.lds_epb, B * E, sum_table_min_chunk(1, 4), 131072);
          table.grid = (unsigned)((B * E + table.epb - 1) / table.epb);
        }
        launch_binned_add<int32_t>(a, bp.p, s, three_way, false, table);
        table_launched = table.grid != 0;
        a.skip_flag = bp.p.unsorted;
        binned = true;
      }
    }
    // the sizes from which the sum of one float per entry goes through the accumulator table (a hub otherwise
    // costs an atomic on one address per entry: 4 M entries under a Zipf(1.2) index 1.3 ms against 0.08 ms)
    const bool contended = a.lds_cache == 2 || (a.lds_cache == 1 && sum_table_by_size(B, E, 1, N, 4));
    if (binned) {
      // behind the buckets: the table kernel for a skewed index (flag 2), the run kernel for a sorted one (flag 0)
      if (three_way && !table_launched) {
        ScatterArgs t = a;
        t.skip_want = 2;
        const int64_t epb = per_cu_chunk_edges(a.lds_epb, B * E, sum_table_min_chunk(1, 4), 131072);
        hipLaunchKernelGGL(scatter_add_lds_kernel<int32_t>, dim3((unsigned)((B * E + epb - 1) / epb)), dim3(kLdsAddBlock),
                           0, s, t, kLdsAccRows - 1, epb);
      }
      const RunGrid g = run_grid(B * E, 1, 1, 4);
      launch_add_run<int32_t, 1, 1>(a, g, s);
    } else if (contended && B * N < 0x7FFFFFFFll) {
      const int64_t epb = per_cu_chunk_edges(a.lds_epb, B * E, sum_table_min_chunk(1, 4), 131072);
      hipLaunchKernelGGL(scatter_add_lds_kernel<int32_t>, dim3((unsigned)((B * E + epb - 1) / epb)), dim3(kLdsAddBlock), 0,
                         s, a, kLdsAccRows - 1, epb);
    } else if (env_int("TS_SCATTER_RUNS", 1) && B * N < 0x7FFFFFFFll) {
      // runs of equal neighbouring indices (sorted input) are counted in the wavefront first
      const RunGrid g = run_grid(B * E, 1, 1, 4);
      launch_add_run<int32_t, 1, 1>(a, g, s);
    } else {
      hipLaunchKernelGGL(scatter_count_kernel, dim3(grid_for(B * E)), dim3(kBlock), 0, s, index, count, B, E, N,
                         index_stride_b, index_stride_e);
    }
  }
  return hipGetLastError() == hipSuccess ? TS_OK : TS_ERR_LAUNCH;
}

size_t ts_scatter_sum_count_workspace_bytes(int64_t B, int64_t E, int64_t K, int64_t N, int dtype) {
  const size_t sum = ts_scatter_workspace_bytes(B, E, K, N, dtype, TS_SUM);
  const size_t cnt = ts_scatter_count_workspace_bytes(B, E, N);
  return sum > cnt ? sum : cnt;
}

int ts_scatter_sum_count_with_workspace(const void *src, const int64_t *index, void *out, int32_t *count, int64_t B,
                                        int64_t E, int64_t K, int64_t N, int64_t index_stride_b,
                                        int64_t index_stride_e, int dtype, int out_given, void *workspace,
                                        size_t workspace_bytes, ts_stream_t stream) {
  if (!valid_dtype(dtype) || !sizes_ok(B, N, E, K)) return TS_ERR_BAD_ARG;
  if (B * N == 0) return TS_OK;
  if (!count) return TS_ERR_BAD_ARG;
  hipStream_t s = static_cast<hipStream_t>(stream);
  // The sum. If it goes through the buckets, their adding pass counts as well (one pass over the index for both) and
  // leaves the buckets' flag here: 1 = the buckets took the call.
  const int *flag = nullptr;
  bool may_fuse = B * E * K > 0 && workspace != nullptr && B * N < 0x7FFFFFFFll && env_int("TS_SCATTER_RUNS", 1) &&
                  env_int("TS_SCATTER_LDS", 1) && env_int("TS_SCATTER_BINNED", 1);
  if (may_fuse) {  // only where the sum has a plan for the buckets (else count is cleared by its own call below)
    const bool any_size = env_int("TS_SCATTER_BINNED", 1) == 2;
    may_fuse = K <= kBinPayloadCols && (dtype == TS_F32 || dtype == TS_I32) &&
               bin_plan_payload(B, E, K, N, 4, workspace, workspace_bytes, any_size).ok;
  }
  if (may_fuse)
    hipLaunchKernelGGL(fill_kernel<int32_t>, dim3(grid_for(B * N)), dim3(kBlock), 0, s, count, B * N, (int32_t)0);
  // (a small sum clears and counts by itself, in the launches that clear out and add: then `counted` reads 1)
  int counted = 0;
  const int rc = scatter_ws_impl(src, index, out, nullptr, B, E, K, N, index_stride_b, index_stride_e, 0, dtype, TS_SUM,
                                 out_given, workspace, workspace_bytes, stream, count, may_fuse ? &flag : nullptr, &counted);
  if (rc != TS_OK || counted == 1) return rc;
  if (flag == nullptr)  // another route: the count on its own (with its own fill)
    return ts_scatter_count_with_workspace(index, count, B, E, N, index_stride_b, index_stride_e, workspace, workspace_bytes,
                                           stream);
  // the kernels behind the buckets, for the counts: the table for a skewed index (flag 2, single values only), runs for
  // a sorted one (flag 0)
  ScatterArgs c;
  c.src = nullptr;
  c.index = index;
  c.out = count;
  c.arg_out = nullptr;
  c.B = B;
  c.E = E;
  c.K = 1;
  c.N = N;
  c.sb = index_stride_b;
  c.se = index_stride_e;
  c.sk = 0;
  c.out_given = 1;
  c.precheck = 1;
  c.lds_cache = env_int("TS_SCATTER_LDS", 1);
  c.lds_epb = env_int("TS_SCATTER_EPB", 0);
  c.skip_flag = flag;
  if (K <= kBinPayloadCols && counted != 2) {  // (the plans whose sample can answer "skewed"; 2: the sum's table counted)
    ScatterArgs t = c;
    t.skip_want = 2;
    const int64_t epb = per_cu_chunk_edges(c.lds_epb, B * E, sum_table_min_chunk(1, 4), 131072);
    hipLaunchKernelGGL(scatter_add_lds_kernel<int32_t>, dim3((unsigned)((B * E + epb - 1) / epb)), dim3(kLdsAddBlock), 0, s,
                       t, kLdsAccRows - 1, epb);
  }
  const RunGrid g = run_grid(B * E, 1, 1, 4);
  launch_add_run<int32_t, 1, 1>(c, g, s);
  return hipGetLastError() == hipSuccess ? TS_OK : TS_ERR_LAUNCH;
}

int ts_divide_by_count(void *out, const int32_t *count, int64_t B, int64_t N, int64_t K, int dtype,
                       ts_stream_t stream) {
  if (!valid_dtype(dtype) || B < 0 || N < 0 || K < 0) return TS_ERR_BAD_ARG;
  if (B * N * K == 0) return TS_OK;
  if (!out || !count) return TS_ERR_BAD_ARG;
  return dispatch_divide(dtype, out, count, B * N, K, static_cast<hipStream_t>(stream));
}

int ts_arg_backward(const void *grad_out, const int64_t *arg, void *grad_in, int64_t B, int64_t N, int64_t E,
                    int64_t K, int dtype, ts_stream_t stream) {
  if (!valid_dtype(dtype) || B < 0 || N < 0 || E < 0 || K < 0) return TS_ERR_BAD_ARG;
  if (B * E * K == 0) return TS_OK;
  if (!grad_in || (B * N * K > 0 && (!grad_out || !arg))) return TS_ERR_BAD_ARG;
  return dispatch_arg_backward(dtype, grad_out, arg, grad_in, B, N, E, K, static_cast<hipStream_t>(stream));
}

size_t ts_arg_backward_rows_workspace_bytes(int64_t B, int64_t E, int64_t K, int64_t N, int dtype) {
  if (!valid_dtype(dtype) || !is_float_dtype(dtype) || !sizes_ok(B, N, E, K) || B * E == 0 || N == 0) return 0;
  const int mode = env_int("TS_SCATTER_BINNED", 1);  // tuning aid: 0 never, 2 at any size
  const int64_t row_bytes = K * kElemBytes[dtype];
  if (mode == 0 || row_bytes < 64 || K >= (int64_t)1 << 20) return 0;
  // As long as grad_in fits the 256 MB of the memory-side cache, the second pass over it is cheap (us of ts_arg_backward /
  // this call, even index and a hub: 1 M x 64 floats, 10 a row 90 / 92 and 65 / 90). Beyond it the elements of grad_out, 14 ps
  // each in the scatter, outweigh the sort (25 ps an entry and 30 us at the least) from B N K = 2.1 M + 1.8 B E on under an
  // even index. Under a hub fewer of them win, so the line lies at about twice that: 2.3 M entries, 10 a row, 64 floats 414 /
  // 196 and 188 / 168, 128 bf16 458 / 313 and 226 / 238; 30 a row, left to the scatter, 281 / 164 and 160 / 167, 368 / 225 and
  // 176 / 236. Rows that fill no 16-byte vector do not gain (33 doubles, 2 M, 4 a row 458 / 480 and 223 / 348).
  if (mode != 2 && (row_bytes < 256 || row_bytes % kVecBytes != 0 || B * E * row_bytes < 384000000 ||
                    B * N * K < ((int64_t)4 << 20) + 3 * B * E))
    return 0;
  return row_sort_plan(B, E, N, nullptr, 0, true).bytes;
}

int ts_arg_backward_rows(const void *grad_out, const int64_t *arg, const int64_t *index, void *grad_in, int64_t B, int64_t N,
                         int64_t E, int64_t K, int64_t index_stride_b, int64_t index_stride_e, int dtype, void *workspace,
                         size_t workspace_bytes, ts_stream_t stream) {
  const size_t need = ts_arg_backward_rows_workspace_bytes(B, E, K, N, dtype);
  if (need == 0) return TS_ERR_UNSUPPORTED;
  if (!grad_out || !arg || !index || !grad_in) return TS_ERR_BAD_ARG;
  if (!workspace || workspace_bytes < need || !aligned16(workspace)) return TS_ERR_WORKSPACE;
  RowSortPlan sp = row_sort_plan(B, E, N, workspace, workspace_bytes, true);
  if (!sp.ok) return TS_ERR_WORKSPACE;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int rc = launch_row_sort(sp.p, index, index_stride_b, index_stride_e, false, next_nonce(), s);
  if (rc != TS_OK) return rc;
  RowSortArgs p = sp.p;
  p.index = index;
  p.sb = index_stride_b;
  p.se = index_stride_e;
  p.flat = B == 1 && index_stride_e == 1;
  const int es = kElemBytes[dtype], full = kVecBytes / es;
  const bool wide = K % full == 0 && aligned16(grad_out) && aligned16(arg) && aligned16(grad_in);
  if (es == 2)
    return wide ? launch_arg_rows<uint16_t, 8>(p, grad_out, arg, grad_in, K, s)
                : launch_arg_rows<uint16_t, 1>(p, grad_out, arg, grad_in, K, s);
  if (es == 4)
    return wide ? launch_arg_rows<uint32_t, 4>(p, grad_out, arg, grad_in, K, s)
                : launch_arg_rows<uint32_t, 1>(p, grad_out, arg, grad_in, K, s);
  return wide ? launch_arg_rows<uint64_t, 2>(p, grad_out, arg, grad_in, K, s)
              : launch_arg_rows<uint64_t, 1>(p, grad_out, arg, grad_in, K, s);
}

namespace {
// std / logsumexp backward with a workspace of ts_group_softmax_workspace_bytes(): the values an entry needs of its group
// are laid side by side first (one more launch over [B, N, K]) when there are at least as many entries as groups
bool group_coef_ok(int64_t B, int64_t E, int64_t N, int64_t K, int dtype, const void *ws, size_t ws_bytes) {
  if (ws == nullptr || (reinterpret_cast<uintptr_t>(ws) & 31) != 0 || !env_int("TS_GROUP_COEF", 1)) return false;
  if (E < N) return false;
  return ws_bytes >= (size_t)(B * N * K) * 2 * (kElemBytes[dtype] == 8 ? 8 : 4);
}
// columns per lane of the bucket kernels: 16 bytes when the row allows it
int group_bins_vec(int64_t K, int dtype, bool aligned) {
  const int full = kVecBytes / kElemBytes[dtype];
  return (full > 1 && K % full == 0 && aligned) ? full : 1;
}
// TS_GROUP_BINS (tuning aid): 0 the buckets of groups never take a call, 2 they take it at any size
GroupBinPlan group_bins_plan(int64_t B, int64_t E, int64_t K, int64_t N, int dtype, bool aligned, void *ws, size_t ws_bytes) {
  const int mode = env_int("TS_GROUP_BINS", 1);
  if (mode == 0) {
    GroupBinPlan r;
    r.ok = false;
    r.bytes = 0;
    return r;
  }
  // the buckets' scratch lies behind the workspace of the three passes (softmax keeps its keys, sums and flag there)
  const size_t front = group_workspace_bytes(B, N, K, kElemBytes[dtype]);
  GroupBinPlan r = group_bin_plan(B, E, K, N, kElemBytes[dtype], group_bins_vec(K, dtype, aligned),
                                  ws != nullptr && ws_bytes > front ? static_cast<char *>(ws) + front : nullptr,
                                  ws_bytes > front ? ws_bytes - front : 0, mode == 2);
  if (r.bytes > 0) r.bytes += front;
  return r;
}
// std / logsumexp: the one-pass tiles for an index in order, their scratch behind that of the buckets (at ws + skip).
// TS_GROUP_FUSED (tuning aid): 0 never, 2 at any size and whatever the index looks like.
FusedReducePlan group_tiles_plan(int64_t B, int64_t E, int64_t K, int64_t N, int dtype, bool aligned, void *ws,
                                 size_t ws_bytes, size_t skip) {
  const int mode = env_int("TS_GROUP_FUSED", 1);
  if (mode == 0 || skip == 0) {
    FusedReducePlan r;
    r.ok = false;
    r.bytes = 0;
    return r;
  }
  return group_reduce_fused_plan(B, E, K, N, kElemBytes[dtype], aligned,
                                 ws != nullptr && ws_bytes > skip ? static_cast<char *>(ws) + skip : nullptr,
                                 ws_bytes > skip ? ws_bytes - skip : 0, mode == 2);
}
}  // namespace

namespace {
int run_group_softmax(const void *src, const void *grad, const int64_t *index, void *out, int64_t B, int64_t E,
                      int64_t K, int64_t N, int64_t sb, int64_t se, int dtype, int mode, double eps, void *workspace,
                      size_t workspace_bytes, hipStream_t stream) {
  if (!valid_dtype(dtype) || !sizes_ok(B, N, E, K)) return TS_ERR_BAD_ARG;
  if (!is_float_dtype(dtype)) return TS_ERR_UNSUPPORTED;
  if (B * E * K == 0) return TS_OK;
  if (!src || !index || !out) return TS_ERR_BAD_ARG;
  if ((mode == GS_SOFTMAX_BWD || mode == GS_LOG_SOFTMAX_BWD) && !grad) return TS_ERR_BAD_ARG;
  if (N == 0 || B * N >= 0x7FFFFFFFll) return TS_ERR_UNSUPPORTED;
  const size_t need = group_workspace_bytes(B, N, K, kElemBytes[dtype]);
  if (!workspace || workspace_bytes < need || !aligned16(workspace)) return TS_ERR_WORKSPACE;
  GroupArgs g;
  g.src = src;
  g.grad = grad;
  g.index = index;
  g.out = out;
  g.gmax = workspace;
  // forward: a group's keys and sums side by side (the finish reads both with one line); backward: sums only
  const bool with_keys = mode == GS_SOFTMAX || mode == GS_LOG_SOFTMAX;
  g.gs = with_keys ? 2 * K : K;
  g.gsum = static_cast<char *>(workspace) + (with_keys ? (size_t)K * (kElemBytes[dtype] == 8 ? 8 : 4) : 0);
  g.B = B;
  g.E = E;
  g.K = K;
  g.N = N;
  g.sb = sb;
  g.se = se;
  g.eps = eps;
  g.node_out = nullptr;
  g.node_grad = nullptr;
  g.from_neg_inf = 0;
  g.total = nullptr;
  g.count = nullptr;
  g.unbiased = 0;
  g.ws_bytes = group_three_pass_bytes(B, N, K, kElemBytes[dtype]);
  g.flag = reinterpret_cast<int *>(static_cast<char *>(workspace) + g.ws_bytes);
  const int full = kVecBytes / kElemBytes[dtype];
  const bool al = aligned16(src) && aligned16(out) && (!grad || aligned16(grad));
  const int vec = (full > 1 && K % full == 0 && al) ? full : 1;
  // forward with a workspace of ts_group_bins_workspace_bytes(): an index that is not in order goes through buckets of groups
  GroupBinPlan plan;
  plan.ok = false;
  if (with_keys) {
    plan = group_bins_plan(B, E, K, N, dtype, al, workspace, workspace_bytes);
    // (rows of up to 128 bytes, where the one-pass tiles take an index in order: for wider rows the three passes are
    // ahead under a sorted index, 1 M x 128 floats 570 against 741 us, and behind under a random one, 663 against 449)
    // (nor for few groups of many entries in rows of more than 64 bytes, which the tiles decline as well: 4 M x 64 bf16
    // in 4 k groups, sorted, 890 against 1116 us)
    const int64_t row_bytes = K * kElemBytes[dtype];
    const bool tiles_cover = row_bytes <= 64 || (row_bytes <= kFusedRowBytes && E <= 64 * N);
    if (plan.ok && group_bins_vec(K, dtype, al) == vec && (tiles_cover || env_int("TS_GROUP_BINS", 1) == 2))
      g.bins = &plan.p;
  }
  // a workspace of ts_group_workspace_bytes(): what lies behind the three passes' (and the buckets') part is scratch
  // for the one-pass tiles
  const size_t used = plan.ok ? plan.bytes : need;
  if (workspace_bytes > used) {
    g.fused_ws = static_cast<char *>(workspace) + used;
    g.fused_ws_bytes = workspace_bytes - used;
  }
  return dispatch_group_softmax(dtype, g, mode, vec, stream);
}
}  // namespace

namespace {
// Softmax over entries sorted by group (row_sort.h, group_rows.h, the ordered tiles of group_fused.h). Where the tiles for an index in
// order apply they come first, behind a sample of the index, and what follows returns at once if they took the call: an
// index in order costs what it did without the sort (and the sort of one that is not, 14 us for the launches in front).
// Where the line lies (us without / with, groups of 30; even, Zipf(1.2) hub, both in no order, then both in order):
//   forward, from 8 MB: 300 k x 8 floats 55 88 43 76 / 41 75 30 46, 100 k x 32 45 68 42 65 / 38 70 31 46, 66 k x 32 41 63 40 62 / 35 66
//   28 42; rows above 128 bytes from 10 MB: 33 k x 64 45 54 28 30 / 35 65 29 42, 20 k x 128 49 58 30 32 / 34 51 29 42, 50 k x 64 58 69 34
//   37 / 37 67 31 44. Up to 128 entries a group; below 16 MB 64 in rows above 64 bytes, 32 above 128: groups of 120, 200 k x 16 52 86 44
//   78 / 49 71 39 44, 100 k x 32 65 69 32 34 / 50 70 43 46, 100 k x 64 92 99 56 56 / 62 79 55 54; groups of 60, 50 k x 64 59 64 32 34 /
//   43 70 36 46. With 1000 the tables in LDS hold every group, 300 k x 8 62 82 52 70 / 61 75 49 48, but 300 k x 4 60 95 48 77 / 53 71 40
//   42 against 100 k x 32 52 53 33 34 / 57 79 49 56 and, in order, 3 M x 32 430 550 / 471 1314.
// TS_GROUP_ORDER (tuning aid): 0 never, 2 at any size; 3: at any size, and never the tiles for an index in order.
bool group_order_rule(int64_t B, int64_t E, int64_t K, int64_t N, int dtype) {
  if (!valid_dtype(dtype) || !is_float_dtype(dtype) || !sizes_ok(B, N, E, K) || B * E * K == 0 || N == 0) return false;
  const int mode = env_int("TS_GROUP_ORDER", 1);
  const int64_t row_bytes = K * kElemBytes[dtype], bytes = B * E * row_bytes;
  if (mode == 0 || K >= (int64_t)1 << 20 || row_bytes % kVecBytes != 0) return false;
  if (mode >= 2) return true;
  const int64_t least = (int64_t)(row_bytes <= 128 ? 8 : 10) << 20;
  const int64_t most = bytes >= (int64_t)16 << 20 || row_bytes <= 64 ? 128 : row_bytes <= 128 ? 64 : 32;
  return bytes >= least && E <= most * N;
}
// What else goes over the sorted entries (group_rows.h). op: 0 softmax, 1 logsumexp, 2 std. The passes that it replaces add and
// compare in memory, element by element unless rows are whole 16-byte units, so rows that are not, and 16-bit elements, gain from
// smaller inputs on. us without / with the sort, forward and backward (f: forward alone), entries x columns:
//   softmax    1.7 M x 199 bf16, 4 a group 7719 / 2561; 580 k x 98 floats, 39 a group 1321 / 589; f 1.3 M x 1 bf16, 30 a group 177 / 48;
//              f 29 k x 64 bf16 46 / 30; 18 k x 146 floats, 260 a group 252 / 81. Left: f 950 k x 1 floats in order 30 / 53; 5.4 M x 1
//              floats under a hub, 280 a group 412 / 612; 4.8 M x 128 floats in order, 147 a group (2.3 GB) 3886 / 5101
//   logsumexp  606 k x 256 floats 1793 / 685, f 348 k x 32 floats 128 / 63, f 8.1 M x 3 f16 359 / 247. Left: 3.3 M x 1 floats, 46 a
//              group 159 / 207; f 4.8 M x 256 bf16 in order (2.3 GB) 2342 / 3118
//   std        f 2.65 M x 64 floats, 207 a group 897 / 476; 484 k x 128 floats under a hub 518 / 320. Left: f 580 k x 256 floats in
//              order 253 / 402; 5.1 M x 100 floats in order (2 GB) 2295 / 3334; 1.7 M x 100 floats, 297 a group 865 / 1198 (pieces that
//              are not lines); 19 M x 4 floats under a hub, 359 a group 1204 / 1868
// 440 drawn calls of all sizes, those that stay among them: 0.86 of the time in the geometric mean.
bool group_rows_rule(int64_t B, int64_t E, int64_t K, int64_t N, int dtype, int op) {
  if (!valid_dtype(dtype) || !is_float_dtype(dtype) || !sizes_ok(B, N, E, K) || B * E * K == 0 || N == 0) return false;
  if (op < 0 || op > 2 || K >= (int64_t)1 << 20) return false;
  const int mode = env_int("TS_GROUP_ORDER", 1);
  if (mode == 0) return false;
  if (mode >= 2) return true;
  const int es = kElemBytes[dtype];
  const int64_t row_bytes = K * es, bytes = B * E * row_bytes, MB = (int64_t)1 << 20;
  if (op == 0) {
    if (group_order_rule(B, E, K, N, dtype)) return true;
    if (E > 128 * N && (bytes > 1024 * MB || row_bytes < 32)) return false;
    if (row_bytes >= 128) return bytes >= (es == 2 ? MB : 8 * MB);
    return bytes >= (es == 2 ? 2 * MB : 8 * MB) && E <= (K <= 2 ? 32 : 512) * N;
  }
  if (op == 1 && es == 2 && bytes > 1024 * MB) return false;
  if (op == 2) {
    if (row_bytes > 512 || bytes > 1024 * MB || E > (row_bytes < 64 ? 128 : 4096) * N) return false;
    if (row_bytes > 256 && row_bytes % 128 != 0 && bytes > 256 * MB) return false;
  }
  if (K == 1) return bytes >= 4 * MB && E <= 16 * N;
  return bytes >= (row_bytes >= 128 ? 4 * MB : 8 * MB);
}
// plan of the tiles for an index in order, their records at ws; false: they do not apply
bool group_order_tiles(GroupArgs &g, int dtype, int mode, void *ws, size_t ws_bytes, int *flag, FusedArgs &f) {
  if (env_int("TS_GROUP_FUSED", 1) == 0 || env_int("TS_GROUP_ORDER", 1) == 3) return false;
  const bool backward = mode == GS_SOFTMAX_BWD || mode == GS_LOG_SOFTMAX_BWD;
  if (!group_fused_plan(g, mode, kElemBytes[dtype], ws, ws_bytes, backward, f)) return false;
  f.flag = flag;
  return true;
}
// 16-bit rows of whole 16-byte units: the forward pass of softmax takes the tiles of group_fused.h over the sorted entries,
// whose lanes hold eight elements (128 columns of bf16 in groups of 20, 2.6 M entries: 884 us, 1059 with the rows in registers;
// 64 columns in groups of 5, 5.1 M entries: 873 / 938), and whose tiles are longer where groups are (128 floats in groups of 117,
// 1.3 M entries: 611 / 766). Other rows the other way round: 128 floats, groups of 6, 1.3 M entries, forward and backward 1537 / 842.
bool group_rows_in_tiles(int64_t B, int64_t E, int64_t K, int64_t N, int dtype, int mode) {
  return (mode == GS_SOFTMAX || mode == GS_LOG_SOFTMAX) && (kElemBytes[dtype] == 2 || E > 64 * N) &&
         group_order_rule(B, E, K, N, dtype) && group_fused_ordered_plan(B * E, K, kElemBytes[dtype], nullptr).bytes > 0;
}
size_t group_rows_records(int64_t B, int64_t E, int64_t K, int64_t N, int dtype) {
  size_t most = group_rows_plan(B * E, B * N, K, kElemBytes[dtype], nullptr).bytes;  // (one after the other)
  auto with = [&](size_t bytes) { most = bytes > most ? bytes : most; };
  with(group_fused_scratch_bytes(B, E, K, kElemBytes[dtype]));
  with(group_reduce_fused_plan(B, E, K, N, kElemBytes[dtype], true, nullptr, 0, false).bytes);
  if (group_rows_in_tiles(B, E, K, N, dtype, GS_SOFTMAX)) with(group_fused_ordered_plan(B * E, K, kElemBytes[dtype], nullptr).bytes);
  return most;
}
// sorted: the order, made by a forward call and read by a backward call. g: the call's own arrays, for one list of entries and
// groups still to be described. sorted.state[4] reads 0 if the tiles for an index in order took the forward call: then there is
// no order.
int run_group_rows(GroupArgs g, int64_t B, int64_t E, int64_t K, int64_t N, int64_t sb, int64_t se, int dtype, int mode,
                   const RowSortArgs &sorted, void *records, size_t records_bytes, hipStream_t stream) {
  const bool softmax = mode == GS_SOFTMAX || mode == GS_LOG_SOFTMAX || mode == GS_SOFTMAX_BWD || mode == GS_LOG_SOFTMAX_BWD;
  const bool backward = mode == GS_SOFTMAX_BWD || mode == GS_LOG_SOFTMAX_BWD || mode == GS_STD_BWD || mode == GS_LSE_BWD;
  const int es = kElemBytes[dtype];
  GroupRowsPlan p = group_rows_plan(B * E, B * N, K, es, records);
  if (p.bytes == 0) return TS_ERR_UNSUPPORTED;
  g.B = B;
  g.E = E;
  g.K = K;
  g.N = N;
  g.sb = sb;
  g.se = se;
  bool tried = false;  // the tiles for an index in order, in front
  int *const flag = sorted.state + 4;
  const bool al = aligned16(g.src) && aligned16(g.out) && (g.grad == nullptr || aligned16(g.grad));
  if (softmax && K * es <= 64) {  // (rows that the tiles of either direction hold)
    FusedArgs tiles;
    GroupArgs any = g;  // (do the sizes allow them?)
    any.src = any.grad = any.out = nullptr;
    const int fwd_mode = mode == GS_SOFTMAX_BWD ? GS_SOFTMAX : mode == GS_LOG_SOFTMAX_BWD ? GS_LOG_SOFTMAX : mode;
    tried = group_order_tiles(any, dtype, fwd_mode, records, records_bytes, flag, tiles);
    if (tried && backward && !al) return TS_ERR_UNSUPPORTED;  // (they may hold the only way to the result)
    tried = tried && al;
    if (tried) {
      if (!group_order_tiles(g, dtype, mode, records, records_bytes, flag, tiles)) return TS_ERR_UNSUPPORTED;
      g.in_order = &tiles;
      g.in_order_sample = backward ? 0 : 1;
      const int full = kVecBytes / es;
      const int rc = dispatch_group_softmax(dtype, g, mode, K % full == 0 ? full : 1, stream);
      if (rc != TS_OK) return rc;
      g.in_order = nullptr;
    }
  } else if ((mode == GS_LSE || mode == GS_STD) && K * es <= kFusedRowBytes && env_int("TS_GROUP_FUSED", 1) != 0 &&
             env_int("TS_GROUP_ORDER", 1) != 3) {
    // (wider rows: the tiles in front are behind; 64 floats in groups of 91, in order, 8.4 M entries, std forward and backward
    // 2581 us with them, 2217 without; 32 floats in groups of 9, logsumexp forward: 257 / 559)
    FusedReducePlan tiles = group_reduce_fused_plan(B, E, K, N, es, aligned16(g.src), records, records_bytes, false);
    tried = tiles.ok;
    if (tried) {
      tiles.f.flag = flag;
      g.tiles = &tiles.f;
      const int rc = dispatch_group_softmax(dtype, g, mode == GS_STD ? GS_STD_BINS : GS_LSE_BINS,
                                            group_bins_vec(K, dtype, aligned16(g.src)), stream);
      if (rc != TS_OK) return rc;
      g.tiles = nullptr;
    }
  }
  if (!backward) {
    const int rc = launch_row_sort(sorted, g.index, sb, se, false, next_nonce(), stream, tried ? flag : nullptr);
    if (rc != TS_OK) return rc;
  }
  g.B = 1;
  g.E = B * E;
  g.N = B * N;
  if (al && group_rows_in_tiles(B, E, K, N, dtype, mode)) {
    FusedOrderedPlan o = group_fused_ordered_plan(B * E, K, es, records);
    o.f.gate = tried ? flag : nullptr;
    o.f.state = sorted.state;
    o.f.n_sorted = sorted.ptr + B * N;
    o.f.perm = sorted.perm;
    o.f.group = sorted.perm_row;
    o.f.ptr = sorted.ptr;
    o.f.index = g.index;
    o.f.sb = sb;
    o.f.se = se;
    o.f.E0 = E;
    o.f.N0 = N;
    g.ordered = &o.f;
    return dispatch_group_softmax(dtype, g, mode, kVecBytes / es, stream);
  }
  p.f.gate = tried ? flag : nullptr;
  p.f.state = sorted.state;
  p.f.ptr = sorted.ptr;
  p.f.perm = sorted.perm;
  p.f.group = sorted.perm_row;
  p.f.index = g.index;
  p.f.sb = sb;
  p.f.se = se;
  p.f.E0 = E;
  p.f.N0 = N;
  if (!aligned16(g.out)) p.f.stream = 0;
  return dispatch_group_rows(dtype, g, p.f, mode, stream);
}
// (sizes that the rule and the plans take)
bool group_rows_ok(int64_t B, int64_t E, int64_t K, int64_t N, int dtype, int op) {
  return group_rows_rule(B, E, K, N, dtype, op) && row_sort_plan(B, E, N, nullptr, 0, true).bytes > 0 &&
         group_rows_plan(B * E, B * N, K, kElemBytes[dtype], nullptr).bytes > 0;
}
// the order of a backward call, as the forward call left it
int group_rows_saved(const void *order, size_t order_bytes, void *workspace, size_t workspace_bytes, int64_t B, int64_t E,
                     int64_t K, int64_t N, int dtype, int op, RowSortPlan &sp) {
  if (!group_rows_ok(B, E, K, N, dtype, op)) return TS_ERR_UNSUPPORTED;
  sp = row_sort_plan(B, E, N, nullptr, 0, true, const_cast<void *>(order));
  if (!order || order_bytes < sp.kept_bytes || !aligned16(order) || !workspace || !aligned16(workspace) ||
      workspace_bytes < group_rows_records(B, E, K, N, dtype) || !sp.ok)
    return TS_ERR_WORKSPACE;
  return TS_OK;
}
int group_rows_made(void *order, size_t order_bytes, void *workspace, size_t workspace_bytes, int64_t B, int64_t E, int64_t K,
                    int64_t N, int dtype, int op, RowSortPlan &sp) {
  if (!group_rows_ok(B, E, K, N, dtype, op)) return TS_ERR_UNSUPPORTED;
  const size_t records = group_rows_records(B, E, K, N, dtype);
  if (!order || !aligned16(order) || !workspace || !aligned16(workspace) || workspace_bytes < records) return TS_ERR_WORKSPACE;
  sp = row_sort_plan(B, E, N, static_cast<char *>(workspace) + records, workspace_bytes - records, true, order);
  return sp.ok && order_bytes >= sp.kept_bytes ? TS_OK : TS_ERR_WORKSPACE;
}
}  // namespace

size_t ts_group_order_bytes(int64_t B, int64_t E, int64_t K, int64_t N, int dtype) {
  // (a slice of the tiles that this form used to take held 16-byte units of 128 bytes)
  if (!group_order_rule(B, E, K, N, dtype) || (K * kElemBytes[dtype] + 127) / 128 > 65535) return 0;
  return ts_group_rows_order_bytes(B, E, K, N, dtype, 0);
}

size_t ts_group_order_workspace_bytes(int64_t B, int64_t E, int64_t K, int64_t N, int dtype, int backward) {
  if (ts_group_order_bytes(B, E, K, N, dtype) == 0) return 0;
  return ts_group_rows_workspace_bytes(B, E, K, N, dtype, 0, backward);
}

size_t ts_group_rows_order_bytes(int64_t B, int64_t E, int64_t K, int64_t N, int dtype, int op) {
  return group_rows_ok(B, E, K, N, dtype, op) ? row_sort_plan(B, E, N, nullptr, 0, true).kept_bytes : 0;
}

size_t ts_group_rows_workspace_bytes(int64_t B, int64_t E, int64_t K, int64_t N, int dtype, int op, int backward) {
  if (!group_rows_ok(B, E, K, N, dtype, op)) return 0;
  const RowSortPlan sp = row_sort_plan(B, E, N, nullptr, 0, true);
  return group_rows_records(B, E, K, N, dtype) + (backward ? 0 : sp.bytes - sp.kept_bytes);
}

int ts_group_softmax_ordered(const void *src, const int64_t *index, void *out, int64_t B, int64_t E, int64_t K, int64_t N,
                             int64_t index_stride_b, int64_t index_stride_e, int dtype, int log_space, double eps,
                             void *order, size_t order_bytes, void *workspace, size_t workspace_bytes, ts_stream_t stream) {
  RowSortPlan sp;
  if (!group_rows_ok(B, E, K, N, dtype, 0)) return TS_ERR_UNSUPPORTED;
  if (!src || !index || !out) return TS_ERR_BAD_ARG;
  const int rc = group_rows_made(order, order_bytes, workspace, workspace_bytes, B, E, K, N, dtype, 0, sp);
  if (rc != TS_OK) return rc;
  GroupArgs g = {};
  g.src = src;
  g.index = index;
  g.out = out;
  g.eps = eps;
  return run_group_rows(g, B, E, K, N, index_stride_b, index_stride_e, dtype, log_space ? GS_LOG_SOFTMAX : GS_SOFTMAX, sp.p,
                        workspace, group_rows_records(B, E, K, N, dtype), static_cast<hipStream_t>(stream));
}

int ts_group_softmax_ordered_backward(const void *result, const void *grad_out, const int64_t *index, void *grad_in, int64_t B,
                                      int64_t E, int64_t K, int64_t N, int64_t index_stride_b, int64_t index_stride_e,
                                      int dtype, int log_space, const void *order, size_t order_bytes, void *workspace,
                                      size_t workspace_bytes, ts_stream_t stream) {
  RowSortPlan sp;
  if (!group_rows_ok(B, E, K, N, dtype, 0)) return TS_ERR_UNSUPPORTED;
  if (!result || !grad_out || !index || !grad_in) return TS_ERR_BAD_ARG;
  const int rc = group_rows_saved(order, order_bytes, workspace, workspace_bytes, B, E, K, N, dtype, 0, sp);
  if (rc != TS_OK) return rc;
  GroupArgs g = {};
  g.src = result;
  g.grad = grad_out;
  g.index = index;
  g.out = grad_in;
  return run_group_rows(g, B, E, K, N, index_stride_b, index_stride_e, dtype, log_space ? GS_LOG_SOFTMAX_BWD : GS_SOFTMAX_BWD,
                        sp.p, workspace, group_rows_records(B, E, K, N, dtype), static_cast<hipStream_t>(stream));
}

int ts_group_reduce_ordered(const void *src, const int64_t *index, void *out, void *total, int32_t *count, int64_t B, int64_t E,
                            int64_t K, int64_t N, int64_t index_stride_b, int64_t index_stride_e, int dtype, int std_dev,
                            int unbiased, double eps, void *order, size_t order_bytes, void *workspace, size_t workspace_bytes,
                            ts_stream_t stream) {
  RowSortPlan sp;
  const int op = std_dev ? 2 : 1;
  if (!group_rows_ok(B, E, K, N, dtype, op)) return TS_ERR_UNSUPPORTED;
  if (!src || !index || !out || (std_dev && (!total || !count))) return TS_ERR_BAD_ARG;
  const int rc = group_rows_made(order, order_bytes, workspace, workspace_bytes, B, E, K, N, dtype, op, sp);
  if (rc != TS_OK) return rc;
  GroupArgs g = {};
  g.src = src;
  g.index = index;
  g.out = out;
  g.total_w = total;
  g.count_w = count;
  g.unbiased = unbiased ? 1 : 0;
  g.eps = eps;
  return run_group_rows(g, B, E, K, N, index_stride_b, index_stride_e, dtype, std_dev ? GS_STD : GS_LSE, sp.p, workspace,
                        group_rows_records(B, E, K, N, dtype), static_cast<hipStream_t>(stream));
}

int ts_group_reduce_ordered_backward(const void *src, const int64_t *index, const void *out, const void *total,
                                     const int32_t *count, const void *grad_out, void *grad_in, int64_t B, int64_t E, int64_t K,
                                     int64_t N, int64_t index_stride_b, int64_t index_stride_e, int dtype, int std_dev,
                                     int unbiased, const void *order, size_t order_bytes, void *workspace,
                                     size_t workspace_bytes, ts_stream_t stream) {
  RowSortPlan sp;
  const int op = std_dev ? 2 : 1;
  if (!group_rows_ok(B, E, K, N, dtype, op)) return TS_ERR_UNSUPPORTED;
  if (!src || !index || !out || !grad_out || !grad_in || (std_dev && (!total || !count))) return TS_ERR_BAD_ARG;
  const int rc = group_rows_saved(order, order_bytes, workspace, workspace_bytes, B, E, K, N, dtype, op, sp);
  if (rc != TS_OK) return rc;
  GroupArgs g = {};
  g.src = src;
  g.index = index;
  g.out = grad_in;
  g.node_out = out;
  g.node_grad = grad_out;
  g.total = total;
  g.count = count;
  g.unbiased = unbiased ? 1 : 0;
  return run_group_rows(g, B, E, K, N, index_stride_b, index_stride_e, dtype, std_dev ? GS_STD_BWD : GS_LSE_BWD, sp.p, workspace,
                        group_rows_records(B, E, K, N, dtype), static_cast<hipStream_t>(stream));
}

size_t ts_group_softmax_workspace_bytes(int64_t B, int64_t N, int64_t K, int dtype) {
  if (!valid_dtype(dtype) || B < 0 || N < 0 || K < 0) return 0;
  return group_workspace_bytes(B, N, K, kElemBytes[dtype]);
}

int ts_group_softmax(const void *src, const int64_t *index, void *out, int64_t B, int64_t E, int64_t K, int64_t N,
                     int64_t index_stride_b, int64_t index_stride_e, int dtype, int log_space, double eps,
                     void *workspace, size_t workspace_bytes, ts_stream_t stream) {
  return run_group_softmax(src, nullptr, index, out, B, E, K, N, index_stride_b, index_stride_e, dtype,
                           log_space ? GS_LOG_SOFTMAX : GS_SOFTMAX, eps, workspace, workspace_bytes,
                           static_cast<hipStream_t>(stream));
}

int ts_group_softmax_backward(const void *result, const void *grad_out, const int64_t *index, void *grad_in,
                              int64_t B, int64_t E, int64_t K, int64_t N, int64_t index_stride_b,
                              int64_t index_stride_e, int dtype, int log_space, void *workspace,
                              size_t workspace_bytes, ts_stream_t stream) {
  return run_group_softmax(result, grad_out, index, grad_in, B, E, K, N, index_stride_b, index_stride_e, dtype,
                           log_space ? GS_LOG_SOFTMAX_BWD : GS_SOFTMAX_BWD, 0.0, workspace, workspace_bytes,
                           static_cast<hipStream_t>(stream));
}

int ts_group_logsumexp(const void *src, const int64_t *index, void *out, int64_t B, int64_t E, int64_t K, int64_t N,
                       int64_t index_stride_b, int64_t index_stride_e, int dtype, double eps, void *workspace,
                       size_t workspace_bytes, ts_stream_t stream) {
  if (!valid_dtype(dtype) || !sizes_ok(B, N, E, K)) return TS_ERR_BAD_ARG;
  if (!is_float_dtype(dtype)) return TS_ERR_UNSUPPORTED;
  if (B * N * K == 0) return TS_OK;
  if (!out || (B * E * K > 0 && (!src || !index))) return TS_ERR_BAD_ARG;
  if (B * N >= 0x7FFFFFFFll) return TS_ERR_UNSUPPORTED;
  const size_t need = group_workspace_bytes(B, N, K, kElemBytes[dtype]);
  if (!workspace || workspace_bytes < need || !aligned16(workspace)) return TS_ERR_WORKSPACE;
  GroupArgs g = {};
  g.src = src;
  g.index = index;
  g.out = out;
  if (B * E * K > 0) {
    // a workspace of ts_group_bins_workspace_bytes(): one gather of src through buckets of groups
    const GroupBinPlan plan = group_bins_plan(B, E, K, N, dtype, aligned16(src), workspace, workspace_bytes);
    if (plan.ok) {
      g.B = B;
      g.E = E;
      g.K = K;
      g.N = N;
      g.sb = index_stride_b;
      g.se = index_stride_e;
      g.eps = eps;
      g.bins = &plan.p;
      const FusedReducePlan tiles = group_tiles_plan(B, E, K, N, dtype, aligned16(src), workspace, workspace_bytes, plan.bytes);
      if (tiles.ok) {
        g.tiles = &tiles.f;
        g.tiles_force = env_int("TS_GROUP_FUSED", 1) == 2;
      }
      return dispatch_group_softmax(dtype, g, GS_LSE_BINS, group_bins_vec(K, dtype, aligned16(src)),
                                    static_cast<hipStream_t>(stream));
    }
  }
  g.gmax = workspace;
  g.gs = 2 * K;  // a group's keys and sums side by side
  g.gsum = static_cast<char *>(workspace) + (size_t)K * (kElemBytes[dtype] == 8 ? 8 : 4);
  g.B = B;
  g.E = E;
  g.K = K;
  g.N = N;
  g.sb = index_stride_b;
  g.se = index_stride_e;
  g.eps = eps;
  g.from_neg_inf = 1;
  const int full = kVecBytes / kElemBytes[dtype];
  const int vec = (full > 1 && K % full == 0 && aligned16(src)) ? full : 1;
  return dispatch_group_softmax(dtype, g, GS_LSE, vec, static_cast<hipStream_t>(stream));
}

size_t ts_group_workspace_bytes(int64_t B, int64_t E, int64_t K, int64_t N, int dtype) {
  if (!valid_dtype(dtype) || !is_float_dtype(dtype) || !sizes_ok(B, N, E, K)) return 0;
  const size_t front = group_workspace_bytes(B, N, K, kElemBytes[dtype]);
  const size_t bins = group_bins_plan(B, E, K, N, dtype, true, nullptr, 0).bytes;
  const size_t base = bins > 0 ? bins : front;
  size_t tail = bins > 0 ? group_tiles_plan(B, E, K, N, dtype, true, nullptr, 0, bins).bytes : 0;
  const size_t soft = env_int("TS_GROUP_FUSED", 1) != 0 ? group_fused_scratch_bytes(B, E, K, kElemBytes[dtype]) : 0;
  if (soft > tail) tail = soft;
  return base + tail;
}

size_t ts_group_bins_workspace_bytes(int64_t B, int64_t E, int64_t K, int64_t N, int dtype) {
  if (!valid_dtype(dtype) || !is_float_dtype(dtype) || !sizes_ok(B, N, E, K)) return 0;
  const size_t bins = group_bins_plan(B, E, K, N, dtype, true, nullptr, 0).bytes;
  return bins + group_tiles_plan(B, E, K, N, dtype, true, nullptr, 0, bins).bytes;
}

size_t ts_group_std_workspace_bytes(int64_t B, int64_t E, int64_t K, int64_t N, int dtype) {
  const size_t bins = ts_group_bins_workspace_bytes(B, E, K, N, dtype);
  if (bins > 0 || !valid_dtype(dtype) || !is_float_dtype(dtype) || !sizes_ok(B, N, E, K)) return bins;
  const RowsRoute rr = rows_route(B, E, K, N, dtype, TS_MEAN);
  return rr.ok ? rr.total() : 0;
}

int ts_group_std_forward(const void *src, const int64_t *index, void *total, int32_t *count, void *out, int64_t B,
                         int64_t E, int64_t K, int64_t N, int64_t index_stride_b, int64_t index_stride_e, int dtype,
                         int unbiased, void *workspace, size_t workspace_bytes, ts_stream_t stream) {
  if (!valid_dtype(dtype) || !sizes_ok(B, N, E, K)) return TS_ERR_BAD_ARG;
  if (!is_float_dtype(dtype)) return TS_ERR_UNSUPPORTED;
  if (B * N * K == 0) return TS_OK;
  if (!out || !total || !count || !src || !index) return TS_ERR_BAD_ARG;
  const bool al = aligned16(src);
  const GroupBinPlan plan = group_bins_plan(B, E, K, N, dtype, al, workspace, workspace_bytes);
  if (plan.bytes == 0) {
    // (an aligned src would have gone through the buckets, and the workspace is theirs: the three-call form has to serve it)
    if (!al && group_bins_plan(B, E, K, N, dtype, true, nullptr, 0).bytes != 0) return TS_ERR_UNSUPPORTED;
    // rows that the buckets do not hold: the entries sorted by group, then two segmented reductions (sums; squared
    // deviations from the means), the counts from the row pointers
    const RowsRoute rr = rows_route(B, E, K, N, dtype, TS_MEAN);
    if (!rr.ok) return TS_ERR_UNSUPPORTED;
    if (!workspace || workspace_bytes < rr.total() || !aligned16(workspace)) return TS_ERR_WORKSPACE;
    RowSortPlan sp = row_sort_plan(B, E, N, workspace, rr.sort_bytes);
    if (!sp.ok) return TS_ERR_WORKSPACE;
    hipStream_t s = static_cast<hipStream_t>(stream);
    void *const ws = static_cast<char *>(workspace) + rr.sort_bytes;
    int rc = launch_row_sort(sp.p, index, index_stride_b, index_stride_e, false, next_nonce(), s);
    if (rc != TS_OK) return rc;
    const uint64_t status_nonce = next_nonce();
    rc = run_rows_reduce(src, sp.p, total, nullptr, B, E, K, N, dtype, TS_SUM, 0, ws, rr.csr_bytes,
                         status_nonce, s);
    if (rc != TS_OK) return rc;
    hipLaunchKernelGGL(row_lengths_kernel, dim3(grid_for(B * N)), dim3(kBlock), 0, s, sp.p.ptr, count, B * N);
    const CsrPlan p = rows_csr_plan(B * N, B * E, K, dtype, al && aligned16(total) && aligned16(out), TS_SUM);
    CsrReduceArgs a;
    rc = rows_reduce_args(a, p, src, sp.p, out, nullptr, B, E, K, N, dtype, TS_SUM, 0, ws, rr.csr_bytes,
                          status_nonce, false);
    if (rc != TS_OK) return rc;
    a.row_total = total;
    a.unbiased = unbiased ? 1 : 0;
    GroupArgs g = {};
    g.rows = &a;
    g.rows_plan = &p;
    return dispatch_group_softmax(dtype, g, GS_STD_ROWS, p.vec, s);
  }
  if (!plan.ok) return TS_ERR_WORKSPACE;
  GroupArgs g = {};
  g.src = src;
  g.index = index;
  g.out = out;
  g.total_w = total;
  g.count_w = count;
  g.unbiased = unbiased ? 1 : 0;
  g.B = B;
  g.E = E;
  g.K = K;
  g.N = N;
  g.sb = index_stride_b;
  g.se = index_stride_e;
  g.bins = &plan.p;
  const FusedReducePlan tiles = group_tiles_plan(B, E, K, N, dtype, al, workspace, workspace_bytes, plan.bytes);
  if (tiles.ok) {
    g.tiles = &tiles.f;
    g.tiles_force = env_int("TS_GROUP_FUSED", 1) == 2;
  }
  return dispatch_group_softmax(dtype, g, GS_STD_BINS, group_bins_vec(K, dtype, al), static_cast<hipStream_t>(stream));
}

int ts_group_logsumexp_backward(const void *src, const int64_t *index, const void *out, const void *grad_out,
                                void *grad_in, int64_t B, int64_t E, int64_t K, int64_t N, int64_t index_stride_b,
                                int64_t index_stride_e, int dtype, ts_stream_t stream) {
  return ts_group_logsumexp_backward_with_workspace(src, index, out, grad_out, grad_in, B, E, K, N, index_stride_b,
                                                    index_stride_e, dtype, nullptr, 0, stream);
}

int ts_group_logsumexp_backward_with_workspace(const void *src, const int64_t *index, const void *out,
                                               const void *grad_out, void *grad_in, int64_t B, int64_t E, int64_t K,
                                               int64_t N, int64_t index_stride_b, int64_t index_stride_e, int dtype,
                                               void *workspace, size_t workspace_bytes, ts_stream_t stream) {
  if (!valid_dtype(dtype) || !sizes_ok(B, N, E, K)) return TS_ERR_BAD_ARG;
  if (!is_float_dtype(dtype)) return TS_ERR_UNSUPPORTED;
  if (B * E * K == 0) return TS_OK;
  if (!src || !index || !out || !grad_out || !grad_in) return TS_ERR_BAD_ARG;
  if (N == 0 || B * N >= 0x7FFFFFFFll) return TS_ERR_UNSUPPORTED;
  GroupArgs g = {};
  g.src = src;
  g.index = index;
  g.out = grad_in;
  g.node_out = out;
  g.node_grad = grad_out;
  g.B = B;
  g.E = E;
  g.K = K;
  g.N = N;
  g.sb = index_stride_b;
  g.se = index_stride_e;
  const int full = kVecBytes / kElemBytes[dtype];
  const bool al = aligned16(src) && aligned16(grad_in) && aligned16(out) && aligned16(grad_out);
  const int vec = (full > 1 && K % full == 0 && al) ? full : 1;
  if (group_coef_ok(B, E, N, K, dtype, workspace, workspace_bytes)) g.coef = workspace;
  return dispatch_group_softmax(dtype, g, GS_LSE_BWD, vec, static_cast<hipStream_t>(stream));
}

int ts_group_std(const void *src, const int64_t *index, const void *total, const int32_t *count, void *out, int64_t B,
                 int64_t E, int64_t K, int64_t N, int64_t index_stride_b, int64_t index_stride_e, int dtype,
                 int unbiased, void *workspace, size_t workspace_bytes, ts_stream_t stream) {
  if (!valid_dtype(dtype) || !sizes_ok(B, N, E, K)) return TS_ERR_BAD_ARG;
  if (!is_float_dtype(dtype)) return TS_ERR_UNSUPPORTED;
  if (B * N * K == 0) return TS_OK;
  if (!out || !total || !count || (B * E * K > 0 && (!src || !index))) return TS_ERR_BAD_ARG;
  if (B * N >= 0x7FFFFFFFll) return TS_ERR_UNSUPPORTED;
  const size_t need = group_workspace_bytes(B, N, K, kElemBytes[dtype]);
  if (!workspace || workspace_bytes < need || !aligned16(workspace)) return TS_ERR_WORKSPACE;
  GroupArgs g = {};
  g.src = src;
  g.index = index;
  g.out = out;
  g.gmax = workspace;
  g.gs = K;  // sums only
  g.gsum = workspace;
  g.total = total;
  g.count = count;
  g.unbiased = unbiased ? 1 : 0;
  g.B = B;
  g.E = E;
  g.K = K;
  g.N = N;
  g.sb = index_stride_b;
  g.se = index_stride_e;
  const int full = kVecBytes / kElemBytes[dtype];
  const int vec = (full > 1 && K % full == 0 && aligned16(src) && aligned16(total)) ? full : 1;
  return dispatch_group_softmax(dtype, g, GS_STD, vec, static_cast<hipStream_t>(stream));
}

int ts_group_std_backward(const void *src, const int64_t *index, const void *total, const int32_t *count,
                          const void *out, const void *grad_out, void *grad_in, int64_t B, int64_t E, int64_t K,
                          int64_t N, int64_t index_stride_b, int64_t index_stride_e, int dtype, int unbiased,
                          ts_stream_t stream) {
  return ts_group_std_backward_with_workspace(src, index, total, count, out, grad_out, grad_in, B, E, K, N, index_stride_b,
                                              index_stride_e, dtype, unbiased, nullptr, 0, stream);
}

int ts_group_std_backward_with_workspace(const void *src, const int64_t *index, const void *total, const int32_t *count,
                                         const void *out, const void *grad_out, void *grad_in, int64_t B, int64_t E,
                                         int64_t K, int64_t N, int64_t index_stride_b, int64_t index_stride_e, int dtype,
                                         int unbiased, void *workspace, size_t workspace_bytes, ts_stream_t stream) {
  if (!valid_dtype(dtype) || !sizes_ok(B, N, E, K)) return TS_ERR_BAD_ARG;
  if (!is_float_dtype(dtype)) return TS_ERR_UNSUPPORTED;
  if (B * E * K == 0) return TS_OK;
  if (!src || !index || !total || !count || !out || !grad_out || !grad_in) return TS_ERR_BAD_ARG;
  if (N == 0 || B * N >= 0x7FFFFFFFll) return TS_ERR_UNSUPPORTED;
  GroupArgs g = {};
  g.src = src;
  g.index = index;
  g.out = grad_in;
  g.node_out = out;
  g.node_grad = grad_out;
  g.total = total;
  g.count = count;
  g.unbiased = unbiased ? 1 : 0;
  g.B = B;
  g.E = E;
  g.K = K;
  g.N = N;
  g.sb = index_stride_b;
  g.se = index_stride_e;
  const int full = kVecBytes / kElemBytes[dtype];
  const bool al = aligned16(src) && aligned16(grad_in) && aligned16(out) && aligned16(grad_out) && aligned16(total);
  const int vec = (full > 1 && K % full == 0 && al) ? full : 1;
  if (group_coef_ok(B, E, N, K, dtype, workspace, workspace_bytes)) g.coef = workspace;
  return dispatch_group_softmax(dtype, g, GS_STD_BWD, vec, static_cast<hipStream_t>(stream));
}

// ---- index formats
int ts_index_to_indptr(const int64_t *index, int64_t *indptr, int64_t B, int64_t E, int64_t N,
                       int64_t index_batch_stride, ts_stream_t stream) {
  if (B < 0 || E < 0 || N < 0) return TS_ERR_BAD_ARG;
  if (B == 0) return TS_OK;
  if (!indptr || (E > 0 && !index)) return TS_ERR_BAD_ARG;
  return run_coo_to_indptr(index, indptr, B, E, N, index_batch_stride, static_cast<hipStream_t>(stream));
}

size_t ts_indptr_to_index_workspace_bytes(int64_t B, int64_t N) {
  return B < 0 || N < 0 ? 0 : ((size_t)B * N * 8 + 255) & ~(size_t)255;
}

int ts_indptr_to_index(const int64_t *indptr, int64_t *index, int64_t B, int64_t N, int64_t E,
                       int64_t indptr_batch_stride, void *workspace, size_t workspace_bytes, ts_stream_t stream) {
  if (!sizes_ok(B, N, E, 1)) return TS_ERR_BAD_ARG;
  if (B * E == 0 || N == 0) return TS_OK;
  if (!indptr || !index) return TS_ERR_BAD_ARG;
  if (!workspace || workspace_bytes < ts_indptr_to_index_workspace_bytes(B, N) || !aligned16(workspace))
    return TS_ERR_WORKSPACE;
  hipStream_t s = static_cast<hipStream_t>(stream);
  // the row numbers 0 .. N-1 of every batch, expanded along the row pointers like any other source
  int64_t *rows = static_cast<int64_t *>(workspace);
  hipLaunchKernelGGL(row_numbers_kernel, dim3(index_grid(B * N)), dim3(kBlock), 0, s, rows, B * N, N);
  if (hipGetLastError() != hipSuccess) return TS_ERR_LAUNCH;
  return ts_gather_csr(rows, indptr, index, B, N, E, 1, indptr_batch_stride, TS_I64, stream);
}

static int sort_key_bits(int64_t N) {  // keys are 0 .. N (N: an index outside [0, N))
  int bits = 1;
  while (bits < 32 && ((int64_t)1 << bits) <= N) ++bits;
  return bits;
}
static size_t sort_keys_bytes(int64_t E) { return ((size_t)E * 4 + 255) & ~(size_t)255; }

size_t ts_sort_index_workspace_bytes(int64_t E, int64_t N) {
  if (E < 0 || N < 0 || E >= 0x7FFFFFFFll || N >= 0x7FFFFFFFll) return 0;
  return 2 * sort_keys_bytes(E) + ((sort_keys_temp_bytes(E, sort_key_bits(N)) + 255) & ~(size_t)255);
}

int ts_sort_index(const int64_t *index, int32_t *perm, int64_t *indptr, int64_t E, int64_t N, void *workspace,
                  size_t workspace_bytes, ts_stream_t stream) {
  if (E < 0 || N < 0) return TS_ERR_BAD_ARG;
  if (E >= 0x7FFFFFFFll || N >= 0x7FFFFFFFll) return TS_ERR_UNSUPPORTED;
  if (!indptr || (E > 0 && (!index || !perm))) return TS_ERR_BAD_ARG;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const size_t kb = sort_keys_bytes(E);
  uint32_t *keys_in = static_cast<uint32_t *>(workspace);
  uint32_t *keys_out = reinterpret_cast<uint32_t *>(static_cast<char *>(workspace) + kb);
  if (E > 0) {
    const int bits = sort_key_bits(N);
    const size_t temp = sort_keys_temp_bytes(E, bits);
    if (!workspace || !aligned16(workspace) || workspace_bytes < 2 * kb + temp) return TS_ERR_WORKSPACE;
    hipLaunchKernelGGL(index_keys_kernel, dim3(index_grid(E)), dim3(kBlock), 0, s, index, keys_in, E, N);
    if (hipGetLastError() != hipSuccess) return TS_ERR_LAUNCH;
    const int rc = sort_keys_to_perm(static_cast<char *>(workspace) + 2 * kb, temp, keys_in, keys_out, perm, E, bits, s);
    if (rc != TS_OK) return rc;
  }
  hipLaunchKernelGGL(keys_to_indptr_kernel, dim3((unsigned)((E + 1 + kBlock - 1) / kBlock)), dim3(kBlock), 0, s,
                     keys_out, indptr, N, E);
  return hipGetLastError() == hipSuccess ? TS_OK : TS_ERR_LAUNCH;
}

}  // extern "C"
