// The passes of the value buckets (bin_plan_payload) for up to 8 M entries (included by scatter_binned.h): sums of one to four
// 4-byte values per entry under an index that is not in order. As in row_sort.h nothing is counted in front:
//   place : a workgroup per tile of up to 8192 entries: records (values, row in the bucket) sorted by bucket in LDS leave in one
//           piece, with the offset of every bucket among them
//   add   : a workgroup per bucket collects its runs from all tiles, adds in LDS and writes its rows, whole and once: no atomics
//           on out
//   rest  : a bucket of more than 16384 entries (a hub's) in pieces that meet in out through atomics. The same launch holds
//           the table of hot rows (scatter_add_lds_body), for the third answer of the sample: an idle launch is 3.5 to 4.6 us
// (Measured slower: the workgroups of add that are done take the pieces. 3 M values under a Zipf(1.2) index 270 to 340 against
// 73 us: most have left before a large bucket is known to be one.)
// What bounds it: place the loads and the stage, add the instructions (about 30 an entry and 4 a value). 3 M entries of three
// floats onto 150 k rows, us: place 20, add 23, the call 51; with the passes for larger inputs (count 18, scan 8, place 49, add
// 26) 110, through the table of hot rows 175. 3 M entries of one, two, four floats: 37, 45 to 49, 71 to 75 against 73 to 82, 91 to
// 107, 135 to 157 us before. In order, where these launches return at once: 58 against 66 us (two), 79 against 75 (three).
#pragma once

namespace ts {

constexpr int kVtBlock = 512;          // add
constexpr int kVtStage = 16384;        // words of a tile's records: 64 KB
constexpr int kVtAcc = 4096;           // rows of a bucket x values per entry
constexpr int kVtCap = kRsSortPer * kVtBlock;  // entries of a round
constexpr int kVtBig = kRsSortPer * kLdsAddBlock;  // entries of a piece, and from which a bucket is taken in pieces

struct ValueTiles {
  int ok = 0;
  RowSortArgs t;         // tiles, buckets and offsets
  uint32_t *records;     // [tiles << log][values + 1]
  int max_pieces;        // of buckets above kVtBig entries. t.state: [0] how many there are; t.chunk_big: [max_pieces][2] the
};                       // bucket and which of its pieces

// The table of hot rows behind them (scatter_add_lds_kernel's arguments), if the sample has three answers
struct TableCall {
  int tn_mask = 0;
  int64_t epb = 0;
  unsigned grid = 0;     // 0: none
};

// bytes: 0 if the passes do not apply
inline ValueTiles value_tiles_plan(int64_t B, int64_t E, int64_t K, int64_t N, void *ws, size_t ws_bytes, size_t *bytes) {
  ValueTiles v;
  *bytes = 0;
  RowSortArgs &p = v.t;
  p = RowSortArgs();
  const int64_t n = B * E, rows = B * N;
  if (K < 1 || K > 4 || n > (int64_t)1 << 23 || rows >= 0x7FFFF000ll) return v;
  p.B = B;
  p.E = E;
  p.N = N;
  p.n = n;
  p.rows = rows;
  // buckets of about 6000 entries, up to 1024 (a tile leaves runs of 4 to 8 records), more where one could not hold its rows
  int64_t want = n / 6144;
  want = want > 1024 ? 1024 : (want < 64 ? 64 : want);
  int rs = 0;
  while (((rows + ((int64_t)1 << rs) - 1) >> rs) > want) ++rs;
  while ((K << rs) > kVtAcc) --rs;
  p.rshift = rs;
  const int64_t nb = (rows + ((int64_t)1 << rs) - 1) >> rs;
  if (nb > 2048) return v;
  p.nb = (int)nb;
  const int64_t most = kVtStage / kRsBlock / (K + 1), per = (n + 512 * kRsBlock - 1) / (512 * kRsBlock);
  p.per = (int)(per > most ? most : per);
  p.log = 10;
  while (1 << (p.log - 10) < p.per) ++p.log;
  const int64_t tile = (int64_t)p.per * kRsBlock;
  p.tiles = (int)((n + tile - 1) / tile);
  p.pitch = (p.nb + 2) & ~1;
  v.max_pieces = (int)(2 * (n / kVtBig));  // (entries / kVtBig + 1 of a bucket with more than kVtBig)
  auto up = [](size_t x) { return (x + 255) & ~(size_t)255; };
  const size_t o_off = up((size_t)v.max_pieces * 8 + 16), o_rec = o_off + up((size_t)p.tiles * p.pitch * 2);
  *bytes = o_rec + ((size_t)p.tiles << p.log) * (K + 1) * 4;
  if (ws == nullptr || ws_bytes < *bytes) return v;
  p.state = static_cast<int32_t *>(ws);
  p.chunk_big = p.state + 4;
  p.off = reinterpret_cast<uint16_t *>(static_cast<char *>(ws) + o_off);
  v.records = reinterpret_cast<uint32_t *>(static_cast<char *>(ws) + o_rec);
  v.ok = 1;
  return v;
}

// one: bits of the value of an entry when there is no src (a count)
template <int K, int FLAT>
static __global__ __launch_bounds__(kRsBlock) __attribute__((amdgpu_waves_per_eu(8, 8)))
void vt_place_kernel(ScatterArgs a, ValueTiles vt, const int *flag, uint32_t one) {
  constexpr int PER = kVtStage / kRsBlock / (K + 1), R = K + 1;
  extern __shared__ uint32_t s_cnt[];  // [nb] counts, then the tile's exclusive prefix
  __shared__ uint32_t s_rec[kVtStage];
  __shared__ uint32_t s_wave[kRsBlock / kWave];
  if (*flag != 1) return;
  const RowSortArgs &p = vt.t;
  if (blockIdx.x == 0 && threadIdx.x == 0) p.state[0] = 0;
  const int tile = p.per * kRsBlock;
  const int64_t lo = (int64_t)blockIdx.x * tile;
  const uint32_t left = (uint32_t)(p.n - lo < tile ? p.n - lo : tile);
  int64_t idx[PER];
  uint32_t val[PER][K];
#pragma unroll
  for (int j = 0; j < PER; ++j) {  // (past the end: the last entry again)
    const uint32_t i = threadIdx.x + j * kRsBlock < left ? threadIdx.x + j * kRsBlock : left - 1;
    idx[j] = FLAT ? (p.index + lo)[i] : rs_load<FLAT>(p, lo + i);
  }
  const uint32_t *src = static_cast<const uint32_t *>(a.src);
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const uint32_t i = threadIdx.x + j * kRsBlock < left ? threadIdx.x + j * kRsBlock : left - 1;
#pragma unroll
    for (int k = 0; k < K; ++k) val[j][k] = src != nullptr ? (src + lo * K)[i * K + k] : one;
  }
  for (int i = threadIdx.x; i < p.nb; i += kRsBlock) s_cnt[i] = 0;
  __syncthreads();
  int32_t node[PER];
  uint32_t rank[PER];
  int32_t hot = -1;
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const uint32_t i = threadIdx.x + j * kRsBlock;
    node[j] = i < left ? rs_row<FLAT>(p, lo + i, idx[j]) : -1;
    rank[j] = 0;
    if (j * kRsBlock < (int)left) rank[j] = rs_take(s_cnt, node[j] >> p.rshift, hot);  // (-1 stays -1)
  }
  __syncthreads();
  const int total = (int)rs_scan_lds<kRsBlock>(s_cnt, p.nb, s_wave);
  uint16_t *off = p.off + (size_t)blockIdx.x * p.pitch;
  for (int i = threadIdx.x; i <= p.nb; i += kRsBlock) off[i] = (uint16_t)(i < p.nb ? s_cnt[i] : (uint32_t)total);
  const uint32_t mask = (1u << p.rshift) - 1;
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    if (node[j] < 0) continue;
    uint32_t *rec = s_rec + (s_cnt[(uint32_t)node[j] >> p.rshift] + rank[j]) * R;
#pragma unroll
    for (int k = 0; k < K; ++k) rec[k] = val[j][k];
    rec[K] = (uint32_t)node[j] & mask;
  }
  __syncthreads();
  uint32_t *out = vt.records + ((size_t)blockIdx.x << p.log) * R;
#pragma unroll
  for (int j = 0; j < kVtStage / kRsBlock; ++j) {
    const int i = (int)threadIdx.x + j * kRsBlock;
    if (i < total * R) out[i] = s_rec[i];
  }
}

// the records at places [skip, skip + cnt) of a bucket into the tables in LDS (a0, c0: rs_run_of of tile threadIdx.x)
template <typename T, int K, bool COUNT, int BLOCK>
__device__ __forceinline__ void vt_add_places(const ValueTiles &vt, int bucket, uint32_t skip, int cnt, uint32_t a0, uint32_t c0,
                                              RsRuns<BLOCK> &s_runs, typename BinSlot<T>::type *s_acc, int32_t *s_num) {
  typedef typename BinSlot<T>::type A;
  constexpr int R = K + 1, U = 4;
  uint32_t at[kRsSortPer];
  rs_places<BLOCK>(vt.t, bucket, skip, cnt, a0, c0, s_runs, at);
#pragma unroll
  for (int j0 = 0; j0 < kRsSortPer; j0 += U) {
    if (j0 * BLOCK >= cnt) break;  // (the same for the workgroup)
    uint32_t w[U][R];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint32_t *rec = vt.records + (size_t)at[j0 + u] * R;
#pragma unroll
      for (int k = 0; k < R; ++k) w[u][k] = rec[k];
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if ((j0 + u) * BLOCK + (int)threadIdx.x >= cnt) continue;
#pragma unroll
      for (int k = 0; k < K; ++k) {
        T x;
        __builtin_memcpy(&x, &w[u][k], 4);
        __hip_atomic_fetch_add(&s_acc[w[u][K] * K + k], (A)x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      }
      if (COUNT) __hip_atomic_fetch_add(&s_num[w[u][K]], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
  }
}

template <typename T, int K, bool COUNT>
static __global__ __launch_bounds__(kVtBlock) void vt_add_kernel(ScatterArgs a, ValueTiles vt, const int *flag, int32_t *count) {
  typedef typename BinSlot<T>::type A;
  __shared__ A s_acc[kVtAcc];
  __shared__ int32_t s_num[COUNT ? kVtAcc / K : 1];
  __shared__ RsRuns<kVtBlock> s_runs;
  __shared__ int s_first;
  if (*flag != 1) return;
  const RowSortArgs &p = vt.t;
  // neighbouring buckets, whose runs share lines, on one of the eight dies (workgroups go to them in turn)
  const int per_die = (p.nb + 7) / 8, bucket = (int)(blockIdx.x & 7) * per_die + (int)(blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per_die || bucket >= p.nb) return;
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave, rows = 1 << p.rshift;
  for (int i = tid; i < rows * K; i += kVtBlock) s_acc[i] = (A)0;
  if (COUNT)
    for (int i = tid; i < rows; i += kVtBlock) s_num[i] = 0;
  uint32_t a0, c0, entries;
  rs_run_of(p, bucket, tid, a0, c0);
  {
    uint32_t c = c0;
    for (int t = tid + kVtBlock; t < p.tiles; t += kVtBlock) {
      uint32_t at, ct;
      rs_run_of(p, bucket, t, at, ct);
      c += ct;
    }
    const int32_t ic = wave_inclusive_sum((int32_t)c);
    if (lane == kWave - 1) s_runs.wave[2][wave] = (uint32_t)ic;
    __syncthreads();
    rs_waves_before<kVtBlock>(s_runs.wave[2], entries);
    __syncthreads();
  }
  if (entries > (uint32_t)kVtBig) {  // the rows without their entries here, and a note for the launch behind
    const int m = (int)((entries + kVtBig - 1) / kVtBig);
    if (tid == 0) s_first = atomicAdd(&p.state[0], m);
    __syncthreads();
    for (int c = tid; c < m; c += kVtBlock) {
      p.chunk_big[2 * (s_first + c)] = bucket;
      p.chunk_big[2 * (s_first + c) + 1] = c;
    }
  } else {
    for (uint32_t skip = 0; skip < entries; skip += kVtCap)
      vt_add_places<T, K, COUNT>(vt, bucket, skip, entries - skip < (uint32_t)kVtCap ? (int)(entries - skip) : kVtCap, a0, c0,
                                 s_runs, s_acc, s_num);
    __syncthreads();
  }
  const int64_t row0 = (int64_t)bucket << p.rshift;
  const int n_rows = p.rows - row0 < rows ? (int)(p.rows - row0) : rows;
  T *out = static_cast<T *>(a.out) + row0 * K;
  for (int i = tid; i < n_rows * K; i += kVtBlock) {
    A v = s_acc[i];
    if (a.out_given) v = (A)out[i] + v;
    out[i] = (T)v;
  }
  if (COUNT)
    for (int i = tid; i < n_rows; i += kVtBlock) count[row0 + i] = s_num[i];
}

template <typename T, int K, bool COUNT>
__device__ __forceinline__ void vt_add_piece(const ScatterArgs &a, const ValueTiles &vt, int bucket, uint32_t skip, int32_t *count) {
  typedef typename BinSlot<T>::type A;
  constexpr int BLOCK = kLdsAddBlock;
  __shared__ A s_acc[kVtAcc];
  __shared__ int32_t s_num[COUNT ? kVtAcc / K : 1];
  __shared__ RsRuns<BLOCK> s_runs;
  const RowSortArgs &p = vt.t;
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave, rows = 1 << p.rshift;
  for (int i = tid; i < rows * K; i += BLOCK) s_acc[i] = (A)0;
  if (COUNT)
    for (int i = tid; i < rows; i += BLOCK) s_num[i] = 0;
  uint32_t a0, c0, entries;
  rs_run_of(p, bucket, tid, a0, c0);
  uint32_t c = c0;
  for (int t = tid + BLOCK; t < p.tiles; t += BLOCK) {
    uint32_t at, ct;
    rs_run_of(p, bucket, t, at, ct);
    c += ct;
  }
  const int32_t ic = wave_inclusive_sum((int32_t)c);
  if (lane == kWave - 1) s_runs.wave[2][wave] = (uint32_t)ic;
  __syncthreads();
  rs_waves_before<BLOCK>(s_runs.wave[2], entries);
  __syncthreads();
  vt_add_places<T, K, COUNT>(vt, bucket, skip, entries - skip < (uint32_t)kVtBig ? (int)(entries - skip) : kVtBig, a0, c0, s_runs,
                             s_acc, s_num);
  __syncthreads();
  const int64_t row0 = (int64_t)bucket << p.rshift;
  T *out = static_cast<T *>(a.out) + row0 * K;
  for (int i = tid; i < rows * K; i += BLOCK) {  // (a row that no entry named adds nothing)
    const A v = s_acc[i];
    if (v != (A)0) atomic_add_elem<T>(out + i, (T)v);
  }
  if (COUNT)
    for (int i = tid; i < rows; i += BLOCK)
      if (s_num[i] != 0) atomicAdd(count + row0 + i, s_num[i]);
  __syncthreads();
}

template <typename T, int K, bool COUNT>
static __global__ __launch_bounds__(kLdsAddBlock) void vt_rest_kernel(ScatterArgs a, ValueTiles vt, const int *flag, int32_t *count,
                                                                      TableCall table) {
  const int verdict = *flag;
  if (verdict == 2) {
    if (blockIdx.x < table.grid) scatter_add_lds_body<T, false, COUNT>(a, table.tn_mask, table.epb);
  } else if (verdict == 1) {
    for (int c = blockIdx.x; c < vt.t.state[0]; c += gridDim.x)
      vt_add_piece<T, K, COUNT>(a, vt, vt.t.chunk_big[2 * c], (uint32_t)vt.t.chunk_big[2 * c + 1] * kVtBig, count);
  }
}

template <typename T, int K>
inline void launch_value_tiles_k(const ScatterArgs &a, const ValueTiles &vt, const int *flag, int32_t *count, const TableCall &table,
                               hipStream_t stream) {
  const T unit = (T)1;
  uint32_t one;
  __builtin_memcpy(&one, &unit, 4);
  const RowSortArgs &p = vt.t;
  if (p.flat)
    hipLaunchKernelGGL((vt_place_kernel<K, 1>), dim3((unsigned)p.tiles), dim3(kRsBlock), (size_t)p.nb * 4, stream, a, vt, flag, one);
  else
    hipLaunchKernelGGL((vt_place_kernel<K, 0>), dim3((unsigned)p.tiles), dim3(kRsBlock), (size_t)p.nb * 4, stream, a, vt, flag, one);
  const dim3 g((unsigned)((p.nb + 7) / 8 * 8));
  const unsigned pieces = (unsigned)(vt.max_pieces < 256 ? vt.max_pieces : 256);
  const dim3 rest(table.grid > pieces ? table.grid : pieces);
  if (count != nullptr)
    hipLaunchKernelGGL((vt_add_kernel<T, K, true>), g, dim3(kVtBlock), 0, stream, a, vt, flag, count);
  else
    hipLaunchKernelGGL((vt_add_kernel<T, K, false>), g, dim3(kVtBlock), 0, stream, a, vt, flag, count);
  if (rest.x == 0) return;
  if (count != nullptr)
    hipLaunchKernelGGL((vt_rest_kernel<T, K, true>), rest, dim3(kLdsAddBlock), 0, stream, a, vt, flag, count, table);
  else
    hipLaunchKernelGGL((vt_rest_kernel<T, K, false>), rest, dim3(kLdsAddBlock), 0, stream, a, vt, flag, count, table);
}
// flag: reads 1 if these passes take the call
template <typename T>
inline void launch_value_tiles(const ScatterArgs &a, const ValueTiles &tiles, const int *flag, int32_t *count, const TableCall &table,
                               hipStream_t stream) {
  ValueTiles vt = tiles;
  vt.t.index = a.index;
  vt.t.sb = a.sb;
  vt.t.se = a.se;
  vt.t.flat = a.B == 1 && a.se == 1;
  switch (a.K) {
  case 1: return launch_value_tiles_k<T, 1>(a, vt, flag, count, table, stream);
  case 2: return launch_value_tiles_k<T, 2>(a, vt, flag, count, table, stream);
  case 3: return launch_value_tiles_k<T, 3>(a, vt, flag, count, table, stream);
  default: return launch_value_tiles_k<T, 4>(a, vt, flag, count, table, stream);
  }
}

}  // namespace ts
