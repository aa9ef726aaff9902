// Scatter sum / mean / min / max of a small input (up to 8192 entries and 262144 values) in one launch, e.g. the readout of a
// mini-batch of small graphs. The other kernels clear out, meet there through atomics, and for a mean count the entries and
// divide, for min / max unpack keys: two to five launches of a few microseconds, each of which costs the host more than the
// device. Here a workgroup owns R rows of out: it reads the whole index of its batch, sorts the entries of its rows in LDS,
// reduces their values there (every group of lanes takes an equal share of the entries, whatever their rows; sums in double,
// min / max as keys of value and position, scatter.h), and writes its rows once, empty ones included.
// What bounds it: the chain of one workgroup (index, rank, values, result), about 7 us. 3010 entries x 64 floats onto 128
// rows, mean with its count: 6.8 us and one launch, before 15 us in five and two more for the count in the element type; the
// training step around it 75 -> 45-53 us, most of it the host's. 1188 calls of 200 to 8000 entries: 0.65 of the time in the
// geometric mean (sums 0.76, means 0.53, maxima 0.68).
#pragma once

#include "csr_reduce.h"
#include "row_sort.h"
#include "scatter.h"

namespace ts {

constexpr int kSmallBlock = 512;
constexpr int kSmallPer = 16;          // entries per lane: a batch of up to 8192
constexpr int kSmallRows = 512;        // rows per workgroup at most
constexpr int kSmallAcc = 4096;        // accumulators per workgroup: 32 KB of doubles

struct SmallArgs {
  const void *src;       // [B, E, K]
  const int64_t *index;  // index[b * sb + e * se]
  void *out;             // [B, N, K]
  void *count;           // sum, mean: [B, N] in the element type, at least 1; may be null
  int64_t *arg_out;      // min, max: [B, N, K]
  int64_t sb, se, B, E, K, N;
  int R, C, G;           // rows and columns of a workgroup, lanes of a row
  int mean, out_given;
};

struct SmallPlan {
  bool ok;
  int R, C, G, xchunks, ychunks;
};
inline SmallPlan small_plan(int64_t B, int64_t E, int64_t K, int64_t N, int elem_bytes, int vec, int reduce, bool any_size) {
  SmallPlan p = {false, 0, 0, 0, 0, 0};
  if (B < 1 || E < 1 || K < 1 || N < 1 || E > kSmallPer * kSmallBlock || B > 65535) return p;
  if (elem_bytes > 4 && (reduce == TS_MIN || reduce == TS_MAX)) return p;  // keys of 32 bits
  // Half a megabyte of 16-bit elements, a megabyte of others (all of it may lie in one row, i.e. in one workgroup; us without
  // this kernel / with it, 3000 entries a row, hub: mean of 8000 x 64 bf16 17.0 / 19.5, max 31.6 / 36.7, of 1000 x 512 bf16 onto
  // two rows 20.8 / 55). Sums, which are two launches elsewhere, half of that and up to 4096 entries: 8000 x 4 floats onto 400
  // rows 10.5 / 12.8, 8000 x 64 bf16 10.4 / 14.0.
  const int64_t most = reduce == TS_SUM ? (int64_t)1 << 17 : (int64_t)1 << 18;
  if (!any_size && (B * E * K > most || (reduce == TS_SUM && E > 4096))) return p;
  const int64_t lanes = (K + vec - 1) / vec;
  p.G = 1;
  while (p.G < lanes && p.G < kWave) p.G *= 2;
  p.C = (int)(lanes < p.G ? K : (int64_t)p.G * vec);
  if (p.C > K) p.C = (int)K;
  const int64_t y = (K + p.C - 1) / p.C;
  int64_t R = (B * N * y + 511) / 512;  // about 512 workgroups
  if (R > N) R = N;
  if (R > kSmallRows) R = kSmallRows;
  if (R > kSmallAcc / p.C) R = kSmallAcc / p.C;
  const int64_t x = (N + R - 1) / R;
  // every workgroup reads its batch's index: 32 MB from the L2 caches at most
  if (B * x * y * E > ((int64_t)4 << 20) || B * x > 0x7FFFFFFFll || y > 65535) return p;
  p.R = (int)R;
  p.xchunks = (int)x;
  p.ychunks = (int)y;
  p.ok = true;
  return p;
}

// REDUCE: TS_SUM (and mean, by a.mean), TS_MIN, TS_MAX
template <typename T, int VEC, int REDUCE>
static __global__ __launch_bounds__(kSmallBlock) void scatter_small_kernel(SmallArgs a, int xchunks) {
  constexpr bool kKeys = REDUCE != TS_SUM, kMax = REDUCE == TS_MAX;
  typedef typename std::conditional<kKeys, uint64_t, double>::type A;
  __shared__ A s_acc[kSmallAcc];
  __shared__ uint32_t s_list[kSmallPer * kSmallBlock];  // row << 16 | entry, by row
  __shared__ uint32_t s_start[kSmallRows + 1];
  __shared__ uint32_t s_wave[kSmallBlock / kWave];
  const int tid = threadIdx.x, E = (int)a.E;
  const int64_t b = blockIdx.x / (unsigned)xchunks, r0 = (int64_t)(blockIdx.x - b * xchunks) * a.R;
  const int R = a.N - r0 < a.R ? (int)(a.N - r0) : a.R;
  const int64_t k0 = (int64_t)blockIdx.y * a.C;
  const int C = a.K - k0 < a.C ? (int)(a.K - k0) : a.C;
  const int64_t *idx = a.index + b * a.sb;
  int32_t row[kSmallPer];
  uint32_t rank[kSmallPer];
#pragma unroll
  for (int j = 0; j < kSmallPer; ++j) {
    if (j * kSmallBlock >= E) break;  // (the same for the workgroup)
    const int e = j * kSmallBlock + tid;
    const int64_t at = idx[(int64_t)(e < E ? e : E - 1) * a.se] - r0;
    row[j] = e < E && at >= 0 && at < R ? (int32_t)at : -1;
  }
  T *out = static_cast<T *>(a.out) + (b * a.N + r0) * a.K + k0;
  for (int i = tid; i < R * C; i += kSmallBlock) {
    if constexpr (kKeys) {  // (as scatter_key_init_kernel)
      if (a.out_given) {
        const T prev = out[(int64_t)(i / C) * a.K + i % C];
        s_acc[i] = Key<T>::is_nan(prev) ? ~(uint64_t)0 : pack_key<T, kMax>(prev, kKeepLow);
      } else {
        s_acc[i] = pack_key<T, kMax>(kMax ? ElemLim<T>::lowest() : ElemLim<T>::max(), kKeepLow);
      }
    } else {
      s_acc[i] = 0.0;
    }
  }
  for (int i = tid; i < R; i += kSmallBlock) s_start[i] = 0;
  __syncthreads();
  int32_t hot = -1;
#pragma unroll
  for (int j = 0; j < kSmallPer; ++j) {
    if (j * kSmallBlock >= E) break;
    rank[j] = rs_take(s_start, row[j], hot);
  }
  __syncthreads();
  const int M = (int)rs_scan_lds<kSmallBlock>(s_start, R, s_wave);
  if (tid == 0) s_start[R] = (uint32_t)M;
#pragma unroll
  for (int j = 0; j < kSmallPer; ++j) {
    if (j * kSmallBlock >= E) break;
    if (row[j] >= 0) s_list[s_start[row[j]] + rank[j]] = (uint32_t)row[j] << 16 | (uint32_t)(j * kSmallBlock + tid);
  }
  __syncthreads();
  const int G = a.G, W = kSmallBlock / G, w = tid / G, c0 = (tid - w * G) * VEC;
  const int per = (M + W - 1) / W, m0 = w * per, m1 = m0 + per < M ? m0 + per : M;
  if (c0 < C && m0 < m1) {
    const T *src = static_cast<const T *>(a.src) + b * a.E * a.K + k0 + c0;
    A acc[VEC];
    int32_t cur = (int32_t)(s_list[m0] >> 16);
#pragma unroll
    for (int v = 0; v < VEC; ++v) acc[v] = (A)0;
    auto flush = [&]() {
#pragma unroll
      for (int v = 0; v < VEC; ++v) {
        if constexpr (kKeys)
          __hip_atomic_fetch_max(&s_acc[cur * C + c0 + v], acc[v], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        else
          __hip_atomic_fetch_add(&s_acc[cur * C + c0 + v], acc[v], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        acc[v] = (A)0;
      }
    };
    constexpr int U = 8;  // rows on the way together
    for (int m = m0; m < m1; m += U) {
      uint32_t word[U];
      Vec<T, VEC> x[U];
#pragma unroll
      for (int u = 0; u < U; ++u) word[u] = s_list[m + u < m1 ? m + u : m1 - 1];  // (past the end: the last one again)
#pragma unroll
      for (int u = 0; u < U; ++u) x[u] = load_vec<T, VEC>(src + (int64_t)(word[u] & 0xFFFFu) * a.K);
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (m + u >= m1) break;
        if ((int32_t)(word[u] >> 16) != cur) {
          flush();
          cur = (int32_t)(word[u] >> 16);
        }
        if constexpr (kKeys) {
          uint64_t key[VEC];
          make_keys<T, VEC, kMax>(x[u], (int64_t)(word[u] & 0xFFFFu), key);
#pragma unroll
          for (int v = 0; v < VEC; ++v) acc[v] = key[v] > acc[v] ? key[v] : acc[v];
        } else {
#pragma unroll
          for (int v = 0; v < VEC; ++v) acc[v] += (double)to_acc<T>(x[u].v[v]);
        }
      }
    }
    flush();
  }
  __syncthreads();
  typedef typename Acc<T>::type F;
  for (int i = tid; i < R * C; i += kSmallBlock) {
    const int r = i / C, c = i - r * C;
    T *p = out + (int64_t)r * a.K + c;
    if constexpr (kKeys) {  // (as scatter_key_final_kernel)
      const uint64_t key = s_acc[i];
      const uint32_t low = (uint32_t)key;
      int64_t *arg = a.arg_out + (p - static_cast<T *>(a.out));
      if (low == kKeepLow) {  // nothing beat the initial / previous content
        if (!a.out_given) *p = zero_elem<T>();
        *arg = a.E;
      } else {
        const int64_t e = (int64_t)(0xFFFFFFFEu - low);
        uint32_t k = (uint32_t)(key >> 32);
        if (!kMax) k = ~k;
        // (a zero: from src, to keep the sign of the winning entry)
        *p = k == 0x80000000u ? static_cast<const T *>(a.src)[(b * a.E + e) * a.K + k0 + c] : Key<T>::dec(k);
        *arg = e;
      }
      continue;
    }
    double sum = (double)s_acc[i];
    if (a.out_given) sum += (double)to_acc<T>(*p);
    T t = from_acc<T>((F)sum);
    const int32_t n = (int32_t)(s_start[r + 1] - s_start[r]);
    if (a.mean && n > 1) t = div_elem<T>(t, count_as<T>(n));
    *p = t;
  }
  if (!kKeys && a.count != nullptr && blockIdx.y == 0) {
    for (int r = tid; r < R; r += kSmallBlock) {
      const int64_t n = (int64_t)(s_start[r + 1] - s_start[r]);
      static_cast<T *>(a.count)[b * a.N + r0 + r] = count_as<T>(n > 1 ? n : 1);
    }
  }
}

template <typename T, int VEC>
inline int launch_scatter_small(const SmallArgs &args, const SmallPlan &p, int reduce, hipStream_t stream) {
  SmallArgs a = args;
  a.R = p.R;
  a.C = p.C;
  a.G = p.G;
  const dim3 grid((unsigned)(a.B * p.xchunks), (unsigned)p.ychunks);
  if constexpr (sizeof(T) <= 4) {
    if (reduce == TS_MIN) hipLaunchKernelGGL((scatter_small_kernel<T, VEC, TS_MIN>), grid, dim3(kSmallBlock), 0, stream, a, p.xchunks);
    if (reduce == TS_MAX) hipLaunchKernelGGL((scatter_small_kernel<T, VEC, TS_MAX>), grid, dim3(kSmallBlock), 0, stream, a, p.xchunks);
  }
  if (reduce == TS_SUM) hipLaunchKernelGGL((scatter_small_kernel<T, VEC, TS_SUM>), grid, dim3(kSmallBlock), 0, stream, a, p.xchunks);
  return hipGetLastError() == hipSuccess ? TS_OK : TS_ERR_LAUNCH;
}

}  // namespace ts
