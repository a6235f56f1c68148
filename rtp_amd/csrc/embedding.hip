// Sharded embedding: coalesced row gather and a deterministic (sorted, segmented) scatter-add.
#include <cstring>

#include "common.h"

#include <rocprim/rocprim.hpp>

namespace rtp {

// One wavefront per token, over the columns of all shards of the run: a token's output row is contiguous across the shards
// (V elements per lane, kGatherDepth vectors requested before the first is stored), only the table they come from
// differs.  Bound by memory: at 16368 tokens of 8 shards x 256 bf16 columns a workgroup per (token, shard) moved 512 bytes
// with half of its lanes idle and took 55 us (2.4 TB/s); this form takes 21 us (6.4 TB/s; part of the reads hit the caches).
// With `pos` the row is scaled and a positional row added on the way: out = T(T(table * scale) + pos[t / batch]),
// each step rounded to T as the two separate element-wise operations would round it.
constexpr int kGatherDepth = 4;
template <typename T, int V, bool POS>
__global__ __launch_bounds__(256) void gather_kernel(const T* table, long ld_table, long row_begin, long row_count,
                                                     int per_row, FastDiv d_row, int total, const int64_t* ids, long n, T* out,
                                                     long ld_out, long table_sg, long out_sg, float scale, const T* pos,
                                                     long ld_pos, long pos_sg, FastDiv d_batch) {
  const long t = (long)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (t >= n) return;
  const long row = ids[t] - row_begin;
  if (row < 0 || row >= row_count) return;
  const T* src = table + row * ld_table;
  T* dst = out + t * ld_out;
  const T* prow = POS ? pos + (long)fast_div((unsigned)t, d_batch) * ld_pos : nullptr;
  union Pack {
    uint4 q;
    T e[V == 1 ? 1 : 16 / (int)sizeof(T)];
  };
  auto load = [](const T* p) {
    Pack u;
    if constexpr (V == 1)
      u.e[0] = p[0];
    else
      u.q = *reinterpret_cast<const uint4*>(p);
    return u;
  };
  for (int e0 = threadIdx.x & 63; e0 < total; e0 += kGatherDepth * 64) {
    Pack a[kGatherDepth], b[kGatherDepth];
    long at[kGatherDepth];
#pragma unroll
    for (int d = 0; d < kGatherDepth; ++d) {
      const int e = e0 + d * 64 < total ? e0 + d * 64 : e0;  // past the row: the first vector again, not stored
      const unsigned g = fast_div((unsigned)e, d_row);
      const int c = (e - (int)g * per_row) * V;
      at[d] = g * out_sg + c;
      a[d] = load(src + g * table_sg + c);
      if constexpr (POS) b[d] = load(prow + g * pos_sg + c);
    }
#pragma unroll
    for (int d = 0; d < kGatherDepth; ++d) {
      if (e0 + d * 64 >= total) break;
      if constexpr (POS) {
#pragma clang fp contract(off)
#pragma unroll
        for (int v = 0; v < V; ++v) a[d].e[v] = from_f32<T>(to_f32(from_f32<T>(to_f32(a[d].e[v]) * scale)) + to_f32(b[d].e[v]));
      }
      if constexpr (V == 1)
        dst[at[d]] = a[d].e[0];
      else
        *reinterpret_cast<uint4*>(dst + at[d]) = a[d].q;
    }
  }
}

__global__ __launch_bounds__(256) void sort_prep_kernel(const int64_t* ids, long n, int* keys, int* vals) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i < n) {
    keys[i] = (int)ids[i];
    vals[i] = (int)i;
  }
}

// (id, position) pairs of up to kSortLdsMax token ids sorted by one workgroup in LDS: a bitonic network over the
// 64-bit words id << 32 | position (all different, so the order is total and the result is the stable sort by id).
// A step's 1024 ids take 55 compare-exchange rounds of a few hundred nanoseconds each; a device-wide radix sort
// spends several launches on them.  Slots beyond n hold the largest word and stay at the end.
constexpr int kSortLdsMax = 8192;  // 64 KiB of LDS
constexpr int kSortThreads = 1024;
__global__ __launch_bounds__(kSortThreads) void sort_ids_lds_kernel(const int64_t* ids, int n, int npow2, int* keys,
                                                                    int* vals) {
  extern __shared__ unsigned long long sort_words[];
  for (int i = threadIdx.x; i < npow2; i += kSortThreads)
    sort_words[i] = i < n ? ((unsigned long long)(unsigned)(int)ids[i] << 32) | (unsigned)i : ~0ull;
  __syncthreads();
  for (int k = 2; k <= npow2; k <<= 1) {
    for (int j = k >> 1; j > 0; j >>= 1) {
      for (int t = threadIdx.x; t < (npow2 >> 1); t += kSortThreads) {
        const int lo = ((t & ~(j - 1)) << 1) | (t & (j - 1)), hi = lo | j;
        const unsigned long long a = sort_words[lo], b = sort_words[hi];
        const bool ascending = (lo & k) == 0;
        if ((a > b) == ascending) {
          sort_words[lo] = b;
          sort_words[hi] = a;
        }
      }
      __syncthreads();
    }
  }
  for (int i = threadIdx.x; i < n; i += kSortThreads) {
    const unsigned long long w = sort_words[i];
    keys[i] = (int)(unsigned)(w >> 32);
    vals[i] = (int)(unsigned)(w & 0xffffffffull);
  }
}

__global__ __launch_bounds__(256) void zero_rows_kernel(char* base, long ld_bytes, long row_bytes, long rows,
                                                        long group_bytes) {
  const long r = blockIdx.x;
  if (r >= rows) return;
  char* p = base + blockIdx.z * group_bytes + r * ld_bytes;
  if ((((uintptr_t)p | (uintptr_t)row_bytes) & 15) == 0) {
    uint4* d = reinterpret_cast<uint4*>(p);
    const uint4 z = make_uint4(0, 0, 0, 0);
    for (long i = (long)blockIdx.y * 256 + threadIdx.x; i < (row_bytes >> 4); i += (long)gridDim.y * 256) d[i] = z;
  } else {
    for (long i = (long)blockIdx.y * 256 + threadIdx.x; i < row_bytes; i += (long)gridDim.y * 256) p[i] = 0;
  }
}

// keys: token ids sorted ascending (stable), vals: their positions.  The workgroup at sorted index i
// owns the segment that starts there (if one does) and sums it front to back, i.e. in ascending
// position order, starting from +0.0f exactly like a sequential index_add_ into a zeroed table.
template <typename T, typename G>
__global__ __launch_bounds__(256) void scatter_kernel(const T* grad_out, long ld_go, long n, const int* keys,
                                                      const int* vals, G* grad_table, long ld_gt, long row_begin,
                                                      long row_count, long cols, long padding_idx, int scale_by_freq,
                                                      int overwrite, long go_sg, long gt_sg, float grad_scale,
                                                      float* master, T* weights, float lr, float clip, int store_grad) {
  grad_out += blockIdx.z * go_sg;  // group = shard: its column block of the upstream gradient, its own table
  grad_table += blockIdx.z * gt_sg;
  if (master != nullptr) master += blockIdx.z * gt_sg;
  if (weights != nullptr) weights += blockIdx.z * gt_sg;
  const long i = blockIdx.x;
  const int id = keys[i];
  if (i > 0 && keys[i - 1] == id) return;
  if (id == padding_idx) return;
  const long row = (long)id - row_begin;
  if (row < 0 || row >= row_count) return;
  long end = i + 1;
  while (end < n && keys[end] == id) ++end;
  const float inv = scale_by_freq ? 1.0f / (float)(end - i) : 1.0f;
  for (long c = (long)blockIdx.y * 256 + threadIdx.x; c < cols; c += (long)gridDim.y * 256) {
    float acc = 0.0f;
    if (grad_scale == 1.0f) {
      for (long j = i; j < end; ++j) acc += to_f32(grad_out[(long)vals[j] * ld_go + c]);
    } else {
#pragma clang fp contract(off)
      // the upstream gradient of a scaled embedding: T(grad * scale), rounded as the separate multiplication would
      // (no fused multiply-add: the product is rounded before it joins the sum)
      for (long j = i; j < end; ++j)
        acc += to_f32(from_f32<T>(to_f32(grad_out[(long)vals[j] * ld_go + c]) * grad_scale));
    }
    if (scale_by_freq) acc *= inv;
    G* dst = grad_table + row * ld_gt + c;
    if (master != nullptr) {
      // clip + SGD applied where the row's gradient is produced (the caller guarantees that this is the row's whole
      // gradient of the step): the arithmetic of the separate update on the gradient as its table would hold it.
      // Rows no token names keep a zero gradient, which the update leaves alone, so they are not touched at all.
      const float w = sgd_update<G>(master[row * ld_gt + c], acc, lr, clip);
      master[row * ld_gt + c] = w;
      if (weights != nullptr) weights[row * ld_gt + c] = from_f32<T>(w);
      if (store_grad) *dst = from_f32<G>(acc);
      continue;
    }
    if (!overwrite) acc = to_f32(*dst) + acc;
    *dst = from_f32<G>(acc);
  }
}

// V consecutive elements of type X as floats and back; V > 1 means whole 16-byte vectors (the caller checked alignment).
template <typename X, int V>
__device__ __forceinline__ void vec_load(const X* p, float (&f)[V]) {
  if constexpr (V == 1) {
    f[0] = to_f32(p[0]);
  } else {
    constexpr int NQ = V * (int)sizeof(X) / 16;
    union {
      uint4 q[NQ];
      X e[V];
    } u;
#pragma unroll
    for (int q = 0; q < NQ; ++q) u.q[q] = reinterpret_cast<const uint4*>(p)[q];
#pragma unroll
    for (int v = 0; v < V; ++v) f[v] = to_f32(u.e[v]);
  }
}
template <typename X, int V>
__device__ __forceinline__ void vec_store(X* p, const float (&f)[V]) {
  if constexpr (V == 1) {
    p[0] = from_f32<X>(f[0]);
  } else {
    constexpr int NQ = V * (int)sizeof(X) / 16;
    union {
      uint4 q[NQ];
      X e[V];
    } u;
#pragma unroll
    for (int v = 0; v < V; ++v) u.e[v] = from_f32<X>(f[v]);
#pragma unroll
    for (int q = 0; q < NQ; ++q) reinterpret_cast<uint4*>(p)[q] = u.q[q];
  }
}

// The whole backward of the sharded embedding in ONE launch, for steps of up to kBwdMaxIds tokens: no sort.  Every
// workgroup stages the step's ids in LDS.  Workgroup t < n owns token position t: if an earlier position names the
// same id it leaves at once; otherwise it marks the later positions with that id in an LDS bitmap, lists them in
// ascending order and sums their upstream rows front to back, starting from +0.0f with position t -- the order of a
// sequential index_add_ into a zeroed table, for all shards (groups) of the layer.  With a zero fill requested the
// grid has further workgroups, one per block of table rows: each finds the rows of its block that no token names
// (bitmap over the same ids) and clears them; rows that are named are written in full by their token workgroup, so
// nothing is written twice and no ordering between the two kinds of workgroup is needed.
constexpr int kBwdMaxIds = 4096;
template <typename T, typename G, int V>
__global__ __launch_bounds__(256) void embedding_bwd_kernel(const T* grad_out, long ld_go, int n, const int64_t* ids,
                                                            G* grad_table, long ld_gt, long row_begin, long row_count,
                                                            long cols, long padding_idx, int scale_by_freq,
                                                            int overwrite, int groups, long go_sg, long gt_sg,
                                                            float grad_scale, float* master, T* weights, float lr,
                                                            float clip, int store_grad, int zero_rows) {
  __shared__ int s_ids[kBwdMaxIds];
  __shared__ unsigned s_bits[kBwdMaxIds / 32];
  __shared__ int s_count;
  const int tid = threadIdx.x;
  for (int i = tid; i < n; i += 256) s_ids[i] = (int)ids[i];
  for (int i = tid; i < kBwdMaxIds / 32; i += 256) s_bits[i] = 0u;
  __syncthreads();
  if ((long)blockIdx.x >= n) {
    // ---- rows that no token names: cleared ----
    const long r0 = ((long)blockIdx.x - n) * zero_rows;
    for (int i = tid; i < n; i += 256) {
      const int id = s_ids[i];
      const long r = (long)id - row_begin - r0;
      if (id != padding_idx && r >= 0 && r < zero_rows) atomicOr(&s_bits[r >> 5], 1u << (r & 31));
    }
    __syncthreads();
    const long per_row = cols / V;  // vectors of a row in one group
    const long total = (long)zero_rows * groups * per_row;
    for (long e = tid; e < total; e += 256) {
      const long r = e / (groups * per_row), rem = e - r * (groups * per_row);
      const long g = rem / per_row, c = (rem - g * per_row) * V;
      if (r0 + r >= row_count || ((s_bits[r >> 5] >> (r & 31)) & 1u)) continue;
      G* dst = grad_table + g * gt_sg + (r0 + r) * ld_gt + c;
      if (V == 1) {
        dst[0] = from_f32<G>(0.0f);
      } else {
        constexpr int NQ = V * (int)sizeof(G) / 16;
#pragma unroll
        for (int q = 0; q < NQ; ++q) reinterpret_cast<uint4*>(dst)[q] = make_uint4(0u, 0u, 0u, 0u);
      }
    }
    return;
  }
  // ---- token position t ----
  const int t = blockIdx.x;
  const int id = s_ids[t];
  const long row = (long)id - row_begin;
  if (id == padding_idx || row < 0 || row >= row_count) return;
  int early = 0;
  for (int j = tid; j < t; j += 256) early |= (s_ids[j] == id) ? 1 : 0;
  if (__syncthreads_or(early)) return;  // an earlier position owns this id
  for (int j = t + tid; j < n; j += 256)
    if (s_ids[j] == id) atomicOr(&s_bits[j >> 5], 1u << (j & 31));
  __syncthreads();
  if (tid == 0) {
    // the positions with this id, ascending, written over the ids (which nobody reads any more)
    int cnt = 0;
    for (int w = t >> 5; w < (n + 31) / 32; ++w) {
      unsigned bits = s_bits[w];
      while (bits) {
        const int b = __builtin_ctz(bits);
        bits &= bits - 1;
        s_ids[cnt++] = w * 32 + b;
      }
    }
    s_count = cnt;
  }
  __syncthreads();
  const int cnt = s_count;
  const float inv = scale_by_freq ? 1.0f / (float)cnt : 1.0f;
  const long per_row = cols / V;
  for (long e = tid; e < (long)groups * per_row; e += 256) {
    const long g = e / per_row, c = (e - g * per_row) * V;
    const T* src = grad_out + g * go_sg + c;
    float acc[V];
#pragma unroll
    for (int v = 0; v < V; ++v) acc[v] = 0.0f;
    for (int k = 0; k < cnt; ++k) {
#pragma clang fp contract(off)
      const T* sp = src + (long)s_ids[k] * ld_go;
      union {
        uint4 q;
        T e[16 / sizeof(T)];
      } u;
      if (V == 1)
        u.e[0] = sp[0];
      else
        u.q = *reinterpret_cast<const uint4*>(sp);
#pragma unroll
      for (int v = 0; v < V; ++v) {
        // grad_scale != 1: the upstream gradient of a scaled embedding, T(grad * scale), rounded as the separate
        // multiplication would round it before it joins the sum (no fused multiply-add)
        const float x = grad_scale == 1.0f ? to_f32(u.e[v]) : to_f32(from_f32<T>(to_f32(u.e[v]) * grad_scale));
        acc[v] += x;
      }
    }
    const long off = g * gt_sg + row * ld_gt + c;
    {
#pragma clang fp contract(off)
      if (scale_by_freq) {
#pragma unroll
        for (int v = 0; v < V; ++v) acc[v] *= inv;
      }
      if (master != nullptr) {
        // clip + SGD where the row's gradient is produced (the caller guarantees it is the row's whole gradient)
        float w[V];
        vec_load<float, V>(master + off, w);
#pragma unroll
        for (int v = 0; v < V; ++v) w[v] = sgd_update<G>(w[v], acc[v], lr, clip);
        vec_store<float, V>(master + off, w);
        if (weights != nullptr) vec_store<T, V>(weights + off, w);
        if (store_grad) vec_store<G, V>(grad_table + off, acc);
        continue;
      }
      if (!overwrite) {
        float old[V];
        vec_load<G, V>(grad_table + off, old);
#pragma unroll
        for (int v = 0; v < V; ++v) acc[v] = old[v] + acc[v];
      }
      vec_store<G, V>(grad_table + off, acc);
    }
  }
}

// ---- backward of long steps: ids grouped by table row, no sort ----
// Two launches.  group_ids_kernel: workgroup w owns a slice of the table rows, counts the step's ids that fall into it (LDS
// counters, every workgroup reads all ids), turns the counts into offsets and writes every position into its row's
// segment of `pos` -- in any order -- and the rows with kLongRow positions or more into a list of its own.
// grouped_bwd_kernel: a wavefront per table row orders the row's positions and sums their upstream rows front to back,
// starting from +0.0f (the order of a sequential index_add_), or clears the row when no position names it; a long row
// is dealt over workgroups by columns instead, which start first.
//
// Words of running text are what makes this worth its launches: with ids by word frequency one of 16368 positions in nine
// is the same row, and the sum over that row's positions is a serial chain that only columns can share.  The sorted
// path (radix sort, one workgroup per segment and shard, one row in flight) took 533 us there, this takes 48 (uniform ids: 122
// against 34): 12 us the grouping, 35 the chain of the most frequent row, 36 clocks a position.
//
// kLongRow: with 64 (two rows of a short row's wavefront in flight) 2000 ids by word frequency over 5000 x 1024 took 29 us, with 32
// (four) 20.  kRankRow: 65536 uniform ids over 1000 x 512, rows of 65, 136 us by windows and 53 by counting.
constexpr int kLongRow = 32;             // positions from which a row is dealt over workgroups by columns
constexpr int kRankRow = 512;            // positions up to which such a row's are ordered by counting
constexpr int kGroupSlices = 32;         // workgroups of the grouping pass, at least
constexpr int kGroupRowsMax = 8192;      // table rows per slice, at most (LDS counters)
constexpr int kGroupMaxIds = 1 << 18;    // a long row's bitmap of positions in LDS: 32 KiB
constexpr int kGroupThreads = 1024;

struct GroupLayout {  // int32 arrays in the workspace
  size_t offs, pos, nlong, longs, total;
  int slices, rows_per, long_cap;
};
static GroupLayout group_layout(int64_t n, int64_t rows) {
  GroupLayout L;
  L.slices = (int)std::max<int64_t>(kGroupSlices, ceil_div(rows, kGroupRowsMax));
  L.rows_per = (int)ceil_div(rows, L.slices);
  L.long_cap = (int)(n / kLongRow);
  L.offs = 0;
  L.pos = ((size_t)(rows + 1) * 4 + 255) & ~(size_t)255;
  L.nlong = L.pos + (((size_t)n * 4 + 255) & ~(size_t)255);
  L.longs = L.nlong + (((size_t)L.slices * 4 + 255) & ~(size_t)255);
  L.total = L.longs + (size_t)L.slices * L.long_cap * 4 + 256;
  return L;
}

__global__ __launch_bounds__(kGroupThreads) void group_ids_kernel(const int64_t* ids, int n, long row_begin, int row_count,
                                                                  long padding_idx, int rows_per, int* offs, int* pos,
                                                                  int* nlong, int* longs, int long_cap) {
  __shared__ int cnt[kGroupRowsMax];
  __shared__ int wave_sum_[kGroupThreads / 64];
  __shared__ int s_long;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r0 = blockIdx.x * rows_per, r1 = min(r0 + rows_per, row_count), mine = max(r1 - r0, 0);
  for (int i = tid; i < mine; i += kGroupThreads) cnt[i] = 0;
  if (tid == 0) s_long = 0;
  __syncthreads();
  // row of position i inside the table, or -1
  constexpr int U = 8;
  auto rows_of = [&](int i0, int (&r)[U]) {
    int64_t v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int i = i0 + u * kGroupThreads;
      v[u] = ids[i < n ? i : n - 1];
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t q = (int64_t)(int)v[u] - row_begin;
      r[u] = (i0 + u * kGroupThreads < n && v[u] != padding_idx && q >= 0 && q < row_count) ? (int)q : -1;
    }
  };
  int below = 0;
  for (int i0 = tid; i0 < n; i0 += U * kGroupThreads) {
    int r[U];
    rows_of(i0, r);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (r[u] >= r0 && r[u] < r1) atomicAdd(&cnt[r[u] - r0], 1);
      below += (r[u] >= 0 && r[u] < r0) ? 1 : 0;
    }
  }
  // base = positions of all earlier slices; then the exclusive scan of the slice's counts, in place
  auto block_scan = [&](int v, int& all) {  // exclusive prefix of v over the workgroup, and the sum
    int x = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int y = __shfl_up(x, o, 64);
      if (lane >= o) x += y;
    }
    __syncthreads();
    if (lane == 63) wave_sum_[wave] = x;
    __syncthreads();
    int before = 0;
    all = 0;
#pragma unroll
    for (int w = 0; w < kGroupThreads / 64; ++w) {
      before += w < wave ? wave_sum_[w] : 0;
      all += wave_sum_[w];
    }
    return before + x - v;
  };
  int base = 0, all;
  (void)block_scan(below, base);
  const int per = (mine + kGroupThreads - 1) / kGroupThreads, c0 = min(tid * per, mine), c1 = min(c0 + per, mine);
  int sum = 0;
  for (int c = c0; c < c1; ++c) sum += cnt[c];
  int run = base + block_scan(sum, all);
  for (int c = c0; c < c1; ++c) {
    const int k = cnt[c];
    if (k >= kLongRow) longs[(long)blockIdx.x * long_cap + atomicAdd(&s_long, 1)] = r0 + c;
    cnt[c] = run;
    offs[r0 + c] = run;
    run += k;
  }
  __syncthreads();
  if (tid == 0) {
    nlong[blockIdx.x] = s_long;
    if (r1 == row_count && mine > 0) offs[row_count] = base + all;
  }
  for (int i0 = tid; i0 < n; i0 += U * kGroupThreads) {
    int r[U];
    rows_of(i0, r);
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (r[u] >= r0 && r[u] < r1) pos[atomicAdd(&cnt[r[u] - r0], 1)] = i0 + u * kGroupThreads;
  }
}

template <typename T, typename G>
struct GroupedBwd {
  const T* grad_out;
  long ld_go, go_sg;
  G* grad_table;
  long ld_gt, gt_sg;
  float* master;
  T* weights;
  float grad_scale, lr, clip;
  int scale_by_freq, overwrite, store_grad, zero_fill;
  int n, row_count, groups, cols;
  const int *offs, *pos, *nlong, *longs;
  int slices, long_cap;
  int plain;  // the upstream gradient lies within 2 GiB of its start and is not scaled

  // one upstream value as it joins the sum
  __device__ __forceinline__ float take(T g) const {
#pragma clang fp contract(off)
    return grad_scale == 1.0f ? to_f32(g) : to_f32(from_f32<T>(to_f32(g) * grad_scale));
  }
  // the finished sums of V columns of a row that `cnt` positions name
  template <int V>
  __device__ __forceinline__ void finish(float (&acc)[V], long off, int cnt) const {
#pragma clang fp contract(off)
    if (scale_by_freq) {
      const float inv = 1.0f / (float)cnt;
#pragma unroll
      for (int v = 0; v < V; ++v) acc[v] *= inv;
    }
    if (master != nullptr) {
      float w[V];
      vec_load<float, V>(master + off, w);
#pragma unroll
      for (int v = 0; v < V; ++v) w[v] = sgd_update<G>(w[v], acc[v], lr, clip);
      vec_store<float, V>(master + off, w);
      if (weights != nullptr) vec_store<T, V>(weights + off, w);
      if (store_grad) vec_store<G, V>(grad_table + off, acc);
      return;
    }
    if (!overwrite) {
      float old[V];
      vec_load<G, V>(grad_table + off, old);
#pragma unroll
      for (int v = 0; v < V; ++v) acc[v] = old[v] + acc[v];
    }
    vec_store<G, V>(grad_table + off, acc);
  }
};

// Adds column `src` of the upstream rows at list[0 .. m) + at (ascending positions).  The sum is a serial chain of one wave: kBlocks
// blocks of kBlockRows rows are on their way to registers while the oldest is added, and a row costs the wave five
// instructions: its offset, worked out by 64 lanes at once, becomes the scalar offset of a buffer load, and what is loaded is
// widened and added.  (With the row's 64-bit address from scalar multiplications, and two columns a lane, a row
// took 80 clocks: a wave of 1670 rows 68 us.)  PLAIN: the upstream gradient lies within 2 GiB, so that offsets are 32 bits, and
// joins the sum unscaled.
constexpr int kBlockRows = 16, kBlocks = 4;
template <bool PLAIN, typename T, typename G, typename L>
__device__ __forceinline__ void sum_rows(const GroupedBwd<T, G>& a, long src, const L* list, int at, int m, float& acc) {
  const int lane = threadIdx.x & 63;
  const __amdgpu_buffer_rsrc_t all = __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(a.grad_out), 0, 0x7fffffff, 0x00020000);
  const int mine_col = (int)(src * (long)sizeof(T));
  T g[kBlocks][kBlockRows];
  auto load = [&](int b, auto S) __attribute__((always_inline)) {
    const int mine = (int)list[min(b * kBlockRows + (lane & (kBlockRows - 1)), m - 1)] + at;
    const int ofs = (int)((unsigned)mine * (unsigned)(a.ld_go * (long)sizeof(T)));
#pragma unroll
    for (int u = 0; u < kBlockRows; ++u) {
      T& v = g[decltype(S)::value][u];
      if constexpr (!PLAIN)
        v = a.grad_out[(long)__builtin_amdgcn_readlane(mine, u) * a.ld_go + src];
      else if constexpr (sizeof(T) == 4)
        v = __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b32(all, mine_col, __builtin_amdgcn_readlane(ofs, u), 0));
      else
        v = __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b16(all, mine_col, __builtin_amdgcn_readlane(ofs, u), 0));
    }
  };
  auto add = [&](int b, auto S) __attribute__((always_inline)) {
    const int left = m - b * kBlockRows;
    if (left >= kBlockRows) {
#pragma unroll
      for (int u = 0; u < kBlockRows; ++u) acc += PLAIN ? to_f32(g[decltype(S)::value][u]) : a.take(g[decltype(S)::value][u]);
    } else if (left > 0) {
#pragma unroll
      for (int u = 0; u < kBlockRows; ++u) acc = u < left ? acc + (PLAIN ? to_f32(g[decltype(S)::value][u]) : a.take(g[decltype(S)::value][u])) : acc;
    }
  };
  // blocks behind the last one re-read its last row: with loads under a condition every block would wait for all of them
  [&]<int... S>(std::integer_sequence<int, S...>) __attribute__((always_inline)) {
    (load(S, std::integral_constant<int, S>{}), ...);
  }(std::make_integer_sequence<int, kBlocks - 1>{});
  for (int b = 0; b * kBlockRows < m; b += kBlocks)
    [&]<int... S>(std::integer_sequence<int, S...>) __attribute__((always_inline)) {
      ((load(b + S + kBlocks - 1, std::integral_constant<int, (S + kBlocks - 1) % kBlocks>{}),
        add(b + S, std::integral_constant<int, S>{})),
       ...);
    }(std::make_integer_sequence<int, kBlocks>{});
}

// long_wgs workgroups for the long rows (long row j, column chunk y: j * chunks + y), then one wavefront per table row.
// V: columns per lane of a short row (16-byte vectors, or 1); a lane of a long row has one.
template <typename T, typename G, int V>
__global__ __launch_bounds__(256) void grouped_bwd_kernel(GroupedBwd<T, G> a, int long_wgs, int chunks) {
  extern __shared__ __attribute__((aligned(16))) unsigned bits[];  // a long row's positions as a bitmap, then the window's list
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  if ((int)blockIdx.x < long_wgs) {
    __shared__ int s_row, s_part[4];
    const int want = blockIdx.x / chunks, chunk = blockIdx.x - want * chunks;
    if (wave == 0) {  // long row `want` of all slices: 64 slices' counts at a time
      int left = want, row = -1;
      for (int s0 = 0; s0 < a.slices && row < 0; s0 += 64) {
        const int c = s0 + lane < a.slices ? a.nlong[s0 + lane] : 0;
        int x = c;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
          const int y = __shfl_up(x, o, 64);
          if (lane >= o) x += y;
        }
        const bool here = left < x && left >= x - c;
        if (here) row = a.longs[(long)(s0 + lane) * a.long_cap + left - (x - c)];
        const unsigned long long at = __ballot(here);
        row = at ? __shfl(row, __builtin_ctzll(at), 64) : -1;
        left -= __shfl(x, 63, 64);
      }
      if (lane == 0) s_row = row;
    }
    __syncthreads();
    const int row = s_row;
    if (row < 0) return;
    const int p0 = a.offs[row], cnt = a.offs[row + 1] - p0;
    const int e = chunk * 256 + tid;  // column of the row over all shards
    const bool live = e < a.cols * a.groups;
    const int g = live ? e / a.cols : 0, c = live ? e - g * a.cols : 0;
    const long src = g * a.go_sg + c;
    float acc = 0.0f;
    if (cnt <= kRankRow) {
      // every thread counts the positions below its own; (a window at a time, as below, a row of 65 positions in 65536
      // had a trip to memory for every eight of them)
      int* raw = reinterpret_cast<int*>(bits);
      int* sorted = raw + kRankRow;
      for (int i = tid; i < kRankRow; i += 256) raw[i] = i < cnt ? a.pos[p0 + i] : 0x7fffffff;
      __syncthreads();
      for (int i = tid; i < cnt; i += 256) {
        const int mine = raw[i];
        int rank = 0;
        for (int k = 0; k < cnt; k += 4) {
          const int4 q = *reinterpret_cast<const int4*>(raw + k);
          rank += (q.x < mine) + (q.y < mine) + (q.z < mine) + (q.w < mine);
        }
        sorted[rank] = mine;
      }
      __syncthreads();
      if (a.plain)
        sum_rows<true>(a, src, sorted, 0, cnt, acc);
      else
        sum_rows<false>(a, src, sorted, 0, cnt, acc);
    } else {
      const int words = (a.n + 31) / 32, windows = (words + 255) / 256;
      unsigned short* list = reinterpret_cast<unsigned short*>(bits + windows * 256);
      for (int i = tid; i < windows * 256; i += 256) bits[i] = 0u;
      __syncthreads();
      for (int i = tid; i < cnt; i += 256) {
        const int q = a.pos[p0 + i];
        atomicOr(&bits[q >> 5], 1u << (q & 31));
      }
      for (int win = 0; win < windows; ++win) {
        __syncthreads();  // the bitmap is complete; the previous window's list has been read
        // the window's 8192 positions: a word per thread, listed in ascending order
        unsigned b = bits[win * 256 + tid];
        int x = __popc(b);
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
          const int y = __shfl_up(x, o, 64);
          if (lane >= o) x += y;
        }
        if (lane == 63) s_part[wave] = x;
        __syncthreads();
        int at = x - __popc(b);
#pragma unroll
        for (int w = 0; w < 4; ++w) at += w < wave ? s_part[w] : 0;
        const int m = (s_part[0] + s_part[1]) + (s_part[2] + s_part[3]);
        while (b) {
          list[at++] = (unsigned short)(tid * 32 + __builtin_ctz(b));
          b &= b - 1;
        }
        __syncthreads();
        if (m > 0 && a.plain) sum_rows<true>(a, src, list, win * 8192, m, acc);
        else if (m > 0) sum_rows<false>(a, src, list, win * 8192, m, acc);
      }
    }
    if (!live) return;
    float one[1] = {acc};
    a.template finish<1>(one, g * a.gt_sg + (long)row * a.ld_gt + c, cnt);
    return;
  }
  const int row = (int)(blockIdx.x - long_wgs) * 4 + wave;
  if (row >= a.row_count) return;
  const int p0 = a.offs[row], cnt = a.offs[row + 1] - p0;
  if (cnt >= kLongRow || (cnt == 0 && !a.zero_fill)) return;
  const int per_row = a.cols / V, total = per_row * a.groups;
  // the row's positions in ascending order, one per lane: each lane counts the smaller ones, then they change places
  int sorted = 0;
  if (cnt > 0) {
    const int mine = lane < cnt ? a.pos[p0 + lane] : 0x7fffffff;
    int rank = 0;
    for (int k = 0; k < cnt; ++k) rank += __builtin_amdgcn_readlane(mine, k) < mine ? 1 : 0;
    // lanes beyond the row's positions keep out of the way: each its own slot behind them
    sorted = __builtin_amdgcn_ds_permute((lane < cnt ? rank : lane) * 4, mine);
  }
  constexpr int CB = 4;  // vectors per lane worked on at once
  for (int e0 = lane; e0 < total; e0 += CB * 64) {
    float acc[CB][V];
    long at[CB], to[CB];
#pragma unroll
    for (int d = 0; d < CB; ++d) {
      const int e = e0 + d * 64 < total ? e0 + d * 64 : e0;
      const int g = e / per_row, c = (e - g * per_row) * V;
      at[d] = g * a.go_sg + c, to[d] = g * a.gt_sg + (long)row * a.ld_gt + c;
#pragma unroll
      for (int v = 0; v < V; ++v) acc[d][v] = 0.0f;
    }
    auto add = [&](int k, auto rows_tag) {
      constexpr int R = decltype(rows_tag)::value;
      union {
        uint4 q;
        T e[16 / sizeof(T)];
      } u[R][CB];
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const T* src = a.grad_out + (long)__builtin_amdgcn_readlane(sorted, k + r) * a.ld_go;
#pragma unroll
        for (int d = 0; d < CB; ++d) {
          if constexpr (V == 1)
            u[r][d].e[0] = src[at[d]];
          else
            u[r][d].q = *reinterpret_cast<const uint4*>(src + at[d]);
        }
      }
#pragma unroll
      for (int r = 0; r < R; ++r)
#pragma unroll
        for (int d = 0; d < CB; ++d)
#pragma unroll
          for (int v = 0; v < V; ++v) acc[d][v] += a.take(u[r][d].e[v]);
    };
    int k = 0;
    for (; k + 4 <= cnt; k += 4) add(k, std::integral_constant<int, 4>{});
    if (k + 2 <= cnt) add(k, std::integral_constant<int, 2>{}), k += 2;
    if (k < cnt) add(k, std::integral_constant<int, 1>{});
#pragma unroll
    for (int d = 0; d < CB; ++d) {
      if (e0 + d * 64 >= total) break;
      if (cnt == 0)
        vec_store<G, V>(a.grad_table + to[d], acc[d]);
      else
        a.template finish<V>(acc[d], to[d], cnt);
    }
  }
}

struct SortLayout {
  size_t keys_in, vals_in, keys_out, vals_out, temp, total, temp_bytes;
};

static SortLayout sort_layout(int64_t n) {
  SortLayout L;
  const size_t arr = ((size_t)n * 4 + 255) & ~(size_t)255;
  L.keys_in = 0;
  L.vals_in = arr;
  L.keys_out = 2 * arr;
  L.vals_out = 3 * arr;
  L.temp = 4 * arr;
  size_t tb = 0;
  (void)rocprim::radix_sort_pairs(nullptr, tb, (const int*)nullptr, (int*)nullptr, (const int*)nullptr, (int*)nullptr,
                                  (unsigned)n, 0, 32, (hipStream_t) nullptr);
  L.temp_bytes = tb;
  L.total = L.temp + ((tb + 255) & ~(size_t)255) + 256;
  return L;
}

}  // namespace rtp

using namespace rtp;

static int gather_impl(void* stream, int dtype, const void* table, int64_t ld_table, int64_t row_begin,
                       int64_t row_count, int64_t cols, const int64_t* ids, int64_t n_ids, void* out, int64_t ld_out,
                       int64_t groups, int64_t table_sg, int64_t out_sg, float scale, const void* pos, int64_t ld_pos,
                       int64_t pos_sg, int64_t batch) {
  RTP_REQUIRE(table && ids && out, "rtp_embedding_gather: null pointer");
  RTP_REQUIRE(cols >= 0 && ld_table >= cols && ld_out >= cols && row_count >= 0 && n_ids >= 0,
              "rtp_embedding_gather: bad shape cols=%lld ld_table=%lld ld_out=%lld", (long long)cols,
              (long long)ld_table, (long long)ld_out);
  if (n_ids == 0 || cols == 0) return RTP_OK;
  RTP_REQUIRE(n_ids < (1ll << 31), "rtp_embedding_gather: too many ids");
  RTP_REQUIRE(groups >= 1 && groups < 65536, "rtp_embedding_gather: groups=%lld out of range", (long long)groups);
  const size_t esz = dtype == RTP_F32 ? 4 : 2;
  RTP_REQUIRE(dtype == RTP_F32 || dtype == RTP_BF16, "rtp_embedding_gather: unknown dtype %d", dtype);
  const int vec = ((uintptr_t)table % 16 == 0) && ((uintptr_t)out % 16 == 0) && (ld_table * esz) % 16 == 0 &&
                  (ld_out * esz) % 16 == 0 && (cols * esz) % 16 == 0 && (table_sg * esz) % 16 == 0 &&
                  (out_sg * esz) % 16 == 0 &&
                  (!pos || ((uintptr_t)pos % 16 == 0 && (ld_pos * esz) % 16 == 0 && (pos_sg * esz) % 16 == 0));
  const int64_t per_row = vec ? cols * (int64_t)esz / 16 : cols;
  RTP_REQUIRE(per_row * groups < (1ll << 30), "rtp_embedding_gather: rows too long");
  const dim3 grid((unsigned)ceil_div(n_ids, 4));
  hipStream_t s = (hipStream_t)stream;
  ProfileScope prof(s, "embedding_gather", 0.0, (2.0 * (double)n_ids * cols * esz + 8.0 * n_ids) * groups);
#define RTP_GATHER(T, V, POS)                                                                                          \
  hipLaunchKernelGGL((gather_kernel<T, V, POS>), grid, dim3(256), 0, s, (const T*)table, (long)ld_table, (long)row_begin, \
                     (long)row_count, (int)per_row, make_fastdiv((unsigned)per_row), (int)(per_row * groups), ids, (long)n_ids, \
                     (T*)out, (long)ld_out, (long)table_sg, (long)out_sg, scale, (const T*)pos, (long)ld_pos, (long)pos_sg, \
                     make_fastdiv((unsigned)batch))
#define RTP_GATHER_V(T, V) do { if (pos) RTP_GATHER(T, V, true); else RTP_GATHER(T, V, false); } while (0)
  if (dtype == RTP_F32) {
    if (vec) RTP_GATHER_V(float, 4); else RTP_GATHER_V(float, 1);
  } else {
    if (vec) RTP_GATHER_V(bf16_t, 8); else RTP_GATHER_V(bf16_t, 1);
  }
#undef RTP_GATHER_V
#undef RTP_GATHER
  RTP_LAUNCH_CHECK();
  return RTP_OK;
}

extern "C" int rtp_embedding_gather(void* stream, int dtype, const void* table, int64_t ld_table, int64_t row_begin,
                                    int64_t row_count, int64_t cols, const int64_t* ids, int64_t n_ids, void* out,
                                    int64_t ld_out, int64_t groups, int64_t table_sg, int64_t out_sg) {
  return gather_impl(stream, dtype, table, ld_table, row_begin, row_count, cols, ids, n_ids, out, ld_out, groups,
                     table_sg, out_sg, 1.0f, nullptr, 0, 0, 1);
}

extern "C" int rtp_embedding_gather_scale_pos(void* stream, int dtype, const void* table, int64_t ld_table,
                                              int64_t row_begin, int64_t row_count, int64_t cols, const int64_t* ids,
                                              int64_t n_ids, void* out, int64_t ld_out, int64_t groups,
                                              int64_t table_sg, int64_t out_sg, float scale, const void* pos,
                                              int64_t ld_pos, int64_t pos_sg, int64_t batch) {
  RTP_REQUIRE(pos && batch >= 1 && batch < (1ll << 31) && ld_pos >= cols,
              "rtp_embedding_gather_scale_pos: need a positional table and 1 <= batch < 2^31");
  return gather_impl(stream, dtype, table, ld_table, row_begin, row_count, cols, ids, n_ids, out, ld_out, groups,
                     table_sg, out_sg, scale, pos, ld_pos, pos_sg, batch);
}

extern "C" size_t rtp_embedding_scatter_workspace_bytes(int64_t n_ids) {
  if (n_ids <= 0) return 256;
  return sort_layout(n_ids).total;
}

extern "C" int rtp_embedding_sort_ids(void* stream, const int64_t* ids, int64_t n_ids, void* workspace,
                                      size_t workspace_bytes) {
  RTP_REQUIRE(ids && workspace, "rtp_embedding_sort_ids: null pointer");
  RTP_REQUIRE(n_ids >= 0 && n_ids < (1ll << 31), "rtp_embedding_sort_ids: bad n_ids %lld", (long long)n_ids);
  if (n_ids == 0) return RTP_OK;
  RTP_REQUIRE((uintptr_t)workspace % 256 == 0, "rtp_embedding_sort_ids: workspace must be 256-byte aligned");
  const SortLayout L = sort_layout(n_ids);
  if (workspace_bytes < L.total)
    return fail(RTP_ERR_WORKSPACE, "rtp_embedding_sort_ids: workspace %zu < required %zu", workspace_bytes, L.total);
  char* w = (char*)workspace;
  hipStream_t s = (hipStream_t)stream;
  if (n_ids <= kSortLdsMax) {
    int npow2 = 2;
    while (npow2 < n_ids) npow2 <<= 1;
    ProfileScope prof(s, "embedding_sort_ids", 0.0, 16.0 * (double)n_ids);
    hipLaunchKernelGGL(sort_ids_lds_kernel, dim3(1), dim3(kSortThreads), (size_t)npow2 * 8, s, ids, (int)n_ids, npow2,
                       (int*)(w + L.keys_out), (int*)(w + L.vals_out));
    RTP_LAUNCH_CHECK();
    return RTP_OK;
  }
  // more ids than one workgroup's LDS holds: the device-wide radix sort of rocPRIM
  hipLaunchKernelGGL(sort_prep_kernel, dim3((unsigned)ceil_div(n_ids, 256)), dim3(256), 0, s, ids, (long)n_ids,
                     (int*)(w + L.keys_in), (int*)(w + L.vals_in));
  RTP_LAUNCH_CHECK();
  size_t tb = L.temp_bytes;
  RTP_HIP_TRY(rocprim::radix_sort_pairs((void*)(w + L.temp), tb, (const int*)(w + L.keys_in), (int*)(w + L.keys_out),
                                        (const int*)(w + L.vals_in), (int*)(w + L.vals_out), (unsigned)n_ids, 0, 32,
                                        s));
  return RTP_OK;
}

static int scatter_impl(void* stream, int dtype, const void* grad_out, int64_t ld_grad_out, int64_t n_ids,
                        const void* workspace, void* grad_table, int64_t ld_grad_table, int grad_table_f32,
                        int64_t row_begin, int64_t row_count, int64_t cols, int64_t padding_idx, int scale_by_freq,
                        int zero_fill, int64_t groups, int64_t grad_out_sg, int64_t grad_table_sg, float grad_scale,
                        float* master = nullptr, void* weights = nullptr, float lr = 0.0f, float clip = 0.0f,
                        int store_grad = 1) {
  RTP_REQUIRE(grad_out && workspace && grad_table, "rtp_embedding_scatter_add_det: null pointer");
  if (master != nullptr) {
    // the fused update replaces the dense gradient: nothing to fill unless the gradient is wanted as well
    RTP_REQUIRE(!grad_table_f32 || dtype == RTP_F32, "rtp_embedding_scatter_add_sgd: the gradient table has the table's dtype");
    RTP_REQUIRE(zero_fill || !store_grad, "rtp_embedding_scatter_add_sgd: a stored gradient starts from a zero fill");
    if (!store_grad) zero_fill = 0;
  }
  RTP_REQUIRE(groups >= 1 && groups < 65536, "rtp_embedding_scatter_add_det: groups %lld not in 1..65535",
              (long long)groups);
  RTP_REQUIRE(dtype == RTP_F32 || dtype == RTP_BF16, "rtp_embedding_scatter_add_det: unknown dtype %d", dtype);
  RTP_REQUIRE(cols >= 0 && ld_grad_out >= cols && ld_grad_table >= cols && row_count >= 0 && n_ids >= 0 &&
                  n_ids < (1ll << 31),
              "rtp_embedding_scatter_add_det: bad shape");
  if (cols == 0 || row_count == 0) return RTP_OK;
  hipStream_t s = (hipStream_t)stream;
  const size_t gsz = (dtype == RTP_F32 || grad_table_f32) ? 4 : 2;
  const unsigned chunks = (unsigned)std::min<int64_t>(16, std::max<int64_t>(1, ceil_div(cols, 1024)));
  if (zero_fill) {
    RTP_REQUIRE(row_count < (1ll << 31), "rtp_embedding_scatter_add_det: too many rows");
    ProfileScope prof(s, "embedding_grad_zero_fill", 0.0, (double)groups * row_count * cols * gsz);
    if (ld_grad_table == cols) {
      // a group's table is one contiguous block: fill it as such (a workgroup per 512-byte row slice is mostly idle)
      const int64_t bytes = row_count * cols * gsz;
      const unsigned wgs = (unsigned)std::min<int64_t>(2048, std::max<int64_t>(1, ceil_div(bytes, 16384)));
      hipLaunchKernelGGL(zero_rows_kernel, dim3(1, wgs, (unsigned)groups), dim3(256), 0, s, (char*)grad_table,
                         (long)bytes, (long)bytes, 1l, (long)(grad_table_sg * gsz));
    } else {
      hipLaunchKernelGGL(zero_rows_kernel, dim3((unsigned)row_count, chunks, (unsigned)groups), dim3(256), 0, s,
                         (char*)grad_table, (long)(ld_grad_table * gsz), (long)(cols * gsz), (long)row_count,
                         (long)(grad_table_sg * gsz));
    }
    RTP_LAUNCH_CHECK();
  }
  if (n_ids == 0) return RTP_OK;
  const SortLayout L = sort_layout(n_ids);
  const char* w = (const char*)workspace;
  const int* keys = (const int*)(w + L.keys_out);
  const int* vals = (const int*)(w + L.vals_out);
  dim3 grid((unsigned)n_ids, chunks, (unsigned)groups);
  // After a zero fill the rows can simply be overwritten; otherwise the sum is added to what is there.
  const int overwrite = zero_fill ? 1 : 0;
#define RTP_SCATTER(T, G)                                                                                         \
  hipLaunchKernelGGL((scatter_kernel<T, G>), grid, dim3(256), 0, s, (const T*)grad_out, (long)ld_grad_out,         \
                     (long)n_ids, keys, vals, (G*)grad_table, (long)ld_grad_table, (long)row_begin, (long)row_count, \
                     (long)cols, (long)padding_idx, scale_by_freq, overwrite, (long)grad_out_sg, (long)grad_table_sg,  \
                     grad_scale, master, (T*)weights, lr, clip, store_grad)
  // algorithmic bytes: read every upstream row once, write (or read-modify-write) every touched row once
  ProfileScope prof(s, "embedding_scatter_add", (double)groups * n_ids * cols,
                    (double)groups * n_ids * cols * ((dtype == RTP_F32 ? 4.0 : 2.0) + (zero_fill ? 1.0 : 2.0) * gsz) + 8.0 * n_ids);
  if (dtype == RTP_F32)
    RTP_SCATTER(float, float);
  else if (grad_table_f32)
    RTP_SCATTER(bf16_t, float);
  else
    RTP_SCATTER(bf16_t, bf16_t);
#undef RTP_SCATTER
  RTP_LAUNCH_CHECK();
  return RTP_OK;
}

extern "C" int rtp_embedding_scatter_add_det(void* stream, int dtype, const void* grad_out, int64_t ld_grad_out,
                                             int64_t n_ids, const void* workspace, void* grad_table,
                                             int64_t ld_grad_table, int grad_table_f32, int64_t row_begin,
                                             int64_t row_count, int64_t cols, int64_t padding_idx, int scale_by_freq,
                                             int zero_fill, int64_t groups, int64_t grad_out_sg,
                                             int64_t grad_table_sg) {
  return scatter_impl(stream, dtype, grad_out, ld_grad_out, n_ids, workspace, grad_table, ld_grad_table, grad_table_f32,
                      row_begin, row_count, cols, padding_idx, scale_by_freq, zero_fill, groups, grad_out_sg,
                      grad_table_sg, 1.0f);
}

extern "C" int rtp_embedding_scatter_add_scaled(void* stream, int dtype, const void* grad_out, int64_t ld_grad_out,
                                                int64_t n_ids, const void* workspace, void* grad_table,
                                                int64_t ld_grad_table, int grad_table_f32, int64_t row_begin,
                                                int64_t row_count, int64_t cols, int64_t padding_idx,
                                                int scale_by_freq, int zero_fill, int64_t groups, int64_t grad_out_sg,
                                                int64_t grad_table_sg, float grad_scale) {
  return scatter_impl(stream, dtype, grad_out, ld_grad_out, n_ids, workspace, grad_table, ld_grad_table, grad_table_f32,
                      row_begin, row_count, cols, padding_idx, scale_by_freq, zero_fill, groups, grad_out_sg,
                      grad_table_sg, grad_scale);
}

extern "C" int rtp_embedding_scatter_add_sgd(void* stream, int dtype, const void* grad_out, int64_t ld_grad_out,
                                             int64_t n_ids, const void* workspace, void* grad_table,
                                             int64_t ld_grad_table, int64_t row_begin, int64_t row_count, int64_t cols,
                                             int64_t padding_idx, int scale_by_freq, int64_t groups,
                                             int64_t grad_out_sg, int64_t grad_table_sg, float grad_scale,
                                             float* master, void* weights, float lr, float clip, int store_grad) {
  RTP_REQUIRE(master != nullptr, "rtp_embedding_scatter_add_sgd: null master");
  RTP_REQUIRE(dtype == RTP_F32 ? weights == nullptr || weights == (void*)master : true,
              "rtp_embedding_scatter_add_sgd: fp32 tables are their own master");
  return scatter_impl(stream, dtype, grad_out, ld_grad_out, n_ids, workspace, grad_table, ld_grad_table, 0, row_begin,
                      row_count, cols, padding_idx, scale_by_freq, store_grad ? 1 : 0, groups, grad_out_sg,
                      grad_table_sg, grad_scale, master, dtype == RTP_F32 ? nullptr : weights, lr, clip, store_grad);
}

extern "C" int rtp_embedding_backward_supported(int64_t n_ids) { return n_ids >= 0 && n_ids <= kBwdMaxIds ? 1 : 0; }

extern "C" int rtp_embedding_backward(void* stream, int dtype, const void* grad_out, int64_t ld_grad_out, int64_t n_ids,
                                      const int64_t* ids, void* grad_table, int64_t ld_grad_table, int grad_table_f32,
                                      int64_t row_begin, int64_t row_count, int64_t cols, int64_t padding_idx,
                                      int scale_by_freq, int zero_fill, int64_t groups, int64_t grad_out_sg,
                                      int64_t grad_table_sg, float grad_scale, float* master, void* weights, float lr,
                                      float clip, int store_grad) {
  RTP_REQUIRE(grad_out && grad_table && (ids || n_ids == 0), "rtp_embedding_backward: null pointer");
  RTP_REQUIRE(rtp_embedding_backward_supported(n_ids), "rtp_embedding_backward: %lld ids, at most %d (sort + scatter beyond)",
              (long long)n_ids, kBwdMaxIds);
  RTP_REQUIRE(dtype == RTP_F32 || dtype == RTP_BF16, "rtp_embedding_backward: unknown dtype %d", dtype);
  RTP_REQUIRE(groups >= 1 && groups < 65536, "rtp_embedding_backward: groups %lld not in 1..65535", (long long)groups);
  RTP_REQUIRE(cols >= 0 && ld_grad_out >= cols && ld_grad_table >= cols && row_count >= 0 && row_count < (1ll << 31),
              "rtp_embedding_backward: bad shape");
  if (master != nullptr) {
    RTP_REQUIRE(!grad_table_f32 || dtype == RTP_F32, "rtp_embedding_backward: with an update the gradient table has the table's dtype");
    RTP_REQUIRE(dtype != RTP_F32 || weights == nullptr || weights == (void*)master,
                "rtp_embedding_backward: fp32 tables are their own master");
    RTP_REQUIRE(zero_fill || !store_grad, "rtp_embedding_backward: a stored gradient beside the update starts from a zero fill");
    if (!store_grad) zero_fill = 0;  // the update replaces the dense gradient: nothing to fill
    if (dtype == RTP_F32) weights = nullptr;
  } else {
    store_grad = 1;
  }
  if (cols == 0 || row_count == 0 || (n_ids == 0 && !zero_fill)) return RTP_OK;
  hipStream_t s = (hipStream_t)stream;
  const size_t esz = dtype == RTP_F32 ? 4 : 2, gsz = (dtype == RTP_F32 || grad_table_f32) ? 4 : 2;
  // 16-byte accesses when every row of every operand allows them
  const int64_t vec = 16 / (int64_t)esz;
  const bool aligned = cols % vec == 0 && (uintptr_t)grad_out % 16 == 0 && (ld_grad_out * esz) % 16 == 0 &&
                       (grad_out_sg * esz) % 16 == 0 && (uintptr_t)grad_table % 16 == 0 &&
                       (ld_grad_table * gsz) % 16 == 0 && (grad_table_sg * gsz) % 16 == 0 &&
                       (master == nullptr || (uintptr_t)master % 16 == 0) &&
                       (weights == nullptr || (uintptr_t)weights % 16 == 0);
  // a zero-fill workgroup clears about 64 KiB: a block of rows over all groups
  int64_t zero_rows = 0, zero_wgs = 0;
  if (zero_fill) {
    zero_rows = std::max<int64_t>(1, std::min<int64_t>(kBwdMaxIds, 65536 / std::max<int64_t>(1, groups * cols * (int64_t)gsz)));
    zero_wgs = ceil_div(row_count, zero_rows);
  }
  RTP_REQUIRE(n_ids + zero_wgs < (1ll << 31), "rtp_embedding_backward: grid too large");
  const dim3 grid((unsigned)(n_ids + zero_wgs));
  // algorithmic bytes: every upstream row read once, every named row written (or read, modified and written) once;
  // the fill of the rows nobody names is extra
  ProfileScope prof(s, "embedding_backward", (double)groups * n_ids * cols,
                    (double)groups * n_ids * cols * (esz + (zero_fill || master ? 1.0 : 2.0) * gsz) + 8.0 * n_ids);
#define RTP_EMB_BWD(T, G, V)                                                                                          \
  hipLaunchKernelGGL((embedding_bwd_kernel<T, G, V>), grid, dim3(256), 0, s, (const T*)grad_out, (long)ld_grad_out,    \
                     (int)n_ids, ids, (G*)grad_table, (long)ld_grad_table, (long)row_begin, (long)row_count, (long)cols, \
                     (long)padding_idx, scale_by_freq, zero_fill ? 1 : 0, (int)groups, (long)grad_out_sg,               \
                     (long)grad_table_sg, grad_scale, master, (T*)weights, lr, clip, store_grad, (int)zero_rows)
  if (dtype == RTP_F32) {
    if (aligned) RTP_EMB_BWD(float, float, 4); else RTP_EMB_BWD(float, float, 1);
  } else if (grad_table_f32) {
    if (aligned) RTP_EMB_BWD(bf16_t, float, 8); else RTP_EMB_BWD(bf16_t, float, 1);
  } else {
    if (aligned) RTP_EMB_BWD(bf16_t, bf16_t, 8); else RTP_EMB_BWD(bf16_t, bf16_t, 1);
  }
#undef RTP_EMB_BWD
  RTP_LAUNCH_CHECK();
  return RTP_OK;
}

extern "C" int rtp_embedding_backward_grouped_supported(int64_t n_ids, int64_t row_count) {
  return n_ids > 0 && n_ids <= kGroupMaxIds && row_count > 0 && row_count < (1ll << 26) ? 1 : 0;
}

extern "C" size_t rtp_embedding_backward_grouped_workspace_bytes(int64_t n_ids, int64_t row_count) {
  if (!rtp_embedding_backward_grouped_supported(n_ids, row_count)) return 256;
  return group_layout(n_ids, row_count).total;
}

extern "C" int rtp_embedding_backward_grouped(void* stream, int dtype, const void* grad_out, int64_t ld_grad_out,
                                              int64_t n_ids, const int64_t* ids, void* grad_table, int64_t ld_grad_table,
                                              int grad_table_f32, int64_t row_begin, int64_t row_count, int64_t cols,
                                              int64_t padding_idx, int scale_by_freq, int zero_fill, int64_t groups,
                                              int64_t grad_out_sg, int64_t grad_table_sg, float grad_scale, float* master,
                                              void* weights, float lr, float clip, int store_grad, void* workspace,
                                              size_t workspace_bytes) {
  const char* who = "rtp_embedding_backward_grouped";
  RTP_REQUIRE(grad_out && grad_table && ids && workspace, "%s: null pointer", who);
  RTP_REQUIRE(rtp_embedding_backward_grouped_supported(n_ids, row_count), "%s: %lld ids, %lld rows out of range", who,
              (long long)n_ids, (long long)row_count);
  RTP_REQUIRE(dtype == RTP_F32 || dtype == RTP_BF16, "%s: unknown dtype %d", who, dtype);
  RTP_REQUIRE(groups >= 1 && groups < 65536 && cols >= 0 && cols * groups < (1ll << 30) && ld_grad_out >= cols &&
                  ld_grad_table >= cols,
              "%s: bad shape", who);
  if (master != nullptr) {
    RTP_REQUIRE(!grad_table_f32 || dtype == RTP_F32, "%s: with an update the gradient table has the table's dtype", who);
    RTP_REQUIRE(dtype != RTP_F32 || weights == nullptr || weights == (void*)master, "%s: fp32 tables are their own master", who);
    RTP_REQUIRE(zero_fill || !store_grad, "%s: a stored gradient beside the update starts from a zero fill", who);
    if (!store_grad) zero_fill = 0;  // the update replaces the dense gradient: nothing to fill
    if (dtype == RTP_F32) weights = nullptr;
  } else {
    store_grad = 1;
  }
  if (cols == 0) return RTP_OK;
  RTP_REQUIRE((uintptr_t)workspace % 256 == 0, "%s: workspace must be 256-byte aligned", who);
  const GroupLayout L = group_layout(n_ids, row_count);
  if (workspace_bytes < L.total) return fail(RTP_ERR_WORKSPACE, "%s: workspace %zu < required %zu", who, workspace_bytes, L.total);
  char* w = (char*)workspace;
  int *offs = (int*)(w + L.offs), *pos = (int*)(w + L.pos), *nlong = (int*)(w + L.nlong), *longs = (int*)(w + L.longs);
  hipStream_t s = (hipStream_t)stream;
  const size_t esz = dtype == RTP_F32 ? 4 : 2, gsz = (dtype == RTP_F32 || grad_table_f32) ? 4 : 2;
  {
    ProfileScope prof(s, "embedding_group_ids", 0.0, 8.0 * (double)n_ids);
    hipLaunchKernelGGL(group_ids_kernel, dim3((unsigned)L.slices), dim3(kGroupThreads), 0, s, ids, (int)n_ids, (long)row_begin,
                       (int)row_count, (long)padding_idx, L.rows_per, offs, pos, nlong, longs, L.long_cap);
    RTP_LAUNCH_CHECK();
  }
  const int64_t vec = 16 / (int64_t)esz;
  const bool aligned = cols % vec == 0 && (uintptr_t)grad_out % 16 == 0 && (ld_grad_out * esz) % 16 == 0 &&
                       (grad_out_sg * esz) % 16 == 0 && (uintptr_t)grad_table % 16 == 0 &&
                       (ld_grad_table * gsz) % 16 == 0 && (grad_table_sg * gsz) % 16 == 0 &&
                       (master == nullptr || (uintptr_t)master % 16 == 0) &&
                       (weights == nullptr || (uintptr_t)weights % 16 == 0);
  const int64_t reach = ((n_ids - 1) * ld_grad_out + (groups - 1) * grad_out_sg + cols) * (int64_t)esz;
  const int plain = grad_scale == 1.0f && grad_out_sg >= 0 && reach < (1ll << 31) - 4;
  const int64_t chunks = ceil_div(cols * groups, 256), long_wgs = n_ids / kLongRow * chunks;
  RTP_REQUIRE(long_wgs + ceil_div(row_count, 4) < (1ll << 31), "%s: grid too large", who);
  const dim3 grid((unsigned)(long_wgs + ceil_div(row_count, 4)));
  const size_t lds = (size_t)ceil_div(ceil_div(n_ids, 32), 256) * 1024 + 8192 * 2;
  ProfileScope prof(s, "embedding_backward_grouped", (double)groups * n_ids * cols,
                    (double)groups * cols * ((double)n_ids * esz + (zero_fill ? (double)row_count : 2.0 * n_ids) * gsz));
#define RTP_EMB_GROUPED(T, G, V)                                                                                    \
  do {                                                                                                                \
    GroupedBwd<T, G> a{(const T*)grad_out, (long)ld_grad_out, (long)grad_out_sg, (G*)grad_table, (long)ld_grad_table,   \
                       (long)grad_table_sg, master, (T*)weights, grad_scale, lr, clip, scale_by_freq, zero_fill ? 1 : 0, \
                       store_grad, zero_fill, (int)n_ids, (int)row_count, (int)groups, (int)cols, offs, pos, nlong,      \
                       longs, L.slices, L.long_cap, plain};                                                                \
    hipLaunchKernelGGL((grouped_bwd_kernel<T, G, V>), grid, dim3(256), lds, s, a, (int)long_wgs, (int)chunks);      \
  } while (0)
  if (dtype == RTP_F32) {
    if (aligned) RTP_EMB_GROUPED(float, float, 4); else RTP_EMB_GROUPED(float, float, 1);
  } else if (grad_table_f32) {
    if (aligned) RTP_EMB_GROUPED(bf16_t, float, 8); else RTP_EMB_GROUPED(bf16_t, float, 1);
  } else {
    if (aligned) RTP_EMB_GROUPED(bf16_t, bf16_t, 8); else RTP_EMB_GROUPED(bf16_t, bf16_t, 1);
  }
#undef RTP_EMB_GROUPED
  RTP_LAUNCH_CHECK();
  return RTP_OK;
}
