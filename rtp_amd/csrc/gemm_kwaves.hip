// Products with few output tiles and a long contraction, the contraction split over the waves of a workgroup.
#include "gemm_tile.h"

namespace rtp {

// A product of few tiles is a serial chain of K slabs in each of a few workgroups: 64 x 4096 outputs over K = 4096 are 64 tiles of
// 64 x 64, 64 busy CUs and 64 slabs of 167 ns one behind the other, at 1.8 TB/s of weights.  Here a workgroup owns 32 x 32 outputs and its
// eight waves an eighth of the contraction each.  A wave streams the slabs of its own part into LDS that nobody else touches --
// one slab in flight while one is multiplied, 64 KB in flight per CU, no barrier in the loop -- and the eight partial sums meet in
// LDS once, added in wave order; then the epilogue of the other kernels.  Bound by the loads' latency and, from some hundred
// workgroups on, by memory (bf16), by the fp32 MFMAs (fp32, exact products: 256 flops a clock and CU).  Slabs of 64 bytes a row, four
// stages, instead of 128 and two: the same on row-contiguous operands, 14 -> 19 us on 64 x 2048 x 8192 in bf16.
// us in a replayed graph on operands that are not in the caches, 64 x 64 tiles -> this: bf16 64 x 1024 x 1024 7.0 -> 4.9, 32 x 4096 x 4096
// 18.9 -> 9.9, 32 x 1024 x 8192 31.1 -> 13.9, input gradient 64 x 4096 x 4096 19.5 -> 14.7; fp32 (split tiles before) 64 x 1024 x 1024
// 18.4 -> 8.7, 64 x 4096 x 4096 57.7 -> 26.7.  Eight short sums: error against fp64 below that of one long one.
//
// MT = 2: tiles of 64 x 32, slabs of 64 bytes a row and three stages, where 32 x 32 would be two workgroups a CU (fp32 256 x 2048 x 512
// 13.1 -> 11.0 us, 100 x 3072 x 384 10.5 -> 8.2; bf16 100 x 3072 x 8192 32.6 -> 27.3, weight gradient 250 x 2048 x 4096 37.6 -> 24.5).
// REG: operands of any alignment, through registers into the wave's LDS, three slabs ahead (bf16 255 x 1023 x 3333 24.0 -> 17.6 us,
// 64 x 1001 x 2048 10.7 -> 7.8, its weight gradient 22.5 -> 14.4; fp32 255 x 1023 x 3333 65.6 -> 28.5, 1 x 1303 x 1364 29.4 -> 11.7); RAG: the epilogue for any alignment
// (an output, addend or mask that is not vector-aligned).
template <typename T, int MT, bool AKC, bool BKC, bool REG, bool RAG>
__global__ __launch_bounds__(512) void gemm_kwaves_kernel(GemmArgs p) {
  constexpr int BM = 32 * MT, SB = MT == 1 ? 128 : 64, NST = MT == 1 ? 2 : 3;  // bytes of a slab's row, stages per wave
  using DA = DmaOperand<T, BM, AKC, 1, SB>;
  using DB = DmaOperand<T, 32, BKC, 1, SB>;
  constexpr int WAVES = 8, BK = SB / (int)sizeof(T), KS = BK / (2 * DA::VEC);
  constexpr int STAGE = DA::BYTES + DB::BYTES, NI = DA::NI + DB::NI;
  constexpr int PITCH = 33, PART = WAVES * BM * PITCH * 4;
  static_assert((NST - 1) * NI < 64, "vmcnt is a 6-bit counter");
  static_assert(WAVES * NST * STAGE <= 160 * 1024 && PART + BM * 36 * 4 + WAVES * BM * 4 <= WAVES * NST * STAGE,
                "160 KiB of LDS; the sums reuse the slabs' memory");
  __shared__ __attribute__((aligned(1024))) char lds[WAVES * NST * STAGE];

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 31, g = lane >> 5;
  // the row tiles of a column tile, and column tiles that share memory lines, on one XCD
  unsigned bid = blockIdx.x;
  const unsigned nb = gridDim.x;
  if ((nb & 7) == 0) bid = (bid & 7) * (nb >> 3) + (bid >> 3);
  const int n0 = (int)(bid / (unsigned)p.tiles_m) * 32, m0 = (int)(bid % (unsigned)p.tiles_m) * BM;
  const int grp = blockIdx.y / p.batch, zb = blockIdx.y % p.batch;
  const long zo = zb / p.zdiv, zi = zb % p.zdiv;

  const T* A = reinterpret_cast<const T*>(p.a) + grp * p.a_sg + zo * p.a_so + zi * p.a_si;
  const T* B = reinterpret_cast<const T*>(p.b) + grp * p.b_sg + zo * p.b_so + zi * p.b_si;
  const int nk_seg = (p.k + BK - 1) / BK, nk = nk_seg * p.ksegs;
  const int per = (nk + WAVES - 1) / WAVES;
  const int first = min(wave * per, nk), n = min(per, nk - first);

  constexpr long SZ = (long)sizeof(T);
  const long step_a = (AKC ? (long)BK : (long)BK * p.lda) * SZ, step_b = (BKC ? (long)BK : (long)BK * p.ldb) * SZ;
  const long last_a = step_a + p.a_sk * SZ - nk_seg * step_a, last_b = step_b + p.b_sk * SZ - nk_seg * step_b;
  const int seg = first / nk_seg, in_seg = first - seg * nk_seg;
  char* const mine = lds + wave * (NST * STAGE);

  f32x16 acc[MT];
  float rs[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    rs[t] = 0.0f;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[t][r] = 0.0f;
  }
  const bool rowsum = p.a_rowsum != nullptr && n0 == 0;
  Frag<T> fa[MT][KS], fb[KS];
  auto read = [&](int stage) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < KS; ++q) {
#pragma unroll
      for (int t = 0; t < MT; ++t) fa[t][q] = read_frag_dma<T, BM, AKC, SB>(mine + stage * STAGE, 32 * t, lane, q);
      fb[q] = read_frag_dma<T, 32, BKC, SB>(mine + stage * STAGE + DA::BYTES, 0, lane, q);
    }
    // the stage is free when its reads have returned
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  auto multiply = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < KS; ++q) {
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        mma(fa[t][q], fb[q], acc[t]);
        if (rowsum) rs[t] = frag_sum(fa[t][q], rs[t]);
      }
    }
  };

  if constexpr (REG) {
    // slabs behind the wave's last one re-read it, so that the loop has no branch around a request
    RegOperand<T, BM, AKC, 1, SB> ra;
    RegOperand<T, 32, BKC, 1, SB> rb;
    ra.init(A, p.lda, m0, p.m, 0, lane);
    rb.init(B, p.ldb, n0, p.n, 0, lane);
    struct Place {
      int seg, k0, i;
    };
    Place f{seg, in_seg * BK, 0}, w = f;  // the next slab to request and to write
    auto next = [&](Place& at) __attribute__((always_inline)) {
      if (++at.i >= n) return;
      at.k0 += BK;
      if (at.k0 >= p.k) at.k0 = 0, ++at.seg;
    };
    auto fetch = [&](auto S) __attribute__((always_inline)) {
      ra.template fetch<decltype(S)::value>(f.seg * p.a_sk * SZ, f.k0, p.k);
      rb.template fetch<decltype(S)::value>(f.seg * p.b_sk * SZ, f.k0, p.k);
      next(f);
      asm volatile("" ::: "memory");  // requests stay in this order
      __builtin_amdgcn_sched_barrier(0);
    };
    auto slab = [&](auto S) __attribute__((always_inline)) {
      ra.template store<decltype(S)::value>(mine, 0, lane, w.k0, p.k);
      rb.template store<decltype(S)::value>(mine + DA::BYTES, 0, lane, w.k0, p.k);
      next(w);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      read(0);
      fetch(S);
      multiply();
    };
    constexpr auto ring = std::make_integer_sequence<int, kRegDepth>{};
    if (n > 0) {
      [&]<int... S>(std::integer_sequence<int, S...>) { (fetch(std::integral_constant<int, S>{}), ...); }(ring);
      int i = 0;
      for (; i + kRegDepth <= n; i += kRegDepth)
        [&]<int... S>(std::integer_sequence<int, S...>) { (slab(std::integral_constant<int, S>{}), ...); }(ring);
      [&]<int... S>(std::integer_sequence<int, S...>) {
        ((i + S < n ? slab(std::integral_constant<int, S>{}) : (void)0), ...);
      }(ring);
    }
  } else {
    DA da;
    DB db;
    da.init(p.lda, m0, p.m, 0, lane);
    db.init(p.ldb, n0, p.n, 0, lane);
    const char* ca = DA::slab_base(A, p.lda, m0) + seg * p.a_sk * SZ + in_seg * step_a;
    const char* cb = DB::slab_base(B, p.ldb, n0) + seg * p.b_sk * SZ + in_seg * step_b;
    int left = nk_seg - in_seg;  // slabs left in the K segment, the next one included
    const bool tail = p.k % BK != 0;
    const unsigned lds_mine = (unsigned)(uintptr_t)(lptr_t)lds + (unsigned)(wave * (NST * STAGE));
    auto issue = [&](int stage) __attribute__((always_inline)) {
      const unsigned at = lds_mine + (unsigned)(stage * STAGE);
      if (left != 1 || !tail) {
        da.template issue<false>(at, 0, ca, 0, 0);
        db.template issue<false>(at + DA::BYTES, 0, cb, 0, 0);
      } else {
        da.template issue<true>(at, 0, ca, (nk_seg - 1) * BK, p.k);
        db.template issue<true>(at + DA::BYTES, 0, cb, (nk_seg - 1) * BK, p.k);
      }
      const bool more = left != 1;
      ca += more ? step_a : last_a;
      cb += more ? step_b : last_b;
      left = more ? left - 1 : nk_seg;
    };
#pragma unroll
    for (int s = 0; s < NST; ++s)
      if (s < n) issue(s);
    int i = 0;
    for (; i + 2 * NST <= n; i += NST)
#pragma unroll
      for (int s = 0; s < NST; ++s) {
        asm volatile("s_waitcnt vmcnt(%0)" : : "n"((NST - 1) * NI) : "memory");
        read(s);
        issue(s);
        multiply();
      }
    for (int s = 0; i < n; ++i) {
      if (i + NST <= n)
        asm volatile("s_waitcnt vmcnt(%0)" : : "n"((NST - 1) * NI) : "memory");
      else
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      read(s);
      if (i + NST < n) issue(s);
      multiply();
      s = s + 1 == NST ? 0 : s + 1;
    }
  }

  __syncthreads();  // nobody reads slabs any more, and no load is on its way
  float(*part)[BM][PITCH] = reinterpret_cast<float(*)[BM][PITCH]>(lds);
  float* ct = reinterpret_cast<float*>(lds + PART);
  float* sums = ct + BM * 36;
#pragma unroll
  for (int t = 0; t < MT; ++t) {
#pragma unroll
    for (int r = 0; r < 16; ++r) part[wave][32 * t + 8 * (r >> 2) + 4 * g + (r & 3)][li] = acc[t][r];
    const float both = rs[t] + __shfl_xor(rs[t], 32, kWave);
    if (g == 0) sums[wave * BM + 32 * t + li] = both;
  }
  __syncthreads();
#pragma unroll
  for (int e = 0; e < 2 * MT; ++e) {
    const int row = (tid >> 5) + 16 * e;
    float v = 0.0f;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) v += part[w][row][li];
    ct[row * 36 + li] = v;
  }
  if (rowsum && tid < BM && m0 + tid < p.m) {
    float v = 0.0f;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) v += sums[w * BM + tid];
    T* dst = reinterpret_cast<T*>(p.a_rowsum) + grp * p.rowsum_sg + m0 + tid;
    *dst = from_f32<T>((p.flags & RTP_GEMM_ROWSUM_ACCUM) ? to_f32(*dst) + v : v);
  }
  __syncthreads();
  if (tid >= 128 * MT) return;  // a thread finishes eight outputs
  if (RAG && !(REG && p.vec_c))
    finish_tile_ragged<T, BM, 32, 128 * MT>(p, ct, m0, n0, tid, grp, zo, zi);
  else if (p.sgd_master != nullptr)
    finish_tile_sgd<T, BM, 32, 128 * MT>(p, ct, m0, n0, tid, grp, zo, zi);
  else
    finish_tile<T, BM, 32, 128 * MT>(p, ct, m0, n0, tid, grp, zo, zi);
}

template <typename T, int MT, bool REG, bool RAG>
static void launch_layouts(hipStream_t s, const GemmArgs& a, bool akc, bool bkc, dim3 grid) {
  if (akc && bkc)
    hipLaunchKernelGGL((gemm_kwaves_kernel<T, MT, true, true, REG, RAG>), grid, dim3(512), 0, s, a);
  else if (akc)
    hipLaunchKernelGGL((gemm_kwaves_kernel<T, MT, true, false, REG, RAG>), grid, dim3(512), 0, s, a);
  else if (bkc)
    hipLaunchKernelGGL((gemm_kwaves_kernel<T, MT, false, true, REG, RAG>), grid, dim3(512), 0, s, a);
  else
    hipLaunchKernelGGL((gemm_kwaves_kernel<T, MT, false, false, REG, RAG>), grid, dim3(512), 0, s, a);
}
template <typename T, int MT>
static void launch_kind(hipStream_t s, const GemmArgs& a, bool akc, bool bkc, bool direct, dim3 grid) {
  if (!direct)
    launch_layouts<T, MT, true, true>(s, a, akc, bkc, grid);
  else if (!a.vec_c)
    launch_layouts<T, MT, false, true>(s, a, akc, bkc, grid);
  else
    launch_layouts<T, MT, false, false>(s, a, akc, bkc, grid);
}

int launch_kwaves(hipStream_t s, const GemmArgs& a, int bm, bool bf16, bool akc, bool bkc, bool direct, dim3 grid) {
  if (bf16 && bm == 32)
    launch_kind<bf16_t, 1>(s, a, akc, bkc, direct, grid);
  else if (bf16)
    launch_kind<bf16_t, 2>(s, a, akc, bkc, direct, grid);
  else if (bm == 32)
    launch_kind<float, 1>(s, a, akc, bkc, direct, grid);
  else
    launch_kind<float, 2>(s, a, akc, bkc, direct, grid);
  RTP_LAUNCH_CHECK();
  return RTP_OK;
}

}  // namespace rtp
