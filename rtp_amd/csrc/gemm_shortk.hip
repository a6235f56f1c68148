// Products with a short contraction and many outputs: bound by the stores, not by the matrix cores.
#include "gemm_tile.h"

namespace rtp {

// The weight gradient of a wide layer over few rows (8192 x 8192 outputs, 32 rows) is all output: one or two K slabs a tile.  The
// kernels for long contractions run one workgroup a CU there, whose load, two MFMAs, transposition and stores follow each other: 2.2
// TB/s.  Here a workgroup of four waves has one slab in LDS, no pipeline, and 34 KB, so that four of them share a CU and one's stores
// run under the others' loads; after the products every wave brings its own 64 x 64 outputs through its own LDS, without a barrier.
// The sums are formed in the order of the other kernels, so the results are theirs bit for bit.  Three workgroups a CU (no
// spilled registers) are slower: 47 us instead of 39 on the first line.
// us in a replayed graph, 256 x 128 tiles -> this: bf16 8192 x 8192 x 32 60.2 -> 39.2, 4096 x 4096 x 32 16.3 -> 11.0, 4096 x 3072 x 32
// 16.6 -> 9.9; fp32 8192 x 8192 x 64 154 -> 107, 4096 x 4096 x 32 40.6 -> 36.3.
template <typename T, bool AKC, bool BKC>
__global__ __launch_bounds__(256, 4) void gemm_shortk_kernel(GemmArgs p) {
  constexpr int BM = 128, BN = 128, SB = 128;
  using DA = DmaOperand<T, BM, AKC, 4, SB>;
  using DB = DmaOperand<T, BN, BKC, 4, SB>;
  constexpr int BK = SB / (int)sizeof(T), KS = BK / (2 * DA::VEC);
  constexpr int STAGE = DA::BYTES + DB::BYTES, PART = 32 * (64 + 4) * 4;  // a wave's half of its outputs in fp32
  constexpr int LDS = STAGE > 4 * PART ? STAGE : 4 * PART;
  __shared__ __attribute__((aligned(1024))) char lds[LDS];

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 31, g = lane >> 5, wm = wave >> 1, wn = wave & 1;
  const int tile_m = (int)fast_div(blockIdx.x, p.d_tiles_n), tile_n = (int)(blockIdx.x - tile_m * p.d_tiles_n.d);
  const int m0 = tile_m * BM, n0 = tile_n * BN;
  const int grp = blockIdx.y / p.batch, zb = blockIdx.y % p.batch;
  const long zo = zb / p.zdiv, zi = zb % p.zdiv;
  const T* A = reinterpret_cast<const T*>(p.a) + grp * p.a_sg + zo * p.a_so + zi * p.a_si;
  const T* B = reinterpret_cast<const T*>(p.b) + grp * p.b_sg + zo * p.b_so + zi * p.b_si;

  DA da;
  DB db;
  da.init(p.lda, m0, p.m, wave, lane);
  db.init(p.ldb, n0, p.n, wave, lane);
  f32x16 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;
  float rs[2] = {0.0f, 0.0f};
  const bool rowsum = p.a_rowsum != nullptr && n0 == 0 && wn == 0;
  const unsigned lds0 = (unsigned)(uintptr_t)(lptr_t)lds;
  constexpr long SZ = (long)sizeof(T);
  for (int seg = 0; seg < p.ksegs; ++seg)
    for (int k0 = 0; k0 < p.k; k0 += BK) {
      const char* ca = DA::slab_base(A + seg * p.a_sk + (AKC ? (long)k0 : k0 * p.lda), p.lda, m0);
      const char* cb = DB::slab_base(B + seg * p.b_sk + (BKC ? (long)k0 : k0 * p.ldb), p.ldb, n0);
      if (seg + k0 > 0) __syncthreads();  // everyone has read the slab before
      if (k0 + BK <= p.k) {
        da.template issue<false>(lds0, wave, ca, 0, 0);
        db.template issue<false>(lds0 + DA::BYTES, wave, cb, 0, 0);
      } else {
        da.template issue<true>(lds0, wave, ca, k0, p.k);
        db.template issue<true>(lds0 + DA::BYTES, wave, cb, k0, p.k);
      }
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
#pragma unroll
      for (int q = 0; q < KS; ++q) {
        Frag<T> fa[2], fb[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          fa[i] = read_frag_dma<T, BM, AKC, SB>(lds, wm * 64 + i * 32, lane, q);
          fb[i] = read_frag_dma<T, BN, BKC, SB>(lds + DA::BYTES, wn * 64 + i * 32, lane, q);
        }
#pragma unroll
        for (int i = 0; i < 2; ++i) {
#pragma unroll
          for (int j = 0; j < 2; ++j) mma(fa[i], fb[j], acc[i][j]);
          if (rowsum) rs[i] = frag_sum(fa[i], rs[i]);
        }
      }
    }
  if (rowsum) {
    T* dst = reinterpret_cast<T*>(p.a_rowsum) + grp * p.rowsum_sg;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const float v = rs[i] + __shfl_xor(rs[i], 32, 64);
      const int row = m0 + wm * 64 + i * 32 + li;
      if (g == 0 && row < p.m) dst[row] = from_f32<T>((p.flags & RTP_GEMM_ROWSUM_ACCUM) ? to_f32(dst[row]) + v : v);
    }
  }
  __syncthreads();  // the slab's memory is free; from here every wave is on its own
  float* ct = reinterpret_cast<float*>(lds + wave * PART);
#pragma unroll
  for (int i = 0; i < 2; ++i) {
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) ct[(8 * (r >> 2) + 4 * g + (r & 3)) * 68 + j * 32 + li] = acc[i][j][r];
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    const int row0 = m0 + wm * 64 + i * 32, col0 = n0 + wn * 64;
    if (p.sgd_master != nullptr)
      finish_tile_sgd<T, 32, 64, 64>(p, ct, row0, col0, lane, grp, zo, zi);
    else
      finish_tile<T, 32, 64, 64>(p, ct, row0, col0, lane, grp, zo, zi);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  }
}

template <typename T>
static void launch_layouts(hipStream_t s, const GemmArgs& a, bool akc, bool bkc, dim3 grid) {
  if (akc && bkc)
    hipLaunchKernelGGL((gemm_shortk_kernel<T, true, true>), grid, dim3(256), 0, s, a);
  else if (akc)
    hipLaunchKernelGGL((gemm_shortk_kernel<T, true, false>), grid, dim3(256), 0, s, a);
  else if (bkc)
    hipLaunchKernelGGL((gemm_shortk_kernel<T, false, true>), grid, dim3(256), 0, s, a);
  else
    hipLaunchKernelGGL((gemm_shortk_kernel<T, false, false>), grid, dim3(256), 0, s, a);
}

int launch_shortk(hipStream_t s, const GemmArgs& a, bool bf16, bool akc, bool bkc, dim3 grid) {
  if (bf16)
    launch_layouts<bf16_t>(s, a, akc, bkc, grid);
  else
    launch_layouts<float>(s, a, akc, bkc, grid);
  RTP_LAUNCH_CHECK();
  return RTP_OK;
}

}  // namespace rtp
