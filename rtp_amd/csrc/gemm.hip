// LDS-staged MFMA GEMM for gfx950 (fp32 via v_mfma_f32_32x32x2_f32, long contractions in gemm_split.hip; bf16 via
// v_mfma_f32_32x32x16_bf16)
// with the four operand layouts the rotated layers need (forward X W^T, input gradient dY W, weight
// gradient dY^T X, batched q k^T / p v), a fused epilogue (accumulate, bias, ReLU, ReLU-mask), and two
// ways of covering several rotation shards in ONE launch:
//   groups     : independent problems that differ only by a constant pointer stride per operand
//                (shard s of a column-parallel layer: W_s, b_s and the output column block s);
//   K segments : one output whose contraction runs over several shards in turn
//                (row-parallel outputs, input gradients of column-parallel layers: sum_s dY_s W_s),
//                accumulated in the MFMA accumulators, so the cross-shard sum never leaves registers.
//
// Work decomposition: 256 threads = 4 wavefronts in a 2x2 arrangement over a BM x BN output tile;
// each wavefront owns (BM/2)x(BN/2) as 32x32 MFMA blocks with fp32 accumulators in VGPRs.  The K loop
// moves 128-byte-per-row slabs (64 bf16 / 32 fp32 values of k) global -> registers -> LDS.  LDS is
// double buffered (one barrier per slab) and the global loads run DEPTH slabs ahead of the MFMAs in a
// ring of register buffers, which is what hides HBM/L2 latency when only one workgroup fits a CU.
#include "gemm_tile.h"

#include <algorithm>
#include <atomic>
#include <cstdlib>
#include <type_traits>

namespace rtp {

constexpr int kThreads = 256;
constexpr int kSlabBytes = 128;               // bytes of k per tile row and slab
constexpr int kRowPitchKC = kSlabBytes + 16;  // LDS row pitch when k is contiguous (16 B pad)

// Moves one R x BK operand slab global -> registers -> LDS.
//   KC  (k contiguous in memory): LDS holds [row][k], row pitch 144 bytes.
//   !KC (rows contiguous in memory): LDS holds [k][row], k pitch R*sizeof(T)+16 bytes.
template <typename T, int R, bool KC>
struct Slab {
  static constexpr int VEC = 16 / sizeof(T);
  static constexpr int BK = kSlabBytes / sizeof(T);
  static constexpr int KV = BK / VEC;           // 16-byte vectors per row (= 8)
  static constexpr int NV = R * KV / kThreads;  // vectors per thread
  static constexpr int RV = R / VEC;            // vectors per k line when rows are contiguous
  static constexpr int PITCH = KC ? kRowPitchKC : (R * (int)sizeof(T) + 16);
  static constexpr int BYTES = KC ? R * kRowPitchKC : BK * PITCH;
  uint4 reg[NV];

  // FAST: every 16-byte vector of the slab is either wholly inside the operand or wholly outside it
  // (guaranteed by the host: aligned pointers and strides, extents that are multiples of VEC), so a
  // vector is loaded unconditionally from a clamped address; vectors beyond the contraction length are
  // replaced by zeros later, when the registers are moved to LDS (store with ktail), so nothing here
  // consumes a load result and all loads of a slab stay in flight.  Rows beyond the operand are clamped
  // too: they only feed accumulators the epilogue never stores.
  // !FAST: element-wise guarded loads for ragged or unaligned operands.
  template <bool FAST>
  __device__ __forceinline__ void load(const T* base, long ld, int row0, int rows, int k0, int kdim, int tid) {
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int v = tid + i * kThreads;
      union {
        uint4 q;
        T e[VEC];
      } u;
      if (KC) {
        const int row = row0 + v / KV;
        const int k = k0 + (v % KV) * VEC;
        if (FAST) {
          const int rc = row < rows ? row : rows - 1;
          const int kc = k < kdim ? k : 0;
          u.q = *reinterpret_cast<const uint4*>(base + (long)rc * ld + kc);
        } else {
          const T* src = base + (long)row * ld + k;
#pragma unroll
          for (int e = 0; e < VEC; ++e) u.e[e] = (row < rows && k + e < kdim) ? src[e] : (T)0.0f;
        }
      } else {
        const int k = k0 + v / RV;
        const int row = row0 + (v % RV) * VEC;
        if (FAST) {
          const int kc = k < kdim ? k : 0;
          const int rc = row < rows ? row : 0;
          u.q = *reinterpret_cast<const uint4*>(base + (long)kc * ld + rc);
        } else {
          const T* src = base + (long)k * ld + row;
#pragma unroll
          for (int e = 0; e < VEC; ++e) u.e[e] = (k < kdim && row + e < rows) ? src[e] : (T)0.0f;
        }
      }
      reg[i] = u.q;
    }
  }

  // ktail: the slab that starts at k0 reaches beyond kdim, zero the vectors that lie outside.
  __device__ __forceinline__ void store(char* lds, int tid, bool ktail, int k0, int kdim) const {
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int v = tid + i * kThreads;
      char* dst = KC ? lds + (v / KV) * kRowPitchKC + (v % KV) * 16 : lds + (v / RV) * PITCH + (v % RV) * 16;
      uint4 q = reg[i];
      if (ktail) {
        const int k = KC ? k0 + (v % KV) * VEC : k0 + v / RV;
        const bool live = k < kdim;
        q.x = live ? q.x : 0u;
        q.y = live ? q.y : 0u;
        q.z = live ? q.z : 0u;
        q.w = live ? q.w : 0u;
      }
      *reinterpret_cast<uint4*>(dst) = q;
    }
  }
};

// Lane (li = lane%32, g = lane/32) reads row `row` of the slab, k = (2*ks + g)*VEC .. +VEC-1.
template <typename T, int R, bool KC>
__device__ __forceinline__ Frag<T> read_frag(const char* lds, int row, int ks, int g) {
  constexpr int VEC = 16 / sizeof(T);
  constexpr int PITCH = Slab<T, R, KC>::PITCH;
  union {
    uint4 q;
    T e[VEC];
    Frag<T> f;
  } u;
  if (KC) {
    u.q = *reinterpret_cast<const uint4*>(lds + row * kRowPitchKC + (2 * ks + g) * 16);
  } else {
    const char* p = lds + (2 * ks + g) * VEC * PITCH + row * (int)sizeof(T);
#pragma unroll
    for (int e = 0; e < VEC; ++e) u.e[e] = *reinterpret_cast<const T*>(p + e * PITCH);
  }
  return u.f;
}

template <typename T, int BM, int BN, bool AKC, bool BKC, int DEPTH, bool FAST>
struct GemmTile {
  using LA = Slab<T, BM, AKC>;
  using LB = Slab<T, BN, BKC>;
  static constexpr int BK = LA::BK;
  static constexpr int WM = BM / 2, WN = BN / 2, MT = WM / 32, NT = WN / 32;
  static constexpr int STAGE = LA::BYTES + LB::BYTES;
  static constexpr int KSTEPS = 4;  // slab k extent / (2*VEC)

  const GemmArgs& p;
  const T* A;
  const T* B;
  int m0, n0, tid, nk_seg;
  LA la[DEPTH];
  LB lb[DEPTH];

  __device__ __forceinline__ GemmTile(const GemmArgs& args) : p(args) {}

  template <int R>
  __device__ __forceinline__ void fetch(int slab) {
    const int seg = slab / nk_seg;
    const int k0 = (slab - seg * nk_seg) * BK;
    la[R].template load<FAST>(A + seg * p.a_sk, p.lda, m0, p.m, k0, p.k, tid);
    lb[R].template load<FAST>(B + seg * p.b_sk, p.ldb, n0, p.n, k0, p.k, tid);
  }
  // `slab` is the slab held by register slot R; only the last slab of a K segment can be partial.
  template <int R>
  __device__ __forceinline__ void stash(char* stage, int slab) {
    const int seg = slab / nk_seg;
    const int k0 = (slab - seg * nk_seg) * BK;
    const bool ktail = FAST && k0 + BK > p.k;
    la[R].store(stage, tid, ktail, k0, p.k);
    lb[R].store(stage + LA::BYTES, tid, ktail, k0, p.k);
  }
};

template <typename T, int BM, int BN, bool AKC, bool BKC, int DEPTH, bool FAST>
__global__ __launch_bounds__(kThreads) void gemm_kernel(GemmArgs p) {
  using G = GemmTile<T, BM, BN, AKC, BKC, DEPTH, FAST>;
  constexpr int MT = G::MT, NT = G::NT, WM = G::WM, WN = G::WN, STAGE = G::STAGE;
  __shared__ __attribute__((aligned(16))) char lds[2 * STAGE];

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int li = lane & 31, g = lane >> 5;

  // Consecutive workgroup ids land on different XCDs (round robin over 8); give each XCD a
  // contiguous run of output tiles so its L2 sees neighbouring tiles that share operand rows.
  int bid = blockIdx.x;
  const int nb = p.tiles_m * p.tiles_n;
  if ((nb & 7) == 0) bid = (bid & 7) * (nb >> 3) + (bid >> 3);

  const int grp = blockIdx.y / p.batch, zb = blockIdx.y % p.batch;
  const long zo = zb / p.zdiv, zi = zb % p.zdiv;

  G t(p);
  t.tid = tid;
  t.m0 = (bid / p.tiles_n) * BM;
  t.n0 = (bid % p.tiles_n) * BN;
  t.A = reinterpret_cast<const T*>(p.a) + grp * p.a_sg + zo * p.a_so + zi * p.a_si;
  t.B = reinterpret_cast<const T*>(p.b) + grp * p.b_sg + zo * p.b_so + zi * p.b_si;
  t.nk_seg = (p.k + G::BK - 1) / G::BK;
  const int nk = t.nk_seg * p.ksegs;

  f32x16 acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

  // Prologue: slabs 0..DEPTH-1 into the register ring, slab 0 on into LDS stage 0.
  if (nk > 0) t.template fetch<0>(0);
  if (DEPTH > 1 && nk > 1) t.template fetch<1 % DEPTH>(1);
  if (DEPTH > 2 && nk > 2) t.template fetch<2 % DEPTH>(2);
  if (nk > 0) t.template stash<0>(lds, 0);
  __syncthreads();

  auto compute = [&](int kt) {
    const char* sa = lds + (kt & 1) * STAGE;
    const char* sb = sa + G::LA::BYTES;
#pragma unroll
    for (int ks = 0; ks < G::KSTEPS; ++ks) {
      Frag<T> fa[MT], fb[NT];
#pragma unroll
      for (int i = 0; i < MT; ++i) fa[i] = read_frag<T, BM, AKC>(sa, wm * WM + i * 32 + li, ks, g);
#pragma unroll
      for (int j = 0; j < NT; ++j) fb[j] = read_frag<T, BN, BKC>(sb, wn * WN + j * 32 + li, ks, g);
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) mma(fa[i], fb[j], acc[i][j]);
    }
  };

  // Steady state for slab kt (register slot kt % DEPTH was just emptied into LDS): refill that slot
  // with slab kt+DEPTH, run the MFMAs of slab kt from LDS stage kt&1, move slab kt+1 from its register
  // slot to the other LDS stage, barrier.  While 2*DEPTH slabs remain none of this needs a guard, so the
  // loop body is branch-free and the loads of DEPTH slabs stay in flight across the barriers.
  int kt = 0;
  for (; kt + 2 * DEPTH <= nk; kt += DEPTH) {
    t.template fetch<0>(kt + DEPTH);
    compute(kt);
    t.template stash<1 % DEPTH>(lds + ((kt + 1) & 1) * STAGE, kt + 1);
    __syncthreads();
    if (DEPTH > 1) {
      t.template fetch<1 % DEPTH>(kt + 1 + DEPTH);
      compute(kt + 1);
      t.template stash<2 % DEPTH>(lds + ((kt + 2) & 1) * STAGE, kt + 2);
      __syncthreads();
    }
    if (DEPTH > 2) {
      t.template fetch<2 % DEPTH>(kt + 2 + DEPTH);
      compute(kt + 2);
      t.template stash<0>(lds + ((kt + 3) & 1) * STAGE, kt + 3);
      __syncthreads();
    }
  }
  // Drain: the same phases with guards (kt is a multiple of DEPTH, so the slot assignment continues).
  for (; kt < nk; kt += DEPTH) {
    if (kt + DEPTH < nk) t.template fetch<0>(kt + DEPTH);
    compute(kt);
    if (kt + 1 < nk) t.template stash<1 % DEPTH>(lds + ((kt + 1) & 1) * STAGE, kt + 1);
    __syncthreads();
    if (DEPTH > 1) {
      if (kt + 1 >= nk) break;
      if (kt + 1 + DEPTH < nk) t.template fetch<1 % DEPTH>(kt + 1 + DEPTH);
      compute(kt + 1);
      if (kt + 2 < nk) t.template stash<2 % DEPTH>(lds + ((kt + 2) & 1) * STAGE, kt + 2);
      __syncthreads();
    }
    if (DEPTH > 2) {
      if (kt + 2 >= nk) break;
      if (kt + 2 + DEPTH < nk) t.template fetch<2 % DEPTH>(kt + 2 + DEPTH);
      compute(kt + 2);
      if (kt + 3 < nk) t.template stash<0>(lds + ((kt + 3) & 1) * STAGE, kt + 3);
      __syncthreads();
    }
  }

  store_tile<T, MT, NT, WM, WN>(p, acc, t.m0, t.n0, wm, wn, li, g, grp, zo, zi);
}

// The body of the product kernel: workgroup `id` of the `nwg` that work on the problem `p` (`bx`, `by`: its
// coordinates in a launch that does not use XCD bricks).  `p` lives in the kernel-argument segment.
// REG: the loader waves go through registers (RegOperand) instead of loading straight into LDS.  RAG: the epilogue's operands
// may be unaligned; kernels of their own, since a second epilogue inside every kernel cost the others registers
// and code (1 % of the LM attention's time).
template <typename T, int BM, int BN, bool AKC, bool BKC, int NSTAGE, int SB, int PD, bool REG, bool RAG>
__device__ __forceinline__ void gemm_dma_body(const GemmArgs& p, const unsigned id, const unsigned bx, const unsigned by,
                                              const unsigned nwg) {
  constexpr int NL = 4;  // loader waves (waves 4..7); waves 0..3 compute
  using DA = DmaOperand<T, BM, AKC, NL, SB>;
  using DB = DmaOperand<T, BN, BKC, NL, SB>;
  constexpr int BK = SB / sizeof(T);
  constexpr int KS = SB / 32;  // MFMA k-steps per slab
  // the four MFMA waves form a 2 x 2 grid of wave tiles, or 4 x 1 where half the tile's columns are no whole number
  // of 32-column MFMA blocks (BN = 160)
  constexpr int WGM = (BN / 2) % 32 == 0 ? 2 : 4, WGN = 4 / WGM;
  constexpr int WM = BM / WGM, WN = BN / WGN, MT = WM / 32, NT = WN / 32;
  static_assert(WM % 32 == 0 && WN % 32 == 0, "wave tiles are whole 32 x 32 MFMA blocks");
  constexpr int STAGE = DA::BYTES + DB::BYTES;
  constexpr int NI = DA::NI + DB::NI;  // loads per loader wave and slab
  static_assert((NSTAGE - 2) * NI < 64, "vmcnt is a 6-bit counter");
  static_assert(NSTAGE >= 3, "at least 3 LDS stages");
  static_assert(NSTAGE * STAGE + 1024 <= 160 * 1024, "160 KiB of LDS per workgroup");
  static_assert(BM * (BN + 4) * 4 <= NSTAGE * STAGE, "the epilogue stages the fp32 tile in the slab memory");
  // Stage addresses are compile-time offsets into one array, so LDS reads carry immediate offsets.  The last KiB
  // is where the loads of WarmAhead land.
  __shared__ __attribute__((aligned(1024))) char lds[NSTAGE * STAGE + 1024];

  const int tid = threadIdx.x;
  unsigned long long t_start = 0, t_ready = 0, t_loop = 0;  // phase stamps of thread 0 (an MFMA wave), mode 2 only
  if (p.trace != nullptr && tid == 0) {
    t_start = (unsigned long long)wall_clock64();
    atomicMin(p.trace, t_start);
  }
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = WGM == 2 ? (wave >> 1) & 1 : wave & 3, wn = WGM == 2 ? wave & 1 : 0;
  const int li = lane & 31, g = lane >> 5;

  // Workgroups are handed to the 8 XCDs round-robin in launch order, and every XCD has its own L2.  The
  // host splits the (batch*groups, tiles_m, tiles_n) space into 8 bricks (xg * xm * xn == 8) chosen so that
  // the operand rows one XCD touches are as few as possible; workgroup `id` works on brick id % 8.
  // Both mappings are computed and one is selected, without a branch: every kernel argument is then fetched by
  // one batch of scalar loads at entry instead of three dependent rounds (each a trip to memory on a cold cache).
  const unsigned xcd = id & 7, slot = id >> 3;
  // The ~32 workgroups an XCD runs at a time should cover a compact block of the brick, not a row of it: they
  // share the XCD's L2, and a 4 x 8 block of tiles reads 12 tile-operands where a 1 x 32 row reads 33.  Over the
  // rounds of a long launch the panels walk down a strip of pcol tile columns, whose B operand stays in the L2
  // while the A rows stream past once per strip.
  const unsigned zl = fast_div(slot, p.d_brick);  // entry of the batch*groups axis inside the brick
  const unsigned t = slot - zl * p.d_brick.d;      // tile inside the mbk x nbk brick
  const unsigned q = fast_div(t, p.d_panel), r = t - q * p.d_panel.d;  // panel, tile inside the panel
  const unsigned cn = fast_div(r, p.d_prow), cm = r - cn * p.d_prow.d;
  const unsigned qn = fast_div(q, p.d_pm), qm = q - qn * p.d_pm.d;     // strip, panel inside the strip
  const int tile_n_x = (int)((xcd & ((1u << p.xn_shift) - 1)) * p.nbk + qn * p.pcol + cn);
  const int tile_m_x = (int)(((xcd >> p.xn_shift) & ((1u << p.xm_shift) - 1)) * p.mbk + qm * p.prow + cm);
  const int z_x = (int)((xcd >> (p.xn_shift + p.xm_shift)) * p.zbk + zl);
  const int tile_m_p = (int)fast_div(bx, p.d_tiles_n);
  const int tile_n_p = (int)(bx - tile_m_p * p.d_tiles_n.d);
  const bool bricks = p.xg != 0;
  const int tile_m = bricks ? tile_m_x : tile_m_p, tile_n = bricks ? tile_n_x : tile_n_p;
  const int z = bricks ? z_x : (int)by;
  const int m0 = tile_m * BM;
  const int n0 = tile_n * BN;
  const int grp = (int)fast_div(z, p.d_batch), zb = z - grp * (int)p.d_batch.d;
  const long zo = fast_div(zb, p.d_zdiv), zi = zb - (int)zo * (int)p.d_zdiv.d;
  const int nk_seg = (p.k + BK - 1) / BK;
  const int nk = nk_seg * p.ksegs;

  f32x16 acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

  // Row sums of A: bf16 even and odd k-steps apart, which is the order in which the 256 x 256 kernel's fragments add up.  Both wave columns hold the same
  // rows; in the 256 x 128 tile, whose registers don't hold twice the sums of four blocks, each takes two of them (5085 x 1280 x 5120 as a weight
  // gradient, with or without sums, 108 us where one took all and the loop spilled, 88 so; smaller tiles lose by a second branch).
  constexpr int NSUM = sizeof(T) == 2 && !AKC ? 2 : 1;
  constexpr bool SHARED_SUMS = NSUM == 2 && WGN == 2 && MT == 4;
  constexpr int MS = SHARED_SUMS ? MT / 2 : MT;  // blocks whose rows a wave sums
  float rsum[MS][NSUM];
#pragma unroll
  for (int i = 0; i < MS; ++i)
#pragma unroll
    for (int c = 0; c < NSUM; ++c) rsum[i][c] = 0.0f;

  // Barrier protocol: both paths meet the same nk barriers.  Barrier k is passed when slab k is visible to
  // every wave: a loader reaches it only after its own loads of slab k have landed.  A compute wave reaches
  // barrier k+1 after the MFMAs that consumed the last fragments of slab k-1, so once barrier k+1 is passed
  // the loaders may refill the stage of slab k-1 (with slab k-1+NSTAGE).
  if (wave >= 4) {
    // ---- loader waves: issue slabs strictly in order, NSTAGE-1 ahead of the slab being consumed ----
    const int lw = wave - 4;
    const T* A = reinterpret_cast<const T*>(p.a) + grp * p.a_sg + zo * p.a_so + zi * p.a_si;
    const T* B = reinterpret_cast<const T*>(p.b) + grp * p.b_sg + zo * p.b_so + zi * p.b_si;
    if constexpr (REG) {
      // slab k+1 is written before barrier k+1 -- the stage it takes held slab k+1-NSTAGE, whose last reader passed barrier
      // k+3-NSTAGE -- and slab k+1+kRegDepth requested into its registers.  Slabs behind the last one re-read it, so
      // that the number of loads in flight is known at every wait.
      RegOperand<T, BM, AKC, NL, SB> ra;
      RegOperand<T, BN, BKC, NL, SB> rb;
      ra.init(A, p.lda, m0, p.m, lw, lane);
      rb.init(B, p.ldb, n0, p.n, lw, lane);
      int fs = 0, fk = 0, ws = 0, wk = 0;  // segment and k of the next slab to request and to write
      auto next = [&](int& seg, int& k0) {
        k0 += BK;
        if (k0 < p.k) return;
        if (seg + 1 < p.ksegs) {
          ++seg;
          k0 = 0;
        } else {
          k0 -= BK;
        }
      };
      auto fetch = [&](auto S) {
        ra.template fetch<decltype(S)::value>(fs * p.a_sk * (long)sizeof(T), fk, p.k);
        rb.template fetch<decltype(S)::value>(fs * p.b_sk * (long)sizeof(T), fk, p.k);
        next(fs, fk);
        asm volatile("" ::: "memory");  // requests stay in this order: the waits count them
        __builtin_amdgcn_sched_barrier(0);
      };
      int stage = 0;
      auto write = [&](auto S) {
        ra.template store<decltype(S)::value>(lds + stage * STAGE, lw, lane, wk, p.k);
        rb.template store<decltype(S)::value>(lds + stage * STAGE + DA::BYTES, lw, lane, wk, p.k);
        next(ws, wk);
        stage = stage + 1 == NSTAGE ? 0 : stage + 1;
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      };
      [&]<int... S>(std::integer_sequence<int, S...>) { (fetch(std::integral_constant<int, S>{}), ...); }
      (std::make_integer_sequence<int, kRegDepth>{});
      auto slab = [&](auto S) {
        write(S);
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        fetch(S);
      };
      int k = 0;
      for (; k + kRegDepth <= nk; k += kRegDepth)  // no exit inside a round: the waits of the next one stay exact
        [&]<int... S>(std::integer_sequence<int, S...>) { (slab(std::integral_constant<int, S>{}), ...); }
        (std::make_integer_sequence<int, kRegDepth>{});
      [&]<int... S>(std::integer_sequence<int, S...>) {
        ((k + S < nk ? slab(std::integral_constant<int, S>{}) : (void)0), ...);
      }(std::make_integer_sequence<int, kRegDepth>{});
    } else {
    DA da;
    DB db;
    da.init(p.lda, m0, p.m, lw, lane);
    db.init(p.ldb, n0, p.n, lw, lane);
    const char* ca = DA::slab_base(A, p.lda, m0);  // base of the next slab, uniform: scalar registers
    const char* cb = DB::slab_base(B, p.ldb, n0);
    constexpr long SZ = (long)sizeof(T);
    const long step_a = (AKC ? (long)BK : (long)BK * p.lda) * SZ, step_b = (BKC ? (long)BK : (long)BK * p.ldb) * SZ;
    // after the last slab of a segment the pointers move to the start of the next segment
    const long last_a = step_a + p.a_sk * SZ - nk_seg * step_a, last_b = step_b + p.b_sk * SZ - nk_seg * step_b;
    const int k0_last = (nk_seg - 1) * BK;
    const bool tail = p.k % BK != 0;
    const unsigned lds0 = (unsigned)(uintptr_t)(lptr_t)lds;
    unsigned fill = lds0;  // LDS address of the stage the next slab goes to
    int left = nk_seg;     // slabs left in the current K segment, the next one included
    auto issue = [&]() {
      if (left != 1 || !tail) {
        da.template issue<false>(fill, lw, ca, 0, 0);
        db.template issue<false>(fill + DA::BYTES, lw, cb, 0, 0);
      } else {
        da.template issue<true>(fill, lw, ca, k0_last, p.k);
        db.template issue<true>(fill + DA::BYTES, lw, cb, k0_last, p.k);
      }
      if (left != 1) {
        ca += step_a;
        cb += step_b;
        --left;
      } else {
        ca += last_a;
        cb += last_b;
        left = nk_seg;
      }
      fill += STAGE;
      if (fill == lds0 + NSTAGE * STAGE) fill = lds0;
    };
    const int ahead = nk < NSTAGE - 1 ? nk : NSTAGE - 1;
    for (int s_ = 0; s_ < ahead; ++s_) issue();
    if (nk >= NSTAGE - 1) {
      RTP_WAIT_VM((NSTAGE - 2) * NI);
    } else {
      RTP_WAIT_VM(0);
    }
    __builtin_amdgcn_s_barrier();  // barrier 0
    int k = 0;
    for (; k + NSTAGE - 1 < nk; ++k) {  // slab k+NSTAGE-1 exists: steady state
      RTP_WAIT_VM((NSTAGE - 3) * NI);   // slabs k+2 .. k+NSTAGE-2 may still be in flight
      __builtin_amdgcn_s_barrier();     // barrier k+1
      issue();                          // slab k+NSTAGE-1 into the stage of slab k-1
    }
    for (; k + 1 < nk; ++k) {
      RTP_WAIT_VM(0);
      __builtin_amdgcn_s_barrier();
    }
    }
  } else {
    // ---- compute waves ----
    // Software pipeline over k-steps (KS per slab, numbered through the slabs): the fragments of k-step t + PD are
    // read from LDS right before the MFMAs of k-step t are issued, into one of PD + 1 register sets.  A wave gets
    // one 16-byte LDS read back every ~16 clocks after ~130-200 clocks of latency, so a read needs several k-steps
    // of MFMAs (32 clocks each) to hide behind; PD is chosen per tile shape for that.  The barrier that makes slab
    // k+1 visible sits right before its first fragment read, i.e. PD k-steps before its first MFMA.
    constexpr int NSET = PD + 1;
    static_assert(PD >= 1 && PD <= KS, "prefetch distance of 1..KS k-steps");
    static_assert((NSTAGE * KS) % NSET == 0, "register set of a k-step must not depend on the round");
    Frag<T> fa[NSET][MT], fb[NSET][NT];
    // Row sums of A (a bias gradient) ride along in the waves of the tile row's first tile that own column
    // block 0: each lane adds up the k values of its own row as the fragments pass by.
    const bool rowsum = p.a_rowsum != nullptr && tile_n == 0 && (SHARED_SUMS || wn == 0);
    auto read_step = [&](auto S, auto Q, auto SET) {
      const char* sa = lds + (decltype(S)::value % NSTAGE) * STAGE;
      const char* sb = sa + DA::BYTES;
      constexpr int q = decltype(Q)::value, set = decltype(SET)::value;
#pragma unroll
      for (int i = 0; i < MT; ++i) fa[set][i] = read_frag_dma<T, BM, AKC, SB>(sa, wm * WM + i * 32, lane, q);
#pragma unroll
      for (int j = 0; j < NT; ++j) fb[set][j] = read_frag_dma<T, BN, BKC, SB>(sb, wn * WN + j * 32, lane, q);
    };
    auto mma_step = [&](auto SET, auto Q) {
      constexpr int set = decltype(SET)::value, c = decltype(Q)::value % NSUM;
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) mma(fa[set][i], fb[set][j], acc[i][j]);
      if (rowsum) {
        if (SHARED_SUMS && wn != 0) {
#pragma unroll
          for (int i = 0; i < MS; ++i) rsum[i][c] = frag_sum(fa[set][MT - MS + i], rsum[i][c]);
        } else {
#pragma unroll
          for (int i = 0; i < MS; ++i) rsum[i][c] = frag_sum(fa[set][i], rsum[i][c]);
        }
      }
    };
    // k-step Q of slab k (stage S).  The scheduling fences keep the order written here: left alone, the compiler
    // sinks every LDS read to just before the MFMA that uses it (fewest live registers), which puts the LDS
    // latency in front of each MFMA instead of behind earlier ones.
    auto step = [&](auto S, auto Q, int k, auto STEADY) {
      constexpr bool steady = decltype(STEADY)::value;
      constexpr int s = decltype(S)::value, q = decltype(Q)::value;
      constexpr int t = s * KS + q;                            // k-step number inside the round
      constexpr int tq = (q + PD) % KS, ds = (q + PD) / KS;    // the k-step to prefetch: tq of slab k + ds
      if (steady || k + ds < nk) {
        if (ds == 1 && tq == 0) {
          __builtin_amdgcn_s_barrier();  // barrier k+1: slab k+1 is visible
          __builtin_amdgcn_sched_barrier(0);
        }
        read_step(std::integral_constant<int, (s + ds) % NSTAGE>{}, std::integral_constant<int, tq>{},
                  std::integral_constant<int, (t + PD) % NSET>{});
      }
      mma_step(std::integral_constant<int, t % NSET>{}, Q);
      // Issue order inside the step: one MFMA, then its share of the step's LDS reads, and so on.  A wave issues in
      // order and an MFMA holds the issue port until the matrix pipe takes it, so only what sits between two
      // MFMAs is issued in an MFMA's shadow; reads bunched up before the first MFMA would leave the pipe idle.
      constexpr int RPF_A = AKC ? 1 : (sizeof(T) == 2 ? 2 : 4), RPF_B = BKC ? 1 : (sizeof(T) == 2 ? 2 : 4);
      constexpr int NR = MT * RPF_A + NT * RPF_B, NM = MT * NT * (sizeof(T) == 2 ? 1 : 4);
      constexpr int PER = (NR + NM - 1) / NM;
      [&]<int... I>(std::integer_sequence<int, I...>) {
        ((__builtin_amdgcn_sched_group_barrier(0x008, 1, 0),
          (I * PER < NR ? __builtin_amdgcn_sched_group_barrier(0x100, (I + 1) * PER <= NR ? PER : NR - I * PER, 0)
                        : (void)0)),
         ...);
      }(std::make_integer_sequence<int, NM>{});
      __builtin_amdgcn_sched_barrier(0);
    };
    // A condition a slab holds up loops that issue more for an MFMA than the aligned bf16 ones: 180 x 1024 x 1024 in fp32 26.1 -> 27.5 us,
    // the fp32 cores' batched products 9.5 -> 10.3.  Those ask for everything at their start, and so do the 256 x 128 tile, which has no
    // registers left, and 64 x 64, whose loops are short.
    constexpr bool PACED = sizeof(T) == 2 && !REG && !RAG && BM >= 128 && BM * BN < 256 * 128;
    WarmAhead warm(p, (unsigned)(uintptr_t)(lptr_t)lds + NSTAGE * STAGE, id, nwg, wave, lane, PACED);
    auto phase = [&](auto S, int k, auto STEADY) {
      if (!decltype(STEADY)::value && k >= nk) return;
      if constexpr (PACED) warm.slab();
      [&]<int... Q>(std::integer_sequence<int, Q...>) {
        (step(S, std::integral_constant<int, Q>{}, k, STEADY), ...);
      }(std::make_integer_sequence<int, KS>{});
    };
    // one round = NSTAGE phases with compile-time stage indices
    auto round = [&](int kt, auto STEADY) {
      [&]<int... S>(std::integer_sequence<int, S...>) {
        (phase(std::integral_constant<int, S>{}, kt + S, STEADY), ...);
      }(std::make_integer_sequence<int, NSTAGE>{});
    };
    if constexpr (!PACED) warm.slab();
    if (!RAG || p.vec_c)
      request_epilogue<T, BM, BN>(p, (unsigned)(uintptr_t)(lptr_t)lds + NSTAGE * STAGE, m0, n0, grp, zo, zi, wave, lane);
    __builtin_amdgcn_s_barrier();  // barrier 0
    if (p.trace != nullptr && tid == 0) t_ready = (unsigned long long)wall_clock64();
    [&]<int... Q>(std::integer_sequence<int, Q...>) {
      (read_step(std::integral_constant<int, 0>{}, std::integral_constant<int, Q>{}, std::integral_constant<int, Q>{}),
       ...);
    }(std::make_integer_sequence<int, PD>{});
    __builtin_amdgcn_sched_barrier(0);
    int kt = 0;
    for (; kt + NSTAGE < nk; kt += NSTAGE) round(kt, std::true_type{});
    for (; kt < nk; kt += NSTAGE) round(kt, std::false_type{});
    if (p.trace != nullptr && tid == 0) t_loop = (unsigned long long)wall_clock64();
  }
  const bool computes = wave < 4;
  if (computes && p.a_rowsum != nullptr && tile_n == 0 && (SHARED_SUMS || wn == 0)) {
    // lanes 0..31 and 32..63 hold the two k halves of the same 32 rows
    T* dst = reinterpret_cast<T*>(p.a_rowsum) + grp * p.rowsum_sg;
#pragma unroll
    for (int i = 0; i < MS; ++i) {
      float v = rsum[i][0] + __shfl_xor(rsum[i][0], 32, 64);
      if constexpr (NSUM == 2) v += rsum[i][1] + __shfl_xor(rsum[i][1], 32, 64);
      const int row = m0 + wm * WM + (SHARED_SUMS ? wn * MS + i : i) * 32 + li;
      if (g == 0 && row < p.m) dst[row] = from_f32<T>((p.flags & RTP_GEMM_ROWSUM_ACCUM) ? to_f32(dst[row]) + v : v);
    }
  }

  // Epilogue through LDS: the accumulators (fp32) are laid out as the BM x BN tile, then every thread of the
  // workgroup, loader waves included, finishes 8 consecutive columns of one row and writes them with 16-byte
  // stores.
  __builtin_amdgcn_s_barrier();  // every wave has read its last fragments
  constexpr int CP = BN + 4;     // row pitch in floats
  float* ct = reinterpret_cast<float*>(lds);
  if (computes) {
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          ct[(wm * WM + i * 32 + 8 * (r >> 2) + 4 * g + (r & 3)) * CP + wn * WN + j * 32 + li] = acc[i][j][r];
  }
  __syncthreads();
  if constexpr (RAG) {
    // (the statistics and the vectorised update are only fused into products that are aligned throughout)
    if (REG && p.vec_c)
      finish_tile<T, BM, BN, 512>(p, ct, m0, n0, tid, grp, zo, zi);
    else
      finish_tile_ragged<T, BM, BN, 512>(p, ct, m0, n0, tid, grp, zo, zi);
  } else if (p.sgd_master != nullptr)
    finish_tile_sgd<T, BM, BN, 512>(p, ct, m0, n0, tid, grp, zo, zi);
  else if (p.xent_mode == 1) {
    // (tiles whose width is no multiple of the 64-column statistics blocks are never chosen for this epilogue)
    if constexpr (BN % 64 == 0) finish_tile_xent_stats<T, BM, BN, 512>(p, ct, m0, n0, tid, grp);
  } else
    finish_tile<T, BM, BN, 512>(p, ct, m0, n0, tid, grp, zo, zi);
  if (p.trace != nullptr && tid == 0) {
    const unsigned long long t_end = (unsigned long long)wall_clock64();
    atomicMax(p.trace + 1, t_end);
    // the phase sums come from every 16th workgroup: atomics of all of them on one line would stretch the launch
    if ((id & 15u) != 0u) return;
    atomicAdd(p.trace + 2, t_start);
    atomicAdd(p.trace + 3, t_ready - t_start);
    atomicAdd(p.trace + 4, t_loop - t_ready);
    atomicAdd(p.trace + 5, t_end - t_loop);
    atomicAdd(p.trace + 6, 1ull);
  }
}

template <typename T, int BM, int BN, bool AKC, bool BKC, int NSTAGE, int SB, int PD>
__global__ __launch_bounds__(512) void gemm_dma_kernel(GemmArgs) {
  const GemmArgs& p = fetched_arguments<GemmArgs>();
  gemm_dma_body<T, BM, BN, AKC, BKC, NSTAGE, SB, PD, false, false>(p, blockIdx.x + blockIdx.y * gridDim.x, blockIdx.x,
                                                            blockIdx.y, gridDim.x * gridDim.y);
}

// Operands of any alignment; REG where that includes A or B.
template <typename T, int BM, int BN, bool AKC, bool BKC, int NSTAGE, int SB, int PD, bool REG>
__global__ __launch_bounds__(512) void gemm_unaligned_kernel(GemmArgs) {
  const GemmArgs& p = fetched_arguments<GemmArgs>();
  gemm_dma_body<T, BM, BN, AKC, BKC, NSTAGE, SB, PD, REG, true>(p, blockIdx.x + blockIdx.y * gridDim.x, blockIdx.x, blockIdx.y,
                                                          gridDim.x * gridDim.y);
}

template <typename T, int BM, int BN, int NSTAGE, int SB, int PD>
static int launch_dma(hipStream_t s, const GemmArgs& a, bool akc, bool bkc, dim3 grid) {
  const dim3 block(512);
  // A row-contiguous operand is staged as k lines of R elements, and a 1 KiB load must cover whole lines (or a
  // whole fraction of one): tile extents that are not powers of two only exist for K-contiguous operands.
  constexpr bool A_RC_OK = (BM & (BM - 1)) == 0, B_RC_OK = (BN & (BN - 1)) == 0;
  if constexpr (!A_RC_OK || !B_RC_OK) {
    RTP_REQUIRE((akc || A_RC_OK) && (bkc || B_RC_OK), "gemm: tile %d x %d needs K-contiguous operands", BM, BN);
    if constexpr (!B_RC_OK && A_RC_OK) {
      if (akc)
        hipLaunchKernelGGL((gemm_dma_kernel<T, BM, BN, true, true, NSTAGE, SB, PD>), grid, block, 0, s, a);
      else
        hipLaunchKernelGGL((gemm_dma_kernel<T, BM, BN, false, true, NSTAGE, SB, PD>), grid, block, 0, s, a);
    }
    RTP_LAUNCH_CHECK();
    return RTP_OK;
  } else if (akc && bkc)
    hipLaunchKernelGGL((gemm_dma_kernel<T, BM, BN, true, true, NSTAGE, SB, PD>), grid, block, 0, s, a);
  else if (akc && !bkc)
    hipLaunchKernelGGL((gemm_dma_kernel<T, BM, BN, true, false, NSTAGE, SB, PD>), grid, block, 0, s, a);
  else if (!akc && bkc)
    hipLaunchKernelGGL((gemm_dma_kernel<T, BM, BN, false, true, NSTAGE, SB, PD>), grid, block, 0, s, a);
  else
    hipLaunchKernelGGL((gemm_dma_kernel<T, BM, BN, false, false, NSTAGE, SB, PD>), grid, block, 0, s, a);
  RTP_LAUNCH_CHECK();
  return RTP_OK;
}

template <typename T, int BM, int BN, int NSTAGE, int SB, int PD, bool REG>
static int launch_unaligned(hipStream_t s, const GemmArgs& a, bool akc, bool bkc, dim3 grid) {
  const dim3 block(512);
  if (akc && bkc)
    hipLaunchKernelGGL((gemm_unaligned_kernel<T, BM, BN, true, true, NSTAGE, SB, PD, REG>), grid, block, 0, s, a);
  else if (akc && !bkc)
    hipLaunchKernelGGL((gemm_unaligned_kernel<T, BM, BN, true, false, NSTAGE, SB, PD, REG>), grid, block, 0, s, a);
  else if (!akc && bkc)
    hipLaunchKernelGGL((gemm_unaligned_kernel<T, BM, BN, false, true, NSTAGE, SB, PD, REG>), grid, block, 0, s, a);
  else
    hipLaunchKernelGGL((gemm_unaligned_kernel<T, BM, BN, false, false, NSTAGE, SB, PD, REG>), grid, block, 0, s, a);
  RTP_LAUNCH_CHECK();
  return RTP_OK;
}

// ---------------------------------------------------------------------------------------------
// Tiny batched problems (one attention head at sequence length <= 64: 32 x 32 x 64 per (batch, head)):
// one wavefront per 32 x 32 output block, operands read straight from global memory into MFMA
// fragments (no LDS, no barriers).  Thousands of independent wavefronts hide the load latency.
template <typename T, bool AKC, bool BKC>
__global__ __launch_bounds__(kThreads) void gemm_tiny_kernel(GemmArgs p, long nblocks) {
  constexpr int VEC = 16 / sizeof(T);
  const int lane = threadIdx.x & 63;
  const long blk = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (blk >= nblocks) return;
  const int li = lane & 31, g = lane >> 5;
  const int tiles = p.tiles_m * p.tiles_n;
  const long z = blk / tiles;
  const int tile = (int)(blk % tiles);
  const int m0 = (tile / p.tiles_n) * 32, n0 = (tile % p.tiles_n) * 32;
  const int grp = (int)(z / p.batch), zb = (int)(z % p.batch);
  const long zo = zb / p.zdiv, zi = zb % p.zdiv;
  const T* A = reinterpret_cast<const T*>(p.a) + grp * p.a_sg + zo * p.a_so + zi * p.a_si;
  const T* B = reinterpret_cast<const T*>(p.b) + grp * p.b_sg + zo * p.b_so + zi * p.b_si;

  f32x16 acc[1][1];
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[0][0][r] = 0.0f;

  // fragment of `rows`-row operand X for this lane's row and the VEC k values starting at k
  auto frag = [&](const T* X, long ld, bool kc, bool vec_ok, int row, int rows, int k) {
    union {
      uint4 q;
      T e[VEC];
      Frag<T> f;
    } u;
    if (kc) {
      const T* src = X + (long)row * ld + k;
      if (vec_ok && row < rows && k + VEC <= p.k) {
        u.q = *reinterpret_cast<const uint4*>(src);
      } else {
#pragma unroll
        for (int e = 0; e < VEC; ++e) u.e[e] = (row < rows && k + e < p.k) ? src[e] : (T)0.0f;
      }
    } else {
#pragma unroll
      for (int e = 0; e < VEC; ++e) u.e[e] = (row < rows && k + e < p.k) ? X[(long)(k + e) * ld + row] : (T)0.0f;
    }
    return u.f;
  };

  for (int seg = 0; seg < p.ksegs; ++seg) {
    const T* As = A + seg * p.a_sk;
    const T* Bs = B + seg * p.b_sk;
    for (int k0 = 0; k0 < p.k; k0 += 2 * VEC) {
      const Frag<T> fa = frag(As, p.lda, AKC, p.vec_a, m0 + li, p.m, k0 + g * VEC);
      const Frag<T> fb = frag(Bs, p.ldb, BKC, p.vec_b, n0 + li, p.n, k0 + g * VEC);
      mma(fa, fb, acc[0][0]);
    }
  }
  store_tile<T, 1, 1, 32, 32>(p, acc, m0, n0, 0, 0, li, g, grp, zo, zi);
}

// ---------------------------------------------------------------------------------------------
// fp32 weight gradients with few output tiles and a long contraction (512 x 512 over thousands of tokens): 64 x 64 tiles
// leave most CUs idle, one serial chain each.  Here a workgroup owns 32 x 32 outputs and its eight waves an eighth of the
// contraction each; the partial sums meet in LDS and are added in wave order.  Both operands are row-contiguous, so a lane's
// MFMA operand is one float of a k line: fragments come straight from global memory (two 128-byte lines per load, any
// alignment) and there is no staging and no barrier in the loop.  Bound by the fp32 MFMAs (3.4 ns per k at 2.35 GHz) where
// the loads' latency is hidden: four batches of 16 loads are in flight per wave, as many as the counter of outstanding loads
// (63) can tell apart, with the lines' addresses on the scalar unit (a buffer resource per batch) and the order held by scheduling
// barriers, or the compiler gathers all the loads behind all the products.
// us, 64 x 64 tiles of fp32 MFMAs -> one batch ahead -> this: 512 x 512 x 1600 31 -> 19.8 -> 12.9, 512 x 512 x 2880 51 -> 30.2 -> 17.4,
// 256 x 256 x 1024 21 -> 12.9 -> 9.6, 128 x 128 x 8192 128 -> 74.8 -> 36.0; error against fp64 7.2e-7 -> 2.6e-7 (eight short sums
// instead of one long one).
// waves, MFMAs (two k each) per batch of loads, batches of loads ahead of the MFMAs
constexpr int kSplitWaves = 8, kSplitBatch = 8, kSplitAhead = 4;
__global__ __launch_bounds__(64 * kSplitWaves) void gemm_ksplit_kernel(GemmArgs p) {
  __shared__ float part[kSplitWaves][32][33];
  __shared__ float sums[kSplitWaves][32];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int li = lane & 31, g = lane >> 5;
  int bid = blockIdx.x;
  const int nb = p.tiles_m * p.tiles_n;
  if ((nb & 7) == 0) bid = (bid & 7) * (nb >> 3) + (bid >> 3);  // neighbouring tiles on one XCD
  const int m0 = bid / p.tiles_n * 32, n0 = bid % p.tiles_n * 32;
  const int grp = blockIdx.y / p.batch, zb = blockIdx.y % p.batch;
  const long zo = zb / p.zdiv, zi = zb % p.zdiv;
  const float* A = reinterpret_cast<const float*>(p.a) + grp * p.a_sg + zo * p.a_so + zi * p.a_si;
  const float* B = reinterpret_cast<const float*>(p.b) + grp * p.b_sg + zo * p.b_so + zi * p.b_si;
  // a lane's place from the start of a pair of k lines; rows past the end re-read the last one: they feed accumulators that
  // are never stored
  const unsigned at_a = (unsigned)(min(m0 + li, p.m - 1) + g * (int)p.lda), at_b = (unsigned)(min(n0 + li, p.n - 1) + g * (int)p.ldb);

  f32x16 acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
  float rs = 0.0f;
  constexpr int STEP = 2 * kSplitBatch;
  const int chunk = ((p.k + kSplitWaves * STEP - 1) / (kSplitWaves * STEP)) * STEP;
  const int kb = min(wave * chunk, p.k), ke = min(kb + chunk, p.k);
  const int full = (ke - kb) / STEP;
  struct Batch {
    float a[kSplitBatch], b[kSplitBatch];
  };
  for (int seg = 0; seg < p.ksegs; ++seg) {
    const float* As = A + seg * p.a_sk;
    const float* Bs = B + seg * p.b_sk;
    Batch ring[kSplitAhead];
    auto fetch = [&](int i, Batch& f) {  // batch i, or the last whole one again
      const long k0 = kb + min(i, full - 1) * STEP;
      const auto ra = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(As + k0 * p.lda), 0, 0x7fffffff, 0x00020000);
      const auto rb = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(Bs + k0 * p.ldb), 0, 0x7fffffff, 0x00020000);
#pragma unroll
      for (int e = 0; e < kSplitBatch; ++e) {
        f.a[e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(ra, (int)(4 * at_a), 8 * e * (int)p.lda, 0));
        f.b[e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rb, (int)(4 * at_b), 8 * e * (int)p.ldb, 0));
      }
      __builtin_amdgcn_sched_barrier(0);  // in the order written: the loads of a batch right behind the products of the one before
    };
    auto multiply = [&](const Batch& f) {
#pragma unroll
      for (int e = 0; e < kSplitBatch; ++e) {
        rs += f.a[e];
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(f.a[e], f.b[e], acc, 0, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    };
    if (full > 0) {
#pragma unroll
      for (int u = 0; u < kSplitAhead; ++u) fetch(u, ring[u]);
      int i = 0;
      for (; i + kSplitAhead <= full; i += kSplitAhead)
#pragma unroll
        for (int u = 0; u < kSplitAhead; ++u) {
          multiply(ring[u]);
          fetch(i + u + kSplitAhead, ring[u]);
        }
#pragma unroll
      for (int u = 0; u < kSplitAhead; ++u)
        if (i + u < full) multiply(ring[u]);
    }
    for (int k0 = kb + full * STEP; k0 < ke; k0 += 2) {  // what is no whole batch
      const long k = min(k0 + g, p.k - 1) - g;
      const bool live = k0 + g < ke;
      const float x = live ? As[k * p.lda + at_a] : 0.0f, y = live ? Bs[k * p.ldb + at_b] : 0.0f;
      rs += x;
      acc = __builtin_amdgcn_mfma_f32_32x32x2f32(x, y, acc, 0, 0, 0);
    }
  }
#pragma unroll
  for (int r = 0; r < 16; ++r) part[wave][8 * (r >> 2) + 4 * g + (r & 3)][li] = acc[r];
  const float both = rs + __shfl_xor(rs, 32, kWave);
  if (g == 0) sums[wave][li] = both;
  __syncthreads();

  if (p.a_rowsum != nullptr && n0 == 0 && threadIdx.x < 32 && m0 + (int)threadIdx.x < p.m) {
    float v = 0.0f;
#pragma unroll
    for (int w = 0; w < kSplitWaves; ++w) v += sums[w][threadIdx.x];
    float* dst = reinterpret_cast<float*>(p.a_rowsum) + grp * p.rowsum_sg + m0 + threadIdx.x;
    *dst = (p.flags & RTP_GEMM_ROWSUM_ACCUM) ? *dst + v : v;
  }
  f32x16 whole[1][1];
  if (wave != 0) return;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    float v = 0.0f;
#pragma unroll
    for (int w = 0; w < kSplitWaves; ++w) v += part[w][8 * (r >> 2) + 4 * g + (r & 3)][li];
    whole[0][0][r] = v;
  }
  store_tile<float, 1, 1, 32, 32>(p, whole, m0, n0, 0, 0, li, g, grp, zo, zi);
}

template <typename T, int BM, int BN, int DEPTH, bool FAST>
static int launch_layout(hipStream_t s, const GemmArgs& a, bool akc, bool bkc, dim3 grid) {
  if (akc && bkc)
    hipLaunchKernelGGL((gemm_kernel<T, BM, BN, true, true, DEPTH, FAST>), grid, dim3(kThreads), 0, s, a);
  else if (akc && !bkc)
    hipLaunchKernelGGL((gemm_kernel<T, BM, BN, true, false, DEPTH, FAST>), grid, dim3(kThreads), 0, s, a);
  else if (!akc && bkc)
    hipLaunchKernelGGL((gemm_kernel<T, BM, BN, false, true, DEPTH, FAST>), grid, dim3(kThreads), 0, s, a);
  else
    hipLaunchKernelGGL((gemm_kernel<T, BM, BN, false, false, DEPTH, FAST>), grid, dim3(kThreads), 0, s, a);
  RTP_LAUNCH_CHECK();
  return RTP_OK;
}

static bool mult(int64_t v, int64_t q) { return v % q == 0; }

// Tile shapes, largest first; launch_gemm picks one with a cost model (the 10-layer LM's per-layer problems
// are 1024 x 2048 outputs: 128 tiles of 128x128 but exactly 256, one per CU, of 128x64).
struct TileShape {
  int bm, bn;
  const char* tag;
};
static const TileShape kShapes[7] = {{256, 128, "256x128"}, {128, 128, "128x128"}, {128, 64, "128x64"}, {64, 64, "64x64"},
                                     {128, 192, "128x192"}, {256, 256, "256x256"}, {128, 160, "128x160"}};
constexpr int kNumShapes = 7;

// One wavefront per 32 x 32 block is the better kernel for one attention head at sequence length <= 64.
static bool is_tiny(const rtp_gemm_desc* d) { return d->m <= 64 && d->n <= 64 && d->k * d->ksegs <= 256; }

// Whether the wave-specialised kernel can run the problem.  Its branch-free loads need whole 16-byte vectors:
// aligned operands and extents that are multiples of VEC along each operand's contiguous axis; and a tile's
// byte offsets from its first vector must fit 32 bits (256 rows or k lines of one leading dimension).
// Anything else goes to the guarded small-tile kernel.
template <typename T>
static bool takes_dma_kernel(const rtp_gemm_desc* d) {
  constexpr int VEC = 16 / sizeof(T);
  const bool vec_a = mult((int64_t)(uintptr_t)d->a, 16) && mult(d->lda, VEC) && mult(d->a_so, VEC) &&
                     mult(d->a_si, VEC) && mult(d->a_sg, VEC) && mult(d->a_sk, VEC);
  const bool vec_b = mult((int64_t)(uintptr_t)d->b, 16) && mult(d->ldb, VEC) && mult(d->b_so, VEC) &&
                     mult(d->b_si, VEC) && mult(d->b_sg, VEC) && mult(d->b_sk, VEC);
  const bool akc = d->a_kcontig, bkc = d->b_kcontig;
  const int64_t ld_max = ((int64_t)1 << 24) / (int64_t)sizeof(T) - 64;
  return vec_a && vec_b && ((akc || bkc) ? mult(d->k, VEC) : true) && (akc || mult(d->m, VEC)) &&
         (bkc || mult(d->n, VEC)) && d->k > 0 && d->lda <= ld_max && d->ldb <= ld_max;
}

// Whether the same kernel with register loaders can: any alignment, as long as every row (or k line) holds one vector.
template <typename T>
static bool takes_reg_kernel(const rtp_gemm_desc* d) {
  constexpr int VEC = 16 / sizeof(T);
  const bool akc = d->a_kcontig, bkc = d->b_kcontig;
  const int64_t ld_max = ((int64_t)1 << 24) / (int64_t)sizeof(T) - 64;
  return ((akc || bkc) ? d->k >= VEC : d->k > 0) && (akc || d->m >= VEC) && (bkc || d->n >= VEC) && d->lda <= ld_max &&
         d->ldb <= ld_max;
}

// The fused clip + SGD lives in the epilogue of the wave-specialised kernel; the gradient keeps the compute dtype.
template <typename T>
static bool sgd_fused(const rtp_gemm_desc* d) {
  return !is_tiny(d) && takes_dma_kernel<T>(d) && !(d->flags & (RTP_GEMM_OUT_F32 | RTP_GEMM_RELU)) && !d->c_in &&
         !d->bias && !d->gate;
}

template <typename T>
static bool rowsum_fused(const rtp_gemm_desc* d) {
  return !d->a_kcontig && d->batch == 1 && !is_tiny(d) && (takes_dma_kernel<T>(d) || takes_reg_kernel<T>(d));
}

// Few tiles, whatever the layout: see gemm_kwaves.hip.  256 tiles of 32 x 32 are one workgroup a CU, and up to there it is ahead at
// every contraction from 256 on (measured in a replayed graph on 70 shapes x 3 layouts x 2 types; bf16 1.1 - 2.5 times, fp32 1.5 - 2.3).
// From 257 on some CU has two and only fp32 with K of 768 and more gains, up to 512 (where 64 x 32, below, does not fit).  us, before -> this:
// 256 tiles bf16 64 x 4096, K = 512 5.7 -> 4.6, 4096 19.2 -> 10.3; 288 tiles 384 x 768, K = 256 5.2 -> 6.7, 1024 7.6 -> 8.7, 2048
// 12.1 -> 11.7; 512 tiles fp32 512 x 1024, K = 384 10.8 -> 12.6, 1024 19.6 -> 18.1; 768 tiles 512 x 1536, K = 2048 36 -> 44.
// Operands that are not vector-aligned, 12 shapes: bf16 255 x 1023 x 3333 24.0 -> 17.6, 31 x 2049 x 515 8.6 -> 8.2, one of 25 behind
// (7 x 8101 x 1027, input gradient, 13.4 -> 14.2); fp32 65.6 -> 28.5 and 15.8 -> 11.1.  (Row-contiguous fp32 has gemm_ksplit_kernel.)
// With tiles of 64 x 32 twice as many outputs are one workgroup a CU: in fp32 ahead at any contraction (1.05 - 1.46 times on 24 shapes,
// two of 72 behind by 1 and 3 %), in bf16 only at long ones, with operands that lie alike (K >= 2048: 1.0 - 1.2, unaligned weight gradients
// 1.4 - 1.8; K = 512 0.83 - 0.98; the input gradient's layout 0.95 - 1.09).
// 0: not few, otherwise the tile's rows.
template <typename T>
static int few_tiles(const rtp_gemm_desc* d) {
  const int64_t nz = d->batch * d->groups, k_all = d->k * d->ksegs;
  const int64_t tiles32 = ceil_div(d->m, 32) * ceil_div(d->n, 32) * nz, tiles64 = ceil_div(d->m, 64) * ceil_div(d->n, 32) * nz;
  return tiles32 <= 256                                                                          ? 32
         : tiles64 <= 256 && (sizeof(T) == 4 || (k_all >= 2048 && d->a_kcontig == d->b_kcontig)) ? 64
         : sizeof(T) == 4 && k_all >= 768 && tiles32 <= 512                                      ? 32
                                                                                                 : 0;
}
// Whether gemm_kwaves.hip takes the product, which splits its contraction over the waves of a workgroup.
// A product under a ReLU stays in the order of its sums, here and below: a sum within its rounding of zero decides whether the
// backward pass sees the unit at all, and of 16 M such sums (1000 tokens, 8 experts of 768 x 8064) some ten are that near.
template <typename T>
static bool takes_kwaves(const rtp_gemm_desc* d) {
  const bool direct = takes_dma_kernel<T>(d);
  return (direct || takes_reg_kernel<T>(d)) && !is_tiny(d) && !(d->flags & RTP_GEMM_RELU) && !d->xent_mode && d->batch * d->groups < 65536 &&
         d->k * d->ksegs >= 256 && !(sizeof(T) == 4 && !direct && !d->a_kcontig && !d->b_kcontig) && few_tiles<T>(d) != 0;
}

// rtp_gemm_warm_next: bytes the next product launched by this host thread requests beside its own.  A later call, from any
// thread, ends an earlier hint: a caller holds the memory of the last one only, and a forward pass and its backward pass
// run on two threads.
static std::atomic<unsigned long long> g_warm_call{0};
static thread_local const void* t_warm_src = nullptr;
static thread_local size_t t_warm_bytes = 0;
static thread_local unsigned long long t_warm_call = 0;
static const void* warm_source() {
  return t_warm_src && t_warm_call == g_warm_call.load(std::memory_order_relaxed) ? t_warm_src : nullptr;
}

// rtp_gemm_workspace: the calling thread's source of scratch memory.
static thread_local rtp_alloc_fn t_alloc = nullptr;
static thread_local void* t_alloc_context = nullptr;

// The price of 256 x 256 tiles and of an update, for every rule that weighs them: ns in the units of launch_gemm's table, where only ratios matter.
// 256 x 256 is priced by its ratio to the others with every CU busy.  Every tile forced on 59 products x 3 layouts, operands from memory: with
// these two numbers the shape taken costs 0.1 % over the best one in the mean (with 1350 and 5000 ns, the price of the kernel before this
// one, 0.8 %), the most 12 % (4096 x 2048 x 6144, 128 tiles: 119 us with 256 x 128 against 111); it is the same for 975 - 1100 and 4000 -
// 5000 ns.  Where 256 x 256 is close and not taken: 4096 x 2048 x 2048, 128 tiles, 39 - 43 us against 37 - 38.
constexpr double kLargeSlabNs = 1050.0, kLargeTileNs = 4500.0;
// The kernel finishes the rarer combinations block after block, a trip to memory each: with bias, addend and ReLU 8 of 1024 x 1280 x 520 is 41.3 us
// (19.2 plain) against 41.1 (25.2) with 128 x 160 tiles, x 2048 61.5 (46.3) against 67.2 (58.3).
static bool rare_epilogue(const rtp_gemm_desc* d) {
  return (d->bias != nullptr) + (d->c_in != nullptr) + (d->gate != nullptr) > 1 || ((d->flags & RTP_GEMM_RELU) && !d->bias) ||
         (d->flags & (RTP_GEMM_OUT_F32 | RTP_GEMM_CIN_F32)) || d->xent_mode;
}
static double large_ns(double rounds, double slabs, bool rare) {
  return rounds * (slabs * kLargeSlabNs + kLargeTileNs + (rare ? 3000.0 : 0.0));
}
// An update moves 10 bytes a parameter (12 with the gradient) behind the K loop, a round's tiles together at the memory's 4.9 TB/s, a CU at no
// more than 32 bytes a ns.  So few large tiles are behind where they leave CUs idle: us with 128 x 128 / 256 x 256, K = 1024, 2048 x 2048
// 19.2 / 39, 8 of 1280 x 2048 97 / 101, 6144 x 2048 59.7 / 49.9, 4096 x 4096 75 / 61; 8192 x 2048 x 4096 174 / 145.
static double update_bytes(const rtp_gemm_desc* d) {  // a parameter
  return !d->sgd_master ? 0.0 : 8.0 + (d->sgd_weights ? 2.0 : 0.0) + (d->flags & RTP_GEMM_SGD_SKIP_OUT ? 0.0 : 2.0);
}
static double update_ns(double tiles, double tile_bytes) {
  const auto round_ns = [&](double n) { return std::max(n * tile_bytes / 4900.0, tile_bytes / 32.0); };
  const double rounds = (double)ceil_div((int64_t)tiles, 256);
  return (rounds - 1.0) * round_ns(256.0) + round_ns(tiles - 256.0 * (rounds - 1.0));
}

// Which operands of a bf16 product are copied to whole vectors first.
struct Packing {
  bool a = false, b = false;
  PackShape sa, sb;
};
static Packing pack_plan(const rtp_gemm_desc* d, bool vec_c) {
  Packing p;
  const bool akc = d->a_kcontig, bkc = d->b_kcontig;
  if (t_alloc == nullptr || d->batch != 1 || d->xent_mode || d->sgd_master || d->m < 128 || d->n < 128 || d->k < 8 || takes_dma_kernel<bf16_t>(d) ||
      takes_kwaves<bf16_t>(d))  // (few tiles: that kernel loads at any alignment, and on its own the product keeps the order of its sums)
    return p;
  const int64_t ld_max = ((int64_t)1 << 23) - 64;
  const auto shape = [&](const void* x, int64_t ld, int64_t sg, int64_t sk, bool kc, int64_t rows) {
    PackShape q;
    q.src = (const char*)x, q.ld = ld, q.copy = sg, q.seg = sk;
    q.copies = sg != 0 ? d->groups : 1, q.segs = sk != 0 ? d->ksegs : 1;
    q.lines = kc ? rows : d->k, q.len = kc ? d->k : rows;
    return q;
  };
  const auto fits = [&](const PackShape& q) {
    return mult((int64_t)(uintptr_t)q.src, 16) && mult(q.ld, 8) && mult(q.copy, 8) && mult(q.seg, 8) && mult(q.len, 8);
  };
  p.sa = shape(d->a, d->lda, d->a_sg, d->a_sk, akc, d->m), p.sb = shape(d->b, d->ldb, d->b_sg, d->b_sk, bkc, d->n);
  const bool a = !fits(p.sa), b = !fits(p.sb);
  const int64_t vectors = (a ? p.sa.vectors() : 0) + (b ? p.sb.vectors() : 0);
  if (vectors > (1 << 26) || p.sa.len > ld_max || p.sb.len > ld_max || (!a && d->lda > ld_max) || (!b && d->ldb > ld_max)) return p;
  // It pays where the copies (their bytes in and out at 4.5 TB/s, 8 us each between their neighbours on the stream) take less than what
  // the register loaders add.  ns a slab of 128 x 128, every CU busy: register loaders 600 / 700 / 800 (both operands k-contiguous /
  // one / none), direct-to-LDS 480; outside the slabs 6 and 5 us; 256 x 256, which only aligned results can take, 1.5 times its price (1650 a
  // slab and 6 us were seen).  us without -> with the copies, forward / input gradient / weight gradient (=: not taken): 6546 x 482 x 6400, 8 shards, 460 / 540 /
  // 628 -> 367 / 353 / 407; 4096 x 1023 x 4096 = / 76 / 80 -> = / 47 / 46; 8192 x 33 x 7000, 8 shards, = / 185 / = -> = / 111 / =;
  // 1024 x 3001 x 4096 = / 45.8 (taken: 47.6) / 64 -> = / = / 50; 1250 x 9090 x 1792, 2 shards, = / 187 (taken: 199) / 160 -> = / = / 145; 2001 x 2003 x
  // 2005 = (taken: 35.9 / 42.1 / 47.1 against 32.7 / 38.5 / 44.0).
  const int64_t slabs = ceil_div(d->k, 64) * d->ksegs;
  const auto rounds = [&](int t) { return (double)ceil_div(ceil_div(d->m, t) * ceil_div(d->n, t) * d->groups, 256); };
  const double slow = rounds(128) * ((double)slabs * (akc && bkc ? 600.0 : akc || bkc ? 700.0 : 800.0) + 6000.0);
  double fast = rounds(128) * ((double)slabs * 480.0 + 5000.0);
  if (vec_c && slabs >= 2) fast = std::min(fast, 1.5 * large_ns(rounds(256), (double)slabs, rare_epilogue(d)));
  const double copies = 32.0 * (double)vectors / 4500.0 + (a ? 8000.0 : 0.0) + (b ? 8000.0 : 0.0);
  if (slow - fast > 1.2 * copies) p.a = a, p.b = b;
  return p;
}

// What one of two products would take by itself, and its arguments as a launch of 256 x 256 tiles (none: it cannot be one).
struct PairPlan {
  GemmArgs args;
  bool large = false, rare = false;
  double alone = 0.0;  // ns
  double slabs = 0.0, update_bytes = 0.0, flops = 0.0, bytes = 0.0;
};

// plan: nothing is launched, it is filled instead.  in_order: rows of a product whose others go in another launch, so that the contraction is
// summed in one sequence, as there: equal rows have equal results wherever they are.
template <typename T>
static int launch_gemm(hipStream_t s, const rtp_gemm_desc* d, PairPlan* plan = nullptr, bool in_order = false) {
  if (plan && (sizeof(T) != 2 || d->a_kcontig || d->b_kcontig || d->xent_mode || is_tiny(d) || !takes_dma_kernel<T>(d))) return RTP_OK;
  // the hint of rtp_gemm_warm_next rides in this launch or ends with it
  const void* warm_src = warm_source();
  if (!plan) t_warm_src = nullptr;
  constexpr int VEC = 16 / sizeof(T);
  GemmArgs a;
  {
    auto ok = [](const void* ptr, int64_t ld, int64_t so, int64_t si, int64_t sg) {
      return mult((int64_t)(uintptr_t)ptr, 16) && mult(ld, 8) && mult(so, 8) && mult(si, 8) && mult(sg, 8);
    };
    a.vec_c = mult(d->n, 8) && ok(d->c_out, d->ldc, d->c_so, d->c_si, d->c_sg) &&
              (!d->c_in || ok(d->c_in, d->ld_cin, d->cin_so, d->cin_si, d->cin_sg)) &&
              (!d->gate || ok(d->gate, d->ld_gate, d->gate_so, d->gate_si, d->gate_sg)) &&
              (!d->bias || (ok(d->bias, 8, d->bias_so, d->bias_si, d->bias_sg) && mult(d->bias_sk, 8)));
  }
  bool packed = false;
  rtp_gemm_desc aligned;
  if constexpr (sizeof(T) == 2) {
    if (const Packing p = pack_plan(d, a.vec_c); p.a || p.b) {
      const int64_t bytes_a = p.a ? p.sa.vectors() * 16 : 0, bytes_b = p.b ? p.sb.vectors() * 16 : 0;
      if (char* at = (char*)t_alloc(t_alloc_context, (size_t)(bytes_a + bytes_b)); at != nullptr && (uintptr_t)at % 16 == 0) {
        aligned = *d, packed = true;
        const auto move = [&](const PackShape& q, char* to, const void*& x, int64_t& ld, int64_t& sg, int64_t& sk) {
          x = to, ld = ceil_div(q.len, 8) * 8;
          if (sk != 0) sk = q.lines * ld;
          if (sg != 0) sg = q.segs * q.lines * ld;
          return launch_pack(s, q, to);
        };
        int rc = RTP_OK;
        if (p.a) rc = move(p.sa, at, aligned.a, aligned.lda, aligned.a_sg, aligned.a_sk);
        if (p.b && rc == RTP_OK) rc = move(p.sb, at + bytes_a, aligned.b, aligned.ldb, aligned.b_sg, aligned.b_sk);
        if (rc != RTP_OK) return rc;
        d = &aligned;
      }
    }
  }
  a.a = (const char*)d->a;
  a.b = (const char*)d->b;
  a.c_out = (char*)d->c_out;
  a.c_in = (const char*)d->c_in;
  a.bias = (const char*)d->bias;
  a.gate = (const char*)d->gate;
  a.m = (int)d->m;
  a.n = (int)d->n;
  a.k = (int)d->k;
  a.ksegs = (int)d->ksegs;
  a.lda = d->lda;
  a.ldb = d->ldb;
  a.ldc = d->ldc;
  a.ld_cin = d->ld_cin;
  a.ld_gate = d->ld_gate;
  a.batch = (int)d->batch;
  a.zdiv = (int)d->zdiv;
  a.a_so = d->a_so, a.a_si = d->a_si, a.b_so = d->b_so, a.b_si = d->b_si;
  a.c_so = d->c_so, a.c_si = d->c_si, a.cin_so = d->cin_so, a.cin_si = d->cin_si;
  a.gate_so = d->gate_so, a.gate_si = d->gate_si, a.bias_so = d->bias_so, a.bias_si = d->bias_si;
  a.a_sg = d->a_sg, a.b_sg = d->b_sg, a.c_sg = d->c_sg, a.cin_sg = d->cin_sg;
  a.gate_sg = d->gate_sg, a.bias_sg = d->bias_sg;
  a.a_sk = d->a_sk, a.b_sk = d->b_sk, a.bias_sk = d->bias_sk;
  a.alpha = d->alpha;
  a.flags = d->flags;
  a.vec_a = mult((int64_t)(uintptr_t)d->a, 16) && mult(d->lda, VEC) && mult(d->a_so, VEC) && mult(d->a_si, VEC) &&
            mult(d->a_sg, VEC) && mult(d->a_sk, VEC);
  a.vec_b = mult((int64_t)(uintptr_t)d->b, 16) && mult(d->ldb, VEC) && mult(d->b_so, VEC) && mult(d->b_si, VEC) &&
            mult(d->b_sg, VEC) && mult(d->b_sk, VEC);

  const bool akc = d->a_kcontig, bkc = d->b_kcontig;
  const bool direct = packed || takes_dma_kernel<T>(d), fast = direct || takes_reg_kernel<T>(d);
  const int64_t nz = d->batch * d->groups;
  a.a_rowsum = (char*)d->a_rowsum;
  a.rowsum_sg = d->rowsum_sg;
  a.trace = nullptr;
  a.xent_mode = d->xent_mode;
  a.xent_blocks = (int)(d->groups * d->n / 64);
  a.xent_target = (const long*)d->xent_target;
  a.xent_ignore = (long)d->xent_ignore;
  a.xent_part = (float2*)d->xent_part;
  a.xent_tlogit = d->xent_tlogit;
  a.xent_stats = (const float2*)d->xent_stats;
  a.xent_dloss = d->xent_dloss;
  a.xent_scale = d->xent_scale;
  if (d->xent_mode) {
    RTP_REQUIRE(d->xent_mode == 1 || d->xent_mode == 2, "rtp_gemm: xent_mode is 0, 1 or 2");
    RTP_REQUIRE(takes_dma_kernel<T>(d) && !is_tiny(d) && a.vec_c && d->n % 64 == 0 && d->batch == 1 && d->ksegs >= 1 &&
                    d->c_sg == d->n && !(d->flags & (RTP_GEMM_OUT_F32 | RTP_GEMM_RELU)) && !d->c_in && !d->gate,
                "rtp_gemm: the cross-entropy epilogues need vector-aligned operands, groups of a multiple of 64 columns "
                "laid side by side (c_sg == n), an output in the compute dtype and no c_in / ReLU / mask");
    RTP_REQUIRE(d->xent_target && (d->xent_mode == 1 ? (d->xent_part && d->xent_tlogit) : (d->xent_stats && d->xent_dloss)),
                "rtp_gemm: missing cross-entropy operands for mode %d", d->xent_mode);
    RTP_REQUIRE((uintptr_t)d->xent_part % 8 == 0 && (uintptr_t)d->xent_stats % 8 == 0, "rtp_gemm: 8-byte aligned statistics");
  }
  a.sgd_master = (float*)d->sgd_master;
  a.sgd_w = (char*)d->sgd_weights;
  a.sgd_lr = d->sgd_lr;
  a.sgd_clip = d->sgd_clip;
  RTP_REQUIRE(!d->sgd_master || sgd_fused<T>(d),
              "rtp_gemm: sgd_master needs vector-aligned operands, an output in the compute dtype and no c_in / bias / "
              "ReLU / mask (rtp_gemm_sgd_fused)");
  RTP_REQUIRE(d->sgd_master || (!d->sgd_weights && !(d->flags & RTP_GEMM_SGD_SKIP_OUT)),
              "rtp_gemm: sgd_weights / RTP_GEMM_SGD_SKIP_OUT without sgd_master");
  if (d->sgd_master)  // the update's 16-byte accesses: 8 fp32 columns are two of them
    a.vec_c = a.vec_c && mult((int64_t)(uintptr_t)d->sgd_master, 16) &&
              (!d->sgd_weights || mult((int64_t)(uintptr_t)d->sgd_weights, 16));
  RTP_REQUIRE(!d->a_rowsum || rowsum_fused<T>(d),
              "rtp_gemm: a_rowsum needs A stored K x M, batch == 1, 16 bytes or more along either operand's contiguous axis and a product "
              "beyond 64 x 64 x 256 (rtp_gemm_rowsum_fused)");
  if (is_tiny(d)) {
    // one wavefront per 32 x 32 block
    a.tiles_m = (int)ceil_div(d->m, 32);
    a.tiles_n = (int)ceil_div(d->n, 32);
    const int64_t nblocks = (int64_t)a.tiles_m * a.tiles_n * nz;
    RTP_REQUIRE(ceil_div(nblocks, 4) < (1ll << 31), "gemm grid too large");
    static const char* const tiny_names[2][2][2] = {
        {{"gemm_f32_tiny_rc_rc", "gemm_f32_tiny_rc_kc"}, {"gemm_f32_tiny_kc_rc", "gemm_f32_tiny_kc_kc"}},
        {{"gemm_bf16_tiny_rc_rc", "gemm_bf16_tiny_rc_kc"}, {"gemm_bf16_tiny_kc_rc", "gemm_bf16_tiny_kc_kc"}}};
    const double mn_ = (double)d->m * (double)d->n * (double)nz, kk_ = (double)d->k * (double)d->ksegs;
    ProfileScope prof(s, tiny_names[sizeof(T) == 2][akc][bkc], 2.0 * mn_ * kk_,
                      ((double)d->m + (double)d->n) * kk_ * nz * sizeof(T) + mn_ * sizeof(T));
    dim3 tgrid((unsigned)ceil_div(nblocks, 4));
    if (akc && bkc)
      hipLaunchKernelGGL((gemm_tiny_kernel<T, true, true>), tgrid, dim3(kThreads), 0, s, a, (long)nblocks);
    else if (akc && !bkc)
      hipLaunchKernelGGL((gemm_tiny_kernel<T, true, false>), tgrid, dim3(kThreads), 0, s, a, (long)nblocks);
    else if (!akc && bkc)
      hipLaunchKernelGGL((gemm_tiny_kernel<T, false, true>), tgrid, dim3(kThreads), 0, s, a, (long)nblocks);
    else
      hipLaunchKernelGGL((gemm_tiny_kernel<T, false, false>), tgrid, dim3(kThreads), 0, s, a, (long)nblocks);
    RTP_LAUNCH_CHECK();
    return RTP_OK;
  }
  const bool relu = d->flags & RTP_GEMM_RELU;
  const int64_t k_all = d->k * d->ksegs;
  if (plan && (!a.vec_c || few_tiles<T>(d) != 0 || k_all <= 128)) return RTP_OK;
  if (!packed && !in_order && takes_kwaves<T>(d)) {
    const int kw_bm = few_tiles<T>(d);
    a.tiles_m = (int)ceil_div(d->m, kw_bm);
    a.tiles_n = (int)ceil_div(d->n, 32);
    static const char* const names[2][2][2] = {{{"gemm_f32_kwaves_rc_rc", "gemm_f32_kwaves_rc_kc"}, {"gemm_f32_kwaves_kc_rc", "gemm_f32_kwaves_kc_kc"}},
                                               {{"gemm_bf16_kwaves_rc_rc", "gemm_bf16_kwaves_rc_kc"}, {"gemm_bf16_kwaves_kc_rc", "gemm_bf16_kwaves_kc_kc"}}};
    const double mn_ = (double)d->m * (double)d->n * (double)nz, kk_ = (double)d->k * (double)d->ksegs;
    ProfileScope prof(s, names[sizeof(T) == 2][akc][bkc], 2.0 * mn_ * kk_,
                      ((double)d->m + (double)d->n) * kk_ * nz * sizeof(T) + mn_ * sizeof(T));
    return launch_kwaves(s, a, kw_bm, sizeof(T) == 2, akc, bkc, direct, dim3((unsigned)(a.tiles_m * a.tiles_n), (unsigned)nz));
  }
  // Many outputs, at most two K slabs: see gemm_shortk.hip.  From 384 of its tiles on it is ahead, in every layout; with 256, one
  // workgroup a CU, it is behind (us, before -> this, bf16: 2048 x 2048 x 64 7.0 -> 7.0, 1024 x 4096 x 96 7.6 -> 8.1, 4096 x 1536 x 32
  // 9.0 -> 8.0, 2048 x 8192 x 96 16.7 -> 13.3; three slabs: 8192 x 1536 x 256 18.8 -> 17.0 in bf16, but 66 -> 70 in fp32).
  if (direct && !packed && a.vec_c && !d->xent_mode && nz < 65536 && k_all * (int64_t)sizeof(T) <= 256 &&
      ceil_div(d->m, 128) * ceil_div(d->n, 128) * nz >= 384) {
    a.tiles_m = (int)ceil_div(d->m, 128);
    a.tiles_n = (int)ceil_div(d->n, 128);
    a.d_tiles_n = make_fastdiv((unsigned)a.tiles_n);
    static const char* const names[2][2][2] = {
        {{"gemm_f32_128x128_shortk_rc_rc", "gemm_f32_128x128_shortk_rc_kc"}, {"gemm_f32_128x128_shortk_kc_rc", "gemm_f32_128x128_shortk_kc_kc"}},
        {{"gemm_bf16_128x128_shortk_rc_rc", "gemm_bf16_128x128_shortk_rc_kc"},
         {"gemm_bf16_128x128_shortk_kc_rc", "gemm_bf16_128x128_shortk_kc_kc"}}};
    const double mn_ = (double)d->m * (double)d->n * (double)nz, kk_ = (double)d->k * (double)d->ksegs;
    ProfileScope prof(s, names[sizeof(T) == 2][akc][bkc], 2.0 * mn_ * kk_,
                      ((double)d->m + (double)d->n) * kk_ * nz * sizeof(T) + mn_ * sizeof(T));
    return launch_shortk(s, a, sizeof(T) == 2, akc, bkc, dim3((unsigned)(a.tiles_m * a.tiles_n), (unsigned)nz));
  }
  // few fp32 weight-gradient tiles, long contraction: see gemm_ksplit_kernel.  128 tiles of 64 x 64 are 512 of its workgroups, two a
  // CU, and it is ahead of the tiles of gemm_split_kernel, which take the same time for 65 tiles as for 256; with three it is
  // behind.  us, gemm_split_kernel -> this, K = 512 / 2048 / 4096: 512 x 576 13.7 / 36 / 65 -> 13.3 / 25 / 40, 512 x 1024
  // 14.1 / 36 / 65 -> 13.3 / 32 / 53, 256 x 2048 13.9 / 36 / 65 -> 13.6 / 37 / 61; 768 x 768 (144 tiles) 14.3 / 36 / 65 against
  // 18.9 / 37 / 60.
  if (sizeof(T) == 4 && fast && !akc && !bkc && !d->sgd_master && !d->xent_mode && d->k >= 512 && nz < 65536 &&
      ceil_div(d->m, 64) * ceil_div(d->n, 64) * nz <= 128) {
    a.tiles_m = (int)ceil_div(d->m, 32);
    a.tiles_n = (int)ceil_div(d->n, 32);
    const double mn_ = (double)d->m * (double)d->n * (double)nz, kk_ = (double)d->k * (double)d->ksegs;
    ProfileScope prof(s, "gemm_f32_32x32_ksplit_rc_rc", 2.0 * mn_ * kk_,
                      ((double)d->m + (double)d->n) * kk_ * nz * sizeof(T) + mn_ * sizeof(T));
    hipLaunchKernelGGL(gemm_ksplit_kernel, dim3((unsigned)(a.tiles_m * a.tiles_n), (unsigned)nz), dim3(64 * kSplitWaves), 0, s, a);
    RTP_LAUNCH_CHECK();
    return RTP_OK;
  }
  // Tile choice by a cost model: the launch runs in ceil(tiles / 256 CUs) rounds, a round costs the tile's
  // measured time per K slab (ns, 4096^3 bf16 on MI355X: bigger tiles do ~30 % more outputs per ns, so what
  // decides is mostly how evenly the tile count fills the CUs) plus a fixed prologue / epilogue.  Only the ratios of
  // the prices matter: with every CU busy on operands from memory all shapes take 1.2 - 1.4 times theirs.
  static const int forced = [] {
    const char* e = getenv("RTP_GEMM_TILE");  // debugging aid: index into kShapes
    return e ? atoi(e) : -1;
  }();
  static const double slab_ns[kNumShapes] = {966.0, 470.0, 283.0, 167.0, 800.0, kLargeSlabNs, 545.0};
  static const double fixed_ns[kNumShapes] = {3000.0, 3000.0, 3000.0, 3000.0, 3000.0, kLargeTileNs, 3000.0};  // per tile outside the K loop
  // The two tiles for operands or outputs of any alignment, 64 x 64 and 128 x 128: the register loaders make a slab take nearly twice as
  // long and the larger tile's share outside the loop 10 us; where only the results are unaligned that is 4.  Either tile forced on 20 odd
  // shapes x 3 layouts: with these prices the one taken costs 0.1 % over the better one in the mean (with 14.5 us, the price of an
  // element-wise epilogue, 0.3 %).  us, 64 x 64 / 128 x 128, bf16: 3864 x 321 x 201 10.5 / 12.6, 1024 x 3001 x 4096 55 / 43, 2001 x 2003 x 2005
  // 50 / 33, 1000 x 501 x 512 with 4 shards (weight gradient) 13.3 / 26.3, 4096 x 1023 x 512 15.3 / 11.8 (1024 wide 15.0 / 10.8); fp32 3222 x 4321 x 137 70 / 75.
  static const double odd_slab_ns[2][2] = {{330.0, 750.0}, {480.0, 2100.0}}, odd_fixed_ns[2][2] = {{3600.0, 10000.0}, {3500.0, 4000.0}};
  static const int slab_bytes[kNumShapes] = {128, 128, 128, 128, 128, 128, 128};
  const bool vec = direct && a.vec_c;  // else the kernels for operands of any alignment
  constexpr double kNever = 1e300;
  const bool whole_lines = mult((int64_t)(uintptr_t)d->sgd_master, 128) && mult(d->ldc, 32) && (d->groups == 1 || mult(d->c_sg, 32)) &&
                           (d->batch == 1 || (mult(d->c_so, 32) && mult(d->c_si, 32)));
  // ns of the first `m` rows in tiles of shape i
  const auto price = [&](int i, int64_t m) {
    // the 256 x 256 kernel is built for 16-bit operands and has no statistics epilogue (never routed to it, forced or not)
    if (i == 5 && (sizeof(T) != 2 || d->xent_mode == 1)) return kNever;
    // ... and an update only where it is a weight gradient's and the parameters' rows are whole 128-byte lines in every group: its waves write
    // 64 columns each.  us, 128 x 128 or 256 x 128 tiles / these, parameters from memory: rows that are not, 3000 x 3000 x 512, 38 / 49; 8 groups of 1024 x
    // 2048 x 1024 that lie 32, 64 and 128 bytes beyond a line apart 69.9 / 95.8, 69.3 / 78.0 and 68.9 / 64.9; 2 of 6144 x 2048 118.9 / 133.9, 108.9 / 115.7, 105.0 / 102.6
    if (i == 5 && d->sgd_master && (akc || bkc || !whole_lines)) return kNever;
    if (i == 6 && d->xent_mode == 1) return kNever;  // 160 columns are no whole number of 64-column statistics blocks
    if (!vec && i != 1 && i != 3) return kNever;  // the kernels for unaligned operands: 128 x 128 and 64 x 64
    // 128 x 160 is priced at the rate measured where it is meant for -- products of at most two rounds of tiles, such
    // as the LM's logits layer (shards of 1280 columns); larger products keep the shapes measured on large products
    if (i == 6 && ceil_div(m, 128) * ceil_div(d->n, 160) * nz > 512 && i != forced) return kNever;
    // It needs neither a full round nor a long contraction to pay: on 144 - 255 tiles it is one round where the others take
    // two or more (6000 x 2048 x 2048, 192 tiles: 51 us against 57 with 128 x 128 and 65 with 256 x 128), and at K = 512 it is
    // 89 us against 123 (8192^2).
    if (i == 5 && ceil_div(d->k, 64) * d->ksegs < 2) return kNever;  // its pipeline is primed with two slabs
    // never a tile that is mostly padding: a 32 x 32 problem (one attention head at seq 32) stays at 64 x 64
    if ((!akc && (kShapes[i].bm & (kShapes[i].bm - 1))) || (!bkc && (kShapes[i].bn & (kShapes[i].bn - 1)))) return kNever;
    if (kShapes[i].bm > 64 && kShapes[i].bm > ceil_div(m, 64) * 64) return kNever;
    if (kShapes[i].bn > 64 && kShapes[i].bn > ceil_div(d->n, 64) * 64) return kNever;
    const int64_t tiles = ceil_div(m, kShapes[i].bm) * ceil_div(d->n, kShapes[i].bn) * nz;
    const double nslabs = (double)ceil_div(d->k * (int64_t)sizeof(T), slab_bytes[i]) * (double)d->ksegs;
    const double rounds = (double)ceil_div(tiles, 256);
    const double update = d->sgd_master && vec ? update_ns((double)tiles, (double)kShapes[i].bm * kShapes[i].bn * update_bytes(d)) : 0.0;
    if (i == 5) return large_ns(rounds, nslabs, rare_epilogue(d)) + update;
    const double slab = vec || direct ? slab_ns[i] : odd_slab_ns[sizeof(T) == 4][i == 1];
    return rounds * (nslabs * slab + (vec ? fixed_ns[i] : odd_fixed_ns[direct][i == 1])) + update;
  };
  const auto cheapest = [&](int64_t m, int& shape) {
    double best = kNever;
    shape = 3;  // 64 x 64 unless the model finds something cheaper
    for (int i = 0; fast && i < kNumShapes; ++i) {
      const double cost = price(i, m);
      if (cost != kNever && i == forced) return shape = i, -1.0;
      if (cost < best) best = cost, shape = i;
    }
    return best;
  };
  int shape;
  const double best = cheapest(d->m, shape);
  // A last round of few 256 x 256 tiles takes as long as a full one, and a last row of tiles that is mostly padding as long as the others:
  // whole rounds' rows (or whole tiles' rows) go in those, the others in the tiles that suit them, where the two launches are priced 5 %
  // below the one.  us, one launch -> two, forward / input gradient / weight gradient layouts: 4352 x 4096 x 4096 159 / 165 / 178 -> 120 / 125 / 129, 6144
  // x 3072 x 4096 159 / 165 / 178 -> 127 / 133 / 136, 4608 x 4096 x 2048 84 / 87 / 95 -> 71 / 74 / 76, 6000 x 6144 x 2048 161 / 150 / 157 -> 147 / 139 /
  // 141, 2300 x 8192 x 2048 89 / 92 -> 68 / 71, 3000 x 6144 x 3000 131 / 131 / 143 -> 109 / 105 / 105; level, so not taken: 5632 x 4096 x 1024 47,
  // 4096 x 6144 x 2048 87, 9000 x 5120 x 1536 112.
  // Few rows behind the cut stay with these tiles too, in the order of the sums before it: gemm_kwaves.hip would be faster, us, this / that, 4128 x
  // 4096 x 2048 70 / 73 / 76 against 66 / 70 / 75, 4104 x 4096 x 8192 234 / 245 / 262 against 217 / 236 / 256, but equal rows would differ.
  if (shape == 5 && best > 0.0 && !plan && !packed && !d->xent_mode) {
    const int64_t row_tiles = ceil_div(d->n, 256) * nz, rounds = ceil_div(ceil_div(d->m, 256) * row_tiles, 256);
    double least = 0.95 * best;
    int64_t cut = 0;
    const auto consider = [&](int64_t m) {
      int other;
      if (m <= 0 || m >= d->m) return;
      const double cost = price(5, m) + cheapest(d->m - m, other) + 4000.0;
      if (cost < least) least = cost, cut = m;
    };
    for (int64_t r = std::max<int64_t>(1, rounds - 2); r < rounds; ++r) consider(256 * r / row_tiles * 256);
    consider(d->m / 256 * 256);
    if (cut != 0) {
      rtp_gemm_desc part = *d;
      const int64_t es = (int64_t)sizeof(T);
      part.m = cut;
      if (int rc = launch_gemm<T>(s, &part, nullptr, true)) return rc;
      const auto down = [&](const void* x, int64_t ld, int64_t size) { return x ? (char*)x + cut * ld * size : nullptr; };
      part.m = d->m - cut;
      part.a = down(d->a, akc ? d->lda : 1, es);
      part.c_out = down(d->c_out, d->ldc, d->flags & RTP_GEMM_OUT_F32 ? 4 : es);
      part.c_in = down(d->c_in, d->ld_cin, d->flags & RTP_GEMM_CIN_F32 ? 4 : es);
      part.gate = down(d->gate, d->ld_gate, es);
      part.a_rowsum = down(d->a_rowsum, 1, es);
      part.sgd_master = down(d->sgd_master, d->ldc, 4), part.sgd_weights = down(d->sgd_weights, d->ldc, es);
      return launch_gemm<T>(s, &part, nullptr, true);
    }
  }
  if (plan) {
    if (price(5, d->m) == kNever) return RTP_OK;
    plan->large = true, plan->rare = rare_epilogue(d), plan->alone = best;  // (what fits a round is not cut)
    plan->slabs = (double)ceil_div(d->k, 64) * (double)d->ksegs;
    plan->update_bytes = (double)(ceil_div(d->m, 256) * ceil_div(d->n, 256) * nz) * 65536.0 * update_bytes(d);
    shape = 5;
  }
  // fp32 contractions of 384 and more go to gemm_split.hip, whose K loop is 1.2 - 1.9 times as fast and whose prologue and epilogue
  // are 1 - 2 us longer (a workgroup fills a CU there): us, fp32 MFMA -> this, forward layout: 64 matrices of 420 x 420 with
  // K = 128 76 -> 78, 160 84 -> 81, 320 119 -> 104; 2048 x 512 with K = 224 9.1 -> 9.5, 320 10.5 -> 10.8; 1600 x 512 x 512 12.9 -> 13.0;
  // 1024 x 2048 x 2048 74 -> 60; 8 of 122 x 1088 x 1536 51 -> 35.
  // Its two tiles cost 700 and 430 ns a slab and 4 us a round with every CU busy.  (The launches that take 128 x 160 tiles, two even
  // rounds of an fp32 logits layer, stay with them.)
  const bool split = sizeof(T) == 4 && fast && !relu && k_all >= 384 && shape != 6;
  if (split) {
    const double nslabs = (double)ceil_div(d->k, 32) * (double)d->ksegs;
    const auto cost = [&](int bm, double slab) {
      return (double)ceil_div(ceil_div(d->m, bm) * ceil_div(d->n, 64) * nz, 256) * (nslabs * slab + 4000.0);
    };
    shape = (forced == 2 || forced == 3) ? forced : cost(128, 700.0) < cost(64, 430.0) ? 2 : 3;
  }
  const TileShape& ts = kShapes[shape];
  a.tiles_m = (int)ceil_div(d->m, ts.bm);
  a.tiles_n = (int)ceil_div(d->n, ts.bn);
  const int64_t nb = (int64_t)a.tiles_m * a.tiles_n;
  RTP_REQUIRE(nb < (1ll << 31) && nz < 65536, "gemm grid too large (%lld tiles, %lld batch*groups)", (long long)nb,
              (long long)nz);
  dim3 grid((unsigned)nb, (unsigned)nz, 1);
  // XCD bricks: among the splits xg*xm*xn == 8 that divide the launch evenly, take the one with the fewest
  // operand bytes per XCD (A rows x K of the brick's row tiles, B likewise; an operand that differs per
  // batch/group entry counts once per entry of the brick).
  a.xg = a.xm = a.xn = 0;
  if (fast) {
    const bool a_per_z = d->batch > 1 || (d->groups > 1 && d->a_sg != 0);
    const bool b_per_z = d->batch > 1 || (d->groups > 1 && d->b_sg != 0);
    double best = 0.0;
    for (int xg = 1; xg <= 8; xg *= 2)
      for (int xm = 1; xg * xm <= 8; xm *= 2) {
        const int xn = 8 / (xg * xm);
        if (nz % xg || a.tiles_m % xm || a.tiles_n % xn) continue;
        const double zb = (double)(nz / xg);
        const double cost = (double)(a.tiles_m / xm) * ts.bm * (a_per_z ? zb : 1.0) +
                            (double)(a.tiles_n / xn) * ts.bn * (b_per_z ? zb : 1.0);
        if (a.xg == 0 || cost < best) {
          best = cost;
          a.xg = xg;
          a.xm = xm;
          a.xn = xn;
        }
      }
  }

  a.d_batch = make_fastdiv((unsigned)d->batch);
  a.d_zdiv = make_fastdiv((unsigned)d->zdiv);
  a.d_tiles_n = make_fastdiv((unsigned)a.tiles_n);
  {
    const int nbk = a.xg ? a.tiles_n / a.xn : a.tiles_n, mbk = a.xg ? a.tiles_m / a.xm : a.tiles_m;
    // Panel = prow x pcol tiles, about one round of an XCD's 32 CUs.  pcol: the widest divisor of nbk (at most 32)
    // whose strip of B tiles (pcol * BN rows x all of K) stays within ~3 MB of the XCD's 4 MB L2 -- the A rows stream
    // past the strip once, so the L2 fills are about A * nbk / pcol + B per brick.  prow: the tallest divisor of mbk
    // that keeps the panel within 32 tiles.
    const double b_tile_bytes = (double)ts.bn * (double)d->k * (double)d->ksegs * sizeof(T);
    int pcol = 1;
    for (int c = 2; c <= 32 && c <= nbk; ++c)
      if (nbk % c == 0 && c * b_tile_bytes <= 3.0 * 1024 * 1024) pcol = c;
    // A contraction so long that not even two B tiles fit: nothing stays in the L2 from one panel to the next, and
    // what counts is the block of tiles that run at the same time and walk K side by side -- as square as it gets
    // (a 16 x 1 column shares one B tile but streams 16 A tiles; 8 x 4 streams 12 tile-operands for 32 CUs).
    if (pcol == 1)
      for (int c = 2; c <= 4 && c <= nbk; ++c)
        if (nbk % c == 0) pcol = c;
    int prow = 1;
    for (int r = 2; r * pcol <= 32 && r <= mbk; ++r)
      if (mbk % r == 0) prow = r;
    a.mbk = mbk, a.nbk = nbk;
    a.prow = prow, a.pcol = pcol;
    a.d_brick = make_fastdiv((unsigned)(nbk * mbk));
    a.d_panel = make_fastdiv((unsigned)(prow * pcol));
    a.d_prow = make_fastdiv((unsigned)prow);
    a.d_pm = make_fastdiv((unsigned)(mbk / prow));
  }
  a.xn_shift = a.xn == 8 ? 3 : a.xn == 4 ? 2 : a.xn == 2 ? 1 : 0;
  a.xm_shift = a.xm == 8 ? 3 : a.xm == 4 ? 2 : a.xm == 2 ? 1 : 0;
  a.zbk = a.xg ? (int)(nz / a.xg) : 0;
  a.tiles = (unsigned)(nb * nz);
  a.per_xcd = (unsigned)ceil_div(nb * nz, 8);

  // variant name = the kernel template instance, e.g. gemm_bf16_128x64_kc_kc
  static const char* const layout_tag[2][2] = {{"rc_rc", "rc_kc"}, {"kc_rc", "kc_kc"}};
  static thread_local char names[2][2][kNumShapes + 3][2][2][40];
  char* name = names[sizeof(T) == 2][vec][split ? kNumShapes - 1 + shape : fast ? shape : kNumShapes][akc][bkc];
  if (!name[0])
    snprintf(name, 40, "gemm_%s_%s%s%s_%s", sizeof(T) == 2 ? "bf16" : "f32", fast ? ts.tag : "64x64_guarded",
             split ? "_split" : "", fast && !vec ? "_unaligned" : "", layout_tag[akc][bkc]);
  const double mn = (double)d->m * (double)d->n * (double)nz;
  const double kk = (double)d->k * (double)d->ksegs;
  const double out_sz = (d->flags & RTP_GEMM_OUT_F32) ? 4.0 : (double)sizeof(T);
  const double cin_sz = d->c_in ? ((d->flags & RTP_GEMM_CIN_F32) ? 4.0 : (double)sizeof(T)) : 0.0;
  // operands once + the output (and addend); a fused update reads and writes the fp32 parameters and writes their copy
  const double upd_sz = d->sgd_master ? 8.0 + (d->sgd_weights ? (double)sizeof(T) : 0.0) -
                                            ((d->flags & RTP_GEMM_SGD_SKIP_OUT) ? out_sz : 0.0)
                                      : 0.0;
  // An operand that every group / batch entry / K segment reads from the same address (stride 0: the activations of a
  // column layer's forward and weight-gradient products) is counted once, not once per shard.
  const auto copies = [&](int64_t so, int64_t si, int64_t sg, int64_t sk) {
    const double per_batch = (d->batch > 1 && (so != 0 || si != 0)) ? (double)d->batch : 1.0;
    const double per_group = (d->groups > 1 && sg != 0) ? (double)d->groups : 1.0;
    const double per_kseg = (d->ksegs > 1 && sk != 0) ? (double)d->ksegs : 1.0;
    return per_batch * per_group * per_kseg;
  };
  const double bytes = ((double)d->m * copies(d->a_so, d->a_si, d->a_sg, d->a_sk) +
                        (double)d->n * copies(d->b_so, d->b_si, d->b_sg, d->b_sk)) * (double)d->k * sizeof(T) +
                       mn * (out_sz + cin_sz + upd_sz);
  a.warm = nullptr;
  if (plan) {
    a.trace = nullptr;
    plan->args = a, plan->flops = 2.0 * mn * kk, plan->bytes = bytes;
    return RTP_OK;
  }
  ProfileScope prof(s, name, 2.0 * mn * kk, bytes);
  a.trace = fast ? prof.trace_slot() : nullptr;
  if (!fast) return launch_layout<T, 64, 64, 1, false>(s, a, akc, bkc, grid);
  // Carried by the kernels whose MFMA waves wait for loader waves at their start.  In the others every wave's own loads would queue
  // behind the hint's.  fp32 products lose nothing by it, their slabs take longer than HBM does: us, weights in the memory-side
  // cache / in HBM, 1024 x 2048 x 2048 split 56 - 61 / 58 - 60, with fp32 MFMAs 77 / 71, 1024 x 6144 x 2048 164 / 164 and 196 / 184.
  // Few rows do (bf16 64 x 2048 x 2048 6.3 / 8.5, input gradient 7.0 / 11.9; fp32 13.5 / 15.3), and are ahead of the tiles that
  // carry hints all the same (gemm_kwaves.hip).
  if (shape != 5 && !split && warm_src != nullptr)
    warm_launch(a, warm_src, t_warm_bytes, (int64_t)grid.x * grid.y, ceil_div(d->k, (int64_t)(128 / sizeof(T))) * d->ksegs);
  if (split) return launch_split(s, a, akc, bkc, ts.bm, !vec, grid);
  if (!vec) {
    if (direct)
      return shape == 1 ? launch_unaligned<T, 128, 128, 4, 128, 1, false>(s, a, akc, bkc, grid)
                        : launch_unaligned<T, 64, 64, 4, 128, 3, false>(s, a, akc, bkc, grid);
    return shape == 1 ? launch_unaligned<T, 128, 128, 4, 128, 1, true>(s, a, akc, bkc, grid)
                      : launch_unaligned<T, 64, 64, 4, 128, 3, true>(s, a, akc, bkc, grid);
  }
  switch (shape) {
    case 0:
      return launch_dma<T, 256, 128, 3, 128, 1>(s, a, akc, bkc, grid);
    case 1:
      // prefetch distance 1: as fast as 3 on every measured shape, and 168 instead of 213 registers per wave for
      // the weight-gradient layout -- with two such waves per SIMD the 120-register waves of the LayerNorm backward
      // kernel on the other stream fit beside them instead of waiting for a workgroup to leave the CU
      return launch_dma<T, 128, 128, 4, 128, 1>(s, a, akc, bkc, grid);
    case 2:
      return launch_dma<T, 128, 64, 5, 128, 4>(s, a, akc, bkc, grid);
    case 4:
      return launch_dma<T, 128, 192, 3, 128, 2>(s, a, akc, bkc, grid);
    case 6:
      // 4 x 1 wave tiles of 32 x 160: a layer whose shards are 1280 columns wide (the LM's logits) is 8 tiles per
      // shard and fills the CUs in two even rounds where 128 x 128 tiles need two and a half
      return launch_dma<T, 128, 160, 4, 128, 1>(s, a, akc, bkc, grid);
    case 5:
      if constexpr (sizeof(T) == 2) return launch_large(s, a, akc, bkc);
      return fail(RTP_ERR_ARG, "gemm: no 256 x 256 kernel for this dtype");
    default:
      return launch_dma<T, 64, 64, 4, 128, 3>(s, a, akc, bkc, grid);
  }
}

// ---------------------------------------------------------------------------------------------
// Column sums (bias gradients) in two deterministic passes: 64 columns x a block of rows per
// workgroup into fp32 partials, then a fixed-order sum of the partials.
constexpr int kColsumRows = 64;

template <typename T>
__global__ __launch_bounds__(kThreads) void colsum_partial_kernel(const T* x, long m, long n, long ld, float* part) {
  __shared__ float red[4][64];
  const int c = threadIdx.x & 63, ph = threadIdx.x >> 6;
  const long col = (long)blockIdx.x * 64 + c;
  const long r0 = (long)blockIdx.y * kColsumRows;
  const long r1 = r0 + kColsumRows < m ? r0 + kColsumRows : m;
  float s0 = 0.f, s1 = 0.f, s2 = 0.f, s3 = 0.f;
  if (col < n) {
    long r = r0 + ph;
    for (; r + 12 < r1; r += 16) {
      s0 += to_f32(x[r * ld + col]);
      s1 += to_f32(x[(r + 4) * ld + col]);
      s2 += to_f32(x[(r + 8) * ld + col]);
      s3 += to_f32(x[(r + 12) * ld + col]);
    }
    for (; r < r1; r += 4) s0 += to_f32(x[r * ld + col]);
  }
  red[ph][c] = (s0 + s1) + (s2 + s3);
  __syncthreads();
  if (ph == 0 && col < n) part[(long)blockIdx.y * n + col] = (red[0][c] + red[1][c]) + (red[2][c] + red[3][c]);
}

// Single-pass variant for a few thousand rows: one workgroup of 512 threads owns 32 columns; each thread walks
// its rows with 16-byte loads (VEC columns, 4 loads in flight), and the per-thread sums are combined through LDS
// in a fixed order (row groups in 4 quarters, then the quarters).
constexpr int kOnepassThreads = 512, kOnepassCols = 32;
template <typename T>
__global__ __launch_bounds__(kOnepassThreads) void colsum_onepass_kernel(const T* x, long m, long n, long ld, void* out,
                                                                         long seg, long seg_stride, int out_f32,
                                                                         int accumulate) {
  constexpr int VEC = 16 / sizeof(T), LPR = kOnepassCols / VEC, RG = kOnepassThreads / LPR;
  __shared__ float red[RG][kOnepassCols + 1];
  __shared__ float quarter[4][kOnepassCols];
  const int cl = (threadIdx.x % LPR) * VEC, rg = threadIdx.x / LPR;
  const long col = (long)blockIdx.x * kOnepassCols + cl;
  float acc[VEC];
#pragma unroll
  for (int e = 0; e < VEC; ++e) acc[e] = 0.0f;
  if (col < n) {  // n is a multiple of VEC, so the vector is wholly inside
    union V {
      uint4 q;
      T e[VEC];
    };
    const T* src = x + col;
    long r = rg;
    for (; r + 3 * RG < m; r += 4 * RG) {
      V u0, u1, u2, u3;
      u0.q = *reinterpret_cast<const uint4*>(src + r * ld);
      u1.q = *reinterpret_cast<const uint4*>(src + (r + RG) * ld);
      u2.q = *reinterpret_cast<const uint4*>(src + (r + 2 * RG) * ld);
      u3.q = *reinterpret_cast<const uint4*>(src + (r + 3 * RG) * ld);
#pragma unroll
      for (int e = 0; e < VEC; ++e) acc[e] += (to_f32(u0.e[e]) + to_f32(u1.e[e])) + (to_f32(u2.e[e]) + to_f32(u3.e[e]));
    }
    for (; r < m; r += RG) {
      V u;
      u.q = *reinterpret_cast<const uint4*>(src + r * ld);
#pragma unroll
      for (int e = 0; e < VEC; ++e) acc[e] += to_f32(u.e[e]);
    }
  }
#pragma unroll
  for (int e = 0; e < VEC; ++e) red[rg][cl + e] = acc[e];
  __syncthreads();
  if (threadIdx.x < 4 * kOnepassCols) {
    const int c = threadIdx.x % kOnepassCols, qd = threadIdx.x / kOnepassCols;
    float v = 0.0f;
    for (int r = qd * (RG / 4); r < (qd + 1) * (RG / 4); ++r) v += red[r][c];
    quarter[qd][c] = v;
  }
  __syncthreads();
  const long c = (long)blockIdx.x * kOnepassCols + threadIdx.x;
  if (threadIdx.x < kOnepassCols && c < n) {
    const int t = threadIdx.x;
    const float v = (quarter[0][t] + quarter[1][t]) + (quarter[2][t] + quarter[3][t]);
    const long o = (c / seg) * seg_stride + c % seg;
    if (out_f32) {
      float* dst = reinterpret_cast<float*>(out);
      dst[o] = accumulate ? dst[o] + v : v;
    } else {
      T* dst = reinterpret_cast<T*>(out);
      dst[o] = from_f32<T>(accumulate ? to_f32(dst[o]) + v : v);
    }
  }
}

// out index of column c: (c / seg) * seg_stride + c % seg  (bias slices of consecutive shards sit
// seg_stride elements apart in the flat gradient buffer).
template <typename T>
__global__ __launch_bounds__(kThreads) void colsum_final_kernel(const float* part, long nparts, long n, void* out,
                                                                long seg, long seg_stride, int out_f32,
                                                                int accumulate) {
  const long col = (long)blockIdx.x * kThreads + threadIdx.x;
  if (col >= n) return;
  float v = 0.0f;
  for (long p = 0; p < nparts; ++p) v += part[p * n + col];
  const long o = (col / seg) * seg_stride + col % seg;
  if (out_f32) {
    float* dst = reinterpret_cast<float*>(out);
    dst[o] = accumulate ? dst[o] + v : v;
  } else {
    T* dst = reinterpret_cast<T*>(out);
    dst[o] = from_f32<T>(accumulate ? to_f32(dst[o]) + v : v);
  }
}

}  // namespace rtp

static int check_gemm(const rtp_gemm_desc* d) {
  using namespace rtp;
  RTP_REQUIRE(d != nullptr, "rtp_gemm: null descriptor");
  RTP_REQUIRE(d->a && d->b && d->c_out, "rtp_gemm: null operand pointer");
  RTP_REQUIRE(d->m >= 0 && d->n >= 0 && d->k >= 0, "rtp_gemm: negative extent m=%lld n=%lld k=%lld",
              (long long)d->m, (long long)d->n, (long long)d->k);
  RTP_REQUIRE(d->m < (1ll << 31) && d->n < (1ll << 31) && d->k < (1ll << 31), "rtp_gemm: extent exceeds int32");
  RTP_REQUIRE(d->batch >= 1 && d->zdiv >= 1 && d->groups >= 1 && d->ksegs >= 1,
              "rtp_gemm: batch=%lld zdiv=%lld groups=%lld ksegs=%lld must be >= 1", (long long)d->batch,
              (long long)d->zdiv, (long long)d->groups, (long long)d->ksegs);
  RTP_REQUIRE(d->k * d->ksegs < (1ll << 31), "rtp_gemm: total contraction length exceeds int32");
  RTP_REQUIRE(d->lda >= 1 && d->ldb >= 1 && d->ldc >= 1, "rtp_gemm: leading dimensions must be >= 1");
  RTP_REQUIRE(!d->c_in || d->ld_cin >= 1, "rtp_gemm: ld_cin must be >= 1 when c_in is given");
  RTP_REQUIRE(!d->gate || d->ld_gate >= 1, "rtp_gemm: ld_gate must be >= 1 when gate is given");
  return RTP_OK;
}

extern "C" int rtp_gemm(void* stream, int dtype, const rtp_gemm_desc* d) {
  using namespace rtp;
  if (int rc = check_gemm(d)) return rc;
  if (d->m == 0 || d->n == 0) return RTP_OK;
  hipStream_t s = (hipStream_t)stream;
  if (dtype == RTP_F32) return launch_gemm<float>(s, d);
  if (dtype == RTP_BF16) return launch_gemm<bf16_t>(s, d);
  return fail(RTP_ERR_ARG, "rtp_gemm: unknown dtype %d", dtype);
}

extern "C" int rtp_gemm_pair(void* stream, int dtype, const rtp_gemm_desc* first, const rtp_gemm_desc* second) {
  using namespace rtp;
  RTP_REQUIRE(first && second, "rtp_gemm_pair: null descriptor");
  // A round of 256 x 256 tiles that leaves CUs idle takes a second product's tiles along.  It pays by the prices of the products alone: the
  // longer contraction, one epilogue, both updates at the memory's rate.  us, one after the other -> together, attention layers of width 2048
  // (64 + 192 tiles): causal over 4096 rows, forward + backward, 512 -> 496; padded over 6000 rows 1024 -> 997; LM step of 10 blocks over 992
  // rows, Adam, 4842 -> 4679, over 1024 with the update in the epilogues 3863 -> 3729.
  // Updates of parameters in memory, us, apart / together, tiles: 64 + 192, K = 1024 72.8 / 64.7; 49 + 147 67.3 / 58.3; 64 + 64, K = 640 38.9 / 37.2; 36 +
  // 108, K = 640 44.1 / 41.8, 2048 67.8 / 70.0; the floor of a CU's rate that update_ns has would keep all but the first two apart.
  if (dtype == RTP_BF16 && first->m > 0 && second->m > 0 && first->n > 0 && second->n > 0 && first->k > 0 && second->k > 0) {
    hipStream_t s = (hipStream_t)stream;
    PairPlan p[2];
    for (int i = 0; i < 2; ++i)
      if (int rc = check_gemm(i ? second : first)) return rc;
    for (int i = 0; i < 2; ++i) {
      if (int rc = launch_gemm<bf16_t>(s, i ? second : first, &p[i])) return rc;
      if (!p[i].large) break;
    }
    if (p[0].large && p[1].large && p[0].args.per_xcd + p[1].args.per_xcd <= 32) {
      const double together = large_ns(1.0, std::max(p[0].slabs, p[1].slabs), p[0].rare || p[1].rare) +
                              (p[0].update_bytes + p[1].update_bytes) / 4900.0;
      if (together < p[0].alone + p[1].alone) {
        t_warm_src = nullptr;  // 256 x 256 tiles carry no hint; it ends here
        ProfileScope prof(s, "gemm_bf16_256x256_pair_rc_rc", p[0].flops + p[1].flops, p[0].bytes + p[1].bytes);
        return launch_large_pair(s, p[0].args, p[1].args);
      }
    }
  }
  if (int rc = rtp_gemm(stream, dtype, first)) return rc;
  return rtp_gemm(stream, dtype, second);
}

extern "C" int rtp_gemm_rowsum_fused(int dtype, const rtp_gemm_desc* d) {
  using namespace rtp;
  if (!d || !d->a || !d->b || d->m <= 0 || d->n <= 0 || d->k <= 0 || d->groups < 1 || d->ksegs < 1) return 0;
  if (dtype == RTP_F32) return rowsum_fused<float>(d) ? 1 : 0;
  if (dtype == RTP_BF16) return rowsum_fused<bf16_t>(d) ? 1 : 0;
  return 0;
}

extern "C" int rtp_gemm_warm_next(const void* src, size_t bytes) {
  RTP_REQUIRE(((uintptr_t)src & 15) == 0, "rtp_gemm_warm_next: source must be 16-byte aligned");
  rtp::t_warm_src = bytes ? src : nullptr;
  rtp::t_warm_bytes = bytes;
  rtp::t_warm_call = ++rtp::g_warm_call;
  return RTP_OK;
}

extern "C" int rtp_gemm_workspace(rtp_alloc_fn alloc, void* context) {
  rtp::t_alloc = alloc, rtp::t_alloc_context = context;
  return RTP_OK;
}

extern "C" int rtp_gemm_warm_pending(void) { return rtp::warm_source() != nullptr; }

extern "C" int rtp_gemm_sgd_fused(int dtype, const rtp_gemm_desc* d) {
  using namespace rtp;
  if (!d || !d->a || !d->b || d->m <= 0 || d->n <= 0 || d->k <= 0 || d->groups < 1 || d->ksegs < 1) return 0;
  if (dtype == RTP_F32) return sgd_fused<float>(d) ? 1 : 0;
  if (dtype == RTP_BF16) return sgd_fused<bf16_t>(d) ? 1 : 0;
  return 0;
}

extern "C" size_t rtp_gemm_desc_size(void) { return sizeof(rtp_gemm_desc); }

extern "C" size_t rtp_colsum_workspace_bytes(int64_t m, int64_t n) {
  using namespace rtp;
  if (m <= 0 || n <= 0) return 256;
  return (size_t)(ceil_div(m, kColsumRows) * n * 4 + 256);
}

extern "C" int rtp_colsum(void* stream, int dtype, const void* x, int64_t m, int64_t n, int64_t ld, void* out,
                          int out_f32, int accumulate, int64_t seg, int64_t seg_stride, void* workspace,
                          size_t workspace_bytes) {
  using namespace rtp;
  RTP_REQUIRE(x && out && workspace, "rtp_colsum: null pointer");
  RTP_REQUIRE(m >= 0 && n >= 0 && ld >= n, "rtp_colsum: bad shape m=%lld n=%lld ld=%lld", (long long)m,
              (long long)n, (long long)ld);
  RTP_REQUIRE(dtype == RTP_F32 || dtype == RTP_BF16, "rtp_colsum: unknown dtype %d", dtype);
  if (n == 0) return RTP_OK;
  if (seg <= 0) {
    seg = n;
    seg_stride = n;
  }
  RTP_REQUIRE(seg_stride >= seg, "rtp_colsum: seg_stride %lld < seg %lld", (long long)seg_stride, (long long)seg);
  const int64_t nparts = std::max<int64_t>(1, ceil_div(m, kColsumRows));
  RTP_REQUIRE(nparts < 65536, "rtp_colsum: too many rows");
  if (workspace_bytes < (size_t)(nparts * n * 4))
    return fail(RTP_ERR_WORKSPACE, "rtp_colsum: workspace %zu < required %lld", workspace_bytes,
                (long long)(nparts * n * 4));
  hipStream_t s = (hipStream_t)stream;
  float* part = (float*)workspace;
  ProfileScope prof(s, "colsum", (double)m * n, (double)m * n * (dtype == RTP_F32 ? 4 : 2));
  const int vec = dtype == RTP_F32 ? 4 : 8;
  if (m <= 4096 && (uintptr_t)x % 16 == 0 && ld % vec == 0 && n % vec == 0) {
    dim3 g1((unsigned)ceil_div(n, kOnepassCols));
    if (dtype == RTP_F32)
      hipLaunchKernelGGL(colsum_onepass_kernel<float>, g1, dim3(kOnepassThreads), 0, s, (const float*)x, (long)m, (long)n,
                         (long)ld, out, (long)seg, (long)seg_stride, 1, accumulate);
    else
      hipLaunchKernelGGL(colsum_onepass_kernel<bf16_t>, g1, dim3(kOnepassThreads), 0, s, (const bf16_t*)x, (long)m, (long)n,
                         (long)ld, out, (long)seg, (long)seg_stride, out_f32, accumulate);
    RTP_LAUNCH_CHECK();
    return RTP_OK;
  }
  dim3 grid((unsigned)ceil_div(n, 64), (unsigned)nparts);
  dim3 grid2((unsigned)ceil_div(n, kThreads));
  if (dtype == RTP_F32) {
    hipLaunchKernelGGL(colsum_partial_kernel<float>, grid, dim3(kThreads), 0, s, (const float*)x, (long)m, (long)n,
                       (long)ld, part);
    hipLaunchKernelGGL(colsum_final_kernel<float>, grid2, dim3(kThreads), 0, s, part, (long)nparts, (long)n, out,
                       (long)seg, (long)seg_stride, 1, accumulate);
  } else {
    hipLaunchKernelGGL(colsum_partial_kernel<bf16_t>, grid, dim3(kThreads), 0, s, (const bf16_t*)x, (long)m, (long)n,
                       (long)ld, part);
    hipLaunchKernelGGL(colsum_final_kernel<bf16_t>, grid2, dim3(kThreads), 0, s, part, (long)nparts, (long)n, out,
                       (long)seg, (long)seg_stride, out_f32, accumulate);
  }
  RTP_LAUNCH_CHECK();
  return RTP_OK;
}
