// fp32 products on the bf16 matrix pipes.
//
// An fp32 number is the sum of three bf16 numbers, each the rounding of what the ones before leave (8 + 8 + 8 bits).  It is taken
// apart 2^24 times as large, so that the last bit of the smallest number, 2^-149, is a normal bf16 number and no part is ever rounded
// or flushed, and the sums are scaled back by 2^-48; numbers of 2^103 and sums of 2^80 and more do not fit and are worked out by
// the fp32 MFMA, see the epilogue.  Of the nine products of two such sums the six whose parts i + j <= 2 reach an fp32 product's last bits;
// v_mfma_f32_32x32x16_bf16 does each at 16 times the rate of the fp32 MFMA, so the six cost 6 / 16 of it.  The leading product has
// an accumulator of its own and the five others, 2^-8 of it and less, share another one or two: 16 k of a contraction round the
// large sum once, where the fp32 MFMA rounds it for every k.
//
// The workgroup: four MFMA waves, each with 32 rows and 64 columns of the tile, and four loader waves.  Taking an element apart
// costs 6.5 vector instructions (v_dot2_f32_bf16 would do a remainder in one, but occupies the matrix pipe), and its parts are
// six bytes instead of four, so as little as possible is taken apart twice or staged as parts: an MFMA wave loads its own rows of A
// straight into LDS of its own, needs no barrier for them, and takes them apart between the MFMAs of the step before; B, which the
// waves share, is taken apart once, by the loaders, and staged as three planes laid out like bf16 operands.  In a tile of
// 64 rows two waves share a block of 32 x 64, a step of 16 k each of every slab, and their sums meet in the epilogue.
//
// What bounds it: power.  A slab of 32 k of a 128 x 64 tile takes 700 ns with every CU busy; its MFMAs alone, on random numbers, take
// 522, because the clock goes down to 1.5 GHz for them; without the loads, the LDS reads of B, or the taking apart it is 140 -
// 180 less each, without the scaling 15 - 20.  us, fp32 MFMA -> this, forward / input gradient / weight gradient layout: 1024 x 2048 x
// 2048 74 / 68 / 65 -> 60 / 58 / 60, 4096 x 4096 x 1024 256 / 254 / 262 -> 230 / 234 / 245, 8 of 122 x 1088 x 1536 51 / 50 / 70 -> 35 /
// 36 / 43; error against fp64 of 1024 x 2048 x 2048 8.1e-7 -> 2.7e-7, of K = 384 and 4096 as much smaller.
#include "gemm_tile.h"

namespace rtp {

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));  // global loads take any alignment

// The parts of eight numbers, in operations that can be dealt over the slots between MFMAs: breadth first, so that an
// operation never waits for the one before.  The remainders replace the numbers.
struct Split8 {
  unsigned h[3][4];  // part, pair of elements
  static constexpr int OPS = 36;
  static constexpr float SCALE = 0x1p24f;
  template <int O>
  __device__ __forceinline__ void op(float (&x)[8]) {
    if constexpr (O < 8) {
      x[O] *= SCALE;
    } else if constexpr (O < 12) {
      pair<0, O - 8>(x);
    } else if constexpr (O < 20) {
      rest<0, O - 12>(x);
    } else if constexpr (O < 24) {
      pair<1, O - 20>(x);
    } else if constexpr (O < 32) {
      rest<1, O - 24>(x);
    } else {
      pair<2, O - 32>(x);
    }
  }
  template <int L, int I>
  __device__ __forceinline__ void pair(const float (&x)[8]) {
    h[L][I] = __builtin_bit_cast(unsigned, __builtin_convertvector((f32x2{x[2 * I], x[2 * I + 1]}), bf16x2));
  }
  template <int L, int E>
  __device__ __forceinline__ void rest(float (&x)[8]) {
    x[E] -= __builtin_bit_cast(float, E & 1 ? h[L][E / 2] & 0xffff0000u : h[L][E / 2] << 16);
  }
  template <int FROM, int TO>
  __device__ __forceinline__ void ops(float (&x)[8]) {
    [&]<int... O>(std::integer_sequence<int, O...>) __attribute__((always_inline)) { (op<FROM + O>(x), ...); }
    (std::make_integer_sequence<int, TO - FROM>{});
  }
  __device__ __forceinline__ Frag<bf16_t> part(int l) const {
    union {
      unsigned u[4];
      Frag<bf16_t> f;
    } q;
#pragma unroll
    for (int i = 0; i < 4; ++i) q.u[i] = h[l][i];
    return q.f;
  }
};

// A loader wave's share of B: vectors of four elements along its contiguous axis, read so that neighbouring lanes have
// neighbouring vectors (whole cache lines per load), kept in the stage where a bf16 operand of the same extent keeps them.
template <int R, bool KC, int SLAB, int DEPTH>
struct SplitOperand {
  static constexpr int SB = 2 * SLAB;                        // bytes of a plane's row and slab
  static constexpr int PLANE = R * SB, BYTES = 3 * PLANE;
  static constexpr int NI = R * SLAB / 4 / 256;              // vectors per lane
  static_assert(NI % 2 == 0, "pairs of vectors are taken apart together");
  const float* base;  // element 0 of row row0 (K-contiguous) or of k line 0, row row0
  long ld;
  int left;           // rows from row0 to the operand's end
  unsigned ofs[NI];   // of the lane's vector, in elements
  int koff[NI];       // its first k inside the slab
  int row[NI];        // rows contiguous: its first row inside the tile
  int early[NI];      // rows contiguous: elements it is read early, to stay inside the operand
  int dst[NI];        // its place in a plane
  float val[DEPTH][NI / 2][8];
  bool unshifted[DEPTH];

  __device__ __forceinline__ void init(const float* x, long ld_, int row0, int rows, int lw, int lane) {
    ld = ld_;
    base = KC ? x + (long)row0 * ld : x + row0;
    left = rows - row0;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int v = (lw * NI + i) * 64 + lane;
      if (KC) {
        const int r = v / (SLAB / 4), c = v % (SLAB / 4);
        koff[i] = 4 * c;
        row[i] = early[i] = 0;
        ofs[i] = (unsigned)(min(r, left - 1) * ld) + 4 * c;  // rows past the end re-read the last one
        dst[i] = r * SB + (((c >> 1) ^ kc_swizzle<SB>(r)) << 4) + (c & 1) * 8;
      } else {
        const int c = v % (R / 4);
        koff[i] = v / (R / 4);
        row[i] = 4 * c;
        early[i] = max(4 * c - max(left - 4, 0), 0);
        ofs[i] = (unsigned)(koff[i] * ld) + 4 * c - early[i];
        dst[i] = koff[i] * R * 2 + (((c >> 1) ^ rc_swizzle<bf16_t, R>(koff[i])) << 4) + (c & 1) * 8;
      }
    }
  }
  // whether the vectors of a slab with all of its k can be loaded and need no shift: past the operand's end whole vectors may
  // hold other rows (they feed columns that are never stored), a vector across the end has to be read early and shifted
  __device__ __forceinline__ bool whole() const { return KC || left >= R || left % 4 == 0; }
  // Request the slab whose first k is k0, in a segment that starts `seg` elements from the operand's base.  GUARD: vectors may
  // reach beyond the operand, and beyond the contraction in its last slab, which is loaded element by element.
  template <int S, bool GUARD>
  __device__ __forceinline__ void fetch(long seg, int k0, int kdim) {
    const float* b = base + seg + (KC ? (long)k0 : (long)k0 * ld);
    if (!GUARD || (k0 + SLAB <= kdim && (KC || left >= 4))) {
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        const f32x4u v = *reinterpret_cast<const f32x4u*>(b + ofs[i]);
#pragma unroll
        for (int e = 0; e < 4; ++e) val[S][i / 2][i % 2 * 4 + e] = v[e];
      }
    } else {
#pragma unroll
      for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const bool in = KC ? k0 + koff[i] + e < kdim : k0 + koff[i] < kdim && row[i] + e < left;
          val[S][i / 2][i % 2 * 4 + e] = in ? b[ofs[i] + early[i] + e] : 0.0f;
        }
      unshifted[S] = false;
      return;
    }
    unshifted[S] = GUARD && !whole();
  }
  // the slab's vectors that were read early, put in place
  template <int S>
  __device__ __forceinline__ void shift() {
    if (KC || !unshifted[S]) return;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      float(&x)[8] = val[S][i / 2];
      const int o = i % 2 * 4, n = early[i];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float v = 0.0f;
#pragma unroll
        for (int f = e; f < 4; ++f) v = n == f - e ? x[o + f] : v;
        x[o + e] = v;
      }
    }
  }
};

// An MFMA wave's 32 rows of A: lane (li, g) holds row li, k = 16 q + 8 g + 0 .. 7 of step q.  By register loads, for operands of
// any alignment.
template <bool KC, int SLAB, int STEPS, int DEPTH>
struct SplitRows {
  const float* base;  // element k = 0 of the lane's row, k offset of the lane and of the wave's first step included
  long ld;
  int koff;           // that k offset
  float val[DEPTH][STEPS][8];

  __device__ __forceinline__ void init(const float* x, long ld_, int row, int koff_) {
    ld = ld_;
    koff = koff_;
    base = KC ? x + (long)row * ld + koff : x + (long)koff * ld + row;
  }
  template <int S, bool GUARD>
  __device__ __forceinline__ void fetch(long seg, int k0, int kdim) {
    const float* b = base + seg + (KC ? (long)k0 : (long)k0 * ld);
    if (!GUARD || k0 + SLAB <= kdim) {
#pragma unroll
      for (int q = 0; q < STEPS; ++q) {
        if (KC) {
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const f32x4u v = *reinterpret_cast<const f32x4u*>(b + 16 * q + 4 * h);
#pragma unroll
            for (int e = 0; e < 4; ++e) val[S][q][4 * h + e] = v[e];
          }
        } else {
#pragma unroll
          for (int e = 0; e < 8; ++e) val[S][q][e] = b[(16 * q + e) * ld];
        }
      }
    } else {
#pragma unroll
      for (int q = 0; q < STEPS; ++q)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const int k = 16 * q + e;
          val[S][q][e] = k0 + koff + k < kdim ? b[KC ? (long)k : k * ld] : 0.0f;
        }
    }
  }
};

// The same rows by loads straight into a part of the LDS that is the wave's own (whole cache lines per load; the register loads
// above touch 32 lines each and fetch every line from the L1 several times), read back two steps ahead.  For aligned operands.
template <bool KC, int STEPS>
struct DmaRows {
  using D = DmaOperand<float, 32, KC, 1, 64 * STEPS>;
  static constexpr int BYTES = D::BYTES, NI = D::NI;  // per slab
  D d;
  const char* base;
  long ld;
  int koff;  // first k of the wave's first step
  __device__ __forceinline__ void init(const float* x, long ld_, int row0, int rows, int koff_, int lane) {
    ld = ld_;
    koff = koff_;
    d.init(ld, row0, rows, 0, lane);
    base = D::slab_base(x, ld, row0) + (KC ? (long)koff : (long)koff * ld) * 4;
  }
  template <bool GUARD>
  __device__ __forceinline__ void fetch(unsigned to, long seg, int k0, int kdim) const {
    const char* b = base + (seg + (KC ? (long)k0 : (long)k0 * ld)) * 4;
    if (!GUARD || k0 + koff + 16 * STEPS <= kdim)
      d.template issue<false>(to, 0, b, 0, 0);
    else
      d.template issue<true>(to, 0, b, k0 + koff, kdim);
  }
  // part I of N of the lane's eight k of step U
  template <int I, int N, int U>
  __device__ __forceinline__ static void read(float (&x)[8], const char* slab, int lane) {
    const int li = lane & 31, g = lane >> 5;
    if constexpr (KC) {
      static_assert(N == 2, "two vectors");
      constexpr int SB = 64 * STEPS;
      const float4 v = *reinterpret_cast<const float4*>(slab + li * SB + (((4 * U + 2 * g + I) ^ kc_swizzle<SB>(li)) << 4));
      x[4 * I] = v.x, x[4 * I + 1] = v.y, x[4 * I + 2] = v.z, x[4 * I + 3] = v.w;
    } else {
#pragma unroll
      for (int e = I * 8 / N; e < (I + 1) * 8 / N; ++e)
        x[e] = *reinterpret_cast<const float*>(slab + (U * 16 + g * 8 + e) * 128 + li * 4);
    }
  }
};

// The position of a contraction that runs over K segments, slab by slab; behind the last slab it stays there.
template <int SLAB>
struct SlabAt {
  int seg = 0, k0 = 0;
  __device__ __forceinline__ void next(const GemmArgs& p) {
    k0 += SLAB;
    if (k0 >= p.k) {
      const bool more = seg + 1 < p.ksegs;
      seg += more ? 1 : 0;
      k0 = more ? 0 : k0 - SLAB;
    }
    // (left alone the compiler may choose with vector instructions, and the loads' base is a scalar operand)
    seg = __builtin_amdgcn_readfirstlane(seg);
    k0 = __builtin_amdgcn_readfirstlane(k0);
  }
};

// RAG: an operand is not vector-aligned (A by register loads, the epilogue for any alignment).
template <int BM, bool AKC, bool BKC, bool RAG>
__global__ __launch_bounds__(512) void gemm_split_kernel(GemmArgs p) {
  constexpr int BN = 64, NT = BN / 32, NW = 4;              // MFMA waves
  constexpr int WK = NW * 32 / BM, STEPS = 2 / WK;          // of them on the same rows, and a wave's steps in a slab
  constexpr int SLAB = 32, NSTAGE = 4, DEPTH = 4;           // k per slab, stages of the LDS, slabs of A in flight
  constexpr int CP = BN + 4;                                // row pitch of the epilogue's fp32 tile, in floats
  using OB = SplitOperand<BN, BKC, SLAB, 3>;
  using RA = DmaRows<AKC, STEPS>;
  constexpr int STAGE = OB::BYTES, LDS_B = RAG ? 0 : NW * DEPTH * RA::BYTES, LDS_ALL = LDS_B + NSTAGE * STAGE;
  static_assert(BM == 128 || BM == 64, "four or two blocks of 32 rows");
  static_assert(NSTAGE % DEPTH == 0 && DEPTH * STEPS % 2 == 0, "register slots and sets of a step do not depend on the round");
  static_assert(BM * CP * 4 <= LDS_ALL, "the epilogue stages the fp32 tile in the slab memory");
  __shared__ __attribute__((aligned(1024))) char lds[LDS_ALL + 1024];  // the last KiB: where request loads land

  touch_kernel_arguments<sizeof(GemmArgs)>();
  const int tid = threadIdx.x;
  unsigned long long t_start = 0, t_ready = 0, t_loop = 0;  // phase stamps of thread 0 (an MFMA wave), mode 2 only
  if (p.trace != nullptr && tid == 0) {
    t_start = (unsigned long long)wall_clock64();
    atomicMin(p.trace, t_start);
  }
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 31, g = lane >> 5;
  const int wrow = wave % (BM / 32) * 32, wk = wave / (BM / 32);  // an MFMA wave's rows, and which of the waves on them it is

  // tile mapping: as in gemm_dma_kernel
  const unsigned id = blockIdx.x + blockIdx.y * gridDim.x;
  const unsigned xcd = id & 7, slot = id >> 3;
  const unsigned zl = fast_div(slot, p.d_brick);
  const unsigned t_ = slot - zl * p.d_brick.d;
  const unsigned q_ = fast_div(t_, p.d_panel), r_ = t_ - q_ * p.d_panel.d;
  const unsigned cn = fast_div(r_, p.d_prow), cm = r_ - cn * p.d_prow.d;
  const unsigned qn = fast_div(q_, p.d_pm), qm = q_ - qn * p.d_pm.d;
  const int tile_n_x = (int)((xcd & ((1u << p.xn_shift) - 1)) * p.nbk + qn * p.pcol + cn);
  const int tile_m_x = (int)(((xcd >> p.xn_shift) & ((1u << p.xm_shift) - 1)) * p.mbk + qm * p.prow + cm);
  const int z_x = (int)((xcd >> (p.xn_shift + p.xm_shift)) * p.zbk + zl);
  const int tile_m_p = (int)fast_div(blockIdx.x, p.d_tiles_n);
  const int tile_n_p = (int)(blockIdx.x - tile_m_p * p.d_tiles_n.d);
  const bool bricks = p.xg != 0;
  const int tile_m = bricks ? tile_m_x : tile_m_p, tile_n = bricks ? tile_n_x : tile_n_p;
  const int z = bricks ? z_x : (int)blockIdx.y;
  const int m0 = tile_m * BM;
  const int n0 = tile_n * BN;
  const int grp = (int)fast_div(z, p.d_batch), zb = z - grp * (int)p.d_batch.d;
  const long zo = fast_div(zb, p.d_zdiv), zi = zb - (int)zo * (int)p.d_zdiv.d;
  const int nk = (p.k + SLAB - 1) / SLAB * p.ksegs;
  const float* A = reinterpret_cast<const float*>(p.a) + grp * p.a_sg + zo * p.a_so + zi * p.a_si;
  const float* B = reinterpret_cast<const float*>(p.b) + grp * p.b_sg + zo * p.b_so + zi * p.b_si;
  const bool exact_k = p.k % SLAB == 0;

  // Row sums of A (a bias gradient) ride along in the tile row's first tile.
  const bool rowsum = !AKC && p.a_rowsum != nullptr && tile_n == 0;
  f32x16 acc[NT];
  float rsum = 0.0f;

  // Barrier protocol: both paths meet the same nk + 1 barriers, barrier k when slab k is visible (behind the last one the
  // MFMA waves read what they never use).  The loaders write slab k + 1 between barriers k and k + 1 into the stage
  // of slab k + 1 - NSTAGE, whose fragments every MFMA wave had read when it reached barrier k.
  if (wave >= NW) {
    const int lw = wave - NW;
    constexpr int LD = 3;
    OB ob;
    ob.init(B, p.ldb, n0, p.n, lw, lane);
    auto run = [&](auto GUARD) __attribute__((always_inline)) {
      SlabAt<SLAB> at;
      int stage = 0;
      auto fetch = [&](auto S) __attribute__((always_inline)) {
        ob.template fetch<decltype(S)::value, decltype(GUARD)::value>(at.seg * p.b_sk, at.k0, p.k);
        at.next(p);
        __builtin_amdgcn_sched_barrier(0);
      };
      // the parts of a slab are on their way to the LDS while the next slab is taken apart
      Split8 sp[OB::NI / 2];
      auto split = [&](auto S) __attribute__((always_inline)) {
        if constexpr (decltype(GUARD)::value) ob.template shift<decltype(S)::value>();
#pragma unroll
        for (int i = 0; i < OB::NI / 2; ++i) sp[i].template ops<0, Split8::OPS>(ob.val[decltype(S)::value][i]);
      };
      auto slab = [&](auto S) __attribute__((always_inline)) {
        constexpr int next = (decltype(S)::value + 1) % LD;
        char* st = lds + LDS_B + stage * STAGE;
#pragma unroll
        for (int i = 0; i < OB::NI; ++i)
#pragma unroll
          for (int l = 0; l < 3; ++l)
            *reinterpret_cast<uint2*>(st + l * OB::PLANE + ob.dst[i]) = make_uint2(sp[i / 2].h[l][i % 2 * 2], sp[i / 2].h[l][i % 2 * 2 + 1]);
        stage = stage + 1 == NSTAGE ? 0 : stage + 1;
        __builtin_amdgcn_sched_barrier(0);
        split(std::integral_constant<int, next>{});
        fetch(std::integral_constant<int, next>{});
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
      };
      [&]<int... S>(std::integer_sequence<int, S...>) __attribute__((always_inline)) {
        (fetch(std::integral_constant<int, S>{}), ...);
      }(std::make_integer_sequence<int, LD>{});
      split(std::integral_constant<int, 0>{});
      fetch(std::integral_constant<int, 0>{});
      int k = 0;
      for (; k + LD <= nk; k += LD)
        [&]<int... S>(std::integer_sequence<int, S...>) __attribute__((always_inline)) {
          (slab(std::integral_constant<int, S>{}), ...);
        }(std::make_integer_sequence<int, LD>{});
      [&]<int... S>(std::integer_sequence<int, S...>) __attribute__((always_inline)) {
        ((k + S < nk ? slab(std::integral_constant<int, S>{}) : (void)0), ...);
      }(std::make_integer_sequence<int, LD>{});
    };
    if (exact_k && ob.whole())
      run(std::false_type{});
    else
      run(std::true_type{});
    __builtin_amdgcn_s_barrier();
  } else {
    f32x16 cor[2][NT];  // the products of 2^-8 and those of 2^-16, apart: an MFMA does not wait for the one before the last
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[j][r] = cor[0][j][r] = cor[1][j][r] = 0.0f;
    SplitRows<AKC, SLAB, STEPS, DEPTH> rr;
    RA rd;
    float x[2][8];  // the rows of a step, as read from the LDS
    const int own = wave * (DEPTH * RA::BYTES);  // the wave's own slabs
    if constexpr (RAG)
      rr.init(A, p.lda, min(m0 + wrow + li, p.m - 1), 16 * wk + 8 * g);
    else
      rd.init(A, p.lda, m0 + wrow < p.m ? m0 + wrow : m0, p.m, 16 * wk, lane);  // (rows all past the end: the tile's first)
    Frag<bf16_t> fb[3][NT];
    Split8 sp[2];
    auto read_b = [&](auto L, int j, int stage, int q) __attribute__((always_inline)) {
      constexpr int l = decltype(L)::value;
      fb[l][j] = read_frag_dma<bf16_t, BN, BKC, OB::SB>(lds + LDS_B + stage * STAGE + l * OB::PLANE, j * 32, lane, q);
    };
    auto run = [&](auto GUARD) __attribute__((always_inline)) {
      SlabAt<SLAB> at;
      // the slab behind the last one fetched, into register or LDS slot S
      auto fetch = [&](auto S) __attribute__((always_inline)) {
        constexpr int s = decltype(S)::value;
        if constexpr (RAG)
          rr.template fetch<s, decltype(GUARD)::value>(at.seg * p.a_sk, at.k0, p.k);
        else
          rd.template fetch<decltype(GUARD)::value>((unsigned)(uintptr_t)(lptr_t)lds + own + s * RA::BYTES, at.seg * p.a_sk, at.k0, p.k);
        at.next(p);
      };
      auto add_rows = [&](const float(&v)[8], bool exists) __attribute__((always_inline)) {  // before they are taken apart
        if (!AKC && rowsum && exists) {
          float t = 0.0f;
#pragma unroll
          for (int e = 0; e < 8; ++e) t += v[e];
          rsum += t;
        }
      };
      // Step U of the wave in the slab of stage S.  In the slots between the MFMAs: the parts of the next step's rows, the
      // reads of the rows of the step behind it, and the reads of B, each plane as soon as its registers are free:
      // plane 2 and 1 of the next step, plane 0 of this one, which comes last.
      auto step = [&](auto S, auto U, int k) __attribute__((always_inline)) {
        constexpr int s = decltype(S)::value, u = decltype(U)::value;
        constexpr bool last = u == STEPS - 1;  // of the slab
        constexpr int sn = last ? (s + 1) % NSTAGE : s, un = last ? 0 : u + 1;
        constexpr int cur = (s * STEPS + u) & 1;
        constexpr int s2 = (s + 2 / STEPS) % DEPTH;  // slab of the step after the next
        float(&v)[8] = RAG ? rr.val[sn % DEPTH][un] : x[cur ^ 1];
        if constexpr (last) {  // the next slab of B is visible
          __builtin_amdgcn_s_barrier();
          asm volatile("" ::: "memory");
        }
        if constexpr (!RAG && last) fetch(std::integral_constant<int, s % DEPTH>{});  // this slab's rows have been read
        if constexpr (!RAG && u == 0) {
          RTP_WAIT_VM((DEPTH - 2) * RA::NI);  // the rows of slab s2 have landed
          asm volatile("" ::: "memory");
        }
        add_rows(v, !last || k + 1 < nk);
        __builtin_amdgcn_sched_barrier(0);
        constexpr int PA[6] = {0, 0, 1, 0, 2, 1}, PB[6] = {2, 1, 1, 0, 0, 0};
        constexpr int NM = 6 * NT, NR = AKC ? 2 : 8;
        [&]<int... M>(std::integer_sequence<int, M...>) __attribute__((always_inline)) {
          ([&] __attribute__((always_inline)) {
            constexpr int t = M / NT, j = M % NT;
            mma(sp[cur].part(PA[t]), fb[PB[t]][j], t == 3 ? acc[j] : cor[PA[t] + PB[t] == 1 ? 0 : 1][j]);
            sp[cur ^ 1].template ops<M * Split8::OPS / NM, (M + 1) * Split8::OPS / NM>(v);
            if constexpr (t == 0) read_b(std::integral_constant<int, 0>{}, j, s, wk + u);
            if constexpr (t == 1) read_b(std::integral_constant<int, 2>{}, j, sn, wk + un);
            if constexpr (t == 3) read_b(std::integral_constant<int, 1>{}, j, sn, wk + un);
            if constexpr (!RAG && M >= NM - NR)
              RA::template read<M - (NM - NR), NR, u>(x[cur], lds + own + s2 * RA::BYTES, lane);
            __builtin_amdgcn_sched_barrier(0);
          }(),
           ...);
        }(std::make_integer_sequence<int, NM>{});
        if constexpr (RAG && un == STEPS - 1) fetch(std::integral_constant<int, sn % DEPTH>{});  // the slot's last rows are taken apart
        __builtin_amdgcn_sched_barrier(0);
      };
      auto slab = [&](auto S, int k) __attribute__((always_inline)) {
        step(S, std::integral_constant<int, 0>{}, k);
        if constexpr (STEPS == 2) step(S, std::integral_constant<int, 1>{}, k);
      };
      using I0 = std::integral_constant<int, 0>;
      if (!RAG) request_epilogue<float, BM, BN>(p, (unsigned)(uintptr_t)(lptr_t)lds + LDS_ALL, m0, n0, grp, zo, zi, wave, lane);
      [&]<int... S>(std::integer_sequence<int, S...>) __attribute__((always_inline)) {
        (fetch(std::integral_constant<int, S>{}), ...);
      }(std::make_integer_sequence<int, DEPTH>{});
      if constexpr (RAG) {
        add_rows(rr.val[0][0], true);
        sp[0].template ops<0, Split8::OPS>(rr.val[0][0]);
        if constexpr (STEPS == 1) fetch(I0{});
      } else {
        constexpr int NR = AKC ? 2 : 8;
        RTP_WAIT_VM((DEPTH - 2) * RA::NI);  // the rows of the first two slabs have landed
        asm volatile("" ::: "memory");
        [&]<int... I>(std::integer_sequence<int, I...>) __attribute__((always_inline)) {
          (RA::template read<I, NR, 0>(x[0], lds + own, lane), ...);
          (RA::template read<I, NR, STEPS - 1>(x[1], lds + own + (STEPS == 1 ? RA::BYTES : 0), lane), ...);
        }(std::make_integer_sequence<int, NR>{});
        add_rows(x[0], true);
        sp[0].template ops<0, Split8::OPS>(x[0]);
      }
      __builtin_amdgcn_s_barrier();  // barrier 0
      asm volatile("" ::: "memory");
      if (p.trace != nullptr && tid == 0) t_ready = (unsigned long long)wall_clock64();
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        read_b(std::integral_constant<int, 2>{}, j, 0, wk);
        read_b(std::integral_constant<int, 1>{}, j, 0, wk);
      }
      __builtin_amdgcn_sched_barrier(0);
      int k = 0;
      for (; k + NSTAGE <= nk; k += NSTAGE)
        [&]<int... S>(std::integer_sequence<int, S...>) __attribute__((always_inline)) {
          (slab(std::integral_constant<int, S>{}, k + S), ...);
        }(std::make_integer_sequence<int, NSTAGE>{});
      [&]<int... S>(std::integer_sequence<int, S...>) __attribute__((always_inline)) {
        ((k + S < nk ? slab(std::integral_constant<int, S>{}, k + S) : (void)0), ...);
      }(std::make_integer_sequence<int, NSTAGE>{});
    };
    if (exact_k)
      run(std::false_type{});
    else
      run(std::true_type{});
    if (!RAG) RTP_WAIT_VM(0);  // slabs behind the last one still land where the epilogue writes
    if (p.trace != nullptr && tid == 0) t_loop = (unsigned long long)wall_clock64();
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[j][r] = (acc[j][r] + (cor[0][j][r] + cor[1][j][r])) * (1.0f / (Split8::SCALE * Split8::SCALE));
  }

  // Epilogue through LDS, as in gemm_dma_kernel
  __builtin_amdgcn_s_barrier();  // every wave has read its last fragments
  float* ct = reinterpret_cast<float*>(lds);
  auto at_tile = [&](int j, int r) -> float& { return ct[(wrow + 8 * (r >> 2) + 4 * g + (r & 3)) * CP + j * 32 + li]; };
  if constexpr (WK > 1) {
    if (wave < NW && wk > 0) {
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) at_tile(j, r) = acc[j][r];
      const float both = rsum + __shfl_xor(rsum, 32, 64);
      if (g == 0) ct[(wrow + li) * CP + BN] = both;
    }
    __syncthreads();
  }
  if (wave < NW && wk == 0) {
    if constexpr (WK > 1) {
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[j][r] += at_tile(j, r);
    }
    // What the parts cannot stand for: a number that is infinite, or is when scaled, has no remainder, and a scaled sum may overflow
    // where the sum itself does not.  Either leaves an infinity or a NaN in every output it reaches: a wave that finds one does
    // its part of the tile again with the fp32 MFMA.  (Not pipelined: with such an output in every wave 1024 x 2048 x 2048 takes 370 -
    // 635 us instead of 58 - 66.)
    float bad = 0.0f;
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) bad = fmaf(acc[j][r], 0.0f, bad);
    if (__any(bad != 0.0f)) {  // NaN
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[j][r] = 0.0f;
      for (int seg = 0; seg < p.ksegs; ++seg)
        for (int k0 = 0; k0 < p.k; k0 += 8) {
          auto part = [&](const float* x, long ld, bool kc, int row) {
            Frag<float> f;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const int k = k0 + 4 * g + e, kr = k < p.k ? k : 0;
              const float v = kc ? x[(long)row * ld + kr] : x[(long)kr * ld + row];
              f.f[e] = k < p.k ? v : 0.0f;
            }
            return f;
          };
          const Frag<float> xa = part(A + seg * p.a_sk, p.lda, AKC, min(m0 + wrow + li, p.m - 1));
#pragma unroll
          for (int j = 0; j < NT; ++j) mma(xa, part(B + seg * p.b_sk, p.ldb, BKC, min(n0 + j * 32 + li, p.n - 1)), acc[j]);
        }
    }
    if (rowsum) {
      // lanes 0..31 and 32..63 hold the two k halves of the same 32 rows
      float* dst = reinterpret_cast<float*>(p.a_rowsum) + grp * p.rowsum_sg;
      const float v = rsum + __shfl_xor(rsum, 32, 64) + (WK > 1 ? ct[(wrow + li) * CP + BN] : 0.0f);
      const int row = m0 + wrow + li;
      if (g == 0 && row < p.m) dst[row] = (p.flags & RTP_GEMM_ROWSUM_ACCUM) ? dst[row] + v : v;
    }
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) at_tile(j, r) = acc[j][r];
  }
  __syncthreads();
  if constexpr (RAG) {
    // (the statistics and the vectorised update are only fused into products that are aligned throughout)
    if (p.vec_c && p.sgd_master == nullptr)
      finish_tile<float, BM, BN, 512>(p, ct, m0, n0, tid, grp, zo, zi);
    else
      finish_tile_ragged<float, BM, BN, 512>(p, ct, m0, n0, tid, grp, zo, zi);
  } else if (p.sgd_master != nullptr)
    finish_tile_sgd<float, BM, BN, 512>(p, ct, m0, n0, tid, grp, zo, zi);
  else if (p.xent_mode == 1)
    finish_tile_xent_stats<float, BM, BN, 512>(p, ct, m0, n0, tid, grp);
  else
    finish_tile<float, BM, BN, 512>(p, ct, m0, n0, tid, grp, zo, zi);
  if (p.trace != nullptr && tid == 0) {
    const unsigned long long t_end = (unsigned long long)wall_clock64();
    atomicMax(p.trace + 1, t_end);
    if ((id & 15u) != 0u) return;  // phase sums from every 16th workgroup, as in gemm_dma_kernel
    atomicAdd(p.trace + 2, t_start);
    atomicAdd(p.trace + 3, t_ready - t_start);
    atomicAdd(p.trace + 4, t_loop - t_ready);
    atomicAdd(p.trace + 5, t_end - t_loop);
    atomicAdd(p.trace + 6, 1ull);
  }
}

template <int BM>
static int launch_shape(hipStream_t s, const GemmArgs& a, bool akc, bool bkc, bool ragged, dim3 grid) {
  auto go = [&](auto AKC, auto BKC, auto RAG) {
    hipLaunchKernelGGL((gemm_split_kernel<BM, decltype(AKC)::value, decltype(BKC)::value, decltype(RAG)::value>), grid,
                       dim3(512), 0, s, a);
  };
  auto layout = [&](auto RAG) {
    using T = std::true_type;
    using F = std::false_type;
    akc ? (bkc ? go(T{}, T{}, RAG) : go(T{}, F{}, RAG)) : (bkc ? go(F{}, T{}, RAG) : go(F{}, F{}, RAG));
  };
  ragged ? layout(std::true_type{}) : layout(std::false_type{});
  RTP_LAUNCH_CHECK();
  return RTP_OK;
}

int launch_split(hipStream_t s, const GemmArgs& a, bool akc, bool bkc, int bm, bool ragged, dim3 grid) {
  return bm == 128 ? launch_shape<128>(s, a, akc, bkc, ragged, grid) : launch_shape<64>(s, a, akc, bkc, ragged, grid);
}

}  // namespace rtp
