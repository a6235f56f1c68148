// bf16 products in tiles of 256 x 256.
#include "gemm_tile.h"

namespace rtp {

// What bounds the kernels of gemm.hip on a large product is the stream of operand bytes from the L2 into the LDS, and that stream is
// (1/BM + 1/BN) bytes per flop: a 256 x 256 tile moves two thirds of what 256 x 128 moves.  Its 256 KiB of fp32 accumulators need all
// eight waves of the workgroup as MFMA waves (2 x 4 wave tiles of 128 x 64, 128 accumulator registers each), so here the waves issue
// the direct-to-LDS loads themselves.
//
// A SIMD holds two of the waves, and their work alternates: a K slab (128 bytes of k per row) is four phases, a phase is a
// read half -- fragments of half an operand into registers, two load instructions -- and an MFMA half of sixteen MFMAs,
// each closed by a workgroup barrier.  The waves of the lower tile half (wm = 1, the second wave of every SIMD) pass one
// barrier more at the start of a tile, so they read while the others multiply and the other way round: LDS reads, loads and scalar
// work of one wave lie under the MFMAs of the other, and neither waits for its own.  That holds as long as a read half takes no
// longer than sixteen MFMAs (256 clocks): it is some 25 instructions, addresses in registers and offsets in the instructions, and its
// rare events are branches that are not taken.
//
// An operand's slab is two half tiles of 128 rows (16 KiB each, stored like a 128-row operand), and a wave tile takes half of
// its rows (columns) from each, so a phase multiplies one quadrant of the wave tile by all of the slab's k:
//   phase    reads               multiplies        loads (into the half tile freed two phases before)
//   1        A half 0            A0 x B0           A half 1 of slab k + 1
//   2        B half 1            A0 x B1           B half 0 of slab k + 2
//   3        A half 1            A1 x B1           A half 0 of slab k + 2
//   4        B half 0 of k + 1   A1 x B0           B half 1 of slab k + 2
// Two barrier-separated halves make phase p's reads complete in every wave before the read half of phase p + 2 begins (the
// reads have returned when the MFMA half ends), which is where that half tile may be overwritten; and a load has six
// phases from its issue to its read.  Before a read half ends, a wave waits until its loads of five phases ago have
// landed (the ten youngest may be on their way); the next phase's reads lie two barriers behind, so that holds for every
// wave's share.
//
// On random operands the matrix pipes' power sets the clock, and 16 x 16 x 32 is the cheaper MFMA: for the same flops it reads and writes its
// accumulators half as often as 32 x 32 x 16, and least where the second k-step of an output follows its first directly (a loop of MFMAs
// in registers, two waves a SIMD, random operands, TF/s: 32 x 32 x 16 1600 in any order; 16 x 16 x 32 with the k-steps apart 1800, back to back
// 1850; zeros 2210 / 2150 / 2195).  The results have the same bits.  us, 32 x 32 x 16 -> this, forward / input gradient / weight gradient layout:
// 8 of 1024 x 8192 x 2048 228 / 233 / 246 -> 214 / 220 / 235, 4096^3 103.5 / 108.5 / 112.5 -> 97.5 / 102 / 109.5, 4096 x 6144 x 2048 93 / - / - -> 87,
// 8192^3 773 / - / - -> 729 (cards differ: on a slower one 4096^3 112 -> 104 as a weight gradient).  It takes 11 % more clocks (the same LDS accesses and
// conflicts, longer waits for them), which costs where the clock is free: half a round of tiles, 4096 x 2048 x 2048 39.1 / 38.8 / - -> 40.0 / 39.0,
// 135 tiles, 1280 x 6912 x 8192, 132.5 / 137 / 150 -> 139.5 / 147 / 165, 155 tiles of four slabs 12.0 / 12.1 / 12.7 -> 12.3 / 12.7 / 13.4; from 192 tiles on it gains.
//
// A workgroup stays on its CU and goes through its tiles (the tile number advances by the number of workgroups), and the loads run on
// into the next tile: when a tile's last MFMAs are done, the first slab and a half of the next are in the LDS or on their way, and the
// epilogue touches neither.  It brings 32 rows of a wave tile at a time through 4 KiB of the wave's own, without a barrier.  The
// operands of the MFMA are exchanged, so that a lane holds four neighbouring columns of a row, and the results are bf16 before they
// are written there: 8 bytes a lane in, 16 bytes out, whole 128-byte lines to memory.  (Stores straight from the registers, 32 bytes
// of a line each, take 9 - 20 us a tile: the L2 takes a request, not a byte, per clock.)  vmcnt counts loads and stores in the
// order of their issue, so the first phases behind an epilogue let its 16 stores be on their way too.
//
// Time stamps in the kernel with 32 x 32 x 16 MFMAs, 8192 x 8192 x 1024 on zeros (at the full clock), us a tile: before (a workgroup a tile, the epilogue
// through 64 KiB of slab memory in four passes between barriers) prologue 2.8, 16 slabs 21 - 22, epilogue 7.9, gap 1.2; now 0.8, 21 -
// 24 (the stores of the tile before drain beside its loads), 1.7 - 2.5.  On one tile a CU (4096 x 4096 x 2048) 49.9 -> 40.7.  Random
// operands cost power, and the clock follows (1.5 - 1.9 us a slab instead of 1.1), so they gain less.  us, forward / input gradient /
// weight gradient layout, before -> now: 8 of 1024 x 8192 x 2048 256 / 261 -> 232 / 238, 8 of 8192 x 2048 x 1024 - / - / 318 -> 286,
// 4096 x 6144 x 2048 114 -> 99, 6000 x 6144 x 2048 169 -> 148, 6000 x 2048 x 2048 55 -> 51, 6144 x 2048 x 6000 - / - / 148 -> 141,
// 8192^3 846 -> 798.
// Closing the MFMA half before its last two MFMAs, so that the waves' MFMAs overlap, costs 10 - 20 %: the two waves of a SIMD then
// drift into the same half.

// The half tile of the rows r' = 0 .. 127 holds tile rows half_row<BLK>(r', h): blocks of BLK rows, every other one.
template <int BLK>
__device__ __forceinline__ constexpr int half_row(int r, int h) {
  return ((r & ~(BLK - 1)) << 1) | (h * BLK) | (r & (BLK - 1));
}

// The kernel's arguments where they stand, in the kernel-argument segment, through a pointer that the compiler knows nothing
// about: what is fetched through it is not kept in scalar registers over the K loops (all of them together do not fit).
typedef const __attribute__((address_space(4))) GemmArgs* KernArgs;
__device__ __forceinline__ KernArgs kernel_args_at(unsigned bytes) {
  KernArgs q = (KernArgs)((const __attribute__((address_space(4))) char*)__builtin_amdgcn_kernarg_segment_ptr() + bytes);
  asm volatile("" : "+s"(q));
  return q;
}
__device__ __forceinline__ unsigned fast_div(unsigned n, const __attribute__((address_space(4))) FastDiv& f) {
  const unsigned t = __umulhi(n, f.mul);
  return (t + ((n - t) >> f.s1)) >> f.s2;
}

// The lane's number, worked out anew: what is derived from it stands in registers only where it is used.  (Addresses of an epilogue
// held over the K loop spill, and a spilled register's way back waits for all loads on their way to the LDS.)
__device__ __forceinline__ int lane_now() {
  int l;
  asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(l));
  return l;
}

typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

// LDS by byte address: base registers and constant offsets, which an LDS instruction adds by itself.
typedef __attribute__((address_space(3))) char* lds_t;
template <typename V>
__device__ __forceinline__ V lds_load(unsigned at) {
  return *(const __attribute__((address_space(3))) V*)(uintptr_t)at;
}
template <typename V>
__device__ __forceinline__ void lds_store(unsigned at, V v) {
  *(__attribute__((address_space(3))) V*)(uintptr_t)at = v;
}

// Where a lane's fragments of a half tile (128 rows, as DmaOperand leaves them) are: of BLOCKS blocks of 16 rows from `row0` on, in
// the slab at `at`.  k-contiguous: an address for every k-step, the blocks at constant distances; row-contiguous the other way round.
template <bool KC, int BLOCKS>
struct FragPlace {
  unsigned v[KC ? 2 : BLOCKS];
  __device__ __forceinline__ void init(unsigned at, int row0, int lane) {
    const int li = lane & 15, g = lane >> 4;
    if (KC) {
#pragma unroll
      for (int q = 0; q < 2; ++q) v[q] = at + (row0 + li) * 128 + (((4 * q + g) ^ kc_swizzle<128>(li)) << 4);
    } else {
      const int kl = g * 8 + (li >> 2);
#pragma unroll
      for (int i = 0; i < BLOCKS; ++i) {
        const int rb = (row0 + i * 16 + 4 * (li & 3)) * 2;
        v[i] = at + kl * 256 + (((rb >> 4) ^ rc_swizzle<bf16_t, 128, 16>(kl)) << 4) + (rb & 15);
      }
    }
  }
  __device__ __forceinline__ void other_slab(unsigned bytes) {
#pragma unroll
    for (int i = 0; i < (KC ? 2 : BLOCKS); ++i) v[i] ^= bytes;
  }
  // block i, k-step q of the half tile `half` bytes into the slab
  __device__ __forceinline__ Frag<bf16_t> read(int half, int i, int q) const {
    Frag<bf16_t> f;
    if (KC) {
      f.v = __builtin_bit_cast(bf16x8, lds_load<u32x4>(v[q] + half + i * 2048));
    } else {
      typedef short short8_t __attribute__((ext_vector_type(8)));
      typedef __attribute__((address_space(3))) short4_t* tr_t;
      const short4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((tr_t)(uintptr_t)(v[i] + half + q * 8192));
      const short4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((tr_t)(uintptr_t)(v[i] + half + q * 8192 + 1024));
      f.v = __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    }
    return f;
  }
};

// Two products in one launch: workgroups 0 .. split - 1 have the first one's tiles, the others the second one's (split: a multiple of 8, so
// that a workgroup's XCD is its number's in either).
struct GemmPair {
  GemmArgs product[2];
  unsigned split;
};

template <bool AKC, bool BKC, bool PAIR>
__device__ __forceinline__ void large_body() {
  using T = bf16_t;
  constexpr int BM = 256, BN = 256, NL = 8, SB = 128;
  constexpr int WM = 128, WN = 64, MT = 8, NT = 4;  // wave tile, blocks of 16 x 16
  constexpr int BLKA = WM / 2, BLKB = WN / 2;
  using DA = DmaOperand<T, BM / 2, AKC, NL, SB, 16>;
  using DB = DmaOperand<T, BN / 2, BKC, NL, SB, 16>;
  constexpr int BK = SB / sizeof(T);
  constexpr int KS = SB / 64;          // k-steps of a slab
  constexpr int HALF = DA::BYTES, SLAB = 4 * HALF;
  constexpr int NI = DA::NI;           // load instructions per wave and half tile
  constexpr int NSTORE = MT * NT / 2;  // stores of a wave in a whole tile's epilogue, at least
  constexpr int PAGE = 4096;           // a wave's own LDS: 32 rows of its 64 columns in bf16, or the bias of its columns
  constexpr bool kUpdates = !AKC && !BKC;  // weight gradients may come with an update
  constexpr int kBiasSegs = 16;        // K segments whose biases are brought there
  static_assert(DB::BYTES == HALF && DB::NI == NI && 5 * NI + NSTORE < 64, "half tiles of one size; vmcnt is a 6-bit counter");
  static_assert(2 * SLAB + NL * PAGE <= 160 * 1024 && kBiasSegs * WN * 2 <= PAGE, "160 KiB of LDS");
  __shared__ __attribute__((aligned(1024))) char lds[2 * SLAB + NL * PAGE];  // [slab & 1][A0, A1, B0, B1], pages

  const unsigned split = PAIR ? ((const __attribute__((address_space(4))) GemmPair*)kernel_args_at(0))->split : 0;
  const bool second = PAIR && blockIdx.x >= split;
  const unsigned block = second ? blockIdx.x - split : blockIdx.x, blocks = PAIR && !second ? split : gridDim.x - split;
  const unsigned at = second ? (unsigned)sizeof(GemmArgs) : 0;
  touch_kernel_arguments<sizeof(GemmArgs)>(at);
  auto kernel_args = [=] { return kernel_args_at(at); };
  const KernArgs args = kernel_args();
  const int tid = threadIdx.x;
  if (args->trace != nullptr && tid == 0) atomicMin(args->trace, (unsigned long long)wall_clock64());
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 2, wn = wave & 3;

  // ---- the tiles of this workgroup ----
  const unsigned xcd = block & 7, stride = blocks >> 3;
  const unsigned chunk = args->xg != 0 ? 0 : xcd * args->per_xcd;  // where no split into bricks fits: an eighth of the tiles
  const unsigned mine = args->xg != 0 ? args->per_xcd : chunk >= args->tiles ? 0 : min(args->per_xcd, args->tiles - chunk);
  unsigned slot = block >> 3;
  if (slot >= mine) return;
  struct Tile {
    int m0, n0, grp, zo, zi;
    const char *a, *b;
  };
  auto tile_at = [&](unsigned s) {
    const KernArgs p = kernel_args();
    const unsigned in_brick = p->xg != 0 ? ~0u : 0u;
    s += chunk;
    const unsigned zl = fast_div(s, p->d_brick), t = s - zl * p->d_brick.d;
    const unsigned q = fast_div(t, p->d_panel), r = t - q * p->d_panel.d;
    const unsigned cn = fast_div(r, p->d_prow), cm = r - cn * p->d_prow.d;
    const unsigned qn = fast_div(q, p->d_pm), qm = q - qn * p->d_pm.d;
    const unsigned bn = xcd & ((1u << p->xn_shift) - 1), bm = (xcd >> p->xn_shift) & ((1u << p->xm_shift) - 1);
    const unsigned bz = xcd >> (p->xn_shift + p->xm_shift);
    const int tn = (int)((in_brick & (bn * p->nbk)) + qn * p->pcol + cn);
    const int tm = (int)((in_brick & (bm * p->mbk)) + qm * p->prow + cm);
    const int z = (int)((in_brick & (bz * p->zbk)) + zl);
    Tile w;
    w.m0 = tm * BM, w.n0 = tn * BN;
    w.grp = (int)fast_div(z, p->d_batch);
    const int zb = z - w.grp * (int)p->d_batch.d;
    w.zo = (int)fast_div(zb, p->d_zdiv), w.zi = zb - w.zo * (int)p->d_zdiv.d;
    w.a = DA::slab_base(reinterpret_cast<const T*>(p->a) + w.grp * p->a_sg + w.zo * p->a_so + w.zi * p->a_si, p->lda, w.m0);
    w.b = DB::slab_base(reinterpret_cast<const T*>(p->b) + w.grp * p->b_sg + w.zo * p->b_so + w.zi * p->b_si, p->ldb, w.n0);
    return w;
  };
  const int kdim = args->k, rows_a = args->m, rows_b = args->n;
  const long lda = args->lda, ldb = args->ldb;
  const int nk_seg = (kdim + BK - 1) / BK;
  const int nk = nk_seg * args->ksegs;

  f32x4 acc[MT][NT];
  float rsum[2] = {0.0f, 0.0f};
  auto clear = [&] {
    rsum[0] = rsum[1] = 0.0f;
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[i][j][r] = 0.0f;
  };

  // ---- this wave's share of the loads, which run ahead of the products and into the next tile ----
  Tile here = tile_at(slot), next = here;
  DA da[2];
  DB db[2];
  auto init_a = [&](const Tile& w) {
#pragma unroll
    for (int h = 0; h < 2; ++h) da[h].init(lda, w.m0, kernel_args()->m, wave, lane_now(), [=](int r) { return half_row<BLKA>(r, h); });
  };
  auto init_b = [&](const Tile& w) {
#pragma unroll
    for (int h = 0; h < 2; ++h) db[h].init(ldb, w.n0, kernel_args()->n, wave, lane_now(), [=](int r) { return half_row<BLKB>(r, h); });
  };
  init_a(here);
  init_b(here);
  const char *ca = here.a, *cb = here.b;
  constexpr long SZ = (long)sizeof(T);
  const long step_a = (AKC ? (long)BK : (long)BK * lda) * SZ, step_b = (BKC ? (long)BK : (long)BK * ldb) * SZ;
  const int k0_last = (nk_seg - 1) * BK;
  const int tail = kdim % BK != 0;
  const unsigned lds0 = (unsigned)(uintptr_t)(lptr_t)lds;
  // Slabs behind the one at ca / cb in its K segment; segments behind that one; the lanes whose vectors lie inside the contraction.
  int left = nk_seg, segs = args->ksegs - 1;
  unsigned long long in_a[NI], in_b[NI];
  int ragged = 0;  // not all of them do
  auto inside = [&](auto KC, unsigned long long(&m)[NI]) {
    const int l = lane_now();
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int j = wave * NI + i, k = decltype(KC)::value ? ((l & 7) ^ kc_swizzle<SB>(j * 8 + (l >> 3))) * 8 : j * 4 + (l >> 4);
      m[i] = __ballot(k0_last + k < kdim);
    }
    ragged = 1;
  };
  auto all_inside = [&] {
#pragma unroll
    for (int i = 0; i < NI; ++i) in_a[i] = in_b[i] = ~0ull;
    ragged = 0;
  };
  // To the next slab of the tile or the first of the next tile.  The loop around the products is one piece of code, whose rare
  // events are short branches that are not taken: a second copy of its MFMAs (for slabs without events, say) joins the
  // first in 128 accumulators, and the compiler then moves those about.
  auto step = [&] {
    if (__builtin_expect(left <= 1, 0)) {
      if (left == 0) {
        const KernArgs p = kernel_args();
        if (segs != 0) {
          ca += p->a_sk * SZ - nk_seg * step_a, cb += p->b_sk * SZ - nk_seg * step_b;
          --segs;
        } else {
          if (rows_a % BM != 0) init_a(next);
          if (rows_b % BN != 0) init_b(next);
          ca = next.a - step_a, cb = next.b - step_b, segs = p->ksegs - 1;
        }
        left = nk_seg;
        all_inside();
      }
      if (tail && left == 1) inside(std::bool_constant<AKC>{}, in_a), inside(std::bool_constant<BKC>{}, in_b);
    }
    ca += step_a, cb += step_b, --left;
  };
  // Half tile h of an operand into the slab at byte `at` of the LDS; vectors beyond the contraction become zeros.
  auto issue = [&](const auto& d, const unsigned long long(&m)[NI], unsigned at, const char* base) {
    const unsigned to = lds0 + at + wave * (NI * 1024);
    static_assert(NI == 2, "two loads");
    asm volatile("s_mov_b32 m0, %0\n\ts_mov_b64 exec, %2\n\tglobal_load_lds_dwordx4 %4, %6\n\t"
                 "s_mov_b32 m0, %1\n\ts_mov_b64 exec, %3\n\tglobal_load_lds_dwordx4 %5, %6\n\ts_mov_b64 exec, -1"
                 :
                 : "s"(to), "s"(to + 1024), "s"(m[0]), "s"(m[1]), "v"(d.ofs[0]), "v"(d.ofs[1]), "s"(base)
                 : "memory");
    if (__builtin_expect(ragged, 0)) {
      const int l = lane_now();
      unsigned zero;
      asm volatile("v_mov_b32 %0, 0" : "=v"(zero));
#pragma unroll
      for (int i = 0; i < NI; ++i)
        if (!(m[i] >> l & 1)) lds_store<u32x4>(to + i * 1024 + l * 16, u32x4{zero, zero, zero, zero});
    }
  };
  auto issue_a = [&](unsigned at, auto H) { issue(da[decltype(H)::value], in_a, at + decltype(H)::value * HALF, ca); };
  auto issue_b = [&](unsigned at, auto H) { issue(db[decltype(H)::value], in_b, at + (2 + decltype(H)::value) * HALF, cb); };

  using I0 = std::integral_constant<int, 0>;
  using I1 = std::integral_constant<int, 1>;
  Frag<T> fa[4][KS], fb0[2][KS], fb0n[2][KS], fb1[2][KS];  // B half 0 of the next slab is read while this slab's is multiplied
  FragPlace<AKC, 4> pa;
  FragPlace<BKC, 2> pb;
  auto place = [&](unsigned slab_at) {
    pa.init(lds0 + slab_at, wm * BLKA, lane_now());
    pb.init(lds0 + slab_at + 2 * HALF, wn * BLKB, lane_now());
  };
  // The block of 32 rows whose sums of A this wave adds up beside the products, or -1.  The additions are one chain behind the MFMAs of a phase, and
  // the waves go in step: a phase with sums is 250 clocks longer for the tile.  So the four blocks of a wave tile's rows go to the first four tile
  // columns, a wave each (with two or three columns two in the same phase), instead of all to the first.  us without sums / all in the first /
  // so: 8 of 8192 x 2048 x 1024 242 / 257 / 245, 2 of 3888 x 3112 x 5139 245 / 264 / 247, 6144 x 2048 x 4096 92 / 98 / 92, 4096^3 108 / 116 / 110.
  // (In the read halves of the phases behind: 239 / - / 262, 246 / - / 263, 92 / - / 98, 108 / - / 114.)
  int sum_block = -1;
  auto read_a = [&](auto H) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int q = 0; q < KS; ++q) fa[i][q] = pa.read(decltype(H)::value * HALF, i, q);
  };
  auto read_b = [&](auto H, Frag<T>(&fb)[2][KS]) {
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int q = 0; q < KS; ++q) fb[j][q] = pb.read(decltype(H)::value * HALF, j, q);
  };
  auto row_sums = [&](auto H) {
    if (!AKC && sum_block >> 1 == decltype(H)::value) {
      if (sum_block & 1) {
#pragma unroll
        for (int q = 0; q < KS; ++q) rsum[0] = frag_sum(fa[2][q], rsum[0]), rsum[1] = frag_sum(fa[3][q], rsum[1]);
      } else {
#pragma unroll
        for (int q = 0; q < KS; ++q) rsum[0] = frag_sum(fa[0][q], rsum[0]), rsum[1] = frag_sum(fa[1][q], rsum[1]);
      }
    }
  };
  auto barrier = [] {
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  // the barrier that ends a read half, the MFMA half and its end, where this wave's reads have returned (the first MFMAs
  // wait only for their own fragments)
  auto multiply = [&](auto H, auto J, const Frag<T>(&fb)[2][KS], auto SUMS) {
    constexpr int h = decltype(H)::value, j = decltype(J)::value;
    __builtin_amdgcn_sched_barrier(0);
    barrier();
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int n = 0; n < 8; ++n) {
      const int i = n >> 1, jj = (n ^ i) & 1;
#pragma unroll
      for (int q = 0; q < KS; ++q) {
        mma(fb[jj][q], fa[i][q], acc[h * 4 + i][j * 2 + jj]);  // transposed: a lane holds columns of one row
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    __builtin_amdgcn_s_setprio(0);
    if constexpr (decltype(SUMS)::value) row_sums(H);
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    barrier();
  };
  int behind = 0;    // phases whose loads are older than the last epilogue's stores
  unsigned cur = 0;  // byte of the LDS where the slab being multiplied is
  // the loads of five phases ago have landed
  auto landed = [&] {
    RTP_WAIT_VM(5 * NI + NSTORE);
    if (__builtin_expect(behind == 0, 1)) RTP_WAIT_VM(5 * NI);
    behind = behind != 0 ? behind - 1 : 0;
  };
  // A slab.  REST: slabs of this and the following tile behind it (2: two or more).
  auto slab = [&](auto REST) {
    constexpr int rest = decltype(REST)::value;
    const unsigned other = cur ^ SLAB;
    read_a(I0{});
    if constexpr (rest >= 1) issue_a(other, I1{});
    if constexpr (rest >= 1) landed();
    else RTP_WAIT_VM(NI);
    multiply(I0{}, I0{}, fb0, std::true_type{});

    read_b(I1{}, fb1);
    if constexpr (rest >= 2) step();
    if constexpr (rest >= 2) issue_b(cur, I0{});
    pb.other_slab(SLAB);
    if constexpr (rest >= 2) landed();
    else if constexpr (rest == 1) RTP_WAIT_VM(4 * NI);
    else RTP_WAIT_VM(0);
    multiply(I0{}, I1{}, fb1, std::false_type{});

    read_a(I1{});
    if constexpr (rest >= 2) issue_a(cur, I0{});
    if constexpr (rest >= 2) landed();
    else if constexpr (rest == 1) RTP_WAIT_VM(3 * NI);
    multiply(I1{}, I1{}, fb1, std::true_type{});

    if constexpr (rest >= 1) read_b(I0{}, fb0n);
    if constexpr (rest >= 2) issue_b(cur, I1{});
    pa.other_slab(SLAB);
    if constexpr (rest >= 2) landed();
    else if constexpr (rest == 1) RTP_WAIT_VM(2 * NI);
    multiply(I1{}, I0{}, fb0, std::false_type{});
    if constexpr (rest >= 1) {
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int q = 0; q < KS; ++q) fb0[j][q] = fb0n[j][q];
    }
    cur = other;
  };

  const unsigned page = lds0 + 2 * SLAB + wave * PAGE;
  // Eight neighbouring columns of a row per lane: of two blocks side by side, columns 16 (g & 1) + 8 (g >> 1) of the 32, after
  // neighbouring groups of 16 lanes have exchanged four of them.
  auto columns = [&](const f32x4& left, const f32x4& right, float(&v)[8]) {
    typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const u32x2 r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(unsigned, (float)left[e]),
                                                       __builtin_bit_cast(unsigned, (float)right[e]), false, false);
      const unsigned lo = r.x, hi = r.y;  // (the cast of a vector's element itself would be one of element 0)
      v[e] = __builtin_bit_cast(float, lo), v[4 + e] = __builtin_bit_cast(float, hi);
    }
  };
  // the bias of a lane's eight of the 32 columns from col on: by scalar loads, which no vector load or store has to be waited for
  auto bias8 = [&](KernArgs p, const Tile& w, int col, int g, float(&v)[8]) {
    typedef const __attribute__((address_space(4))) u32x4* scalar_t;
    const T* bias = reinterpret_cast<const T*>(p->bias) + w.grp * p->bias_sg + w.zo * p->bias_so + w.zi * p->bias_si;
    const int nb_seg = p->bias_sk ? p->ksegs : 1;  // a bias per K segment is summed in segment order
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = 0.0f;
#pragma unroll 1
    for (int sgm = 0; sgm < nb_seg; ++sgm) {
      u32x4 s[4];
#pragma unroll
      for (int c = 0; c < 4; ++c) s[c] = *(scalar_t)(uintptr_t)(bias + (col + 8 * c < rows_b ? col + 8 * c : 0) + sgm * p->bias_sk);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const unsigned two = g & 1 ? g & 2 ? s[3][e] : s[2][e] : g & 2 ? s[1][e] : s[0][e];
        v[2 * e] += __builtin_bit_cast(float, two << 16);
        v[2 * e + 1] += __builtin_bit_cast(float, two & 0xffff0000u);
      }
    }
  };
  // Results in bf16, addend (ADD) or mask (MASK) or bias or none: 32 rows at a time go through the wave's page, so that
  // loads and stores are whole lines (8 lanes a row, 16 bytes a lane).  An addend passes it in the other direction first.  Lanes outside the
  // product load its first vector and store nothing.
  // Tiles across the product's edge too: through the general loop below, where a bias comes by scalar loads, they set the time of a launch of one
  // round.  us, before that loop / with it / this, forward with a bias: 2766 rows, 8 groups of 384, K = 1024 34.7 / 36.6 / 28.2, 5000 x 2504 x 1000
  // 39.2 / 40.4 / 32.7, 4104 x 3808 x 264 24.2 / 27.5 / 19.3; input gradient with an addend, 4104 x 3808 x 1024 47.5 / 44.1 / 39.3.
  // EDGE: the product's edge may cross the tile.  Whole tiles have code of their own: the choice of a place for each load costs 4096 x 6144 x 512 with
  // an addend 38.4 -> 40.5 us, the conditions on the stores cost forward products 1 - 2 % (8192 x 4096 x 1024 57.8 -> 58.9).  Weight
  // gradients without an addend keep the conditions, and with them the stores where they stand: 8 of 8192 x 2048 x 1024 with row sums, eight tiles a
  // workgroup, 287 us without and 278 with them.
  auto finish = [&](const Tile& w, auto ADD, auto MASK, auto BIAS, auto RELU, auto EDGE) {
    constexpr bool add = decltype(ADD)::value, mask = decltype(MASK)::value, bias = decltype(BIAS)::value, relu = decltype(RELU)::value;
    constexpr bool edge = decltype(EDGE)::value;
    typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
    typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
    const KernArgs p = kernel_args();
    const int lane = lane_now(), li = lane & 15, g = lane >> 4;
    const bool stream_out = p->flags & RTP_GEMM_STREAM_OUT;
    const int row0 = w.m0 + wm * WM, col0 = w.n0 + wn * WN;
    if (edge && (row0 >= rows_a || col0 >= rows_b)) return;
    const int lr = lane >> 3, lc = (lane & 7) * 8;  // row (and + 8, 16, 24) and column of this lane's lines
    const int rows = !edge ? WM : col0 + lc < rows_b ? rows_a - (row0 + lr) : 0;  // of the product from this lane's first on
    const long ldc = p->ldc, ld_in = mask ? p->ld_gate : p->ld_cin;
    T* dst = reinterpret_cast<T*>(p->c_out) + w.grp * p->c_sg + w.zo * p->c_so + w.zi * p->c_si + (row0 + lr) * ldc + col0 + lc;
    u32x4 in[MT / 2][4];
    if constexpr (add || mask) {
      const T* first = mask ? reinterpret_cast<const T*>(p->gate) + w.grp * p->gate_sg + w.zo * p->gate_so + w.zi * p->gate_si
                            : reinterpret_cast<const T*>(p->c_in) + w.grp * p->cin_sg + w.zo * p->cin_so + w.zi * p->cin_si;
      const T* src = first + (row0 + lr) * ld_in + col0 + lc;
#pragma unroll
      for (int i = 0; i < MT / 2; ++i)
#pragma unroll
        for (int s = 0; s < 4; ++s)
          in[i][s] = *reinterpret_cast<const u32x4*>(!edge || i * 32 + s * 8 < rows ? src + (i * 32 + s * 8) * ld_in : first);
    }
    float b[NT][4];  // of columns 16 j + 4 g ..
    if constexpr (bias) {
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) b[j][e] = 0.0f;
      const int nb_seg = p->bias_sk ? p->ksegs : 1;  // a bias per K segment is summed in segment order
#pragma unroll 1
      for (int sgm = 0; sgm < nb_seg; ++sgm)
#pragma unroll
        for (int j = 0; j < NT; ++j) {
          const bf16x4 x = __builtin_bit_cast(bf16x4, lds_load<u32x2>(page + sgm * (WN * 2) + (j * 16 + 4 * g) * 2));
#pragma unroll
          for (int e = 0; e < 4; ++e) b[j][e] += (float)x[e];
        }
    }
    const unsigned wr = page + li * 128 + 8 * (g & 1), rd = page + lr * 128;  // 16-byte chunk c of row r is at chunk c ^ (r >> 1 & 7)
    const unsigned swz = ((li >> 1) & 7) ^ (g >> 1);
#pragma unroll
    for (int i = 0; i < MT / 2; ++i) {
      if constexpr (add) {
#pragma unroll
        for (int s = 0; s < 4; ++s)
          lds_store<u32x4>(rd + s * 1024 + (((lane & 7) ^ (((lr + s * 8) >> 1) & 7)) << 4), in[i][s]);
      }
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int j = 0; j < NT; ++j) {
          const unsigned at = wr + t * 2048 + ((unsigned)((j * 2) ^ swz) << 4);
          float v[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = acc[2 * i + t][j][e];
          if constexpr (add) {
            const bf16x4 x = __builtin_bit_cast(bf16x4, lds_load<u32x2>(at));
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] += (float)x[e];
          }
          if constexpr (bias) {
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] += b[j][e];
          }
          if constexpr (relu) {
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = fmaxf(v[e], 0.0f);
          }
          bf16x4 o;
#pragma unroll
          for (int e = 0; e < 4; ++e) o[e] = from_f32<T>(v[e]);
          lds_store<u32x2>(at, __builtin_bit_cast(u32x2, o));
        }
      u32x4 o[4];
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        o[s] = lds_load<u32x4>(rd + s * 1024 + (((lane & 7) ^ (((lr + s * 8) >> 1) & 7)) << 4));
        if constexpr (mask) {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const unsigned two = in[i][s][e], lo = two << 16, hi = two & 0xffff0000u;
            o[s][e] = (__builtin_bit_cast(float, lo) > 0.0f ? o[s][e] & 0xffffu : 0u) |
                      (__builtin_bit_cast(float, hi) > 0.0f ? o[s][e] & 0xffff0000u : 0u);
          }
        }
      }
      if (stream_out) {
#pragma unroll
        for (int s = 0; s < 4; ++s)
          if (i * 32 + s * 8 < rows) __builtin_nontemporal_store(o[s], reinterpret_cast<u32x4*>(dst + s * 8 * ldc));
      } else {
#pragma unroll
        for (int s = 0; s < 4; ++s)
          if (i * 32 + s * 8 < rows) *reinterpret_cast<u32x4*>(dst + s * 8 * ldc) = o[s];
      }
      dst += 32 * ldc;
    }
  };
  // Clip + SGD on the tile's parameters (the arithmetic of finish_tile_sgd): the gradients pass the wave's page in bf16, which is what the
  // update takes them as, the fp32 parameters of 32 rows are requested while the 32 before them are finished.
  auto finish_update = [&](const Tile& w, bool whole) {
    typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
    typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
    const KernArgs p = kernel_args();
    const int lane = lane_now(), li = lane & 15, g = lane >> 4;
    const bool stream_out = p->flags & RTP_GEMM_STREAM_OUT, skip_out = p->flags & RTP_GEMM_SGD_SKIP_OUT, copy = p->sgd_w != nullptr;
    const float lr_ = p->sgd_lr, clip = p->sgd_clip;
    // this lane's row (and + 8, 16, 24) and columns (4 of the first 32, 4 of the others): eight lanes cover a line of fp32 parameters
    const int lr = lane >> 3, l8 = lane & 7;
    const int row0 = w.m0 + wm * WM + lr, col0 = w.n0 + wn * WN + 4 * l8;
    const long ldc = p->ldc, zoff = w.grp * p->c_sg + w.zo * p->c_so + w.zi * p->c_si;
    float* const master = p->sgd_master + zoff;
    T* const wcopy = reinterpret_cast<T*>(p->sgd_w) + zoff;
    T* const out = reinterpret_cast<T*>(p->c_out) + zoff;
    const unsigned wr = page + li * 128 + 8 * (g & 1), swz = ((li >> 1) & 7) ^ (g >> 1);
    auto inside = [&](int row, int h) { return whole || (row < rows_a && col0 + 32 * h < rows_b); };
    f32x4 par[2][2][2];  // of 16 rows
    auto request = [&](int u) {
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int row = row0 + (u >> 1) * 32 + (2 * (u & 1) + s) * 8;
          par[u & 1][s][h] =
              __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(master + (inside(row, h) ? (long)row * ldc + col0 + 32 * h : 0)));
        }
      asm volatile("" ::: "memory");
    };
    request(0);
#pragma unroll
    for (int u = 0; u < MT; ++u) {
      if (u + 1 < MT) request(u + 1);
      if (u % 2 == 0) {
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int j = 0; j < NT; ++j) {
            bf16x4 o;
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = from_f32<T>(acc[u + t][j][e]);
            lds_store<u32x2>(wr + t * 2048 + ((unsigned)((j * 2) ^ swz) << 4), __builtin_bit_cast(u32x2, o));
          }
      }
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int r = lr + (2 * (u & 1) + s) * 8, row = row0 + (u >> 1) * 32 + (2 * (u & 1) + s) * 8;
          const u32x2 grad = lds_load<u32x2>(page + r * 128 + (((l8 >> 1) + 4 * h) ^ ((r >> 1) & 7)) * 16 + (l8 & 1) * 8);
          const bf16x4 gr = __builtin_bit_cast(bf16x4, grad);
          f32x4 x;
          bf16x4 c;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            x[e] = sgd_update<T>(par[u & 1][s][h][e], (float)gr[e], lr_, clip);
            c[e] = from_f32<T>(x[e]);
          }
          if (inside(row, h)) {
            const long off = (long)row * ldc + col0 + 32 * h;
            __builtin_nontemporal_store(x, reinterpret_cast<f32x4*>(master + off));
            if (copy) __builtin_nontemporal_store(__builtin_bit_cast(u32x2, c), reinterpret_cast<u32x2*>(wcopy + off));
            if (!skip_out) {
              u32x2* to = reinterpret_cast<u32x2*>(out + off);
              if (stream_out)
                __builtin_nontemporal_store(grad, to);
              else
                *to = grad;
            }
          }
        }
    }
  };
  // everything else, 16 rows after 16 rows in a loop
  auto finish_any = [&](const Tile& w, bool whole) {
    const KernArgs p = kernel_args();
    const int lane = lane_now(), li = lane & 15, g = lane >> 4;
    const int flags = p->flags;
    const bool stream_out = flags & RTP_GEMM_STREAM_OUT, relu = flags & RTP_GEMM_RELU;
    const bool out_f32 = flags & RTP_GEMM_OUT_F32, cin_f32 = flags & RTP_GEMM_CIN_F32;
    char* cbase = p->c_out + (w.grp * p->c_sg + w.zo * p->c_so + w.zi * p->c_si) * (out_f32 ? 4 : SZ);
    const char* cin = p->c_in ? p->c_in + (w.grp * p->cin_sg + w.zo * p->cin_so + w.zi * p->cin_si) * (cin_f32 ? 4 : SZ) : nullptr;
    const T* gate =
        p->gate ? reinterpret_cast<const T*>(p->gate) + w.grp * p->gate_sg + w.zo * p->gate_so + w.zi * p->gate_si : nullptr;
#pragma unroll 1
    for (int blk = 0; blk < MT; ++blk) {
      f32x4 part[NT];
      // (an empty instruction per copy: merged into one copy from a computed place, the accumulators would have to be in memory)
      auto take = [&](const f32x4(&from)[NT]) {
#pragma unroll
        for (int j = 0; j < NT; ++j) {
          part[j] = from[j];
          asm volatile("" : "+v"(part[j]));
        }
      };
      switch (blk) {
        case 0: take(acc[0]); break;
        case 1: take(acc[1]); break;
        case 2: take(acc[2]); break;
        case 3: take(acc[3]); break;
        case 4: take(acc[4]); break;
        case 5: take(acc[5]); break;
        case 6: take(acc[6]); break;
        default: take(acc[7]);
      }
      const int row = w.m0 + wm * WM + blk * 16 + li, col0 = w.n0 + wn * WN, mine8 = 16 * (g & 1) + 8 * (g >> 1);
      const long rowc = row < rows_a ? row : rows_a - 1;
      Raw8<T> rg[2];
      Raw8<float> rc[2];  // (an addend in bf16 in its first vector)
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const int col = col0 + 32 * c + mine8, colc = col < rows_b ? col : 0;
        if (cin) {
          if (cin_f32)
            rc[c].load(reinterpret_cast<const float*>(cin) + rowc * p->ld_cin + colc);
          else
            rc[c].q[0] = *reinterpret_cast<const uint4*>(reinterpret_cast<const T*>(cin) + rowc * p->ld_cin + colc);
        }
        if (gate) rg[c].load(gate + rowc * p->ld_gate + colc);
      }
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const int col = col0 + 32 * c + mine8;
        float v[8], t[8];
        columns(part[2 * c], part[2 * c + 1], v);
        if (cin) {
          if (cin_f32)
            rc[c].get(t);
          else
            Raw8<T>{{rc[c].q[0]}}.get(t);
#pragma unroll
          for (int e = 0; e < 8; ++e) v[e] += t[e];
        }
        if (p->bias) {
          bias8(p, w, col0 + 32 * c, g, t);
#pragma unroll
          for (int e = 0; e < 8; ++e) v[e] += t[e];
        }
        if (relu) {
#pragma unroll
          for (int e = 0; e < 8; ++e) v[e] = fmaxf(v[e], 0.0f);
        }
        if (gate) {
          rg[c].get(t);
#pragma unroll
          for (int e = 0; e < 8; ++e) v[e] = t[e] > 0.0f ? v[e] : 0.0f;
        }
        if (whole || (row < rows_a && col < rows_b)) {
          if (p->xent_mode == 2) xent_gradient8<T>(*p, v, row, col, w.grp);
          const long off = (long)row * p->ldc + col;
          if (out_f32)
            store8(reinterpret_cast<float*>(cbase) + off, v, stream_out);
          else
            store8(reinterpret_cast<T*>(cbase) + off, v, stream_out);
        }
      }
    }
  };
  // how a tile is finished: 0 by the loop above, 1 plainly, 2 with a bias, 3 with a bias and a ReLU, 4 an addend, 5 a mask, 6 by an update
  auto finish_form = [&](const Tile& w) {
    const KernArgs p = kernel_args();
    const bool add = p->c_in != nullptr, mask = p->gate != nullptr, bias = p->bias != nullptr, relu = p->flags & RTP_GEMM_RELU;
    if (kUpdates && p->sgd_master != nullptr) return 6;
    if ((int)add + (int)mask + (int)bias > 1 || (relu && !bias) || (p->flags & RTP_GEMM_OUT_F32) || (add && (p->flags & RTP_GEMM_CIN_F32)) ||
        p->xent_mode != 0 || (bias && p->bias_sk && p->ksegs > kBiasSegs))
      return 0;
    return add ? 4 : mask ? 5 : relu ? 3 : bias ? 2 : 1;
  };
  // the biases of the wave's columns on their way to its page: 128 bytes a K segment, two of them a load; they have landed when
  // the loads of the tile's second slab have
  auto request_bias = [&](const Tile& w) {
    const KernArgs p = kernel_args();
    const int lane = lane_now(), li = lane & 31, g = lane >> 5;
    const T* bias = reinterpret_cast<const T*>(p->bias) + w.grp * p->bias_sg + w.zo * p->bias_so + w.zi * p->bias_si;
    const int nb_seg = p->bias_sk ? p->ksegs : 1, col = w.n0 + wn * WN + 2 * li;
    for (int s0 = 0; s0 < nb_seg; s0 += 2) {
      const int s = s0 + g < nb_seg ? s0 + g : s0;
      const T* src = bias + s * p->bias_sk + (col < rows_b ? col : 0);
      asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, off" : : "s"(page + s0 * (WN * 2)), "v"(src) : "memory");
    }
  };
  auto finish_lines = [&](const Tile& w, int form, auto EDGE) {
    using Yes = std::true_type;
    using No = std::false_type;
    constexpr bool all = AKC || decltype(EDGE)::value;  // (see finish: a weight gradient's whole tiles come here without EDGE for forms 4 and 5 alone)
    if (all && form == 1)
      finish(w, No{}, No{}, No{}, No{}, EDGE);
    else if (all && form == 2)
      finish(w, No{}, No{}, Yes{}, No{}, EDGE);
    else if (all && form == 3)
      finish(w, No{}, No{}, Yes{}, Yes{}, EDGE);
    else if (form == 4)
      finish(w, Yes{}, No{}, No{}, No{}, EDGE);
    else
      finish(w, No{}, Yes{}, No{}, No{}, EDGE);
  };
  auto epilogue = [&](const Tile& w, int form) {
    const KernArgs p = kernel_args();
    using Yes = std::true_type;
    using No = std::false_type;
    if (!AKC && sum_block >= 0) {
      const int lane = lane_now(), li = lane & 31;
      T* dst = reinterpret_cast<T*>(p->a_rowsum) + w.grp * p->rowsum_sg;
      float v = 0.0f;
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const float h = rsum[t] + __shfl_xor(rsum[t], 16, 64);
        const float f = h + __shfl_xor(h, 32, 64);
        v = li >> 4 == t ? f : v;
      }
      const int row = w.m0 + wm * WM + sum_block * 32 + li;
      if (lane < 32 && row < rows_a) dst[row] = from_f32<T>((p->flags & RTP_GEMM_ROWSUM_ACCUM) ? to_f32(dst[row]) + v : v);
    }
    if (p->alpha != 1.0f) {
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[i][j][r] *= p->alpha;
    }
    const bool whole = w.m0 + BM <= rows_a && w.n0 + BN <= rows_b;
    if (form == 0)
      finish_any(w, whole);
    else if (kUpdates && form == 6)
      finish_update(w, whole);
    else if (whole && (AKC || form >= 4))
      finish_lines(w, form, No{});
    else
      finish_lines(w, form, Yes{});
  };

  // what phases before the first would have issued, in their order; the host sends no problem of a single slab here
  all_inside();
  if (left == 1 && tail) inside(std::bool_constant<AKC>{}, in_a), inside(std::bool_constant<BKC>{}, in_b);
  --left;
  issue_b(0, I0{});
  issue_a(0, I0{});
  issue_b(0, I1{});
  issue_a(0, I1{});
  step();
  issue_b(SLAB, I0{});
  issue_a(SLAB, I0{});
  issue_b(SLAB, I1{});
  clear();
  RTP_WAIT_VM(5 * NI);  // halves 0 of slab 0 have landed
  barrier();
  place(0);
  read_b(I0{}, fb0);
  __builtin_amdgcn_sched_barrier(0);
  for (;;) {
    const bool more = slot + stride < mine;
    slot += stride;
    if (more) next = tile_at(slot);
    const int form = finish_form(here);
    if (form == 2 || form == 3) request_bias(here);
    if (!AKC) {
      const int part = rows_b > 3 * BN ? wn : rows_b > BN ? wn >> 1 : 0;  // the tile column that has block wn's sums
      sum_block = kernel_args()->a_rowsum != nullptr && here.n0 == part * BN ? wn : -1;
    }
    if (wm == 1) __builtin_amdgcn_s_barrier();
    // (The loop at the start of a line of instructions: 4096 x 6144 x 2048 91.8 -> 91.0 us; weight gradients, whose loop is longer, lose 1 % by it.)
    if constexpr (AKC) asm volatile(".p2align 6");
    for (int todo = more ? nk : nk - 2; todo > 0; --todo) slab(std::integral_constant<int, 2>{});
    if (!more) {
      slab(I1{});
      slab(I0{});
    }
    if (wm == 0) __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    epilogue(here, form);
    if (!more) break;
    asm volatile("" ::: "memory");
    behind = here.m0 + BM <= rows_a && here.n0 + BN <= rows_b ? 5 : 0;
    clear();
    place(cur);  // (anew: held over the epilogue the addresses spill)
    here = next;
  }
  if (kernel_args()->trace != nullptr && tid == 0) atomicMax(kernel_args()->trace + 1, (unsigned long long)wall_clock64());
}

template <bool AKC, bool BKC>
__global__ __launch_bounds__(512) void gemm_large_kernel(GemmArgs) {
  large_body<AKC, BKC, false>();
}
__global__ __launch_bounds__(512) void gemm_large_pair_kernel(GemmPair) { large_body<false, false, true>(); }

int launch_large_pair(hipStream_t s, const GemmArgs& a, const GemmArgs& b) {
  GemmPair pair;
  pair.product[0] = a, pair.product[1] = b, pair.split = 8 * a.per_xcd;
  hipLaunchKernelGGL(gemm_large_pair_kernel, dim3(8 * (a.per_xcd + b.per_xcd)), dim3(512), 0, s, pair);
  RTP_LAUNCH_CHECK();
  return RTP_OK;
}

int launch_large(hipStream_t s, const GemmArgs& a, bool akc, bool bkc) {
  const dim3 block(512), grid(8 * (a.per_xcd < 32 ? a.per_xcd : 32));
  if (akc && bkc)
    hipLaunchKernelGGL((gemm_large_kernel<true, true>), grid, block, 0, s, a);
  else if (akc && !bkc)
    hipLaunchKernelGGL((gemm_large_kernel<true, false>), grid, block, 0, s, a);
  else if (!akc && bkc)
    hipLaunchKernelGGL((gemm_large_kernel<false, true>), grid, block, 0, s, a);
  else
    hipLaunchKernelGGL((gemm_large_kernel<false, false>), grid, block, 0, s, a);
  RTP_LAUNCH_CHECK();
  return RTP_OK;
}

}  // namespace rtp
