// Attention core for any number of queries and keys, bf16, without the probabilities in memory.  (In fp32 the backward
// pass's probabilities, recomputed from a rounded log-sum-exp, were further from fp64 than stored ones -- input gradients 3 - 7 %,
// the key bias's up to 20 % --, for 4 - 7 % of a layer's time: fp32 keeps the products and the softmax kernel.)
//
//   forward : S^T = K Q^T (MFMA) -> running softmax over keys (fp32, in registers) -> O^T += V^T P^T (MFMA);
//             keeps O and the log-sum-exp per query
//   backward: recomputes P from the log-sum-exp, once in a pass that owns queries (dQ, and the row dot products
//             delta = sum_d dO*O) and once in a pass that owns keys (dK, dV): no atomics, fixed summation order
//
// A workgroup of NW waves owns 32 * NW rows of one (group, batch, head) -- 32 a wave, their operand fragments and
// accumulators in registers -- and walks the other axis in blocks of ROWS rows, which all waves read from LDS: two
// stages, filled by direct-to-LDS loads that run one block ahead, one barrier a block.  Scores are formed with the
// owned axis in the lanes, so a lane's accumulator registers run over the block's rows: softmax reductions are in-lane
// operations and one half-wave exchange, and P / dS are, as they stand, operands of the next product (an MFMA
// contracts over slots, and which row sits in which slot is free as long as both operands agree).
//
// With one wave per tile and wave-private LDS copies every 32 x 32 block of scores had 16 KB (D = 128) to fetch and to
// wait for.  Shared blocks need a quarter of that and their latency is hidden; the loop is then bound by LDS
// reads, MFMA and the softmax's vector instructions in equal parts (about 1000 clocks each for a wave's 32 x 64 scores at
// D = 128, bf16), which two or more waves per SIMD overlap.
// Measured (one wave per tile -> shared blocks -> this; forward, backward): 64 heads of 1500 x 128 in bf16 261 -> 113 -> 106 us (690 TFLOP/s),
// 636 -> 309 -> 269 us; 256 causal heads of 512 x 64 28 -> 22 -> 21 us, 78 -> 72 -> 65 us; with a [512, 512] mask, D = 32, 42 us and 116 ->
// 90 -> 87 us.
#include "common.h"

#include <type_traits>

namespace rtp {

typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) short s16x4;

struct FlashArgs {
  const char *q, *k, *v, *o, *dout;
  char *dq, *dk, *dv, *out;
  long q_l, q_b, q_h, q_g;  // BYTE strides of q / dq: sequence, batch, head, group
  long k_l, k_b, k_h, k_g;  // of k / v / dk / dv
  long o_l, o_b, o_h, o_g;  // of o / dout
  float* lse;               // [G*N*H][L] log-sum-exp of the scaled, masked scores
  float* delta;             // [G*N*H][L] row dot products dO . O (written by the dQ pass, read by the dK/dV pass)
  const float* mask;        // additive [L][S] or null
  const float* kbias;       // additive per (batch, key) [N][S] or null
  int causal;
  float scale;
  int L, S, N, H, nblk;  // nblk: workgroups along the owned axis
  int nprob;             // G * N * H; nprob * nblk < 2^31
  float empty;           // forward: what a query without a visible key gets, in o and in lse
};

constexpr float kLog2e = 1.44269504088896340736f;
constexpr float kLn2 = 0.69314718055994530942f;

// ---- operand fragments ----
// Row-major fragment: 16 bytes of a tile row.  Accumulator-order fragment m of a 32-row group: the lane owns a
// column, its slots are the rows that accumulator registers MR*m .. MR*m + MR - 1 of that lane group hold (register r of
// lane (li, g) is row 8*(r/4) + 4*g + r%4).
template <typename T>
struct Op;
template <>
struct Op<bf16_t> {
  typedef bf16x8 Frag;
  static constexpr int ROWS = 64, MR = 8;
  static __device__ __forceinline__ f32x16 mma(Frag a, Frag b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  }
};

// A block of ROWS x D elements in LDS, row after row, the 16-byte chunks of a row permuted by XOR with swz(row) so that
// both ways of reading it spread over all banks: 16 lanes on the same chunk of 16 consecutive rows (row-major fragments),
// and rows r .. r+3 (transposing read of 4 x 16 blocks) side by side.  swz is linear over XOR of disjoint row bits, which
// lets the constant part of an address be folded in with one XOR.
template <typename T, int D, int NW>
struct Block {
  static constexpr int ROWS = Op<T>::ROWS, PITCH = D * (int)sizeof(T), CPR = PITCH / 16, BYTES = ROWS * PITCH;
  static constexpr int NI = BYTES / 1024 / NW;  // 1 KiB loads per wave
  static_assert(NI * NW * 1024 == BYTES, "whole loads");
  static_assert(sizeof(T) == 2, "the transposing read is for 16-bit elements");
  typedef typename Op<T>::Frag Frag;

  static __host__ __device__ constexpr int swz(int row) {
    return CPR == 16 ? ((row & 3) << 2) | ((row >> 2) & 3) : CPR == 8 ? (((row >> 1) & 1) << 2) | ((row >> 2) & 3) : (row >> 2) & 3;
  }

  unsigned ofs[NI];  // of the lane's chunk inside a block, per load
  __device__ __forceinline__ void prepare(long stride, int wave, int lane) {
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int pos = (wave * NI + i) * 64 + lane, row = pos / CPR;
      ofs[i] = (unsigned)(row * stride) + (unsigned)(((pos % CPR) ^ swz(row)) * 16);
    }
  }
  // Start the loads of a block whose first row is at `base` into LDS address `dst`; rows beyond the `rows` that exist
  // re-read the last one (their scores are discarded).
  __device__ __forceinline__ void issue(unsigned dst, const char* base, long stride, int rows, int wave, int lane) const {
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      unsigned o = ofs[i];
      if (rows < ROWS) {
        const int pos = (wave * NI + i) * 64 + lane, row = pos / CPR;
        o = (unsigned)(min(row, rows - 1) * stride) + (unsigned)(((pos % CPR) ^ swz(row)) * 16);
      }
      // inline assembly: the compiler must not wait for this load, the kernel's barriers do
      asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                   :
                   : "s"(dst + (unsigned)((wave * NI + i) * 1024)), "v"(o), "s"(base)
                   : "memory");
    }
  }

  // lane parts of the fragment addresses
  static __device__ __forceinline__ int lane_rows(int lane) {
    const int li = lane & 31, g = lane >> 5;
    return li * PITCH + ((g ^ swz(li)) << 4);
  }
  static __device__ __forceinline__ int lane_cols(int lane) {
    const int g = lane >> 5, t = lane & 15;
    const int row = 4 * g + (t >> 2), chunk = 2 * ((lane >> 4) & 1) + ((t & 3) >> 1);
    return row * PITCH + ((chunk ^ swz(row)) << 4) + (t & 1) * 8;
  }
  static __device__ __forceinline__ int at(int lane_part, int row, int chunk) {
    return (lane_part ^ ((chunk ^ swz(row)) << 4)) + row * PITCH;
  }
  // row li of row group h, elements 2*ks*VEC + g*VEC ...
  static __device__ __forceinline__ Frag rows(const char* blk, int lane_part, int h, int ks) {
    return *reinterpret_cast<const Frag*>(blk + at(lane_part, 32 * h, 2 * ks));
  }
  // accumulator-order fragment m of row group h, columns 32*db ...
  static __device__ __forceinline__ Frag cols(const char* blk, int lane_part, int h, int m, int db) {
    typedef __attribute__((address_space(3))) s16x4* lds_ptr;
    union {
      s16x4 h2[2];
      Frag f;
    } u;
#pragma unroll
    for (int x = 0; x < 2; ++x)
      u.h2[x] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(blk + at(lane_part, 32 * h + 16 * m + 8 * x, 4 * db)));
    return u.f;
  }
};

// the lane's row of a global operand as row-major fragments
template <typename T, int NK>
__device__ __forceinline__ void load_rows(const char* row, int g, typename Op<T>::Frag (&f)[NK]) {
#pragma unroll
  for (int ks = 0; ks < NK; ++ks) f[ks] = *reinterpret_cast<const typename Op<T>::Frag*>(row + (2 * ks + g) * 16);
}

// The loads of f have landed.  Said before the loop: the wait at their first use, inside it, would be for every load in
// flight, the next block's among them, in every round.
template <typename F, int NK>
__device__ __forceinline__ void landed(F (&f)[NK]) {
#pragma unroll
  for (int ks = 0; ks < NK; ++ks) asm volatile("" : "+v"(f[ks]));
}

// x combined with the value of the lane's partner in the other half of the wave
__device__ __forceinline__ void halves(float x, float& lo, float& hi) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  lo = __uint_as_float(r[0]), hi = __uint_as_float(r[1]);
}

template <typename T, int NF>
__device__ __forceinline__ void pack(const float* v, typename Op<T>::Frag (&f)[NF]) {
#pragma unroll
  for (int m = 0; m < NF; ++m)
#pragma unroll
    for (int e = 0; e < Op<T>::MR; ++e) f[m][e] = from_f32<T>(v[Op<T>::MR * m + e]);
}

// Accumulators (registers = features, lanes = rows) of a wave's 32 rows -> memory, through LDS of the wave's own (32 rows of D elements;
// the 16-byte chunks of a row permuted by XOR), whole lines at a time.  With a lane's own 4 features a store (16 bytes of each of 32 rows)
// the stores of a workgroup took 3.8 - 5.2 us, a quarter of a workgroup's time at 512 keys.  us, such stores -> these: 256 causal heads of
// 512 x 64 22.1 -> 21.4 forward, 72 -> 66 backward; of 512 x 128 45.8 -> 42.3, 154 -> 128.
template <typename T, int D>
__device__ __forceinline__ void store_rows(char* own, const f32x16 (&acc)[D / 32], float scale, char* first, long stride, int rows, int lane) {
  constexpr int PITCH = D * (int)sizeof(T), CPR = PITCH / 16;
  const int li = lane & 31, g = lane >> 5;
#pragma unroll
  for (int db = 0; db < D / 32; ++db)
#pragma unroll
    for (int a4 = 0; a4 < 4; ++a4) {
      T e[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) e[i] = from_f32<T>(acc[db][4 * a4 + i] * scale);
      *reinterpret_cast<uint2*>(own + li * PITCH + (((4 * db + a4) ^ (li % CPR)) << 4) + 8 * g) = *reinterpret_cast<const uint2*>(e);
    }
  wave_lds_fence();
#pragma unroll
  for (int i = 0; i < CPR / 2; ++i) {
    const int row = (i * 64 + lane) / CPR, chunk = lane % CPR;
    const uint4 v = *reinterpret_cast<const uint4*>(own + row * PITCH + ((chunk ^ (row % CPR)) << 4));
    if (row < rows) *reinterpret_cast<uint4*>(first + row * stride + chunk * 16) = v;
  }
}

struct FlashItem {
  int z, b, blk;
  long q, k, o;
};
// One workgroup's item, scalar throughout.  Block index major: with a causal mask the items of one block index are
// equally long, so the grid runs from the longest to the shortest; and with a multiple of 8 problems all blocks of one
// problem, which read the same rows, meet in one XCD's L2.
__device__ __forceinline__ FlashItem flash_item(const FlashArgs& a) {
  FlashItem it;
  const unsigned w = blockIdx.x, blk = w / (unsigned)a.nprob, z = w - blk * (unsigned)a.nprob;
  const unsigned zh = z / (unsigned)a.H, h = z - zh * (unsigned)a.H;
  const unsigned g = zh / (unsigned)a.N, b = zh - g * (unsigned)a.N;
  it.z = (int)z, it.b = (int)b, it.blk = (int)blk;
  it.q = (long)b * a.q_b + (long)h * a.q_h + (long)g * a.q_g;
  it.k = (long)b * a.k_b + (long)h * a.k_h + (long)g * a.k_g;
  it.o = (long)b * a.o_b + (long)h * a.o_h + (long)g * a.o_g;
  return it;
}

// the block's loads have landed and this wave's LDS writes are visible; then everyone's
__device__ __forceinline__ void block_barrier() {
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// The stage that the last of `blocks` blocks is not in: its own block is the one before, which every wave had left when the last one's barrier
// was passed, and no loads go there any more.  So a wave's results pass through its part of it (32 rows: NW * 32 of 128) without a barrier, and
// waves that are done early, on a causal diagonal or behind the last row, don't wait for the others (64 causal heads of 33 x 128, backward, 13.95 -> 13.6 us).
template <typename B>
__device__ __forceinline__ char* free_stage(char* lds, int blocks) {
  return lds + (blocks & 1) * 2 * B::BYTES;
}

// Fragment addresses are one XOR away from the lane's part: recomputed in every block, not kept in registers across blocks.
__device__ __forceinline__ void keep_in_loop(int& lrow, int& lcol) { asm volatile("" : "+v"(lrow), "+v"(lcol)); }

// 64 floats at src (index clamped to the n that exist) -> LDS, one per lane
__device__ __forceinline__ void issue_floats(unsigned dst, const float* src, int first, int n, int lane) {
  const unsigned o = (unsigned)min(first + lane, n - 1) * 4u;
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" : : "s"(dst), "v"(o), "s"(src) : "memory");
}

// factor * mask[mine][base + 8*(r/4) + 4*g + r%4] (KEYS_IN_REGS false: the transposed entry), clamped into the matrix
template <bool KEYS_IN_REGS>
__device__ __forceinline__ void add_mask(const FlashArgs& a, int mine, int base, int g, float factor, float (&v)[16]) {
  if (!a.mask) return;
  const int own = min(mine, (KEYS_IN_REGS ? a.L : a.S) - 1), last = (KEYS_IN_REGS ? a.S : a.L) - 1;
  if (KEYS_IN_REGS && a.S % 4 == 0 && reinterpret_cast<uintptr_t>(a.mask) % 16 == 0) {
#pragma unroll
    for (int a4 = 0; a4 < 4; ++a4) {
      const f32x4 m = *reinterpret_cast<const f32x4*>(a.mask + (long)own * a.S + min(base + 8 * a4 + 4 * g, last - 3));
#pragma unroll
      for (int e = 0; e < 4; ++e) v[4 * a4 + e] = fmaf(m[e], factor, v[4 * a4 + e]);
    }
  } else {
    float m[16];
    // A whole block in a column: one offset for all sixteen rows.  With sixteen clamped ones the key pass at D = 32 had no registers left for the
    // values, and took them one by one: backward of 256 heads of 512 with a mask 149 us, 86.7 so.
    if (!KEYS_IN_REGS && base + 32 <= last + 1) {
      const unsigned at = (unsigned)(4 * g * a.S + own);
#pragma unroll
      for (int r = 0; r < 16; ++r) m[r] = (a.mask + (long)(base + 8 * (r >> 2) + (r & 3)) * a.S)[at];
    } else {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int other = min(base + 8 * (r >> 2) + 4 * g + (r & 3), last);
        m[r] = a.mask[KEYS_IN_REGS ? (long)own * a.S + other : (long)other * a.S + own];
      }
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) v[r] = fmaf(m[r], factor, v[r]);
  }
}

// 16 values of a 32-entry LDS vector: entries 8*(r/4) + 4*g + r%4
__device__ __forceinline__ void lds_values(const float* src, int g, float (&v)[16]) {
#pragma unroll
  for (int a4 = 0; a4 < 4; ++a4) {
    const f32x4 q = *reinterpret_cast<const f32x4*>(src + 8 * a4 + 4 * g);
#pragma unroll
    for (int e = 0; e < 4; ++e) v[4 * a4 + e] = q[e];
  }
}

// Waves per SIMD the register allocation aims at.
template <typename T, int D, bool ADD>
constexpr int fwd_waves() {
  return D == 128 ? 2 : D == 64 && ADD ? 3 : 4;
}
template <int D, bool INTERLEAVE>
constexpr int dq_waves() {
  return D == 128 || INTERLEAVE ? 2 : D == 64 ? 3 : 4;
}
template <typename T, int D>
constexpr int dkv_waves() {
  return D == 128 ? 1 : D == 64 ? 2 : 3;
}
// Whether blocks without edges or masks go through loops of their own that put the vector work between the MFMAs of the other half of the
// block.  An MFMA leaves 28 of its 32 clocks to other instructions of its wave, but instructions that depend on each other take 8.5
// clocks each, a read of an accumulation register 8 and an LDS read 14, so such a wave gains where no other one fills the gaps: one or two
// a SIMD.  dQ at D = 128 needs 290 registers that way, one wave a SIMD instead of two: 139 -> 144 us for 64 heads of 1500.  At D = 32 the four
// waves a SIMD that it costs are worth more (256 causal heads of 512 50.5 -> 51.4).  dK / dV of 64 heads of 1500 x 128 208 -> 180 us.
template <int D>
constexpr bool kInterleaveDq = D == 64;
template <int D>
constexpr bool kInterleaveDkv = D >= 64;

// ADD: something joins the scaled scores (a mask, a key bias), or the scale is not positive and their order turns round: scores
// are brought to the log2 domain first and their maximum is subtracted there, exactly: a mask may lower all keys of a query by
// 1e9 or more, where a maximum rounded after the change of base is off by 2^6 and the exponential by 2^(2^6).  The key bias
// arrives in LDS already in that domain.  A score of less than -FLT_MAX / log2(e) is a hidden key's.
// Otherwise scores stay raw and scale * log2(e) is applied inside the exponential's FMA.
template <typename T, int D, int NW, bool ADD>
__global__ __launch_bounds__(NW * 64) __attribute__((amdgpu_waves_per_eu(fwd_waves<T, D, ADD>()))) void flash_fwd_kernel(
    FlashArgs a) {
  touch_kernel_arguments<sizeof(FlashArgs)>();
  typedef Block<T, D, NW> B;
  typedef typename B::Frag Frag;
  constexpr int ROWS = B::ROWS, NH = ROWS / 32, NK = B::CPR / 2, NM = 16 / Op<T>::MR, DB = D / 32;
  __shared__ __attribute__((aligned(1024))) char lds[4 * B::BYTES + 512];
  const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) void*)lds;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, li = lane & 31, g = lane >> 5;
  const FlashItem it = flash_item(a);
  const int wg_q0 = (a.nblk - 1 - it.blk) * 32 * NW;  // the long (causal) items first
  const int q0 = wg_q0 + wave * 32, query = q0 + li;
  const char *kp = a.k + it.k, *vp = a.v + it.k;
  const long step = ROWS * a.k_l;
  const float* kbias = a.kbias ? a.kbias + (long)it.b * a.S : nullptr;
  B blk;
  blk.prepare(a.k_l, wave, lane);
  auto issue = [&](int kb) {
    const unsigned dst = lds0 + (kb & 1) * 2 * B::BYTES;
    blk.issue(dst, kp + kb * step, a.k_l, a.S - kb * ROWS, wave, lane);
    blk.issue(dst + B::BYTES, vp + kb * step, a.k_l, a.S - kb * ROWS, wave, lane);
  };
  int nkb = (a.S + ROWS - 1) / ROWS;
  if (a.causal) nkb = min(nkb, (min(wg_q0 + 32 * NW, a.L) - 1) / ROWS + 1);
  // wave 0 writes the key bias of a block into LDS a block ahead of its use and holds the one after that in a register
  float* const bias_lds = reinterpret_cast<float*>(lds + 4 * B::BYTES);
  const bool writes_bias = ADD && kbias && wave == 0;
  auto bias_of = [&](int kb) { return kbias[min(kb * ROWS + lane, a.S - 1)]; };
  const float bias_first = writes_bias ? bias_of(0) : 0.0f;
  float bias_next = writes_bias ? bias_of(1) : 0.0f;
  issue(0);
  Frag qf[NK];
  load_rows<T>(a.q + it.q + min(query, a.L - 1) * a.q_l, g, qf);
  landed(qf);
  if (writes_bias) bias_lds[lane] = bias_first * kLog2e;
  int lrow = B::lane_rows(lane), lcol = B::lane_cols(lane);
  const float c = a.scale * kLog2e;
  // The running maximum (log2 domain) follows the true one: the largest P of a query is then 1, which bf16 holds exactly (with
  // a maximum that may lag behind by 2^8 and fewer rescales, peaked rows lost up to 1 % of the result's accuracy).
  float m_run = -INFINITY, l_run = 0.0f;
  f32x16 acc[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[db][r] = 0.0f;

  auto compute = [&](auto NHc, int kb) {
    constexpr int H = decltype(NHc)::value;
    const char* ks = lds + (kb & 1) * 2 * B::BYTES;
    const char* vs = ks + B::BYTES;
    const int k0 = kb * ROWS;
    float add[ADD ? H : 1][16];
    if constexpr (ADD) {  // requested before the products they wait behind
#pragma unroll
      for (int h = 0; h < H; ++h) {
        if (kbias)
          lds_values(bias_lds + (kb & 1) * 64 + 32 * h, g, add[h]);
        else
#pragma unroll
          for (int r = 0; r < 16; ++r) add[h][r] = 0.0f;
        add_mask<true>(a, query, k0 + 32 * h, g, kLog2e, add[h]);
      }
    }
    f32x16 s[H];
#pragma unroll
    for (int h = 0; h < H; ++h)
#pragma unroll
      for (int r = 0; r < 16; ++r) s[h][r] = 0.0f;
#pragma unroll
    for (int i = 0; i < NK; ++i)
#pragma unroll
      for (int h = 0; h < H; ++h) s[h] = Op<T>::mma(B::rows(ks, lrow, h, i), qf[i], s[h]);
    float val[H][16];
#pragma unroll
    for (int h = 0; h < H; ++h)
#pragma unroll
      for (int r = 0; r < 16; ++r) val[h][r] = ADD ? fmaf(s[h][r], c, add[ADD ? h : 0][r]) : s[h][r];
    if (k0 + 32 * H > a.S || (a.causal && k0 + 32 * H - 1 > q0)) {  // wave-uniform: only these blocks hold hidden keys
#pragma unroll
      for (int h = 0; h < H; ++h)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int key = k0 + 32 * h + 8 * (r >> 2) + 4 * g + (r & 3);
          const bool visible = (key < a.S) & (!a.causal | (key <= query));
          val[h][r] = visible ? val[h][r] : -INFINITY;
        }
    }
    float bm = val[0][0];
#pragma unroll
    for (int h = 0; h < H; ++h)
#pragma unroll
      for (int r = 0; r < 16; ++r) bm = fmaxf(bm, val[h][r]);
    float lo, hi;
    halves(bm, lo, hi);
    bm = ADD ? fmaxf(lo, hi) : fmaxf(lo, hi) * c;
    if (__any(bm > m_run)) {
      const float m_new = fmaxf(m_run, bm);
      const float alpha = __builtin_amdgcn_exp2f(m_run - (m_new == -INFINITY ? 0.0f : m_new));
      m_run = m_new;
      l_run *= alpha;
#pragma unroll
      for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[db][r] *= alpha;
    }
    const float m_ref = m_run == -INFINITY ? 0.0f : m_run;  // everything hidden so far: 2^(-inf - 0) = 0 all round
    float rs[2] = {0.0f, 0.0f};
    Frag pf[H][NM];
#pragma unroll
    for (int h = 0; h < H; ++h) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        val[h][r] = __builtin_amdgcn_exp2f(ADD ? val[h][r] - m_ref : fmaf(val[h][r], c, -m_ref));
        rs[r & 1] += val[h][r];
      }
      pack<T>(val[h], pf[h]);
    }
    l_run += rs[0] + rs[1];  // of the lane's own keys; the halves meet after the loop
#pragma unroll
    for (int h = 0; h < H; ++h)
#pragma unroll
      for (int m = 0; m < NM; ++m)
#pragma unroll
        for (int db = 0; db < DB; ++db) acc[db] = Op<T>::mma(B::cols(vs, lcol, h, m, db), pf[h][m], acc[db]);
  };

  for (int kb = 0; kb < nkb; ++kb) {
    block_barrier();  // block kb is there, and every wave has left block kb - 1
    keep_in_loop(lrow, lcol);
    if (writes_bias && kb + 1 < nkb) {
      asm volatile("" : "+v"(bias_next));  // it landed with the barrier: waited for here, before the next block's loads
      bias_lds[((kb + 1) & 1) * 64 + lane] = bias_next * kLog2e;
      bias_next = bias_of(kb + 2);
    }
    if (kb + 1 < nkb) issue(kb + 1);
    const int k0 = kb * ROWS;
    int keys = a.S - k0;
    if (a.causal) keys = min(keys, q0 + 32 - k0);
    if (q0 >= a.L || keys <= 0) continue;
    if (NH == 2 && keys > 32)
      compute(std::integral_constant<int, NH>{}, kb);
    else
      compute(std::integral_constant<int, 1>{}, kb);
  }
  float lo, hi;
  halves(l_run, lo, hi);
  const float l = lo + hi;
  store_rows<T, D>(free_stage<B>(lds, nkb) + wave * 32 * B::PITCH, acc, l > 0.0f ? 1.0f / l : a.empty, a.out + it.o + q0 * a.o_l, a.o_l, a.L - q0, lane);
  if (query < a.L) {
    if (g == 0) a.lse[(long)it.z * a.L + query] = l > 0.0f ? (m_run + __builtin_amdgcn_logf(l)) * kLn2 : a.empty;
  }
}

// The scores of row group h (registers: keys or queries) and dP -> P and dS / scale.  off[r] is what joins the scaled
// score before the exponential: bias and mask minus the query's log-sum-exp.
template <bool KEYS_IN_REGS>
__device__ __forceinline__ void p_and_ds(const FlashArgs& a, const f32x16& s, const f32x16& dp, const float (&off)[16],
                                         const float (&delta)[KEYS_IN_REGS ? 1 : 16], int mine, int base, int g, bool edge,
                                         float (&p)[16], float (&ds)[16]) {
#pragma unroll
  for (int r = 0; r < 16; ++r) p[r] = __builtin_amdgcn_exp2f(fmaf(s[r], a.scale, off[r]) * kLog2e);
  if (edge) {
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int other = base + 8 * (r >> 2) + 4 * g + (r & 3);
      const int query = KEYS_IN_REGS ? mine : other, key = KEYS_IN_REGS ? other : mine;
      const bool visible = (query < a.L) & (key < a.S) & (!a.causal | (key <= query));
      p[r] = visible ? p[r] : 0.0f;
    }
  }
#pragma unroll
  for (int r = 0; r < 16; ++r) ds[r] = p[r] * (dp[r] - delta[KEYS_IN_REGS ? 0 : r]);
}

// N MFMAs in a row, one slot each: read(n) is MFMA n's operand from LDS, AHEAD slots before its use, between(n) a share of the vector
// work, which a wave issues in the MFMA's shadow.
template <typename Frag, int N, int AHEAD, typename Read, typename Mul, typename Between>
__device__ __forceinline__ void mfma_stream(Read read, Mul mul, Between between) {
  constexpr int R = AHEAD + 1;
  Frag f[R];
  [&]<int... I>(std::integer_sequence<int, I...>) __attribute__((always_inline)) {
    ((f[I] = read(std::integral_constant<int, I>{})), ...);
  }(std::make_integer_sequence<int, AHEAD>{});
  __builtin_amdgcn_sched_barrier(0);
  [&]<int... I>(std::integer_sequence<int, I...>) __attribute__((always_inline)) {
    ([&] __attribute__((always_inline)) {
      if constexpr (I + AHEAD < N) f[(I + AHEAD) % R] = read(std::integral_constant<int, I + AHEAD>{});
      mul(std::integral_constant<int, I>{}, f[I % R]);
      between(std::integral_constant<int, I>{});
      __builtin_amdgcn_sched_barrier(0);
    }(),
     ...);
  }(std::make_integer_sequence<int, N>{});
}
template <int D>
constexpr int kAhead = D == 128 ? 6 : 3;
// Both groups of a block in one stream: 2 * NA products that form their scores, 2 * NC that use them.  The vector work on the first group's
// 16 scores a lane lies under the products that form the second's, that on the second's under the products that use the first's.
// begin(): what the elements need besides the scores; settle(h): group h's scores are read from here on.
template <typename Frag, int NA, int NC, int AHEAD, typename Read, typename Mul, typename Begin, typename Settle, typename Element>
__device__ __forceinline__ void block_stream(Read read, Mul mul, Begin begin, Settle settle, Element element) {
  mfma_stream<Frag, 2 * NA + 2 * NC, AHEAD>(read, mul, [&](auto N) __attribute__((always_inline)) {
    constexpr int n = decltype(N)::value, EA = 16 / NA, EC = 16 / NC;
    using I0 = std::integral_constant<int, 0>;
    using I1 = std::integral_constant<int, 1>;
    if constexpr (n == NA - 4) begin();
    if constexpr (n == NA) settle(I0{});
    if constexpr (n == 2 * NA) settle(I1{});
    if constexpr (n >= NA && n < 2 * NA)
      [&]<int... E>(std::integer_sequence<int, E...>) __attribute__((always_inline)) {
        (element(I0{}, std::integral_constant<int, (n - NA) * EA + E>{}), ...);
      }(std::make_integer_sequence<int, EA>{});
    if constexpr (n >= 2 * NA && n < 2 * NA + NC)
      [&]<int... E>(std::integer_sequence<int, E...>) __attribute__((always_inline)) {
        (element(I1{}, std::integral_constant<int, (n - 2 * NA) * EC + E>{}), ...);
      }(std::make_integer_sequence<int, EC>{});
  });
}

// Scores that vector instructions take next, in vector registers.  A kernel of one wave per SIMD has its MFMA results in accumulation
// registers otherwise, each of which costs a vector instruction of 8 clocks to read.  The compiler does not know what is inside, so it
// does not wait for the results: scores_settle() does, and hands the registers on, so that no reader can be moved in front of it.
template <bool ONE_WAVE, bool FIRST>
__device__ __forceinline__ void mma_scores(bf16x8 a, bf16x8 b, f32x16& c) {
  if constexpr (ONE_WAVE && FIRST)
    asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, 0" : "=&v"(c) : "v"(a), "v"(b));
  else if constexpr (ONE_WAVE)
    asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(c) : "v"(a), "v"(b));
  else
    c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, FIRST ? f32x16{} : c, 0, 0, 0);
}
// (twelve wait states between a 32 x 32 x 16 MFMA and the first vector instruction that takes its results)
template <bool ONE_WAVE>
__device__ __forceinline__ void scores_settle(f32x16& s, f32x16& dp) {
  if constexpr (ONE_WAVE) asm volatile("s_nop 11" : "+v"(s), "+v"(dp));
}

// INTERLEAVE: blocks all of whose keys the wave's queries see go through a loop of their own, see kInterleaveDq.
template <typename T, int D, int NW, bool INTERLEAVE>
__global__ __launch_bounds__(NW * 64) __attribute__((amdgpu_waves_per_eu(dq_waves<D, INTERLEAVE>()))) void flash_dq_kernel(
    FlashArgs a) {
  touch_kernel_arguments<sizeof(FlashArgs)>();
  typedef Block<T, D, NW> B;
  typedef typename B::Frag Frag;
  constexpr int ROWS = B::ROWS, NH = ROWS / 32, NK = B::CPR / 2, NM = 16 / Op<T>::MR, DB = D / 32;
  __shared__ __attribute__((aligned(1024))) char lds[4 * B::BYTES + 512];
  const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) void*)lds;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, li = lane & 31, g = lane >> 5;
  const FlashItem it = flash_item(a);
  const int wg_q0 = (a.nblk - 1 - it.blk) * 32 * NW;
  const int q0 = wg_q0 + wave * 32, query = q0 + li, row = min(query, a.L - 1);
  const char *kp = a.k + it.k, *vp = a.v + it.k;
  const long step = ROWS * a.k_l;
  const float* kbias = a.kbias ? a.kbias + (long)it.b * a.S : nullptr;
  B blk;
  blk.prepare(a.k_l, wave, lane);
  auto issue = [&](int kb) {
    const unsigned dst = lds0 + (kb & 1) * 2 * B::BYTES;
    blk.issue(dst, kp + kb * step, a.k_l, a.S - kb * ROWS, wave, lane);
    blk.issue(dst + B::BYTES, vp + kb * step, a.k_l, a.S - kb * ROWS, wave, lane);
    if (kbias && wave == 0) issue_floats(lds0 + 4 * B::BYTES + (kb & 1) * 256, kbias, kb * ROWS, a.S, lane);
  };
  int nkb = (a.S + ROWS - 1) / ROWS;
  if (a.causal) nkb = min(nkb, (min(wg_q0 + 32 * NW, a.L) - 1) / ROWS + 1);
  issue(0);
  Frag qf[NK], gf[NK];
  load_rows<T>(a.dout + it.o + row * a.o_l, g, gf);
  float delta[1] = {0.0f};
  {
    load_rows<T>(a.o + it.o + row * a.o_l, g, qf);
#pragma unroll
    for (int i = 0; i < NK; ++i)
#pragma unroll
      for (int e = 0; e < (int)(sizeof(Frag) / sizeof(T)); ++e) delta[0] += to_f32((T)gf[i][e]) * to_f32((T)qf[i][e]);
    float lo, hi;
    halves(delta[0], lo, hi);
    delta[0] = lo + hi;
    if (query < a.L && g == 0) a.delta[(long)it.z * a.L + query] = delta[0];
  }
  load_rows<T>(a.q + it.q + row * a.q_l, g, qf);
  float lse = a.lse[(long)it.z * a.L + row];
  landed(qf);
  landed(gf);
  asm volatile("" : "+v"(lse));
  if (INTERLEAVE && !kbias && wave == 0) {  // both stages of the bias are read all the same
    reinterpret_cast<float*>(lds + 4 * B::BYTES)[lane] = 0.0f;
    reinterpret_cast<float*>(lds + 4 * B::BYTES)[64 + lane] = 0.0f;
  }
  int lrow = B::lane_rows(lane), lcol = B::lane_cols(lane);
  f32x16 acc[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[db][r] = 0.0f;

  auto next = [&](int kb) __attribute__((always_inline)) {
    block_barrier();
    keep_in_loop(lrow, lcol);
    if (kb + 1 < nkb) issue(kb + 1);
    return lds + (kb & 1) * 2 * B::BYTES;
  };
  int kb = 0;
  // blocks whose keys all of the wave's queries see (a loop of its own: two ways through one loop would move the accumulators about)
  if constexpr (INTERLEAVE) {
    auto both = [&](const char* ks, const char* vs, const float* bias) __attribute__((always_inline)) {
      constexpr int NA = 2 * NK, NC = NM * DB;
      f32x16 s[2], dp[2];
      Frag df[2][NM];
      f32x4 off[2];
      auto offsets = [&](int quarter) __attribute__((always_inline)) {
        off[quarter & 1] = *reinterpret_cast<const f32x4*>(bias + 8 * quarter + 4 * g);
      };
      auto element = [&](auto Hc, auto R) __attribute__((always_inline)) {
        constexpr int h = decltype(Hc)::value, r = decltype(R)::value;
        const float p = __builtin_amdgcn_exp2f(fmaf(s[h][r], a.scale, -lse + off[r / 4 & 1][r % 4]) * kLog2e);
        df[h][r / Op<T>::MR][r % Op<T>::MR] = from_f32<T>(p * (dp[h][r] - delta[0]));
        if constexpr (r % 4 == 3 && 4 * h + r / 4 + 2 < 8) offsets(4 * h + r / 4 + 2);
      };
      block_stream<Frag, NA, NC, kAhead<D>>(
          [&](auto N) __attribute__((always_inline)) {
            constexpr int n = decltype(N)::value, c = n - 2 * NA;
            if constexpr (n < 2 * NA)
              return B::rows(n & 1 ? vs : ks, lrow, n / NA, n % NA / 2);
            else
              return B::cols(ks, lcol, c / NC, c % NC / DB, c % DB);
          },
          [&](auto N, const Frag& f) __attribute__((always_inline)) {
            constexpr int n = decltype(N)::value, c = n - 2 * NA;
            if constexpr (n < 2 * NA) {
              constexpr int h = n / NA, i = n % NA / 2;
              if constexpr (n & 1)
                dp[h] = Op<T>::mma(f, gf[i], i == 0 ? f32x16{} : dp[h]);
              else
                s[h] = Op<T>::mma(f, qf[i], i == 0 ? f32x16{} : s[h]);
            } else {
              constexpr int h = c / NC, m = c % NC / DB, db = c % DB;
              acc[db] = Op<T>::mma(f, df[h][m], acc[db]);
            }
          },
          [&]() __attribute__((always_inline)) { offsets(0), offsets(1); }, [](auto) {}, element);
    };
    const int whole = q0 >= a.L ? 0 : min(a.causal ? (q0 + 1) / ROWS : nkb, a.S / ROWS);
    for (; kb < whole; ++kb) {
      const char* ks = next(kb);
      both(ks, ks + B::BYTES, reinterpret_cast<const float*>(lds + 4 * B::BYTES) + (kb & 1) * 64);
    }
  }
  for (; kb < nkb; ++kb) {
    const char* ks = next(kb);
    const char* vs = ks + B::BYTES;
#pragma unroll
    for (int h = 0; h < NH; ++h) {
      const int k0 = kb * ROWS + 32 * h;
      if (q0 >= a.L || k0 >= a.S || (a.causal && k0 > q0 + 31)) continue;  // wave-uniform
      float off[16];
#pragma unroll
      for (int r = 0; r < 16; ++r) off[r] = -lse;
      if (kbias) {
        float kb16[16];
        lds_values(reinterpret_cast<const float*>(lds + 4 * B::BYTES) + (kb & 1) * 64 + 32 * h, g, kb16);
#pragma unroll
        for (int r = 0; r < 16; ++r) off[r] += kb16[r];
      }
      if constexpr (!INTERLEAVE) add_mask<true>(a, query, k0, g, 1.0f, off);
      f32x16 s, dp;
#pragma unroll
      for (int r = 0; r < 16; ++r) s[r] = dp[r] = 0.0f;
#pragma unroll
      for (int i = 0; i < NK; ++i) {
        s = Op<T>::mma(B::rows(ks, lrow, h, i), qf[i], s);
        dp = Op<T>::mma(B::rows(vs, lrow, h, i), gf[i], dp);
      }
      const bool edge = k0 + 32 > a.S || (a.causal && k0 + 31 > q0);
      float p[16], ds[16];
      p_and_ds<true>(a, s, dp, off, delta, query, k0, g, edge, p, ds);
      Frag df[NM];
      pack<T>(ds, df);
      // dQ^T[dd][query] += sum_key K[key][dd] dS[query][key]
#pragma unroll
      for (int m = 0; m < NM; ++m)
#pragma unroll
        for (int db = 0; db < DB; ++db) acc[db] = Op<T>::mma(B::cols(ks, lcol, h, m, db), df[m], acc[db]);
    }
  }
  store_rows<T, D>(free_stage<B>(lds, nkb) + wave * 32 * B::PITCH, acc, a.scale, a.dq + it.q + q0 * a.q_l, a.q_l, a.L - q0, lane);
}

// Key pass.  Scores are formed as S[query][key] (A = Q rows, B = K rows), so a lane is a KEY and its 16 accumulator
// registers run over queries: P and dS are then, as they stand, the B operands "lane = key, slots = queries" of
// dV^T = dO^T P and dK^T = Q^T dS, and the per-query statistics come in from LDS, 16 values per lane.
// INTERLEAVE: blocks whose queries all see all of the wave's keys go through a loop of their own, see kInterleaveDkv.
template <typename T, int D, int NW, bool INTERLEAVE>
__global__ __launch_bounds__(NW * 64) __attribute__((amdgpu_waves_per_eu(dkv_waves<T, D>()))) void flash_dkv_kernel(
    FlashArgs a) {
  touch_kernel_arguments<sizeof(FlashArgs)>();
  typedef Block<T, D, NW> B;
  typedef typename B::Frag Frag;
  constexpr int ROWS = B::ROWS, NH = ROWS / 32, NK = B::CPR / 2, NM = 16 / Op<T>::MR, DB = D / 32;
  __shared__ __attribute__((aligned(1024))) char lds[4 * B::BYTES + 1024];
  const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) void*)lds;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, li = lane & 31, g = lane >> 5;
  const FlashItem it = flash_item(a);
  const int wg_k0 = it.blk * 32 * NW;  // causal: the first keys meet every query, so the long items come first
  const int k0 = wg_k0 + wave * 32, key = k0 + li;
  const char *qp = a.q + it.q, *gp = a.dout + it.o;
  const long q_step = ROWS * a.q_l, g_step = ROWS * a.o_l;
  B bq, bg;
  bq.prepare(a.q_l, wave, lane);
  bg.prepare(a.o_l, wave, lane);
  const float *lse_row = a.lse + (long)it.z * a.L, *delta_row = a.delta + (long)it.z * a.L;
  auto issue = [&](int qb) {
    const unsigned dst = lds0 + (qb & 1) * 2 * B::BYTES, stat = lds0 + 4 * B::BYTES + (qb & 1) * 512;
    bq.issue(dst, qp + qb * q_step, a.q_l, a.L - qb * ROWS, wave, lane);
    bg.issue(dst + B::BYTES, gp + qb * g_step, a.o_l, a.L - qb * ROWS, wave, lane);
    if (wave == 0) issue_floats(stat, lse_row, qb * ROWS, a.L, lane);
    if (wave == 1) issue_floats(stat + 256, delta_row, qb * ROWS, a.L, lane);
  };
  const int nqb = (a.L + ROWS - 1) / ROWS, first = a.causal ? wg_k0 / ROWS : 0;
  if (first < nqb) issue(first);
  const long row = min(key, a.S - 1);
  Frag kf[NK], vf[NK];
  load_rows<T>(a.k + it.k + row * a.k_l, g, kf);
  load_rows<T>(a.v + it.k + row * a.k_l, g, vf);
  float kb = a.kbias ? a.kbias[(long)it.b * a.S + row] : 0.0f;
  landed(kf);
  landed(vf);
  asm volatile("" : "+v"(kb));
  int lrow = B::lane_rows(lane), lcol = B::lane_cols(lane);
  f32x16 dk[DB], dv[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int r = 0; r < 16; ++r) dk[db][r] = dv[db][r] = 0.0f;

  auto next = [&](int qb) __attribute__((always_inline)) {
    block_barrier();
    keep_in_loop(lrow, lcol);
    if (qb + 1 < nqb) issue(qb + 1);
    return lds + (qb & 1) * 2 * B::BYTES;
  };
  auto any = [&](int qb) __attribute__((always_inline)) {
    const char* qs = next(qb);
    const char* gs = qs + B::BYTES;
    const float* stat = reinterpret_cast<const float*>(lds + 4 * B::BYTES) + (qb & 1) * 128;
#pragma unroll
    for (int h = 0; h < NH; ++h) {
      const int q0 = qb * ROWS + 32 * h;
      if (k0 >= a.S || q0 >= a.L || (a.causal && k0 > q0 + 31)) continue;  // wave-uniform
      f32x16 s, dp;
#pragma unroll
      for (int r = 0; r < 16; ++r) s[r] = dp[r] = 0.0f;
#pragma unroll
      for (int i = 0; i < NK; ++i) {
        s = Op<T>::mma(B::rows(qs, lrow, h, i), kf[i], s);
        dp = Op<T>::mma(B::rows(gs, lrow, h, i), vf[i], dp);
      }
      float off[16], delta[16], p[16], ds[16];
      lds_values(stat + 32 * h, g, off);
      lds_values(stat + 64 + 32 * h, g, delta);
#pragma unroll
      for (int r = 0; r < 16; ++r) off[r] = kb - off[r];
      if constexpr (!INTERLEAVE) add_mask<false>(a, key, q0, g, 1.0f, off);
      const bool edge = q0 + 32 > a.L || (a.causal && k0 + 31 > q0);
      p_and_ds<false>(a, s, dp, off, delta, key, q0, g, edge, p, ds);
      Frag pf[NM], df[NM];
      pack<T>(p, pf);
      pack<T>(ds, df);
      // dV^T[dd][key] += sum_query dO[query][dd] P[query][key];  dK^T[dd][key] += sum_query Q[query][dd] dS[query][key]
#pragma unroll
      for (int m = 0; m < NM; ++m)
#pragma unroll
        for (int db = 0; db < DB; ++db) {
          dv[db] = Op<T>::mma(B::cols(gs, lcol, h, m, db), pf[m], dv[db]);
          dk[db] = Op<T>::mma(B::cols(qs, lcol, h, m, db), df[m], dk[db]);
        }
    }
  };
  int qb = first;
  // blocks whose queries all see all of the wave's keys (loops of their own: two ways through one loop would move the accumulators about)
  if constexpr (INTERLEAVE) {
    auto both = [&](const char* qs, const char* gs, const float* stat) __attribute__((always_inline)) {
      constexpr int NA = 2 * NK, NC = 2 * NM * DB;
      constexpr bool ONE_WAVE = dkv_waves<T, D>() == 1;
      f32x16 s[2], dp[2];
      Frag pf[2][NM], df[2][NM];
      f32x4 off[2], delta[2];
      auto stats = [&](int quarter) __attribute__((always_inline)) {  // of the block's queries: eight, four of them this lane's
        off[quarter & 1] = *reinterpret_cast<const f32x4*>(stat + 8 * quarter + 4 * g);
        delta[quarter & 1] = *reinterpret_cast<const f32x4*>(stat + 64 + 8 * quarter + 4 * g);
      };
      auto element = [&](auto Hc, auto R) __attribute__((always_inline)) {
        constexpr int h = decltype(Hc)::value, r = decltype(R)::value;
        const float p = __builtin_amdgcn_exp2f(fmaf(s[h][r], a.scale, kb - off[r / 4 & 1][r % 4]) * kLog2e);
        const float ds = p * (dp[h][r] - delta[r / 4 & 1][r % 4]);
        constexpr int MR = Op<T>::MR;
        pf[h][r / MR][r % MR] = from_f32<T>(p);
        df[h][r / MR][r % MR] = from_f32<T>(ds);
        if constexpr (r % 4 == 3 && 4 * h + r / 4 + 2 < 8) stats(4 * h + r / 4 + 2);
      };
      block_stream<Frag, NA, NC, kAhead<D>>(
          [&](auto N) __attribute__((always_inline)) {
            constexpr int n = decltype(N)::value, c = n - 2 * NA, w = n & 1;
            if constexpr (n < 2 * NA)
              return B::rows(w ? gs : qs, lrow, n / NA, n % NA / 2);
            else
              return B::cols(w ? qs : gs, lcol, c / NC, c % NC / (2 * DB), c % (2 * DB) / 2);
          },
          [&](auto N, const Frag& f) __attribute__((always_inline)) {
            constexpr int n = decltype(N)::value, c = n - 2 * NA, w = n & 1;
            if constexpr (n < 2 * NA) {
              constexpr int h = n / NA, i = n % NA / 2;
              if constexpr (w)
                mma_scores<ONE_WAVE, i == 0>(f, vf[i], dp[h]);
              else
                mma_scores<ONE_WAVE, i == 0>(f, kf[i], s[h]);
            } else {
              constexpr int h = c / NC, m = c % NC / (2 * DB), db = c % (2 * DB) / 2;
              if constexpr (w)
                dk[db] = Op<T>::mma(f, df[h][m], dk[db]);
              else
                dv[db] = Op<T>::mma(f, pf[h][m], dv[db]);
            }
          },
          [&]() __attribute__((always_inline)) { stats(0), stats(1); },
          [&](auto Hc) __attribute__((always_inline)) { scores_settle<ONE_WAVE>(s[decltype(Hc)::value], dp[decltype(Hc)::value]); }, element);
    };
    const int whole0 = k0 >= a.S ? nqb : a.causal ? (k0 + 31 + ROWS - 1) / ROWS : first, whole1 = a.L / ROWS;
    for (; qb < min(whole0, nqb); ++qb) any(qb);
    for (; qb < whole1; ++qb) {
      const char* qs = next(qb);
      both(qs, qs + B::BYTES, reinterpret_cast<const float*>(lds + 4 * B::BYTES) + (qb & 1) * 128);
    }
  }
  for (; qb < nqb; ++qb) any(qb);
  char* own = free_stage<B>(lds, nqb) + wave * 32 * B::PITCH;
  store_rows<T, D>(own, dk, a.scale, a.dk + it.k + k0 * a.k_l, a.k_l, a.S - k0, lane);
  wave_lds_fence();
  store_rows<T, D>(own, dv, 1.0f, a.dv + it.k + k0 * a.k_l, a.k_l, a.S - k0, lane);
}

static constexpr int64_t kFlashMaxLen = 1 << 20;

// Rows of a workgroup: 128, or 64 where the owned axis is short or 128 would leave compute units idle.
static int flash_waves(int64_t nprob, int64_t own) { return own <= 64 || nprob * ceil_div(own, 128) < 256 ? 2 : 4; }

template <typename T, int D>
struct FlashFwd {
  template <int NW>
  static void run(hipStream_t st, const FlashArgs& a, dim3 grid) {
    if (a.mask || a.kbias || !(a.scale > 0.0f))
      hipLaunchKernelGGL((flash_fwd_kernel<T, D, NW, true>), grid, dim3(64 * NW), 0, st, a);
    else
      hipLaunchKernelGGL((flash_fwd_kernel<T, D, NW, false>), grid, dim3(64 * NW), 0, st, a);
  }
};
// Calls none of whose blocks are whole for any wave, those with a mask and short ones, have kernels without the second loop, of the registers
// and waves that they had before there was one.  us, backward with a mask, one kernel before the second loop / with it / a kernel without: 256 heads of
// 320 x 64 62.6 / 67.4 / 58.9, of 1024 x 64 406 / 408 / 382.
template <typename T, int D>
struct FlashDq {
  template <int NW>
  static void run(hipStream_t st, const FlashArgs& a, dim3 grid) {
    if (kInterleaveDq<D> && !a.mask && a.S >= Op<T>::ROWS && (!a.causal || a.L > Op<T>::ROWS))
      hipLaunchKernelGGL((flash_dq_kernel<T, D, NW, kInterleaveDq<D>>), grid, dim3(64 * NW), 0, st, a);
    else
      hipLaunchKernelGGL((flash_dq_kernel<T, D, NW, false>), grid, dim3(64 * NW), 0, st, a);
  }
};
template <typename T, int D>
struct FlashDkv {
  template <int NW>
  static void run(hipStream_t st, const FlashArgs& a, dim3 grid) {
    if (kInterleaveDkv<D> && !a.mask && a.L >= (a.causal ? 2 : 1) * Op<T>::ROWS)
      hipLaunchKernelGGL((flash_dkv_kernel<T, D, NW, kInterleaveDkv<D>>), grid, dim3(64 * NW), 0, st, a);
    else
      hipLaunchKernelGGL((flash_dkv_kernel<T, D, NW, false>), grid, dim3(64 * NW), 0, st, a);
  }
};
template <class Pass>
static void flash_pass(hipStream_t st, FlashArgs a, int64_t own) {
  const int nw = flash_waves(a.nprob, own);
  a.nblk = (int)ceil_div(own, 32 * nw);
  const dim3 grid((unsigned)(a.nprob * (int64_t)a.nblk));
  if (nw == 2)
    Pass::template run<2>(st, a, grid);
  else
    Pass::template run<4>(st, a, grid);
}
// `own`: rows of the axis whose blocks the workgroups own
template <template <typename, int> class Pass>
static int flash_launch(hipStream_t st, int64_t D, const FlashArgs& a, int64_t own) {
  if (D == 32)
    flash_pass<Pass<bf16_t, 32>>(st, a, own);
  else if (D == 64)
    flash_pass<Pass<bf16_t, 64>>(st, a, own);
  else
    flash_pass<Pass<bf16_t, 128>>(st, a, own);
  RTP_LAUNCH_CHECK();
  return RTP_OK;
}

static int flash_args(const char* who, FlashArgs& a, int dtype, const int64_t (&qs)[4], const int64_t (&ks)[4],
                      const int64_t (&os)[4], const float* mask, const float* key_bias, int causal, float scale, int64_t L,
                      int64_t S, int64_t N, int64_t H, int64_t D, int64_t G) {
  RTP_REQUIRE(rtp_attn_flash_kv_supported(dtype, L, S, D), "%s: dtype %d with L = %lld, S = %lld, head dimension %lld", who,
              dtype, (long long)L, (long long)S, (long long)D);
  RTP_REQUIRE(N >= 1 && H >= 1 && G >= 1, "%s: batch, heads and groups must be >= 1", who);
  const int64_t esz = 2;
  for (const auto& s : {&qs, &ks, &os}) {
    for (int i = 0; i < 4; ++i)
      RTP_REQUIRE((*s)[i] * esz % 16 == 0, "%s: strides must be multiples of 16 bytes", who);
    // a lane's byte offsets inside one block are kept in 32 bits
    RTP_REQUIRE((*s)[0] >= 0 && (*s)[0] < (1ll << 25), "%s: sequence stride out of range", who);
  }
  RTP_REQUIRE(G * N * H * ceil_div(L > S ? L : S, 32) < (1ll << 31), "%s: too many (head, block) work items", who);
  a.q_l = qs[0] * esz, a.q_b = qs[1] * esz, a.q_h = qs[2] * esz, a.q_g = qs[3] * esz;
  a.k_l = ks[0] * esz, a.k_b = ks[1] * esz, a.k_h = ks[2] * esz, a.k_g = ks[3] * esz;
  a.o_l = os[0] * esz, a.o_b = os[1] * esz, a.o_h = os[2] * esz, a.o_g = os[3] * esz;
  a.mask = mask, a.kbias = key_bias, a.causal = causal, a.scale = scale;
  a.L = (int)L, a.S = (int)S, a.N = (int)N, a.H = (int)H, a.nprob = (int)(G * N * H);
  return RTP_OK;
}

}  // namespace rtp

using namespace rtp;

extern "C" int rtp_attn_flash_kv_supported(int dtype, int64_t L, int64_t S, int64_t D) {
  return dtype == RTP_BF16 && L >= 1 && L <= kFlashMaxLen && S >= 1 && S <= kFlashMaxLen &&
         (D == 32 || D == 64 || D == 128);
}

static int flash_forward(void* stream, int dtype, const void* q, const int64_t (&qs)[4], const void* k, const void* v,
                         const int64_t (&ks)[4], void* o, const int64_t (&os)[4], float* lse, const float* mask,
                         const float* key_bias, int causal, float scale, int64_t L, int64_t S, int64_t N, int64_t H,
                         int64_t D, int64_t G, float empty) {
  RTP_REQUIRE(q && k && v && o && lse, "rtp_attn_flash_fwd: null pointer");
  RTP_REQUIRE(((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)o) % 16 == 0,
              "rtp_attn_flash_fwd: q, k, v, o must be 16-byte aligned");
  FlashArgs a{};
  if (int rc = flash_args("rtp_attn_flash_fwd", a, dtype, qs, ks, os, mask, key_bias, causal, scale, L, S, N, H, D, G))
    return rc;
  a.q = (const char*)q, a.k = (const char*)k, a.v = (const char*)v, a.out = (char*)o, a.lse = lse, a.empty = empty;
  hipStream_t st = (hipStream_t)stream;
  const double np = (double)a.nprob, vis = causal ? 0.5 : 1.0, esz = 2.0;
  ProfileScope prof(st, "attn_flash_fwd", 4.0 * np * L * S * D * vis, np * (2.0 * (L + S) * D * esz + 4.0 * L));
  return flash_launch<FlashFwd>(st, D, a, L);
}

extern "C" int rtp_attn_flash_kv_fwd(void* stream, int dtype, const void* q, int64_t q_l, int64_t q_b, int64_t q_h,
                                     int64_t q_g, const void* k, const void* v, int64_t k_l, int64_t k_b, int64_t k_h,
                                     int64_t k_g, void* o, int64_t o_l, int64_t o_b, int64_t o_h, int64_t o_g, float* lse,
                                     const float* mask, const float* key_bias, int causal, float scale, int64_t L,
                                     int64_t S, int64_t N, int64_t H, int64_t D, int64_t G) {
  return flash_forward(stream, dtype, q, {q_l, q_b, q_h, q_g}, k, v, {k_l, k_b, k_h, k_g}, o, {o_l, o_b, o_h, o_g}, lse, mask,
                       key_bias, causal, scale, L, S, N, H, D, G, __builtin_nanf(""));
}

extern "C" int rtp_attn_flash_kv_bwd(void* stream, int dtype, const void* q, int64_t q_l, int64_t q_b, int64_t q_h,
                                     int64_t q_g, const void* k, const void* v, int64_t k_l, int64_t k_b, int64_t k_h,
                                     int64_t k_g, const void* o, const void* dout, int64_t o_l, int64_t o_b, int64_t o_h,
                                     int64_t o_g, const float* lse, float* delta, void* dq, void* dk, void* dv,
                                     const float* mask, const float* key_bias, int causal, float scale, int64_t L,
                                     int64_t S, int64_t N, int64_t H, int64_t D, int64_t G) {
  RTP_REQUIRE(q && k && v && o && dout && lse && delta && dq && dk && dv, "rtp_attn_flash_bwd: null pointer");
  RTP_REQUIRE(((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)o | (uintptr_t)dout | (uintptr_t)dq |
               (uintptr_t)dk | (uintptr_t)dv) % 16 == 0,
              "rtp_attn_flash_bwd: q, k, v, o, dout, dq, dk, dv must be 16-byte aligned");
  FlashArgs a{};
  if (int rc = flash_args("rtp_attn_flash_bwd", a, dtype, {q_l, q_b, q_h, q_g}, {k_l, k_b, k_h, k_g}, {o_l, o_b, o_h, o_g},
                          mask, key_bias, causal, scale, L, S, N, H, D, G))
    return rc;
  a.q = (const char*)q, a.k = (const char*)k, a.v = (const char*)v;
  a.dq = (char*)dq, a.dk = (char*)dk, a.dv = (char*)dv;
  a.o = (const char*)o, a.dout = (const char*)dout;
  a.lse = const_cast<float*>(lse), a.delta = delta;
  hipStream_t st = (hipStream_t)stream;
  const double np = (double)a.nprob, vis = causal ? 0.5 : 1.0, esz = 2.0;
  {
    // the query pass writes delta, the key pass reads it: same stream, in this order
    ProfileScope prof(st, "attn_flash_dq", 6.0 * np * L * S * D * vis, np * ((4.0 * L + 2.0 * S) * D * esz + 8.0 * L));
    if (int rc = flash_launch<FlashDq>(st, D, a, L)) return rc;
  }
  ProfileScope prof(st, "attn_flash_dkv", 8.0 * np * L * S * D * vis, np * ((2.0 * L + 4.0 * S) * D * esz + 8.0 * L));
  return flash_launch<FlashDkv>(st, D, a, S);
}

// q, k and v packed side by side with common strides, as many keys as queries
extern "C" int rtp_attn_flash_supported(int dtype, int64_t L, int64_t D) {
  return rtp_attn_flash_kv_supported(dtype, L, L, D);
}

extern "C" int rtp_attn_flash_fwd(void* stream, int dtype, const void* q, const void* k, const void* v, int64_t s_l,
                                  int64_t s_b, int64_t s_h, int64_t s_g, void* o, int64_t o_l, int64_t o_b,
                                  int64_t o_h, int64_t o_g, float* lse, const float* mask, const float* key_bias,
                                  int causal, float scale, int64_t L, int64_t N, int64_t H, int64_t D, int64_t G) {
  return flash_forward(stream, dtype, q, {s_l, s_b, s_h, s_g}, k, v, {s_l, s_b, s_h, s_g}, o, {o_l, o_b, o_h, o_g}, lse, mask,
                       key_bias, causal, scale, L, L, N, H, D, G, 0.0f);
}

extern "C" int rtp_attn_flash_bwd(void* stream, int dtype, const void* q, const void* k, const void* v, int64_t s_l,
                                  int64_t s_b, int64_t s_h, int64_t s_g, const void* o, const void* dout, int64_t o_l,
                                  int64_t o_b, int64_t o_h, int64_t o_g, const float* lse, float* delta, void* dq,
                                  void* dk, void* dv, const float* mask, const float* key_bias, int causal, float scale,
                                  int64_t L, int64_t N, int64_t H, int64_t D, int64_t G) {
  return rtp_attn_flash_kv_bwd(stream, dtype, q, s_l, s_b, s_h, s_g, k, v, s_l, s_b, s_h, s_g, o, dout, o_l, o_b, o_h, o_g,
                               lse, delta, dq, dk, dv, mask, key_bias, causal, scale, L, L, N, H, D, G);
}
