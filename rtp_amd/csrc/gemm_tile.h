// What the product kernels share: their arguments, MFMA fragments, direct-to-LDS loads and epilogues.
#pragma once

#include <type_traits>

#include "common.h"

namespace rtp {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(4))) float f32x4;

struct GemmArgs {
  const char* a;
  const char* b;
  char* c_out;
  const char* c_in;
  const char* bias;
  const char* gate;
  int m, n, k, ksegs;
  long lda, ldb, ldc, ld_cin, ld_gate;
  int batch, zdiv;
  long a_so, a_si, b_so, b_si, c_so, c_si, cin_so, cin_si, gate_so, gate_si, bias_so, bias_si;
  long a_sg, b_sg, c_sg, cin_sg, gate_sg, bias_sg;
  long a_sk, b_sk, bias_sk;
  float alpha;
  int flags;
  int vec_a, vec_b;
  int tiles_m, tiles_n;
  int vec_c;       // every epilogue operand allows 16-byte accesses of 8 columns
  int xg, xm, xn;  // split of the (batch*groups, tiles_m, tiles_n) space over the 8 XCDs; xg == 0: none
  char* a_rowsum;  // bias gradient output (sum over k of A's rows), or null
  long rowsum_sg;
  // wave-specialised kernel: tile mapping without run-time divisions
  // A brick is mbk x nbk tiles; its tiles are handed out panel by panel, a panel being prow x pcol tiles with the
  // row running fastest, and the panels of a strip of pcol tile columns follow each other down the rows before
  // the next strip starts -- see the kernel.
  FastDiv d_batch, d_zdiv, d_tiles_n, d_brick, d_panel, d_prow, d_pm;  // divisors mbk*nbk, prow*pcol, prow, mbk/prow
  int mbk, nbk, prow, pcol;
  int xn_shift, xm_shift, zbk;  // log2 of xn and xm, batch*groups entries per brick
  unsigned long long* trace;    // null, or two words: earliest start / latest end of the launch on the wall clock
  float* sgd_master;            // null, or the fp32 parameters the product updates (indexed like c_out)
  char* sgd_w;                  // null, or the compute-dtype copy of the parameters
  float sgd_lr, sgd_clip;
  // softmax cross-entropy over the product's rows (the product is the logits of a column-parallel layer):
  // mode 1 leaves per-(row, 64-column block) {max, sum exp} and the target's logit instead of the logits,
  // mode 2 turns the logits into their gradient before they are stored
  int xent_mode, xent_blocks;   // blocks: 64-column blocks per row over all groups
  const long* xent_target;
  long xent_ignore;
  float2* xent_part;            // mode 1: [m][xent_blocks]
  float* xent_tlogit;           // mode 1: [m]
  const float2* xent_stats;     // mode 2: [m] {max, sum exp} of the whole row
  const float* xent_dloss;      // mode 2: upstream gradient, one scalar
  const float* xent_scale;      // mode 2: second scalar factor (1 / rows counted), or null
  // bytes that some later launch will read from HBM (the next layer's shards): requested here, see WarmAhead
  const char* warm;
  unsigned warm_pieces;         // KiB
  int warm_each, warm_slab;     // pieces of a wave at most, and those that it asks for in a slab
  unsigned tiles, per_xcd;  // gemm_large.hip: all tiles of the launch, an XCD's share of them (rounded up)
};

// The per-lane MFMA operand: VEC consecutive k values of one tile row.
template <typename T>
struct Frag;
template <>
struct Frag<bf16_t> {
  bf16x8 v;
};
template <>
struct Frag<float> {
  float f[4];
};

__device__ __forceinline__ void mma(const Frag<bf16_t>& a, const Frag<bf16_t>& b, f32x16& c) {
  c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.v, b.v, c, 0, 0, 0);
}
// 16 x 16 outputs over 32 k: lane group g = lane / 16 holds k = 8g + e in element e and rows 4g + r of the results in register r.
__device__ __forceinline__ void mma(const Frag<bf16_t>& a, const Frag<bf16_t>& b, f32x4& c) {
  c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.v, b.v, c, 0, 0, 0);
}
__device__ __forceinline__ void mma(const Frag<float>& a, const Frag<float>& b, f32x16& c) {
  // Lane group g holds k = 4g+e in element e, so MFMA number e contracts k in {e, 4+e}.
#pragma unroll
  for (int e = 0; e < 4; ++e) c = __builtin_amdgcn_mfma_f32_32x32x2f32(a.f[e], b.f[e], c, 0, 0, 0);
}

// Sum of the fragment's k values in fp32 (the lane's share of a row sum of A).
__device__ __forceinline__ float frag_sum(const Frag<bf16_t>& a, float s) {
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  const bf16x2 one = {(__bf16)1.0f, (__bf16)1.0f};
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const bf16x2 pr = {a.v[2 * e], a.v[2 * e + 1]};
    s = __builtin_amdgcn_fdot2_f32_bf16(pr, one, s, false);
  }
  return s;
}
__device__ __forceinline__ float frag_sum(const Frag<float>& a, float s) {
  return s + ((a.f[0] + a.f[1]) + (a.f[2] + a.f[3]));
}

// Fused epilogue shared by the GEMM kernels.  Accumulator register r of lane (li, g) is output row
// 8*(r/4) + 4*g + r%4, column li of its 32x32 block.
template <typename T, int MT, int NT, int WM, int WN>
__device__ __forceinline__ void store_tile(const GemmArgs& p, f32x16 (&acc)[MT][NT], int m0, int n0, int wm, int wn,
                                           int li, int g, int grp, long zo, long zi) {
  const bool out_f32 = p.flags & RTP_GEMM_OUT_F32;
  const bool cin_f32 = p.flags & RTP_GEMM_CIN_F32;
  const bool relu = p.flags & RTP_GEMM_RELU;
  char* cbase = p.c_out + (grp * p.c_sg + zo * p.c_so + zi * p.c_si) * (out_f32 ? 4 : (long)sizeof(T));
  const char* cin =
      p.c_in ? p.c_in + (grp * p.cin_sg + zo * p.cin_so + zi * p.cin_si) * (cin_f32 ? 4 : (long)sizeof(T)) : nullptr;
  const T* bias =
      p.bias ? reinterpret_cast<const T*>(p.bias) + grp * p.bias_sg + zo * p.bias_so + zi * p.bias_si : nullptr;
  const T* gate =
      p.gate ? reinterpret_cast<const T*>(p.gate) + grp * p.gate_sg + zo * p.gate_so + zi * p.gate_si : nullptr;

#pragma unroll
  for (int i = 0; i < MT; ++i) {
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const int col = n0 + wn * WN + j * 32 + li;
      if (col >= p.n) continue;
      float bv = 0.0f;
      if (bias) {
        // a bias per K segment (row-parallel shards each carry bias/ws): summed in segment order
        const int nb_seg = p.bias_sk ? p.ksegs : 1;
        for (int sgm = 0; sgm < nb_seg; ++sgm) bv += to_f32(bias[sgm * p.bias_sk + col]);
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int row = m0 + wm * WM + i * 32 + 8 * (r >> 2) + 4 * g + (r & 3);
        if (row >= p.m) continue;
        float v = p.alpha * acc[i][j][r];
        if (cin) {
          const long off = (long)row * p.ld_cin + col;
          v += cin_f32 ? reinterpret_cast<const float*>(cin)[off] : to_f32(reinterpret_cast<const T*>(cin)[off]);
        }
        v += bv;
        if (relu) v = fmaxf(v, 0.0f);
        if (gate) v = to_f32(gate[(long)row * p.ld_gate + col]) > 0.0f ? v : 0.0f;
        const long off = (long)row * p.ldc + col;
        if (out_f32)
          reinterpret_cast<float*>(cbase)[off] = v;
        else
          reinterpret_cast<T*>(cbase)[off] = from_f32<T>(v);
      }
    }
  }
}

// Epilogue of the direct-to-LDS kernel.  `ct` is the BM x BN tile of raw accumulators in LDS (row pitch BN+4
// floats).  Thread `tid` of NTHR finishes chunks of 8 consecutive columns: alpha * acc (+ c_in) (+ bias) -> ReLU ->
// gate mask -> store, the same order of operations as store_tile.  p.vec_c holds (16-byte aligned operands and
// n % 8 == 0, checked by the host): every global access of a chunk is a 16-byte vector.
template <typename T>
__device__ __forceinline__ void load8(const T* src, float (&v)[8]) {
  if (sizeof(T) == 2) {
    union {
      uint4 q;
      T e[8];
    } u;
    u.q = *reinterpret_cast<const uint4*>(src);
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = to_f32(u.e[e]);
  } else {
    const float4 lo = reinterpret_cast<const float4*>(src)[0], hi = reinterpret_cast<const float4*>(src)[1];
    v[0] = lo.x, v[1] = lo.y, v[2] = lo.z, v[3] = lo.w, v[4] = hi.x, v[5] = hi.y, v[6] = hi.z, v[7] = hi.w;
  }
}
template <typename T>
__device__ __forceinline__ void store8(T* dst, const float (&v)[8], bool stream) {
  if (sizeof(T) == 2) {
    union {
      uint4 q;
      T e[8];
    } u;
#pragma unroll
    for (int e = 0; e < 8; ++e) u.e[e] = from_f32<T>(v[e]);
    if (stream)
      nt_store(u.q, reinterpret_cast<uint4*>(dst));
    else
      *reinterpret_cast<uint4*>(dst) = u.q;
  } else if (stream) {
    nt_store(make_float4(v[0], v[1], v[2], v[3]), reinterpret_cast<float4*>(dst));
    nt_store(make_float4(v[4], v[5], v[6], v[7]), reinterpret_cast<float4*>(dst) + 1);
  } else {
    reinterpret_cast<float4*>(dst)[0] = make_float4(v[0], v[1], v[2], v[3]);
    reinterpret_cast<float4*>(dst)[1] = make_float4(v[4], v[5], v[6], v[7]);
  }
}

// Raw 16-byte-vector image of 8 consecutive epilogue operand values (c_in in `dtype` or fp32, bias, gate): what a thread
// requests for all of its chunks before it consumes any of them.
template <typename T>
struct Raw8 {
  uint4 q[sizeof(T) == 2 ? 1 : 2];
  __device__ __forceinline__ void load(const T* src) {
    q[0] = reinterpret_cast<const uint4*>(src)[0];
    if (sizeof(T) == 4) q[sizeof(T) == 2 ? 0 : 1] = reinterpret_cast<const uint4*>(src)[1];
  }
  __device__ __forceinline__ void get(float (&v)[8]) const {
    if (sizeof(T) == 2) {
      union {
        uint4 q;
        T e[8];
      } u;
      u.q = q[0];
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = to_f32(u.e[e]);
    } else {
      union {
        uint4 q[2];
        float f[8];
      } u;
      u.q[0] = q[0], u.q[1] = q[sizeof(T) == 2 ? 0 : 1];
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = u.f[e];
    }
  }
};

// Eight logits -> their cross-entropy gradient: (softmax - onehot(target)) * dloss (* scale); rows whose target is the
// ignore index or outside the classes get zeros.
template <typename T, typename Args>  // (the arguments in either address space)
__device__ __forceinline__ void xent_gradient8(Args& p, float (&v)[8], long row, int col, int grp) {
  const long tg = p.xent_target[row];
  const bool live = tg != p.xent_ignore && tg >= 0 && tg < (long)p.xent_blocks * 64;
  const float2 st = p.xent_stats[row];
  const float inv = 1.0f / st.y;
  const float sc = live ? p.xent_dloss[0] * (p.xent_scale ? p.xent_scale[0] : 1.0f) : 0.0f;
  const long gcol = (long)grp * p.n + col;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    float gq = expf(to_f32(from_f32<T>(v[e])) - st.x) * inv;
    if (gcol + e == tg) gq -= 1.0f;
    v[e] = gq * sc;
  }
}

template <typename T, int BM, int BN, int NTHR>
__device__ __forceinline__ void finish_tile(const GemmArgs& p, const float* ct, int m0, int n0, int tid, int grp,
                                            long zo, long zi) {
  constexpr int CP = BN + 4, CPR = BN / 8, CHUNKS = BM * CPR;
  const bool stream_out = p.flags & RTP_GEMM_STREAM_OUT;
  const bool out_f32 = p.flags & RTP_GEMM_OUT_F32;
  const bool cin_f32 = p.flags & RTP_GEMM_CIN_F32;
  const bool relu = p.flags & RTP_GEMM_RELU;
  char* cbase = p.c_out + (grp * p.c_sg + zo * p.c_so + zi * p.c_si) * (out_f32 ? 4 : (long)sizeof(T));
  const char* cin =
      p.c_in ? p.c_in + (grp * p.cin_sg + zo * p.cin_so + zi * p.cin_si) * (cin_f32 ? 4 : (long)sizeof(T)) : nullptr;
  const T* bias =
      p.bias ? reinterpret_cast<const T*>(p.bias) + grp * p.bias_sg + zo * p.bias_so + zi * p.bias_si : nullptr;
  const T* gate =
      p.gate ? reinterpret_cast<const T*>(p.gate) + grp * p.gate_sg + zo * p.gate_so + zi * p.gate_si : nullptr;
  const int nb_seg = p.bias_sk ? p.ksegs : 1;  // a bias per K segment is summed in segment order

  if constexpr (CHUNKS % NTHR == 0) {
    // The common form (vector-aligned operands, one bias vector): a thread requests the bias, the addend and the mask
    // of ALL its chunks before it consumes the first -- one trip to memory for the whole epilogue instead of one per
    // chunk (a store to c_out may alias a later chunk's c_in as far as the compiler knows, so left alone the loads of
    // chunk i + 1 wait behind the store of chunk i).  When the thread count is a multiple of the chunks per row all of
    // a thread's chunks lie in the same 8 columns and share one bias vector.
    if (nb_seg == 1 && p.xent_mode == 0) {
      constexpr int NCH = CHUNKS / NTHR;
      constexpr bool SAMECOL = NTHR % CPR == 0;
      constexpr int NB = SAMECOL ? 1 : NCH;
      Raw8<T> rb[NB], rg[NCH], rc16[NCH];
      Raw8<float> rc32[NCH];
#pragma unroll
      for (int i = 0; i < NCH; ++i) {
        const int c = tid + i * NTHR;
        const int row = m0 + c / CPR, col = n0 + (c % CPR) * 8;
        const int colc = col < p.n ? col : 0;
        const long rowc = row < p.m ? row : p.m - 1;
        if (bias && (i == 0 || !SAMECOL)) rb[SAMECOL ? 0 : i].load(bias + colc);
        if (cin) {
          if (cin_f32)
            rc32[i].load(reinterpret_cast<const float*>(cin) + rowc * p.ld_cin + colc);
          else
            rc16[i].load(reinterpret_cast<const T*>(cin) + rowc * p.ld_cin + colc);
        }
        if (gate) rg[i].load(gate + rowc * p.ld_gate + colc);
      }
#pragma unroll
      for (int i = 0; i < NCH; ++i) {
        const int c = tid + i * NTHR;
        const int lr = c / CPR, lc = (c % CPR) * 8;
        const int row = m0 + lr, col = n0 + lc;
        const bool col_ok = col < p.n;
        float v[8], t[8];
        const float4 lo = *reinterpret_cast<const float4*>(ct + lr * CP + lc);
        const float4 hi = *reinterpret_cast<const float4*>(ct + lr * CP + lc + 4);
        v[0] = lo.x, v[1] = lo.y, v[2] = lo.z, v[3] = lo.w, v[4] = hi.x, v[5] = hi.y, v[6] = hi.z, v[7] = hi.w;
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] *= p.alpha;
        if (cin) {
          if (cin_f32)
            rc32[i].get(t);
          else
            rc16[i].get(t);
#pragma unroll
          for (int e = 0; e < 8; ++e) v[e] += t[e];
        }
        if (bias) {
          rb[SAMECOL ? 0 : i].get(t);
#pragma unroll
          for (int e = 0; e < 8; ++e) v[e] += t[e];
        }
        if (relu) {
#pragma unroll
          for (int e = 0; e < 8; ++e) v[e] = fmaxf(v[e], 0.0f);
        }
        if (gate) {
          rg[i].get(t);
#pragma unroll
          for (int e = 0; e < 8; ++e) v[e] = t[e] > 0.0f ? v[e] : 0.0f;
        }
        if (row >= p.m || !col_ok) continue;
        const long off = (long)row * p.ldc + col;
        if (out_f32)
          store8(reinterpret_cast<float*>(cbase) + off, v, stream_out);
        else
          store8(reinterpret_cast<T*>(cbase) + off, v, stream_out);
      }
      return;
    }
  }

  for (int c = tid; c < CHUNKS; c += NTHR) {
    const int lr = c / CPR, lc = (c % CPR) * 8;
    const int row = m0 + lr, col = n0 + lc;
    if (row >= p.m || col >= p.n) continue;
    float v[8], t[8];
    {
      const float4 lo = *reinterpret_cast<const float4*>(ct + lr * CP + lc);
      const float4 hi = *reinterpret_cast<const float4*>(ct + lr * CP + lc + 4);
      v[0] = lo.x, v[1] = lo.y, v[2] = lo.z, v[3] = lo.w, v[4] = hi.x, v[5] = hi.y, v[6] = hi.z, v[7] = hi.w;
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] *= p.alpha;
    if (cin) {
      const long off = (long)row * p.ld_cin + col;
      if (cin_f32)
        load8(reinterpret_cast<const float*>(cin) + off, t);
      else
        load8(reinterpret_cast<const T*>(cin) + off, t);
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] += t[e];
    }
    if (bias) {
      // The per-segment biases of a row-parallel layer sit in eight different home rows, far from any cache: the
      // loads of eight segments are issued together (segments past the last re-read segment 0 and count as zero)
      // and then added in segment order -- one trip to memory instead of one per segment.
      float bv[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
      for (int s0 = 0; s0 < nb_seg; s0 += 8) {
        float bt[8][8];
#pragma unroll
        for (int j = 0; j < 8; ++j) load8(bias + (s0 + j < nb_seg ? s0 + j : 0) * p.bias_sk + col, bt[j]);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const float on = s0 + j < nb_seg ? 1.0f : 0.0f;
#pragma unroll
          for (int e = 0; e < 8; ++e) bv[e] += on * bt[j][e];
        }
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] += bv[e];
    }
    if (relu) {
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = fmaxf(v[e], 0.0f);
    }
    if (gate) {
      load8(gate + (long)row * p.ld_gate + col, t);
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = t[e] > 0.0f ? v[e] : 0.0f;
    }
    if (p.xent_mode == 2) {
      xent_gradient8<T>(p, v, row, col, grp);
    }
    const long off = (long)row * p.ldc + col;
    if (out_f32)
      store8(reinterpret_cast<float*>(cbase) + off, v, stream_out);
    else
      store8(reinterpret_cast<T*>(cbase) + off, v, stream_out);
  }
}

// Up to eight consecutive values at any alignment, as fp32; those from `n` (at least 1) on, which may lie outside the operand, are left out:
// the last one is read in their place, so that the loads are without branches and wait together.
template <typename S>
__device__ __forceinline__ void load8_any(const S* src, int n, float (&v)[8]) {
  constexpr int VEC = 16 / (int)sizeof(S);
  typedef S vec_t __attribute__((ext_vector_type(VEC), aligned(sizeof(S))));
  if (n >= 8) {
#pragma unroll
    for (int h = 0; h < 8 / VEC; ++h) {
      const vec_t q = *reinterpret_cast<const vec_t*>(src + h * VEC);
#pragma unroll
      for (int e = 0; e < VEC; ++e) v[h * VEC + e] = to_f32((S)q[e]);
    }
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = to_f32(src[min(e, n - 1)]);
  }
}
template <typename S>
__device__ __forceinline__ void store8_any(S* dst, int n, const float (&v)[8]) {
  constexpr int VEC = 16 / (int)sizeof(S);
  typedef S vec_t __attribute__((ext_vector_type(VEC), aligned(sizeof(S))));
  if (n >= 8) {
#pragma unroll
    for (int h = 0; h < 8 / VEC; ++h) {
      vec_t q;
#pragma unroll
      for (int e = 0; e < VEC; ++e) q[e] = from_f32<S>(v[h * VEC + e]);
      *reinterpret_cast<vec_t*>(dst + h * VEC) = q;
    }
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e)
      if (e < n) dst[e] = from_f32<S>(v[e]);
  }
}

// The epilogue where an operand of it is not vector-aligned (an odd width, a shard of odd size): the operations of finish_tile on
// 16-byte accesses of any alignment, element by element only in the eight columns that the product's last ones lie in.
// (Its predecessor went element by element throughout: 14.5 us outside the K loop of a 128 x 128 tile in bf16, now 6 - 10.  us, before ->
// now, forward / weight gradient: 1250 x 9090 x 1792, 2 shards, 164 / 206 -> 136 / 160; 2001 x 2003 x 2005 36.9 / 47.9 -> 32.7 /
// 44.1; 992 x 126 x 2048, 8 shards, 18.8 / 20.1 -> 17.8 / 18.1; 255 x 1023 x 3333 16.9 / 18.4 -> 16.4 / 13.3; fp32 3222 x 4321 x 137 79 / 77 -> 70 / 75.)
template <typename T, int BM, int BN, int NTHR>
__device__ __forceinline__ void finish_tile_ragged(const GemmArgs& p, const float* ct, int m0, int n0, int tid, int grp,
                                                   long zo, long zi) {
  constexpr int CP = BN + 4, CPR = BN / 8, NCH = BM * CPR / NTHR;
  static_assert(BM * CPR % NTHR == 0 && NTHR % CPR == 0, "whole chunks, all of a thread's in the same columns");
  const bool out_f32 = p.flags & RTP_GEMM_OUT_F32;
  const bool cin_f32 = p.flags & RTP_GEMM_CIN_F32;
  const bool relu = p.flags & RTP_GEMM_RELU;
  const long zoff = grp * p.c_sg + zo * p.c_so + zi * p.c_si;
  char* cbase = p.c_out + zoff * (out_f32 ? 4 : (long)sizeof(T));
  const char* cin =
      p.c_in ? p.c_in + (grp * p.cin_sg + zo * p.cin_so + zi * p.cin_si) * (cin_f32 ? 4 : (long)sizeof(T)) : nullptr;
  const T* bias =
      p.bias ? reinterpret_cast<const T*>(p.bias) + grp * p.bias_sg + zo * p.bias_so + zi * p.bias_si : nullptr;
  const T* gate =
      p.gate ? reinterpret_cast<const T*>(p.gate) + grp * p.gate_sg + zo * p.gate_so + zi * p.gate_si : nullptr;
  const int nb_seg = p.bias_sk ? p.ksegs : 1;
  float* master = p.sgd_master ? p.sgd_master + zoff : nullptr;
  T* wcopy = p.sgd_w ? reinterpret_cast<T*>(p.sgd_w) + zoff : nullptr;
  const bool skip_out = p.flags & RTP_GEMM_SGD_SKIP_OUT;
  const int lc = (tid % CPR) * 8, col = n0 + lc, live = p.n - col;
  if (live <= 0) return;
  // what the thread's chunks need from memory, requested before the first is finished
  float add[NCH][8], msk[NCH][8], bv[8];
#pragma unroll
  for (int i = 0; i < NCH; ++i) {
    const long row = min(m0 + (tid + i * NTHR) / CPR, p.m - 1);
    if (cin) {
      const long off = row * p.ld_cin + col;
      if (cin_f32)
        load8_any(reinterpret_cast<const float*>(cin) + off, live, add[i]);
      else
        load8_any(reinterpret_cast<const T*>(cin) + off, live, add[i]);
    }
    if (gate) load8_any(gate + row * p.ld_gate + col, live, msk[i]);
    if (master) load8_any(master + row * p.ldc + col, live, add[i]);  // (an update excludes an addend)
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) bv[e] = 0.0f;
  if (bias && nb_seg == 1)
    load8_any(bias + col, live, bv);
  else if (bias)
    for (int s0 = 0; s0 < nb_seg; s0 += 4) {  // four segments' at a time, added in their order
      float bt[4][8];
#pragma unroll
      for (int j = 0; j < 4; ++j) load8_any(bias + (s0 + j < nb_seg ? s0 + j : 0) * p.bias_sk + col, live, bt[j]);
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (s0 + j < nb_seg) {
#pragma unroll
          for (int e = 0; e < 8; ++e) bv[e] += bt[j][e];
        }
    }
#pragma unroll
  for (int i = 0; i < NCH; ++i) {
    const int lr = (tid + i * NTHR) / CPR;
    if (m0 + lr >= p.m) break;  // the rows behind this one as well
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      v[e] = p.alpha * ct[lr * CP + lc + e];
      if (cin) v[e] += add[i][e];
      if (bias) v[e] += bv[e];
      if (relu) v[e] = fmaxf(v[e], 0.0f);
      if (gate) v[e] = msk[i][e] > 0.0f ? v[e] : 0.0f;
    }
    const long off = (long)(m0 + lr) * p.ldc + col;
    if (master) {
      float w[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) w[e] = sgd_update<T>(add[i][e], v[e], p.sgd_lr, p.sgd_clip);
      store8_any(master + off, live, w);
      if (wcopy) store8_any(wcopy + off, live, w);
    }
    if (skip_out) continue;
    if (out_f32)
      store8_any(reinterpret_cast<float*>(cbase) + off, live, v);
    else
      store8_any(reinterpret_cast<T*>(cbase) + off, live, v);
  }
}

// Epilogue of a logits product whose rows only feed a softmax cross-entropy (mode 1): thread r of the first BM
// threads walks row r of the tile in LDS, 64 columns at a time, and leaves {max, sum exp(v - max)} of every
// 64-column block in part[row][block] -- the block index runs over the layer's whole output row, group after
// group, so the layout does not depend on the tile shape -- and the logit of the row's target where this tile
// holds it.  The logits themselves are not stored.  v = alpha * acc + bias, rounded to T as the stored logits would
// be, so that loss and gradient are those of the logits a separate product would have written.
template <typename T, int BM, int BN, int NTHR>
__device__ __forceinline__ void finish_tile_xent_stats(const GemmArgs& p, const float* ct, int m0, int n0, int tid,
                                                       int grp) {
  static_assert(BN % 64 == 0 && BM <= NTHR, "64-column blocks, one thread per tile row");
  constexpr int CP = BN + 4;
  if (tid >= BM) return;
  const int row = m0 + tid;
  if (row >= p.m) return;
  const T* bias = p.bias ? reinterpret_cast<const T*>(p.bias) + grp * p.bias_sg : nullptr;
  const long t = p.xent_target[row];
  const long tcol = t - (long)grp * p.n;  // the target's column inside this group, if it is in [0, n)
  const float* crow = ct + tid * CP;
#pragma unroll
  for (int b = 0; b < BN / 64; ++b) {
    const int col0 = n0 + b * 64;
    if (col0 >= p.n) break;
    float mx = -INFINITY;
    for (int j = 0; j < 64; ++j) {
      float v = p.alpha * crow[b * 64 + j];
      if (bias) v += to_f32(bias[col0 + j]);
      v = to_f32(from_f32<T>(v));
      mx = fmaxf(mx, v);
      if (col0 + j == tcol) p.xent_tlogit[row] = v;
    }
    float sum = 0.0f;
    for (int j = 0; j < 64; ++j) {
      float v = p.alpha * crow[b * 64 + j];
      if (bias) v += to_f32(bias[col0 + j]);
      v = to_f32(from_f32<T>(v));
      sum += expf(v - mx);
    }
    p.xent_part[(long)row * p.xent_blocks + ((long)grp * p.n + col0) / 64] = make_float2(mx, sum);
  }
}

// Epilogue of a product whose result is consumed by the fused clip + SGD update (a weight gradient: no c_in, bias,
// ReLU or mask; 16-byte aligned operands, checked by the host).  The fp32 parameters of up to four of the thread's
// chunks are requested before the first of them is needed, so the trips to memory overlap instead of following
// each other; rows / columns outside the problem read a clamped address and store nothing.
template <typename T, int BM, int BN, int NTHR>
__device__ __forceinline__ void finish_tile_sgd(const GemmArgs& p, const float* ct, int m0, int n0, int tid, int grp,
                                                long zo, long zi) {
  constexpr int CP = BN + 4, CPR = BN / 8, CHUNKS = BM * CPR, NCH = CHUNKS / NTHR;
  constexpr int BATCH = NCH % 4 == 0 ? 4 : (NCH % 3 == 0 ? 3 : (NCH % 2 == 0 ? 2 : 1));
  static_assert(CHUNKS % NTHR == 0 && NCH % BATCH == 0, "every thread owns the same number of chunks");
  const bool stream_out = p.flags & RTP_GEMM_STREAM_OUT;
  const bool skip_out = p.flags & RTP_GEMM_SGD_SKIP_OUT;
  const long zoff = grp * p.c_sg + zo * p.c_so + zi * p.c_si;
  T* cbase = reinterpret_cast<T*>(p.c_out) + zoff;
  float* master = p.sgd_master + zoff;
  T* wcopy = p.sgd_w ? reinterpret_cast<T*>(p.sgd_w) + zoff : nullptr;
#pragma unroll
  for (int b0 = 0; b0 < NCH; b0 += BATCH) {
    float w[BATCH][8];
    long off[BATCH];
    bool live[BATCH];
#pragma unroll
    for (int i = 0; i < BATCH; ++i) {
      const int c = tid + (b0 + i) * NTHR;
      const int row = m0 + c / CPR, col = n0 + (c % CPR) * 8;
      live[i] = row < p.m && col < p.n;
      off[i] = (long)(row < p.m ? row : p.m - 1) * p.ldc + (col < p.n ? col : 0);
      load8(master + off[i], w[i]);
    }
#pragma unroll
    for (int i = 0; i < BATCH; ++i) {
      const int c = tid + (b0 + i) * NTHR;
      const int lr = c / CPR, lc = (c % CPR) * 8;
      float v[8];
      const float4 lo = *reinterpret_cast<const float4*>(ct + lr * CP + lc);
      const float4 hi = *reinterpret_cast<const float4*>(ct + lr * CP + lc + 4);
      v[0] = lo.x, v[1] = lo.y, v[2] = lo.z, v[3] = lo.w, v[4] = hi.x, v[5] = hi.y, v[6] = hi.z, v[7] = hi.w;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        v[e] *= p.alpha;
        w[i][e] = sgd_update<T>(w[i][e], v[e], p.sgd_lr, p.sgd_clip);
      }
      if (!live[i]) continue;
      store8(master + off[i], w[i], true);
      if (wcopy) store8(wcopy + off[i], w[i], true);
      if (!skip_out) store8(cbase + off[i], v, stream_out);
    }
  }
}

// ---------------------------------------------------------------------------------------------
// Direct-to-LDS pipeline (the fast path).  Slabs go global -> LDS with global_load_lds_dwordx4: no
// staging registers, NSTAGE LDS stages, up to NSTAGE-1 slabs in flight while the MFMAs of the current slab
// run.  The compiler does not order these asynchronous LDS writes against later LDS reads, so the kernel
// does it by hand: in the middle of the phase of slab k every wave waits until its own loads of slab k+1
// have landed (s_waitcnt vmcnt(N), loads retire in order) and then meets the workgroup barrier; after the
// barrier slab k+1 may be read, and the stage of slab k-1 (whose fragments every wave consumed in its
// previous phase) is refilled.
//
// A wave-level load writes 64 lanes x 16 B = 1 KiB of consecutive LDS, so rows cannot be padded.  For a
// k-contiguous operand (LDS [row][128 B]) bank conflicts are avoided by an XOR swizzle instead: the
// 16-byte chunk c of row r is kept at chunk position c ^ (r & 7); the lane that fills position cp of row
// r fetches chunk cp ^ (r & 7) from global memory.  A row-contiguous operand is kept as [k][rows].
// Vectors beyond the contraction length are fetched from a 16-byte block of zeros; rows beyond the
// operand are clamped (they only feed accumulators that are never stored).
//
// The workgroup has 8 waves with separate roles: waves 0..3 run the MFMAs of a 2x2 grid of wave tiles and
// issue no global loads; waves 4..7 only issue the loads and count them down.  Scalar bookkeeping for the
// loads therefore does not take issue slots from the MFMA waves.
static __device__ __attribute__((aligned(16))) unsigned int g_zero16[4] = {0u, 0u, 0u, 0u};

// s_waitcnt with vmcnt = VM, lgkmcnt = 0, expcnt untouched (gfx9 encoding).
#define RTP_WAIT_VM_LGKM0(VM) __builtin_amdgcn_s_waitcnt(((VM)&0xF) | (((VM) >> 4) << 14) | (0x7 << 4))
// s_waitcnt with vmcnt = VM only (expcnt and lgkmcnt untouched).
#define RTP_WAIT_VM(VM) __builtin_amdgcn_s_waitcnt(((VM)&0xF) | (((VM) >> 4) << 14) | (0x7 << 4) | (0xF << 8))

typedef __attribute__((address_space(1))) const void* gptr_t;
typedef __attribute__((address_space(3))) void* lptr_t;

// LDS has 64 four-byte banks (256 bytes per clock).  Swizzles keep the lanes that are served in one clock on
// different banks:
//  * k-contiguous operand, [row][128 B]: 16 consecutive rows read the same 16-byte chunk c; row r keeps it at
//    chunk position c ^ ((r >> 1) & 7), which together with the row's parity (rows alternate between the two
//    128-byte halves of the bank space) gives 16 different 16-byte bank slots.
//  * row-contiguous 16-bit operand, [k][rows]: a transposing read touches 4 consecutive k lines x 64 bytes; the
//    chunk index inside k line kl is XORed with rc_swizzle(kl) so that the 4 lines fall on different slots.  Fragments of FR = 16
//    rows take 32 bytes of eight lines at a time, four neighbouring ones from each of two of the fragment's four octets of k.
template <typename T, int R, int FR = 32>
__device__ __forceinline__ constexpr int rc_swizzle(int kl) {
  if (sizeof(T) != 2 || R < 64) return 0;  // (the 64-byte lines of 32 rows fall on different slots as they stand)
  static_assert(FR == 32 || R >= 128, "fragments of 16 rows: lines of 256 bytes");
  if (FR == 16) return (kl & 3) << 2 | ((kl >> 3 ^ kl >> 4) & 1) << 1;
  return R >= 128 ? (kl & 3) << 2 : ((kl >> 1) & 1) << 2;
}

// Chunk swizzle of a k-contiguous operand whose slab rows are SB bytes (128: 8 chunks, 64: 4 chunks): 16
// consecutive rows reading the same chunk must land on 16 different 16-byte slots of the 256-byte bank space.
template <int SB>
__device__ __forceinline__ constexpr int kc_swizzle(int row) {
  return SB == 128 ? (row >> 1) & 7 : (row >> 2) & 3;
}

template <typename T, int R, bool KC, int NL, int SB, int FR = 32>
struct DmaOperand {
  static constexpr int VEC = 16 / sizeof(T);
  static_assert(SB == 128 || SB == 64, "slab rows of 128 or 64 bytes");
  static_assert((R * SB / 1024) % NL == 0, "every loader wave issues the same number of loads");
  static constexpr int NI = R * SB / 1024 / NL;   // load instructions (1 KiB each) per loader wave and slab
  static constexpr int BYTES = R * SB;            // one stage of this operand
  static constexpr int BK_ = SB / (int)sizeof(T);  // k per slab
  static constexpr int LINE = R * (int)sizeof(T); // bytes of one k line when rows are contiguous
  static_assert(KC || 1024 % LINE == 0 || LINE % 1024 == 0, "a 1 KiB load covers whole k lines or a whole fraction of one");
  // The lane's vector sits at `ofs` bytes from the slab's base pointer, which is the same for every lane and lives
  // in scalar registers: the loader's steady state then has no vector-ALU instruction at all.  (A vector add per
  // load has to compete for issue slots with the MFMAs of the compute wave on the same SIMD, and loses: measured,
  // per-lane 64-bit pointers make the loads of a slab take the MFMA time longer.)
  unsigned ofs[NI];
  int koff[NI];  // k of the vector inside its slab

  // Base pointer of the first slab: row row0 of a K-contiguous operand, element row0 of k line 0 otherwise.
  __device__ __forceinline__ static const char* slab_base(const T* x, long ld, int row0) {
    return reinterpret_cast<const char*>(KC ? x + (long)row0 * ld : x + row0);
  }

  struct Same {
    __device__ __forceinline__ int operator()(int r) const { return r; }
  };
  // lw: index of the loader wave (0..NL-1).  The host guarantees that a tile's offsets fit 32 bits.  row_of: which row behind
  // row0 the operand's row r is (runs of a vector's rows or more stay together).
  template <typename RowOf = Same>
  __device__ __forceinline__ void init(long ld, int row0, int rows, int lw, int lane, RowOf row_of = RowOf()) {
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int j = lw * NI + i;  // which KiB of the stage
      if (KC) {
        constexpr int LPR = SB / 16;  // lanes (16-byte chunks) per row
        const int row = j * (64 / LPR) + lane / LPR;
        const int c = (lane % LPR) ^ kc_swizzle<SB>(row);
        const int src = row_of(row);
        const int rr = row0 + src < rows ? src : rows - 1 - row0;  // rows past the end re-read the last one
        ofs[i] = (unsigned)((long)rr * ld * (long)sizeof(T)) + (unsigned)(c * 16);
        koff[i] = c * VEC;
      } else {
        const int byte = lane * 16;
        const int kl = j * (1024 / LINE) + byte / LINE;
        const int chunk = ((byte % LINE) >> 4) ^ rc_swizzle<T, R, FR>(kl);  // which 16 bytes of the k line land here
        int src = row_of(chunk * VEC);
        if (row0 + src >= rows) src = 0;  // past the end: re-read the tile's first rows (a k line that is no whole number of vectors is padded)
        ofs[i] = (unsigned)((long)kl * ld * (long)sizeof(T)) + (unsigned)(src * (int)sizeof(T));
        koff[i] = kl;
      }
    }
  }

  // Start the loads of the slab at `base` into the stage at LDS byte address `lds_stage` (this operand's part).
  // TAIL: the slab is the last of its K segment (first k = k0) and reaches beyond the contraction length kdim;
  // vectors beyond it come from a block of zeros (per-lane addresses, the one case that needs them).
  template <bool TAIL>
  __device__ __forceinline__ void issue(unsigned lds_stage, int lw, const char* base, int k0, int kdim) const {
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      // Inline assembly on purpose: the compiler must not track this instruction (it would make LDS reads wait
      // for all outstanding loads); the kernel's explicit s_waitcnt + barrier protocol is the ordering that counts.
      if (TAIL) {
        const char* src = base + ofs[i];
        if (k0 + koff[i] >= kdim) src = reinterpret_cast<const char*>(g_zero16);
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off"
                     :
                     : "s"(lds_stage + (unsigned)((lw * NI + i) * 1024)), "v"(src)
                     : "memory");
      } else {
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                     :
                     : "s"(lds_stage + (unsigned)((lw * NI + i) * 1024)), "v"(ofs[i]), "s"(base)
                     : "memory");
      }
    }
  }
};

// The next layer's shards arrive while this product computes.  Weights are read once per pass, so at their turn
// they come from HBM, whose latency the NSTAGE - 1 slabs in flight do not cover: measured on the LM's shapes, a
// product takes 15 - 30 % longer on weights from HBM than on weights that sit in the 256 MiB memory-side cache.
// So a product can be handed the bytes that the *next* products will need: its MFMA waves request them, 1 KiB per
// instruction, straight into 1 KiB of LDS that nothing reads (no registers, and nobody ever waits for these loads: an
// MFMA wave next waits for vector memory in the epilogue).  Pieces are dealt round-robin over (workgroup, wave), so
// the launch as a whole reads the region front to back; a wave asks for at most kWarmMax pieces (the counter of
// outstanding loads has 6 bits), the rest of a larger region stays unread.  They are asked for a few a slab, over the
// first three quarters of the K loop: all of them at the start of the kernel stood in front of its own first slabs and
// residual or mask (the language model's step 3544 us against 3509; over a quarter of the loop 3520, half 3510, all of it
// 3522, where the last ones are still on their way when the epilogue waits for its operands).
constexpr int kWarmMax = 48;
inline void warm_launch(GemmArgs& a, const void* src, size_t bytes, int64_t workgroups, int64_t slabs) {
  const int64_t pieces = bytes >> 10 < 1u << 30 ? (int64_t)(bytes >> 10) : 1 << 30, each = ceil_div(pieces, 4 * workgroups), over = slabs - slabs / 4;
  if (pieces == 0) return;
  a.warm = (const char*)src, a.warm_pieces = (unsigned)pieces;
  a.warm_each = each < kWarmMax ? (int)each : kWarmMax;
  a.warm_slab = (int)ceil_div(a.warm_each, over > 0 ? over : 1);
}
struct WarmAhead {
  const char* src;  // the wave's next piece
  long step;        // bytes from one of its pieces to the next
  unsigned off, lds_dst;
  int left, per_slab;
  __device__ __forceinline__ WarmAhead(const GemmArgs& p, unsigned dst, unsigned wg, unsigned nwg, int wave, int lane, bool paced) {
    src = nullptr, step = 0, left = 0, per_slab = 0;
    if (p.warm != nullptr) {  // (the launch has divided: in front of the first MFMA two divisions took 0.2 us of products of four slabs)
      const unsigned piece = wg * 4 + wave, step_pieces = nwg * 4;
      left = piece + (p.warm_each - 1) * step_pieces < p.warm_pieces ? p.warm_each : p.warm_each - 1;
      per_slab = paced ? p.warm_slab : left;
      src = p.warm + ((long)piece << 10);
      step = (long)step_pieces << 10;
    }
    off = (unsigned)lane * 16u;
    lds_dst = dst;
  }
  __device__ __forceinline__ void slab() {
    if (left <= 0) return;
    for (int j = 0; j < per_slab && left > 0; ++j, --left, src += step)
      asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                   :
                   : "s"(lds_dst), "v"(off), "s"(src)
                   : "memory");
  }
};

// Epilogue operands with vector alignment, requested by the MFMA waves before the K loop (into LDS that nothing reads, like the
// loads of WarmAhead).
template <typename T, int BM, int BN>
__device__ __forceinline__ void request_epilogue(const GemmArgs& p, unsigned lds_dst, int m0, int n0, int grp, long zo, long zi,
                                                 int wave, int lane) {
  if (p.bias != nullptr && wave == 0) {
    // the epilogue's bias values (one vector per K segment of a row-parallel layer, each in another home row) are
    // requested now and sit in the L2 when the epilogue asks for them
    const int nb = p.bias_sk ? p.ksegs : 1;
    const T* bs = reinterpret_cast<const T*>(p.bias) + grp * p.bias_sg + zo * p.bias_so + zi * p.bias_si + n0;
    constexpr int LPS = (BN * (int)sizeof(T) + 63) / 64;  // lanes per segment: one per 64 bytes of the tile's columns
    const int sgm = lane / LPS, part = lane % LPS;
    if (sgm < nb && n0 + part * (64 / (int)sizeof(T)) + 4 / (int)sizeof(T) <= p.n) {  // the 4 bytes read lie inside the vector
      const char* src = reinterpret_cast<const char*>(bs + (long)sgm * p.bias_sk) + part * 64;
      asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, off"
                   :
                   : "s"(lds_dst), "v"(src)
                   : "memory");
    }
  }
  if (p.gate != nullptr) {
    // the ReLU mask of the epilogue is an activation saved by the forward pass, long gone from the caches: the
    // tile's part of it is requested now, 16 bytes per lane
    constexpr int CPR = BN * (int)sizeof(T) / 16, NCH = BM * CPR;  // 16-byte chunks per tile row, per tile
    const T* gt = reinterpret_cast<const T*>(p.gate) + grp * p.gate_sg + zo * p.gate_so + zi * p.gate_si;
#pragma unroll
    for (int c0 = 0; c0 < NCH; c0 += 256) {
      const int c = c0 + wave * 64 + lane;
      const int row = m0 + c / CPR, col = n0 + (c % CPR) * (16 / (int)sizeof(T));
      if (c < NCH && row < p.m && col + 16 / (int)sizeof(T) <= p.n) {
        const char* src = reinterpret_cast<const char*>(gt + (long)row * p.ld_gate + col);
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off"
                     :
                     : "s"(lds_dst), "v"(src)
                     : "memory");
      }
    }
  }
}

typedef short short4_t __attribute__((ext_vector_type(4)));

// rowbase: first tile row of the 32-row MFMA block; the lane's own row is rowbase + lane % 32.
template <typename T, int R, bool KC, int SB>
__device__ __forceinline__ Frag<T> read_frag_dma(const char* st, int rowbase, int lane, int ks) {
  constexpr int VEC = 16 / sizeof(T);
  constexpr int LINE = R * (int)sizeof(T);
  const int li = lane & 31, g = lane >> 5;
  union {
    uint4 q;
    T e[VEC];
    short4_t h[2];
    Frag<T> f;
  } u;
  if (KC) {
    const int row = rowbase + li;
    u.q = *reinterpret_cast<const uint4*>(st + row * SB + (((2 * ks + g) ^ kc_swizzle<SB>(row)) << 4));
  } else if (sizeof(T) == 2) {
    // LDS holds [k][rows] (rows contiguous) but the MFMA wants 8 consecutive k per lane.  gfx950's
    // transposing LDS read does the 16-bit transpose inside each group of 16 lanes: lane s of a group
    // supplies the address of 4 consecutive rows at k line (s / 4); the group then receives, in lane j,
    // the 4 consecutive k of row (4 * (s % 4) ... ) + j.  Two such reads give the 8 k of the lane's row.
    const int s16 = lane & 15, blk = (lane >> 4) & 1;
    const int kl = (2 * ks + g) * 8 + (s16 >> 2);         // k line of the first read; the second is kl + 4
    const int rb = (rowbase + 16 * blk + 4 * (s16 & 3)) * 2;  // byte of the lane's 4 rows inside the k line
    const int c0 = (rb >> 4) ^ rc_swizzle<T, R>(kl), c1 = (rb >> 4) ^ rc_swizzle<T, R>(kl + 4);
    const char* p0 = st + kl * LINE + (c0 << 4) + (rb & 15);
    const char* p1 = st + (kl + 4) * LINE + (c1 << 4) + (rb & 15);
    u.h[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) short4_t*)(p0));
    u.h[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) short4_t*)(p1));
  } else {
    const char* p = st + (2 * ks + g) * VEC * LINE + (rowbase + li) * (int)sizeof(T);
#pragma unroll
    for (int e = 0; e < VEC; ++e) u.e[e] = *reinterpret_cast<const T*>(p + e * LINE);
  }
  return u.f;
}

// A 16-byte vector shifted down by `n` elements, zeros moving in from the top: what a vector that was read `n` elements
// before its place (to stay inside the operand) has to undergo.
template <typename T>
__device__ __forceinline__ uint4 shift_down(uint4 q, int n) {
  constexpr int PER = 4 / (int)sizeof(T);  // elements per word
  const int w = n / PER;
  const unsigned d[4] = {q.x, q.y, q.z, q.w};
  unsigned r[5];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    r[i] = 0u;
#pragma unroll
    for (int j = i; j < 4; ++j) r[i] = w == j - i ? d[j] : r[i];
  }
  r[4] = 0u;
  if (PER == 2) {
    const unsigned odd = (n & 1) * 16u;
#pragma unroll
    for (int i = 0; i < 4; ++i) r[i] = odd ? (r[i] >> 16) | (r[i + 1] << 16) : r[i];
  }
  return make_uint4(r[0], r[1], r[2], r[3]);
}

// The loader for operands the direct-to-LDS loads cannot take: rows, extents or base addresses that are no multiples of 16
// bytes (a 1001-class head, shards of odd size).  Vectors are read with unaligned 16-byte loads into registers, kRegDepth
// slabs ahead, and written to the stage in the layout DmaOperand leaves there.  A vector that would reach beyond its row (or k
// line) is read further down, inside it, and shifted into place; this is decided per vector without a branch, and
// the shift only runs in slabs and tiles that have such vectors.  Needs rows (k lines) of at least one vector.
// Bound by the rate of unaligned vector loads: 25 - 28 bytes a clock and CU from the L1 against 56 for aligned ones.  A layer of
// 992 x 1001 x 2048 (bf16, 8 shards, forward + both gradients): 54 us, 185 us with the guarded scalar loads; 4096^3 with
// one extent odd 180 - 290 us.
constexpr int kRegDepth = 3;
template <typename T, int R, bool KC, int NL, int SB>
struct RegOperand {
  using D = DmaOperand<T, R, KC, NL, SB>;
  static constexpr int VEC = D::VEC, NI = D::NI, BYTES = D::BYTES;
  typedef unsigned vec_t __attribute__((ext_vector_type(4), aligned(2)));  // global loads take any alignment
  const char* base;  // the operand's element 0 (K-contiguous: of row row0)
  long ldb;          // leading dimension in bytes
  unsigned ofs[NI];  // K-contiguous: of the lane's row;  else of the lane's rows inside a k line
  int koff[NI];      // k of the vector inside its slab
  int shift[NI];     // !KC: elements the vector was read early
  bool edge;         // !KC: the tile has such vectors
  uint4 val[kRegDepth][NI];

  __device__ __forceinline__ void init(const T* x, long ld, int row0, int rows, int lw, int lane) {
    ldb = ld * (long)sizeof(T);
    base = reinterpret_cast<const char*>(KC ? x + (long)row0 * ld : x);
    edge = !KC && row0 + R > rows;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int j = lw * NI + i;
      if (KC) {
        constexpr int LPR = SB / 16;
        const int row = j * (64 / LPR) + lane / LPR;
        const int rr = row0 + row < rows ? row : rows - 1 - row0;
        ofs[i] = (unsigned)(rr * ldb);
        koff[i] = ((lane % LPR) ^ kc_swizzle<SB>(row)) * VEC;
        shift[i] = 0;
      } else {
        const int byte = lane * 16;
        koff[i] = j * (1024 / D::LINE) + byte / D::LINE;
        const int r = row0 + (((byte % D::LINE) >> 4) ^ rc_swizzle<T, R>(koff[i])) * VEC;
        const int start = min(r, rows - VEC);
        ofs[i] = (unsigned)(start * (int)sizeof(T));
        shift[i] = r - start;
      }
    }
  }
  // request the slab whose first k is k0 (in a segment that starts seg bytes from the operand's base)
  template <int S>
  __device__ __forceinline__ void fetch(long seg, int k0, int kdim) {
    const char* b = base + seg + (KC ? 0 : (long)k0 * ldb);
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const unsigned o = KC ? ofs[i] + (unsigned)(min(k0 + koff[i], kdim - VEC) * (int)sizeof(T))
                            : ofs[i] + (unsigned)(min(koff[i], kdim - 1 - k0) * ldb);
      const vec_t v = *reinterpret_cast<const vec_t*>(b + o);
      val[S][i] = make_uint4(v.x, v.y, v.z, v.w);
    }
  }
  template <int S>
  __device__ __forceinline__ void store(char* stage, int lw, int lane, int k0, int kdim) {
    const bool tail = k0 + D::BK_ > kdim;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      uint4 q = val[S][i];
      if (KC) {
        if (tail) q = shift_down<T>(q, min(max(k0 + koff[i] - (kdim - VEC), 0), VEC));
      } else {
        if (edge) q = shift_down<T>(q, min(shift[i], VEC));
        if (tail && k0 + koff[i] >= kdim) q = make_uint4(0u, 0u, 0u, 0u);
      }
      *reinterpret_cast<uint4*>(stage + (lw * NI + i) * 1024 + lane * 16) = q;
    }
  }
};

// The fp32 products of gemm_split.hip, in tiles of bm (128 or 64) x 64; ragged: an operand is not vector-aligned.
int launch_split(hipStream_t s, const GemmArgs& a, bool akc, bool bkc, int bm, bool ragged, dim3 grid);

// bf16 products in tiles of 256 x 256 by workgroups that stay (gemm_large.hip): vector-aligned operands and results, two K slabs or more, no
// statistics epilogue; an update with both operands row-contiguous alone, and worth it only on parameters whose rows are whole 128-byte lines.
int launch_large(hipStream_t s, const GemmArgs& a, bool akc, bool bkc);
// Two weight gradients at once, a tile a workgroup: per_xcd of both together at most 32.
int launch_large_pair(hipStream_t s, const GemmArgs& a, const GemmArgs& b);

// `copies` x `segs` matrices of `lines` lines of `len` bf16 elements -> lines of whole 16-byte vectors, zeros behind their ends, all
// contiguous (gemm_pack.hip).
struct PackShape {
  const char* src;
  long ld, seg, copy;  // strides in elements
  int64_t copies, segs, lines, len;
  int64_t vectors() const { return copies * segs * lines * ((len + 7) / 8); }
};
int launch_pack(hipStream_t s, const PackShape& p, char* dst);

// Many tiles of 128 x 128 over a K slab or two (gemm_shortk.hip).
int launch_shortk(hipStream_t s, const GemmArgs& a, bool bf16, bool akc, bool bkc, dim3 grid);
// Few tiles of bm (32 or 64) x 32, the contraction over the waves (gemm_kwaves.hip); direct: vector-aligned operands.
int launch_kwaves(hipStream_t s, const GemmArgs& a, int bm, bool bf16, bool akc, bool bkc, bool direct, dim3 grid);

}  // namespace rtp
