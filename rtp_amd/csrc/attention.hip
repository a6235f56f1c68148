// Fused attention core for short sequences (L <= 32), bf16: one wavefront owns one (group, batch, head)
// problem and keeps scores, probabilities and their gradients in registers.
//
//   forward : S^T = K Q^T (MFMA) -> softmax over keys (fp32, in registers) -> P stored (bf16) -> O^T = V^T P^T (MFMA)
//   backward: dP^T = V dO^T -> dS = scale * P o (dP - rowsum(dP o P)) -> dQ^T = K^T dS^T, dK^T = Q^T dS, dV^T = dO^T P
//
// The transposed products are chosen so that the softmax axis (keys) lies along the accumulator REGISTERS
// of a lane: MFMA 32x32 accumulator register r of lane (li, g) is row 8*(r/4) + 4*g + r%4, column li.  With
// rows = keys and columns = queries a lane holds 16 keys of one query, its partner lane (li, 1-g) the other 16,
// so a row reduction is 15 in-lane operations and one cross-lane exchange.  The same registers, rounded to
// bf16, are directly the B operand of the next product: an MFMA contracts over "k slots" (8 per lane and
// instruction), and which key sits in which slot is free as long as A and B agree; the A operand (V^T, K^T)
// is gathered from LDS in the matching order.
#include "common.h"

namespace rtp {

typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;

struct AttnArgs {
  // element (l, b, h, g, dd) of q/k/v (and dq/dk/dv) at base + l*s_l + b*s_b + h*s_h + g*s_g + dd
  const bf16_t *q, *k, *v;
  bf16_t *dq, *dk, *dv;
  long s_l, s_b, s_h, s_g;
  // element (l, b, h, g, dd) of o / dout at base + l*o_l + b*o_b + h*o_h + g*o_g + dd
  bf16_t* o;
  const bf16_t* dout;
  long o_l, o_b, o_h, o_g;
  bf16_t* p;          // probabilities [G][N][H][L][L]
  const float* mask;   // additive [L][L] or null
  const float* kbias;  // additive per (batch, key) [N][L] or null (a key padding mask: 0 / -inf)
  int causal;
  float scale;
  int L, N, H;
  long nprob;  // G * N * H
};

constexpr int kSeqMax = 32;
constexpr int kPPitch = kSeqMax + 8;  // row pitch of the P / dS tiles in LDS

// NT tiles of 32 x D (rows beyond L zero) global -> LDS with 16-byte accesses, row pitch D + 8 elements.  Every
// load of every tile is issued before the first LDS write, and without branches (rows beyond L re-read row 0 and are
// zeroed afterwards): a wave owns its problem alone, so a load that waits for the previous one to land puts a full
// trip to memory on the kernel's critical path, and there would be a dozen of them.
template <int D, int NT>
struct TileRegs {
  static constexpr int CPR = D / 8, NIT = kSeqMax * CPR / kWave;
  uint4 val[NT][NIT];
  __device__ __forceinline__ void fetch(const bf16_t* const (&base)[NT], const long (&s_l)[NT], int L, int lane) {
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int it = 0; it < NIT; ++it) {
        const int c = lane + it * kWave, row = c / CPR, cc = c % CPR;
        val[t][it] = *reinterpret_cast<const uint4*>(base[t] + (row < L ? row : 0) * s_l[t] + cc * 8);
      }
  }
  __device__ __forceinline__ void commit(bf16_t* const (&tile)[NT], int L, int lane) const {
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int it = 0; it < NIT; ++it) {
        const int c = lane + it * kWave, row = c / CPR, cc = c % CPR;
        *reinterpret_cast<uint4*>(tile[t] + row * (D + 8) + cc * 8) = row < L ? val[t][it] : make_uint4(0u, 0u, 0u, 0u);
      }
  }
};

// Operand fragment with the contraction index contiguous in the tile: row li, elements 16*ks + 8*g ...
__device__ __forceinline__ bf16x8 frag_rowmajor(const bf16_t* tile, int pitch, int li, int g, int ks) {
  return *reinterpret_cast<const bf16x8*>(tile + li * pitch + 16 * ks + 8 * g);
}
// Operand fragments whose contraction index is the tile ROW come through the LDS's transposing read: per group of
// 16 lanes it takes a 4 x 16 block (lane t supplies the address of 4 consecutive elements of row t/4 at column
// 4*(t%4)) and hands lane t the 4 elements of column t.  Two of them make the 8 contraction slots of a lane.
typedef __attribute__((ext_vector_type(4))) short s16x4;
__device__ __forceinline__ s16x4 lds_transposed4(const bf16_t* tile, int pitch, int row0, int col0, int t) {
  typedef __attribute__((address_space(3))) s16x4* lds_ptr;
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(tile + (row0 + (t >> 2)) * pitch + col0 + 4 * (t & 3)));
}
__device__ __forceinline__ bf16x8 join(s16x4 lo, s16x4 hi) {
  union {
    s16x4 h[2];
    bf16x8 f;
  } u;
  u.h[0] = lo, u.h[1] = hi;
  return u.f;
}
// Fragment of the lane that owns tile column col0 + (lane & 31).  ACCUMULATOR order: slot e of instruction m in lane
// group g is row 8*(2m + e/4) + 4g + e%4 (the row that accumulator register 8m + e of that lane group holds).
__device__ __forceinline__ bf16x8 gather_acc_order(const bf16_t* tile, int pitch, int col0, int m, int lane) {
  const int t = lane & 15, c = col0 + (lane & 16), g = lane >> 5;
  return join(lds_transposed4(tile, pitch, 16 * m + 4 * g, c, t), lds_transposed4(tile, pitch, 16 * m + 8 + 4 * g, c, t));
}
// Natural order: slot e of instruction m in lane group g is row 16m + 8g + e.
__device__ __forceinline__ bf16x8 gather_natural(const bf16_t* tile, int pitch, int col0, int m, int lane) {
  const int t = lane & 15, c = col0 + (lane & 16), g = lane >> 5;
  return join(lds_transposed4(tile, pitch, 16 * m + 8 * g, c, t), lds_transposed4(tile, pitch, 16 * m + 8 * g + 4, c, t));
}

// Accumulator (rows = feature dd, columns = sequence position li) -> columns 32*db .. of a tile's row li, 4 consecutive dd (8 bytes) per
// store.  The tile is the operand whose columns 32*db .. the product has just read: its results take their place.
__device__ __forceinline__ void put_transposed(bf16_t* tile, int pitch, int db, int li, int g, const f32x16& acc) {
#pragma unroll
  for (int a4 = 0; a4 < 4; ++a4) {
    union {
      uint2 u;
      bf16_t e[4];
    } pk;
#pragma unroll
    for (int e = 0; e < 4; ++e) pk.e[e] = from_f32<bf16_t>(acc[4 * a4 + e]);
    *reinterpret_cast<uint2*>(tile + li * pitch + 32 * db + 8 * a4 + 4 * g) = pk.u;
  }
}
// The tile's `rows` rows of D elements -> memory, 16 bytes a lane, whole lines.  (Straight from the accumulators, 16 bytes of each of 32 rows
// an instruction, the L2 takes four times as many requests.)
template <int D>
__device__ __forceinline__ void store_tile_rows(const bf16_t* tile, bf16_t* dst, long stride, int rows, int lane) {
  constexpr int P = D + 8, CPR = D / 8;
  wave_lds_fence();
#pragma unroll
  for (int i = 0; i < CPR / 2; ++i) {
    const int row = (i * 64 + lane) / CPR, c = lane % CPR;
    const uint4 v = *reinterpret_cast<const uint4*>(tile + row * P + c * 8);
    if (row < rows) *reinterpret_cast<uint4*>(dst + row * stride + c * 8) = v;
  }
}

struct Problem {
  long z, qkv_off, o_off;
  int b;
  bool live;
};
// The wave index is made scalar and the problem index is split by 32-bit divisions (the host keeps nprob below 2^31):
// 64-bit divisions are software loops of ~140 instructions each, in front of the kernel's first load.
__device__ __forceinline__ Problem locate(const AttnArgs& a, int waves_per_block) {
  Problem pr;
  const unsigned wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  unsigned z = blockIdx.x * (unsigned)waves_per_block + wave;
  pr.live = z < (unsigned)a.nprob;
  if (!pr.live) z = (unsigned)a.nprob - 1;  // idle waves redo the last problem and store nothing
  pr.z = z;
  const unsigned zh = z / (unsigned)a.H, h = z - zh * (unsigned)a.H;
  const unsigned g = zh / (unsigned)a.N, b = zh - g * (unsigned)a.N;
  pr.qkv_off = (long)b * a.s_b + (long)h * a.s_h + (long)g * a.s_g;
  pr.o_off = (long)b * a.o_b + (long)h * a.o_h + (long)g * a.o_g;
  pr.b = (int)b;
  return pr;
}

template <int DB, int NWV>
__global__ __launch_bounds__(NWV * 64) void attn_fwd_small_kernel(AttnArgs a) {
  touch_kernel_arguments<sizeof(AttnArgs)>();
  constexpr int D = 32 * DB, P = D + 8;
  __shared__ __attribute__((aligned(16))) bf16_t tiles[NWV][3][kSeqMax * P];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, li = lane & 31, g = lane >> 5;
  const Problem pr = locate(a, NWV);
  bf16_t* Qs = tiles[wave][0];
  bf16_t* Ks = tiles[wave][1];
  bf16_t* Vs = tiles[wave][2];
  // Tiles first, then the additive mask values of this lane's 16 (query li, key) pairs; the mask is not looked at
  // before the softmax, so its loads are in flight during the tile hand-over and the first product.
  const bool qlive = li < a.L;
  // keys come in runs of 4: with L % 4 == 0 whole runs are inside or outside the sequence (8-byte accesses to P)
  const bool quads = a.L % 4 == 0 && reinterpret_cast<uintptr_t>(a.p) % 8 == 0;
  TileRegs<D, 3> regs;
  {
    const bf16_t* const src[3] = {a.q + pr.qkv_off, a.k + pr.qkv_off, a.v + pr.qkv_off};
    const long sl[3] = {a.s_l, a.s_l, a.s_l};
    regs.fetch(src, sl, a.L, lane);
  }
  float mk[16];
  const bool mask_quads = a.L % 4 == 0 && reinterpret_cast<uintptr_t>(a.mask) % 16 == 0;
#pragma unroll
  for (int r = 0; r < 16; ++r) mk[r] = 0.0f;
  if (a.mask) {
    if (mask_quads) {
#pragma unroll
      for (int a4 = 0; a4 < 4; ++a4) {
        const int key0 = 8 * a4 + 4 * g;
        const float4 m4 = *reinterpret_cast<const float4*>(a.mask + ((qlive && key0 < a.L) ? li * a.L + key0 : 0));
        mk[4 * a4 + 0] = m4.x, mk[4 * a4 + 1] = m4.y, mk[4 * a4 + 2] = m4.z, mk[4 * a4 + 3] = m4.w;
      }
    } else {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int key = 8 * (r >> 2) + 4 * g + (r & 3);
        mk[r] = a.mask[(qlive && key < a.L) ? li * a.L + key : 0];
      }
    }
  }
  float kb[16];
#pragma unroll
  for (int r = 0; r < 16; ++r) kb[r] = 0.0f;
  if (a.kbias) {
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int key = 8 * (r >> 2) + 4 * g + (r & 3);
      kb[r] = a.kbias[(long)pr.b * a.L + (key < a.L ? key : 0)];
    }
  }
  {
    bf16_t* const tl[3] = {Qs, Ks, Vs};
    regs.commit(tl, a.L, lane);
  }
  __syncthreads();

  // S^T[key][query]
  f32x16 s;
#pragma unroll
  for (int r = 0; r < 16; ++r) s[r] = 0.0f;
#pragma unroll
  for (int ks = 0; ks < D / 16; ++ks)
    s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(frag_rowmajor(Ks, P, li, g, ks), frag_rowmajor(Qs, P, li, g, ks), s, 0,
                                                0, 0);

  // softmax over the keys of query li, in the log2 domain (scale * log2 e in one FMA, the hardware 2^x)
  constexpr float kLog2eSmall = 1.44269504088896340736f;
  const float scale2 = a.scale * kLog2eSmall;
  float val[16];
  float mx = -INFINITY;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int key = 8 * (r >> 2) + 4 * g + (r & 3);
    const bool visible = key < a.L && (!a.causal || key <= li);
    // outside the sequence: unrelated mask entries
    const float x = fmaf(s[r], scale2, ((qlive && key < a.L) ? (mk[r] + kb[r]) * kLog2eSmall : 0.0f));
    val[r] = visible ? x : -INFINITY;
    mx = fmaxf(mx, val[r]);
  }
  mx = fmaxf(mx, __shfl_xor(mx, 32, kWave));
  float sum = 0.0f;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    val[r] = __builtin_amdgcn_exp2f(val[r] - mx);  // hidden keys: 2^(-inf) = 0; every key hidden: NaN, as torch gives
    sum += val[r];
  }
  sum += __shfl_xor(sum, 32, kWave);
  const float inv = 1.0f / sum;
  bf16x8 pb[2];
#pragma unroll
  for (int r = 0; r < 16; ++r) pb[r >> 3][r & 7] = from_f32<bf16_t>(val[r] * inv);
  if (pr.live && qlive) {
    bf16_t* prow = a.p + (pr.z * a.L + li) * a.L;
    if (quads) {
#pragma unroll
      for (int a4 = 0; a4 < 4; ++a4) {
        union {
          uint2 u;
          bf16_t e[4];
        } pk;
#pragma unroll
        for (int e = 0; e < 4; ++e) pk.e[e] = pb[(4 * a4 + e) >> 3][(4 * a4 + e) & 7];
        if (8 * a4 + 4 * g < a.L) *reinterpret_cast<uint2*>(prow + 8 * a4 + 4 * g) = pk.u;
      }
    } else {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int key = 8 * (r >> 2) + 4 * g + (r & 3);
        if (key < a.L) prow[key] = pb[r >> 3][r & 7];
      }
    }
  }

  // O^T[dd][query] = sum_key V[key][dd] P[query][key]
#pragma unroll
  for (int db = 0; db < DB; ++db) {
    f32x16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
#pragma unroll
    for (int m = 0; m < 2; ++m)
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(gather_acc_order(Vs, P, 32 * db, m, lane), pb[m], acc, 0, 0, 0);
    put_transposed(Vs, P, db, li, g, acc);
  }
  store_tile_rows<D>(Vs, a.o + pr.o_off, a.o_l, pr.live ? a.L : 0, lane);
}

template <int DB, int NWV>
__global__ __launch_bounds__(NWV * 64) void attn_bwd_small_kernel(AttnArgs a) {
  touch_kernel_arguments<sizeof(AttnArgs)>();
  constexpr int D = 32 * DB, P = D + 8;
  __shared__ __attribute__((aligned(16))) bf16_t tiles[NWV][4][kSeqMax * P];
  __shared__ __attribute__((aligned(16))) bf16_t ptiles[NWV][2][kSeqMax * kPPitch];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, li = lane & 31, g = lane >> 5;
  const Problem pr = locate(a, NWV);
  bf16_t* Qs = tiles[wave][0];
  bf16_t* Ks = tiles[wave][1];
  bf16_t* Vs = tiles[wave][2];
  bf16_t* Gs = tiles[wave][3];  // dO
  bf16_t* DSs = ptiles[wave][0];
  bf16_t* Ps = ptiles[wave][1];
  // Tiles first, then this lane's 16 probabilities P[query li][key]: they are not needed before dP is there.
  const bool qlive = li < a.L;
  TileRegs<D, 4> regs;
  {
    const bf16_t* const src[4] = {a.q + pr.qkv_off, a.k + pr.qkv_off, a.v + pr.qkv_off, a.dout + pr.o_off};
    const long sl[4] = {a.s_l, a.s_l, a.s_l, a.o_l};
    regs.fetch(src, sl, a.L, lane);
  }
  const bf16_t* prow = a.p + (pr.z * a.L + (qlive ? li : 0)) * a.L;
  // keys come in runs of 4: with L % 4 == 0 whole runs are inside or outside the sequence (8-byte accesses to P)
  const bool quads = a.L % 4 == 0 && reinterpret_cast<uintptr_t>(a.p) % 8 == 0;
  union {
    uint2 u;
    bf16_t e[4];
  } p4[4];
  bf16_t p1[16];
  if (quads) {
#pragma unroll
    for (int a4 = 0; a4 < 4; ++a4) {
      const int key0 = 8 * a4 + 4 * g;
      p4[a4].u = *reinterpret_cast<const uint2*>(prow + ((qlive && key0 < a.L) ? key0 : 0));
    }
  } else {
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int key = 8 * (r >> 2) + 4 * g + (r & 3);
      p1[r] = prow[(qlive && key < a.L) ? key : 0];
    }
  }
  {
    bf16_t* const tl[4] = {Qs, Ks, Vs, Gs};
    regs.commit(tl, a.L, lane);
  }
  __syncthreads();

  // dP^T[key][query] = sum_dd V[key][dd] dO[query][dd]
  f32x16 dp;
#pragma unroll
  for (int r = 0; r < 16; ++r) dp[r] = 0.0f;
#pragma unroll
  for (int ks = 0; ks < D / 16; ++ks)
    dp = __builtin_amdgcn_mfma_f32_32x32x16_bf16(frag_rowmajor(Vs, P, li, g, ks), frag_rowmajor(Gs, P, li, g, ks), dp, 0,
                                                 0, 0);
  float pv[16];
  float dot = 0.0f;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int key = 8 * (r >> 2) + 4 * g + (r & 3);
    const float pr_ = to_f32(quads ? p4[r >> 2].e[r & 3] : p1[r]);
    pv[r] = (qlive && key < a.L) ? pr_ : 0.0f;
    dot += pv[r] * dp[r];
  }
  dot += __shfl_xor(dot, 32, kWave);
  bf16x8 dsb[2];
#pragma unroll
  for (int r = 0; r < 16; ++r) dsb[r >> 3][r & 7] = from_f32<bf16_t>(a.scale * pv[r] * (dp[r] - dot));
  // dS and P as [query][key] tiles for the products that contract over the queries
#pragma unroll
  for (int a4 = 0; a4 < 4; ++a4) {
    union {
      uint2 u;
      bf16_t e[4];
    } d4, p4;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      d4.e[e] = dsb[(4 * a4 + e) >> 3][(4 * a4 + e) & 7];
      p4.e[e] = from_f32<bf16_t>(pv[4 * a4 + e]);
    }
    *reinterpret_cast<uint2*>(DSs + li * kPPitch + 8 * a4 + 4 * g) = d4.u;
    *reinterpret_cast<uint2*>(Ps + li * kPPitch + 8 * a4 + 4 * g) = p4.u;
  }
  __syncthreads();

#pragma unroll
  for (int db = 0; db < DB; ++db) {
    f32x16 acc;
    // dQ^T[dd][query] = sum_key K[key][dd] dS[query][key]
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
#pragma unroll
    for (int m = 0; m < 2; ++m)
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(gather_acc_order(Ks, P, 32 * db, m, lane), dsb[m], acc, 0, 0, 0);
    put_transposed(Ks, P, db, li, g, acc);
    // dK^T[dd][key] = sum_query Q[query][dd] dS[query][key]
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
#pragma unroll
    for (int m = 0; m < 2; ++m)
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(gather_natural(Qs, P, 32 * db, m, lane),
                                                    gather_natural(DSs, kPPitch, 0, m, lane), acc, 0, 0, 0);
    put_transposed(Qs, P, db, li, g, acc);
    // dV^T[dd][key] = sum_query dO[query][dd] P[query][key]
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
#pragma unroll
    for (int m = 0; m < 2; ++m)
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(gather_natural(Gs, P, 32 * db, m, lane),
                                                    gather_natural(Ps, kPPitch, 0, m, lane), acc, 0, 0, 0);
    put_transposed(Gs, P, db, li, g, acc);
  }
  const int rows = pr.live ? a.L : 0;  // li was the query for dQ and the key for dK / dV; both run to L
  store_tile_rows<D>(Ks, a.dq + pr.qkv_off, a.s_l, rows, lane);
  store_tile_rows<D>(Qs, a.dk + pr.qkv_off, a.s_l, rows, lane);
  store_tile_rows<D>(Gs, a.dv + pr.qkv_off, a.s_l, rows, lane);
}

// Problems (waves) per workgroup.  One wave's 14 - 24 KiB of LDS at D = 64 fit beside the 121 - 129 KiB that a product's workgroup on another
// stream holds, where four waves' 55 - 94 KiB wait for it to leave the CU, and a problem's loads do not wait for its neighbours'.  Many small
// problems are set up faster in groups.  us forward / backward with 1, 2 and 4 a workgroup (before: 4, results by 8-byte stores): 1024 problems of 32 x
// 64 6.2 / 11.1, 6.9 / 10.9, 6.4 / 11.3 (7.2 / 13.1), 3072 of them 16.9 / 26.5, 16.2 / 24.9, 15.6 / 29.7 (17.9 / 35.1); 2048 of 32 x 128 19.4 /
// 33.5, 19.2 / 34.1, 21.5 / 34.1 (26.4 / 41.2); of 32 x 32 1024 5.4 / 7.8, 5.1 / 6.9, 5.1 / 6.8, 4096 16.9 / 26.7, 13.5 / 25.5, 12.6 / 21.7 (14.7 / 25.2).
static int small_waves(int64_t nprob, int64_t D) { return D == 32 ? 4 : D == 64 && nprob > 2048 ? 2 : 1; }

static bool aligned8(int64_t v) { return v % 8 == 0; }

static int check_common(const char* who, int dtype, int64_t L, int64_t N, int64_t H, int64_t D, int64_t G, int64_t s_l,
                        int64_t s_b, int64_t s_h, int64_t s_g, int64_t o_l, int64_t o_b, int64_t o_h, int64_t o_g,
                        int64_t max_len = kSeqMax) {
  RTP_REQUIRE(dtype == RTP_BF16, "%s: only bf16 is implemented (dtype %d)", who, dtype);
  RTP_REQUIRE(L >= 1 && L <= max_len, "%s: sequence length %lld not in 1..%lld", who, (long long)L, (long long)max_len);
  RTP_REQUIRE(D == 32 || D == 64 || D == 128, "%s: head dimension %lld not in {32, 64, 128}", who, (long long)D);
  RTP_REQUIRE(N >= 1 && H >= 1 && G >= 1, "%s: batch, heads and groups must be >= 1", who);
  RTP_REQUIRE(aligned8(s_l) && aligned8(s_b) && aligned8(s_h) && aligned8(s_g) && aligned8(o_l) && aligned8(o_b) &&
                  aligned8(o_h) && aligned8(o_g),
              "%s: strides must be multiples of 8 elements", who);
  RTP_REQUIRE(G * N * H < (1ll << 31), "%s: too many problems", who);
  return RTP_OK;
}

}  // namespace rtp

using namespace rtp;

extern "C" int rtp_attn_supported(int dtype, int64_t L, int64_t D) {
  return dtype == RTP_BF16 && L >= 1 && L <= kSeqMax && (D == 32 || D == 64 || D == 128);
}

extern "C" int rtp_attn_fwd(void* stream, int dtype, const void* q, const void* k, const void* v, int64_t s_l,
                            int64_t s_b, int64_t s_h, int64_t s_g, void* o, int64_t o_l, int64_t o_b, int64_t o_h,
                            int64_t o_g, void* p, const float* mask, const float* key_bias, int causal, float scale,
                            int64_t L, int64_t N, int64_t H, int64_t D, int64_t G) {
  RTP_REQUIRE(q && k && v && o && p, "rtp_attn_fwd: null pointer");
  if (int rc = check_common("rtp_attn_fwd", dtype, L, N, H, D, G, s_l, s_b, s_h, s_g, o_l, o_b, o_h, o_g)) return rc;
  RTP_REQUIRE(((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)o) % 16 == 0,
              "rtp_attn_fwd: q, k, v, o must be 16-byte aligned");
  AttnArgs a{};
  a.q = (const bf16_t*)q, a.k = (const bf16_t*)k, a.v = (const bf16_t*)v;
  a.s_l = s_l, a.s_b = s_b, a.s_h = s_h, a.s_g = s_g;
  a.o = (bf16_t*)o, a.o_l = o_l, a.o_b = o_b, a.o_h = o_h, a.o_g = o_g;
  a.p = (bf16_t*)p, a.mask = mask, a.kbias = key_bias, a.causal = causal, a.scale = scale;
  a.L = (int)L, a.N = (int)N, a.H = (int)H, a.nprob = G * N * H;
  hipStream_t st = (hipStream_t)stream;
  const double np = (double)a.nprob;
  ProfileScope prof(st, "attn_fwd_small", 4.0 * np * L * L * D, np * (4.0 * L * D + (double)L * L) * 2.0);
  const int waves = small_waves(a.nprob, D);
  const dim3 grid((unsigned)ceil_div(a.nprob, waves)), block(64 * waves);
  if (D == 32)
    hipLaunchKernelGGL((attn_fwd_small_kernel<1, 4>), grid, block, 0, st, a);
  else if (D == 64 && waves == 2)
    hipLaunchKernelGGL((attn_fwd_small_kernel<2, 2>), grid, block, 0, st, a);
  else if (D == 64)
    hipLaunchKernelGGL((attn_fwd_small_kernel<2, 1>), grid, block, 0, st, a);
  else
    hipLaunchKernelGGL((attn_fwd_small_kernel<4, 1>), grid, block, 0, st, a);
  RTP_LAUNCH_CHECK();
  return RTP_OK;
}

extern "C" int rtp_attn_bwd(void* stream, int dtype, const void* q, const void* k, const void* v, int64_t s_l,
                            int64_t s_b, int64_t s_h, int64_t s_g, const void* dout, int64_t o_l, int64_t o_b,
                            int64_t o_h, int64_t o_g, const void* p, void* dq, void* dk, void* dv, float scale,
                            int64_t L, int64_t N, int64_t H, int64_t D, int64_t G) {
  RTP_REQUIRE(q && k && v && dout && p && dq && dk && dv, "rtp_attn_bwd: null pointer");
  if (int rc = check_common("rtp_attn_bwd", dtype, L, N, H, D, G, s_l, s_b, s_h, s_g, o_l, o_b, o_h, o_g)) return rc;
  RTP_REQUIRE(((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)dout | (uintptr_t)dq | (uintptr_t)dk |
               (uintptr_t)dv) % 16 == 0,
              "rtp_attn_bwd: q, k, v, dout, dq, dk, dv must be 16-byte aligned");
  AttnArgs a{};
  a.q = (const bf16_t*)q, a.k = (const bf16_t*)k, a.v = (const bf16_t*)v;
  a.dq = (bf16_t*)dq, a.dk = (bf16_t*)dk, a.dv = (bf16_t*)dv;
  a.s_l = s_l, a.s_b = s_b, a.s_h = s_h, a.s_g = s_g;
  a.dout = (const bf16_t*)dout, a.o_l = o_l, a.o_b = o_b, a.o_h = o_h, a.o_g = o_g;
  a.p = (bf16_t*)const_cast<void*>(p), a.scale = scale;
  a.L = (int)L, a.N = (int)N, a.H = (int)H, a.nprob = G * N * H;
  hipStream_t st = (hipStream_t)stream;
  const double np = (double)a.nprob;
  ProfileScope prof(st, "attn_bwd_small", 8.0 * np * L * L * D, np * (7.0 * L * D + (double)L * L) * 2.0);
  const int waves = small_waves(a.nprob, D);
  const dim3 grid((unsigned)ceil_div(a.nprob, waves)), block(64 * waves);
  if (D == 32)
    hipLaunchKernelGGL((attn_bwd_small_kernel<1, 4>), grid, block, 0, st, a);
  else if (D == 64 && waves == 2)
    hipLaunchKernelGGL((attn_bwd_small_kernel<2, 2>), grid, block, 0, st, a);
  else if (D == 64)
    hipLaunchKernelGGL((attn_bwd_small_kernel<2, 1>), grid, block, 0, st, a);
  else
    hipLaunchKernelGGL((attn_bwd_small_kernel<4, 1>), grid, block, 0, st, a);
  RTP_LAUNCH_CHECK();
  return RTP_OK;
}
