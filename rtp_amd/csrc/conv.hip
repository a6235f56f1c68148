// Out-channel-sharded 2-D convolution as an implicit GEMM on the MFMA: the patch matrix
//   patches[(n*Ho + ho)*Wo + wo][(ci*kh + i)*kw + j] = x[n][ci][ho*sh - ph + i*dh][wo*sw - pw + j*dw]   (0 outside)
// is never written to memory.  Three products, one tile kernel  C[m][n] = sum_k A(m, k) * B(n, k):
//   forward          y[img][co][ho][wo] = sum_k W[co][k] * patches[pix][k] + b[co]           (m = co, n = pix)
//   weight gradient  dW[co][k']         = sum_pix dy[img][co][ho][wo] * patches[pix][k']     (m = co, n = k')
//   input gradient   dx[img][ci][h][w]  = sum_(co,i,j) W[co][ci][i][j] * dy[img][co][ho][wo] (m = ci, n = (img,h,w))
// co runs over the channels of all shards of the run: shard s holds channels s*n_s .. of it at s*numel, so a layer whose
// shards own 16 channels each still fills a 64-row tile.  The lanes of the MFMA result run along n, which is the
// contiguous direction of every output (NCHW pixels, or the weight's k'), so stores are coalesced and the forward needs
// no layout copy.
//
// What bounds it is the gather, so an operand element costs an add, a bounds test and a load: a thread keeps its pixel (or
// its rows) for the whole contraction, and everything that depends on k alone -- offset inside an image, kernel position --
// is worked out once per slab by one thread per k and handed round through LDS.  The first version called an index function
// with five integer divisions per element and gave every shard tiles of its own: MNIST's second convolution (64 x 32 x 26 x
// 26 -> 64, four shards, fp32) took 127 + 162 + 196 us forward / input / weight gradient; this one takes 25 + 36 + 30.
#include <algorithm>

#include "common.h"

#include "rtp_hip.h"

namespace rtp {

typedef __attribute__((ext_vector_type(8))) __bf16 conv_bf16x8;
typedef __attribute__((ext_vector_type(16))) float conv_f32x16;

// Sizes and indices are 32-bit on the device (the host checks the ranges); addresses are 64-bit.
struct ConvGeom {
  int n, c, h, w, kh, kw, sh, sw, ph, pw, dh, dw, ho, wo;
};

// Element strides of a 4-D activation (any memory format).
struct Strides {
  long n, c, h, w;
};

constexpr int kConvSlab = 32;  // contraction per slab

template <typename T>
struct ConvFrag;
template <>
struct ConvFrag<bf16_t> {
  conv_bf16x8 v;
  static constexpr int kStep = 16;  // k per MFMA step: lane group g holds k = 8g .. 8g+7
};
template <>
struct ConvFrag<float> {
  float f[4];
  static constexpr int kStep = 8;   // lane group g holds k = 4g .. 4g+3
};

__device__ __forceinline__ void conv_mma(const ConvFrag<bf16_t>& a, const ConvFrag<bf16_t>& b, conv_f32x16& c) {
  c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.v, b.v, c, 0, 0, 0);
}
__device__ __forceinline__ void conv_mma(const ConvFrag<float>& a, const ConvFrag<float>& b, conv_f32x16& c) {
#pragma unroll
  for (int e = 0; e < 4; ++e) c = __builtin_amdgcn_mfma_f32_32x32x2f32(a.f[e], b.f[e], c, 0, 0, 0);
}

enum ConvPass { kConvFwd, kConvDgrad, kConvWgrad };

template <typename T>
struct ConvArgs {
  ConvGeom g;
  FastDiv d_pix_img, d_pix_row;  // pixels per image and per row of the pixel grid (output, or input for the input gradient)
  FastDiv d_khkw, d_kw, d_ns, d_sh, d_sw;
  int M, N, K, splits, kchunk;
  int n_s, kp, khkw;             // channels per shard, weights per channel, kernel positions
  int co;                        // WHOLE: contracted channels
  long numel;                    // elements per shard row
  const T* act;                  // x (forward, weight gradient) or dy (input gradient), at the run's first channel
  Strides s;
  const T* w;                    // weights of the run's first shard
  const T* dy;                   // weight gradient: dy at the run's first channel
  Strides sd;
  // outputs
  T* y;                          // forward: NCHW with co_total channels, at the run's first channel
  const T* bias;
  int co_total;
  void* dx;                      // input gradient, contiguous NCHW
  const void* addend;
  int dx_f32, addend_f32;
  T* grads;                      // weight gradient rows
  long w_off, b_off;
  int accumulate;
  float* part;                   // fp32 partial sums [split][M][kp + 1] (entry kp: the row sum), or null: one split
};

// An operand read element by element at byte offsets from its base: buffer loads with a 32-bit offset, which return zero
// for an offset beyond the buffer -- how an element outside the image or the contraction becomes zero without a branch, a
// mask or a select --, or plain 64-bit addresses for an operand of 4 GiB or more (WIDE).
constexpr unsigned kBeyond = 0xffffff00u;
template <typename T, bool WIDE>
struct Gather {
  typedef unsigned off_t;
  __amdgpu_buffer_rsrc_t r;
  __device__ __forceinline__ explicit Gather(const T* base)
      : r(__builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(base), 0, kBeyond, 0x00020000)) {}
  __device__ __forceinline__ T get(unsigned off, bool ok) const {
    off = ok ? off : kBeyond;
    if constexpr (sizeof(T) == 4)
      return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b32(r, (int)off, 0, 0));
    else
      return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b16(r, (int)off, 0, 0));
  }
  // N words at an offset that 16 bytes divide (two words: 8)
  template <int N>
  __device__ __forceinline__ void run(unsigned (&w)[N], unsigned off) const {
    typedef __attribute__((ext_vector_type(N < 4 ? N : 4))) unsigned vec;
#pragma unroll
    for (int i = 0; i < N; i += 4) {
      vec t;
      if constexpr (N == 2)
        t = __builtin_bit_cast(vec, __builtin_amdgcn_raw_buffer_load_b64(r, (int)off, 0, 0));
      else  // (an offset beyond the buffer stays one: the next 16 bytes' own is not added to it)
        t = __builtin_bit_cast(vec, __builtin_amdgcn_raw_buffer_load_b128(r, (int)(off == kBeyond ? off : off + 4 * i), 0, 0));
#pragma unroll
      for (int e = 0; e < (N < 4 ? N : 4); ++e) w[i + e] = t[e];
    }
  }
};
template <typename T>
struct Gather<T, true> {
  typedef long off_t;
  const char* base;
  __device__ __forceinline__ explicit Gather(const T* b) : base(reinterpret_cast<const char*>(b)) {}
  __device__ __forceinline__ T get(long off, bool ok) const {
    return ok ? *reinterpret_cast<const T*>(base + off) : from_f32<T>(0.0f);
  }
};
// What depends on a k of the slab alone.
template <class Off>
struct alignas(16) KEntry {
  Off b;       // byte offset of the gathered activation relative to the pixel
  int di, dj;  // kernel position in input pixels; di = kOutside: beyond the contraction
};
constexpr int kOutside = 1 << 30;

// BM x BN outputs per workgroup, four waves: 64 x 64 or 64 x 128 as 2 x 2 waves of one or two MFMA blocks, or 32 x 128 as 1 x 4 for
// products of at most 32 rows.  LDS is double buffered and elements are requested two slabs ahead of
// their MFMAs: the grids are small (MNIST's second convolution: two waves per SIMD), so the trip to memory has to
// be covered by the wave itself.  SIMPLE: forward and weight gradient without padding (every gathered element exists),
// input gradient with unit strides.
// Forward: a thread takes NA consecutive weights of a row by one load or two at any alignment instead of NA loads (128 x 64 x 32 x 32 -> 128
// padded in bf16, forward and both gradients 332 -> 317 us, MNIST's second convolution in fp32 96.6 -> 94.9).
// WHOLE (weight gradient): runs of NA output pixels of a plane are whole and aligned in dy and come by one load or two, as the forward's weights
// do (launch_tile has the rule; the same case 317 -> 291 us, in 64-row tiles 1 - 9 %).  In tiles of 32 rows they are read one by one: runs took 2 - 4 %
// longer there in bf16 with kernels of 3 x 3 and 5 x 5 (128 x 40 x 56 x 56 -> 16, 5 x 5, 163 -> 169 us), and in fp32 no less.  The bias gradient's 32 chains
// of additions a row are the same ones on either way.
// WHOLE (input gradient): a slab is 32 channels at one kernel position, so a pixel's neighbour is tested and, with strides, divided
// for once a slab, the rest is scalar and there is no table; a slab's weights lie khkw elements apart, and a wave's lanes run along the input
// channels, where 64 of them share ten lines.  us, forward and both gradients, before -> after (the input gradient's share): MNIST's second
// convolution 102.8 -> 96.9, 128 x 64 x 32 x 32 -> 128 padded in bf16 368 -> 333, 37 x 24 x 31 x 31 -> 80 with strides of 2 128 -> 98.
template <typename T, ConvPass PASS, int BM, int BN, bool SIMPLE, bool WIDE, bool WHOLE = false>
__global__ __launch_bounds__(256) void conv_igemm_kernel(ConvArgs<T> p) {
  typedef typename Gather<T, WIDE>::off_t Off;
  constexpr int PITCH = kConvSlab + 16 / (int)sizeof(T);  // elements; rows stay 16-byte aligned
  constexpr int NA = BM * kConvSlab / 256, NB = BN * kConvSlab / 256;
  constexpr int ES = (int)sizeof(T);
  __shared__ __attribute__((aligned(16))) T As[2][BM * PITCH];
  __shared__ __attribute__((aligned(16))) T Bs[2][BN * PITCH];
  __shared__ KEntry<Off> tab[PASS == kConvWgrad ? 1 : 4][PASS == kConvWgrad ? BN : kConvSlab];
  __shared__ Off tab_a[4][kConvSlab];  // input gradient: offset of the weight
  const ConvGeom& g = p.g;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  constexpr int NT = BM * BN / 4096;  // MFMA blocks of a wave
  const int wm = BM == 64 ? wave >> 1 : 0, wn = (BM == 64 ? wave & 1 : wave) * NT, li = lane & 31, lg = lane >> 5;
  const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
  const int split = blockIdx.z, kb = split * p.kchunk, ke = min(kb + p.kchunk, p.K);
  const Gather<T, WIDE> act(p.act), wts(PASS == kConvWgrad ? p.dy : p.w);  // wts: operand A

  // kernel position and activation offset of contraction index (or weight column) k
  auto entry_of = [&](int k, bool live, Off* a) {
    KEntry<Off> e;
    const unsigned ci = fast_div((unsigned)k, p.d_khkw), ij = k - ci * p.khkw;  // ci: the channel of the gathered operand
    const unsigned i = fast_div(ij, p.d_kw), j = ij - i * g.kw;
    const int di = (int)i * g.dh, dj = (int)j * g.dw;
    e.di = live ? di : kOutside;
    e.dj = dj;
    if (PASS == kConvDgrad) {
      const unsigned sft = fast_div(ci, p.d_ns), co = ci - sft * p.n_s;
      *a = live ? (Off)((sft * p.numel + (long)co * p.kp + ij) * ES) : (Off)0;
      e.b = (Off)((ci * p.s.c - (SIMPLE ? di * p.s.h + dj * p.s.w : 0)) * ES);
    } else {
      e.b = live ? (Off)((ci * p.s.c + di * p.s.h + dj * p.s.w) * ES) : (Off)0;
    }
    return e;
  };
  // of two slabs, by one wave: the slabs `slab` and `slab` + 1 steps behind kb
  auto build_table = [&](int slab) {
    if (PASS != kConvWgrad && !WHOLE && tid < 2 * kConvSlab) {
      const int k = kb + slab * kConvSlab + tid, slot = (slab + tid / kConvSlab) & 3, at = tid & (kConvSlab - 1);
      Off a = 0;
      tab[PASS == kConvWgrad ? 0 : slot][at] = entry_of(min(k, p.K - 1), k < ke, &a);
      if (PASS == kConvDgrad) tab_a[slot][at] = a;
    }
  };

  // ---- operand A: k = tid % 32, rows tid / 32 + 8 q (RUNS: the thread's row, NA consecutive k) ----
  const int ak = tid & 31, ar = tid >> 5;
  // (WHOLE: the thread's row m = tid % BM, k = tid / BM * NA + q, whose neighbours in a wave lie khkw elements apart)
  Off aoff[NA];
  const int am = tid & (BM - 1), akq = tid / BM;
  const unsigned a_row = (unsigned)(min(m0 + am, p.M - 1) * p.khkw);
  int c0 = 0, pi = 0, pj = 0;  // WHOLE: first channel and kernel position of the slab that is requested next
  auto channel_rows = [&] {
#pragma unroll
    for (int q = 0; q < NA; ++q) {
      const int co = min(c0 + akq * NA + q, p.co - 1);
      const unsigned sft = fast_div((unsigned)co, p.d_ns);
      aoff[q] = (Off)((sft * p.numel + (long)(co - sft * p.n_s) * p.kp + a_row) * ES);
    }
  };
  constexpr bool RUNS = PASS == kConvFwd || (PASS == kConvWgrad && WHOLE);
  constexpr int RUNW = NA * ES / 4;
  struct __attribute__((packed, aligned(ES))) AnyRun {  // at the elements' alignment
    unsigned w[RUNW];
  };
  union PackedRun {
    T e[NA];
    unsigned w[RUNW];
  };
  const int rr = tid / (kConvSlab / NA), rk = tid % (kConvSlab / NA) * NA;
  const T* run_row = nullptr;
  if constexpr (PASS == kConvFwd) {
    const unsigned m = (unsigned)min(m0 + rr, p.M - 1), sft = fast_div(m, p.d_ns);
    run_row = p.w + (sft * p.numel + (long)(m - sft * p.n_s) * p.kp);
  }
  if constexpr (RUNS) {
    aoff[0] = (Off)(min(m0 + rr, p.M - 1) * p.sd.c * ES);
  } else if constexpr (PASS == kConvDgrad && WHOLE)
    channel_rows();
  else
#pragma unroll
  for (int q = 0; q < NA; ++q) {
    const int m = min(m0 + ar + 8 * q, p.M - 1);
    if (PASS == kConvDgrad) {
      aoff[q] = (Off)((long)m * p.khkw * ES);
    } else {
      aoff[q] = (Off)(m * p.sd.c * ES);
    }
  }
  // ---- operand B ----
  // forward / input gradient: the thread's pixel n, k = kq*NB + e;  weight gradient: k = tid % 32, rows tid / 32 + 8 q
  const int bn = tid & (BN - 1), kq = tid / BN;
  Off bpix = 0;
  int bh = 0, bw = 0;
  KEntry<Off> brow[PASS == kConvWgrad ? NB : 1];
  // pixel -> offset, row and column of the gathered activation before the kernel position
  auto locate = [&](int pix, int& h, int& w) {
    const unsigned img = fast_div((unsigned)pix, p.d_pix_img);
    const int r = pix - img * p.d_pix_img.d;
    const unsigned y = fast_div((unsigned)r, p.d_pix_row);
    const int x = r - y * p.d_pix_row.d;
    if (PASS == kConvDgrad) {
      h = (int)y + g.ph, w = x + g.pw;
      return (Off)(((long)img * p.s.n + (SIMPLE ? h * p.s.h + w * p.s.w : 0)) * ES);
    }
    h = (int)y * g.sh - g.ph, w = x * g.sw - g.pw;
    return (Off)(((long)img * p.s.n + h * p.s.h + w * p.s.w) * ES);
  };
  if (PASS != kConvWgrad) {
    bpix = locate(min(n0 + bn, p.N - 1), bh, bw);
    if constexpr (!(PASS == kConvDgrad && WHOLE)) {
      build_table(0), build_table(2);
      __syncthreads();
    }
  } else {
    Off unused;
    if (tid < BN) tab[0][tid] = entry_of(min(n0 + tid, p.N - 1), n0 + tid < p.N, &unused);
    __syncthreads();
#pragma unroll
    for (int q = 0; q < NB; ++q) brow[PASS == kConvWgrad ? q : 0] = tab[0][(ar + 8 * q) & (BN - 1)];
  }

  struct Regs {
    T a[NA], b[NB];
    unsigned run[RUNW];  // RUNS, in place of a: kept as it was loaded, so that nothing waits for it before it is stored
  } reg[2];
  // requests a slab (one behind the contraction: nothing but zeros)
  auto fetch = [&](int slab, Regs& v) {
    const int k0 = kb + slab * kConvSlab;
    if constexpr (PASS == kConvDgrad && WHOLE) {  // slabs are requested in sequence
      const int ij = (pi * g.kw + pj) * ES;
#pragma unroll
      for (int q = 0; q < NA; ++q) v.a[q] = wts.get(aoff[q] + ij, c0 + akq * NA + q < p.co);
      const int di = pi * g.dh, dj = pj * g.dw;
      Off at;
      bool in;
      if (SIMPLE) {
        in = ((unsigned)(bh - di) < (unsigned)g.ho) & ((unsigned)(bw - dj) < (unsigned)g.wo);
        at = bpix - (Off)((di * p.s.h + dj * p.s.w) * ES);
      } else {
        const int hn = bh - di, wn_ = bw - dj;
        const int ho = (int)fast_div((unsigned)max(hn, 0), p.d_sh), wo = (int)fast_div((unsigned)max(wn_, 0), p.d_sw);
        in = (hn >= 0) & (wn_ >= 0) & (ho * g.sh == hn) & (wo * g.sw == wn_) & (ho < g.ho) & (wo < g.wo);
        at = bpix + (Off)((ho * p.s.h + wo * p.s.w) * ES);
      }
      const int c = c0 + __builtin_amdgcn_readfirstlane(kq) * NB;
      const unsigned sc = (unsigned)(p.s.c * ES);
#pragma unroll
      for (int q = 0; q < NB; ++q) v.b[q] = act.get(at + (unsigned)(c + q) * sc, in & (c + q < p.co));
      if (++pj == g.kw) {
        pj = 0;
        if (++pi == g.kh) {
          pi = 0, c0 += kConvSlab;
          channel_rows();
        }
      }
      return;
    }
    if (PASS == kConvWgrad) {
      const bool live = k0 + ak < ke;
      const int pix = live ? k0 + ak : p.K - 1;
      int h, w;
      const Off base = locate(pix, h, w);
      const unsigned img = fast_div((unsigned)pix, p.d_pix_img);
      const int r = pix - img * p.d_pix_img.d;
      const unsigned yo = fast_div((unsigned)r, p.d_pix_row);
      const Off d = (Off)(((long)img * p.sd.n + (long)yo * p.sd.h + (long)(r - yo * p.d_pix_row.d) * p.sd.w) * ES);
      if constexpr (PASS == kConvWgrad && RUNS) {  // (a run is inside one image and inside or beyond the contraction)
        const unsigned at = (unsigned)(k0 + rk), rimg = fast_div(at, p.d_pix_img);
        const unsigned off = (unsigned)(((long)rimg * p.sd.n + (at - rimg * p.d_pix_img.d)) * ES) + (unsigned)aoff[0];
        wts.run(v.run, (int)at < ke ? off : kBeyond);
      } else {
#pragma unroll
        for (int q = 0; q < NA; ++q) v.a[q] = wts.get(d + aoff[q], live);
      }
#pragma unroll
      for (int q = 0; q < NB; ++q) {
        const KEntry<Off>& e = brow[PASS == kConvWgrad ? q : 0];
        const bool in = SIMPLE ? e.di != kOutside
                               : ((unsigned)(h + e.di) < (unsigned)g.h) & ((unsigned)(w + e.dj) < (unsigned)g.w);
        v.b[q] = act.get(base + e.b, live & in);
      }
      return;
    }
    const int slot = PASS == kConvWgrad ? 0 : slab & 3;
    if constexpr (RUNS) {
      const int left = p.K - (k0 + rk);  // weights of the row from this run on
      auto whole = [&] {
        const AnyRun run = *reinterpret_cast<const AnyRun*>(run_row + k0 + rk);
#pragma unroll
        for (int q = 0; q < RUNW; ++q) v.run[q] = run.w[q];
      };
      if (k0 + kConvSlab <= p.K) {
        whole();
      } else {  // the slab that the contraction ends in, or one behind it
#pragma unroll
        for (int q = 0; q < RUNW; ++q) v.run[q] = 0;
        if (left >= NA) {
          whole();
        } else if (left > 0) {  // the run that it ends in: the only one that is waited for here
          PackedRun u;
#pragma unroll
          for (int q = 0; q < NA; ++q) {
            const T t = run_row[k0 + rk + min(q, left - 1)];
            u.e[q] = q < left ? t : from_f32<T>(0.0f);
          }
#pragma unroll
          for (int q = 0; q < RUNW; ++q) v.run[q] = u.w[q];
        }
      }
    } else {
      const bool live = k0 + ak < ke;
      const Off off = tab_a[slot][ak];
#pragma unroll
      for (int q = 0; q < NA; ++q) v.a[q] = wts.get(aoff[q] + off, live);
    }
    KEntry<Off> e[NB];
#pragma unroll
    for (int q = 0; q < NB; ++q) e[q] = tab[slot][(kq * NB + q) & (kConvSlab - 1)];
#pragma unroll
    for (int q = 0; q < NB; ++q) {
      if (PASS == kConvFwd) {
        const bool in = SIMPLE ? e[q].di != kOutside
                               : ((unsigned)(bh + e[q].di) < (unsigned)g.h) & ((unsigned)(bw + e[q].dj) < (unsigned)g.w);
        v.b[q] = act.get(bpix + e[q].b, in);
      } else if (SIMPLE) {
        v.b[q] = act.get(bpix + e[q].b, ((unsigned)(bh - e[q].di) < (unsigned)g.ho) & ((unsigned)(bw - e[q].dj) < (unsigned)g.wo));
      } else {
        const int hn = bh - e[q].di, wn_ = bw - e[q].dj;
        const int ho = (int)fast_div((unsigned)max(hn, 0), p.d_sh), wo = (int)fast_div((unsigned)max(wn_, 0), p.d_sw);
        const bool in = (hn >= 0) & (wn_ >= 0) & (ho * g.sh == hn) & (wo * g.sw == wn_) & (ho < g.ho) & (wo < g.wo);
        v.b[q] = act.get(bpix + e[q].b + (Off)((ho * p.s.h + wo * p.s.w) * ES), in);
      }
    }
  };
  float rsum[NA];
#pragma unroll
  for (int q = 0; q < NA; ++q) rsum[q] = 0.0f;
  const bool want_rows = PASS == kConvWgrad && blockIdx.x == 0;
  auto stash = [&](int buf, const Regs& v) {
#pragma unroll
    for (int q = 0; q < NA; ++q) {
      if (!WHOLE && !RUNS) As[buf][(ar + 8 * q) * PITCH + ak] = v.a[q];
      if (PASS == kConvWgrad && !RUNS) rsum[q] += to_f32(v.a[q]);
    }
    if constexpr (PASS == kConvWgrad && RUNS) {
      PackedRun u;
#pragma unroll
      for (int q = 0; q < RUNW; ++q) u.w[q] = v.run[q];
#pragma unroll
      for (int q = 0; q < NA; ++q) rsum[q] += to_f32(u.e[q]);
    }
    if constexpr (WHOLE || RUNS) {
      struct alignas(NA * ES < 16 ? NA * ES : 16) Run {
        unsigned w[RUNW];
      } out;
      if constexpr (RUNS) {
#pragma unroll
        for (int q = 0; q < RUNW; ++q) out.w[q] = v.run[q];
      } else {
        PackedRun u;
#pragma unroll
        for (int q = 0; q < NA; ++q) u.e[q] = v.a[q];
#pragma unroll
        for (int q = 0; q < RUNW; ++q) out.w[q] = u.w[q];
      }
      *reinterpret_cast<Run*>(&As[buf][RUNS ? rr * PITCH + rk : am * PITCH + akq * NA]) = out;
    }
    if (PASS == kConvWgrad) {
#pragma unroll
      for (int q = 0; q < NB; ++q) Bs[buf][(ar + 8 * q) * PITCH + ak] = v.b[q];
    } else {
      constexpr int VEC = 16 / (int)sizeof(T);
#pragma unroll
      for (int u8 = 0; u8 < NB / VEC; ++u8) {
        union {
          uint4 q;
          T e[VEC];
        } u;
#pragma unroll
        for (int e = 0; e < VEC; ++e) u.e[e] = v.b[u8 * VEC + e];
        *reinterpret_cast<uint4*>(&Bs[buf][bn * PITCH + kq * NB + u8 * VEC]) = u.q;
      }
    }
  };

  conv_f32x16 accs[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) accs[t][r] = 0.0f;
  const int slabs = (ke - kb + kConvSlab - 1) / kConvSlab;
  fetch(0, reg[0]);
  fetch(1, reg[1]);
  stash(0, reg[0]);
  __syncthreads();
  // step s: requests slab s + 2 into the registers that slab s left, multiplies slab s, stores slab s + 1.  The tables of slabs
  // s + 3 and s + 4 are built meanwhile by odd s: they are read behind the next barrier, and their slots (s + 3) % 4 and s % 4 by
  // nobody now.
  auto step = [&](int sl, Regs& mine, Regs& next, int buf) {
    fetch(sl + 2, mine);  // unconditionally: the wait for slab s + 1 below counts the loads in flight
    constexpr int STEP = ConvFrag<T>::kStep, VEC = 16 / (int)sizeof(T);
#pragma unroll
    for (int ks = 0; ks < kConvSlab / STEP; ++ks) {
      union {
        uint4 q;
        ConvFrag<T> f;
      } a, b[NT];
      a.q = *reinterpret_cast<const uint4*>(&As[buf][(wm * 32 + li) * PITCH + ks * STEP + lg * VEC]);
#pragma unroll
      for (int t = 0; t < NT; ++t)
        b[t].q = *reinterpret_cast<const uint4*>(&Bs[buf][((wn + t) * 32 + li) * PITCH + ks * STEP + lg * VEC]);
#pragma unroll
      for (int t = 0; t < NT; ++t) conv_mma(a.f, b[t].f, accs[t]);
    }
    if (buf == 1) build_table(sl + 3);
    stash(buf ^ 1, next);
    __syncthreads();
  };
  for (int sl = 0; sl < slabs; sl += 2) {
    step(sl, reg[0], reg[1], 0);
    step(sl + 1, reg[1], reg[0], 1);  // past the last slab: zeros
  }

  // ---- results: accumulator register r of lane (li, lg) is row 8*(r/4) + 4*lg + r%4 of the wave's block, column li ----
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int col = n0 + (wn + t) * 32 + li;
    if (col >= p.N) continue;
    const conv_f32x16& acc = accs[t];
    long at = 0;
    if (PASS != kConvWgrad) {
      const unsigned img = fast_div((unsigned)col, p.d_pix_img);
      const long plane = p.d_pix_img.d;
      at = (long)img * (PASS == kConvFwd ? p.co_total : p.M) * plane + (col - (long)img * plane);
    }
    float bias[16];  // requested together: one trip to memory for the 16 rows
    if (PASS == kConvFwd && p.bias != nullptr) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int m = min(m0 + wm * 32 + 8 * (r >> 2) + 4 * lg + (r & 3), p.M - 1);
        const unsigned sft = fast_div((unsigned)m, p.d_ns);
        bias[r] = to_f32(p.bias[sft * p.numel + (m - sft * p.n_s)]);
      }
    } else {
#pragma unroll
      for (int r = 0; r < 16; ++r) bias[r] = 0.0f;
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int m = m0 + wm * 32 + 8 * (r >> 2) + 4 * lg + (r & 3);
      if (m >= p.M) continue;
      float v = acc[r];
      if (PASS == kConvFwd) {
        v += bias[r];
        p.y[at + (long)m * p.d_pix_img.d] = from_f32<T>(v);
      } else if (PASS == kConvDgrad) {
        // dx = acc + addend, either in T or fp32 (the sum over rotation windows is kept in fp32 and rounded once)
        const long o = at + (long)m * p.d_pix_img.d;
        if (p.addend != nullptr)
          v += p.addend_f32 ? reinterpret_cast<const float*>(p.addend)[o] : to_f32(reinterpret_cast<const T*>(p.addend)[o]);
        if (p.dx_f32)
          reinterpret_cast<float*>(p.dx)[o] = v;
        else
          reinterpret_cast<T*>(p.dx)[o] = from_f32<T>(v);
      } else if (p.part != nullptr) {
        p.part[((long)split * p.M + m) * (p.kp + 1) + col] = v;
      } else {
        const unsigned sft = fast_div((unsigned)m, p.d_ns);
        T* dst = p.grads + sft * p.numel + p.w_off + (long)(m - sft * p.n_s) * p.kp + col;
        if (p.accumulate) v += to_f32(*dst);
        *dst = from_f32<T>(v);
      }
    }
  }
  if (want_rows) {  // bias gradient: the rows' sums over this workgroup's pixels, 32 chains (pixel % 32) each in a fixed order
    if constexpr (RUNS) {
#pragma unroll
      for (int o = 16; o >= NA; o >>= 1)
#pragma unroll
        for (int q = 0; q < NA; ++q) rsum[q] += __shfl_xor(rsum[q], o / NA, 64);
#pragma unroll
      for (int o = NA / 2; o > 0; o >>= 1)
#pragma unroll
        for (int q = 0; q < o; ++q) rsum[q] += rsum[q + o];
    }
#pragma unroll
    for (int q = 0; q < (RUNS ? 1 : NA); ++q) {
      float v = rsum[q];
      if constexpr (!RUNS) {
#pragma unroll
        for (int o = 16; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
      }
      const int m = RUNS ? m0 + rr : m0 + ar + 8 * q;
      if ((RUNS ? rk : ak) != 0 || m >= p.M) continue;
      if (p.part != nullptr) {
        p.part[((long)split * p.M + m) * (p.kp + 1) + p.kp] = v;
      } else if (p.b_off >= 0) {
        const unsigned sft = fast_div((unsigned)m, p.d_ns);
        T* dst = p.grads + sft * p.numel + p.b_off + (m - sft * p.n_s);
        if (p.accumulate) v += to_f32(*dst);
        *dst = from_f32<T>(v);
      }
    }
  }
}

// grads (+)= sum over the splits, ascending, of the partial sums: one thread per entry of the [M, kp + 1] block
template <typename T>
__global__ __launch_bounds__(256) void wgrad_reduce_kernel(ConvArgs<T> o) {
  const int total = o.M * (o.kp + 1), idx = blockIdx.x * 256 + threadIdx.x;
  if (idx >= total) return;
  const int m = idx / (o.kp + 1), n = idx - m * (o.kp + 1);
  const unsigned sft = fast_div((unsigned)m, o.d_ns);
  const int co = m - (int)sft * o.n_s;
  if (n == o.kp && o.b_off < 0) return;
  float v = 0.0f;
  int sp = 0;
  for (; sp + 8 <= o.splits; sp += 8) {
    float t[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) t[u] = o.part[(long)(sp + u) * total + idx];
#pragma unroll
    for (int u = 0; u < 8; ++u) v += t[u];
  }
  for (; sp < o.splits; ++sp) v += o.part[(long)sp * total + idx];
  T* dst = o.grads + sft * o.numel + (n < o.kp ? o.w_off + (long)co * o.kp + n : o.b_off + co);
  if (o.accumulate) v += to_f32(*dst);
  *dst = from_f32<T>(v);
}

static int check_geom(const char* who, const rtp_conv_geom* geom, ConvGeom& g) {
  RTP_REQUIRE(geom, "%s: null geometry", who);
  const rtp_conv_geom& q = *geom;
  RTP_REQUIRE(q.n >= 1 && q.c >= 1 && q.h >= 1 && q.w >= 1 && q.kh >= 1 && q.kw >= 1, "%s: sizes must be >= 1", who);
  RTP_REQUIRE(q.sh >= 1 && q.sw >= 1 && q.dh >= 1 && q.dw >= 1 && q.ph >= 0 && q.pw >= 0,
              "%s: stride and dilation must be >= 1, padding >= 0", who);
  const int64_t lim = (int64_t)1 << 30;  // every index of the three products stays within 32 bits
  RTP_REQUIRE(q.sh < lim && q.sw < lim && q.dh < lim && q.dw < lim && q.ph < lim && q.pw < lim && q.ho >= 1 &&
                  q.wo >= 1 && q.n * q.h * q.w < lim && q.n * q.ho * q.wo < lim && q.c * q.kh * q.kw < lim &&
                  q.dh * q.kh < lim && q.dw * q.kw < lim && q.ho * q.sh < lim && q.wo * q.sw < lim,
              "%s: geometry beyond the 32-bit index range of the kernels", who);
  g = ConvGeom{(int)q.n, (int)q.c, (int)q.h, (int)q.w, (int)q.kh, (int)q.kw, (int)q.sh, (int)q.sw,
               (int)q.ph, (int)q.pw, (int)q.dh, (int)q.dw, (int)q.ho, (int)q.wo};
  const long span_h = (long)g.h + 2 * g.ph - (long)g.dh * (g.kh - 1) - 1, span_w = (long)g.w + 2 * g.pw - (long)g.dw * (g.kw - 1) - 1;
  RTP_REQUIRE(span_h >= 0 && span_w >= 0, "%s: kernel larger than the padded input", who);
  RTP_REQUIRE(g.ho == span_h / g.sh + 1 && g.wo == span_w / g.sw + 1,
              "%s: output size %lld x %lld does not match the geometry (expected %lld x %lld)", who, (long long)g.ho,
              (long long)g.wo, (long long)(span_h / g.sh + 1), (long long)(span_w / g.sw + 1));
  return RTP_OK;
}

static int check_run(const char* who, int dtype, int64_t numel, int64_t shards, int64_t w_off, int64_t bias_off,
                     int64_t n_s, const ConvGeom& g) {
  RTP_REQUIRE(dtype == RTP_F32 || dtype == RTP_BF16, "%s: unknown dtype %d", who, dtype);
  const long kp = (long)g.c * g.kh * g.kw;
  RTP_REQUIRE(shards >= 1 && shards < 65536 && n_s >= 1 && shards * n_s * g.kh * g.kw < ((int64_t)1 << 30),
              "%s: shards %lld, channels per shard %lld", who, (long long)shards, (long long)n_s);
  RTP_REQUIRE(w_off >= 0 && w_off + n_s * kp <= numel, "%s: the weight [%lld, %lld] at %lld does not fit a shard row of %lld",
              who, (long long)n_s, (long long)kp, (long long)w_off, (long long)numel);
  RTP_REQUIRE(bias_off < 0 || bias_off + n_s <= numel, "%s: the bias at %lld does not fit a shard row of %lld", who,
              (long long)bias_off, (long long)numel);
  return RTP_OK;
}

// How the input gradient runs.  whole: slabs of 32 channels at one kernel position each (WHOLE) instead of channels with all their positions.
// They save the tests of every element, are filled up to whole ones, which costs MFMAs, and read a slab's weights khkw elements apart: every
// position touches the same `lines` lines of each of the 32 channels again, and once those no longer stay in the L1 the weights come from the L2
// khkw times.  wider: tiles of 64 x 128 (bf16), which read the weights half as often and are half as many.
// us for the input gradient of 128 x 32 x 32 pixels, channels in -> out (lines of a channel): mixed slabs -> whole ones.
//   fp32, strides of 1: 3 x 3, 32 -> 64 (9) 70 -> 63, 64 -> 64 (18) 110 -> 124, 64 -> 48 88 -> 110; 5 x 5, 16 -> 64 (13) 173 -> 153, 32 -> 64 (25) 175 ->
//   210, 64 -> 64 (50) 272 -> 652; 1 x 1, 64 -> 32 24 -> 25, 64 -> 64 27 -> 25.  Strides of 2: 3 x 3, 64 -> 64 150 -> 125; 5 x 5, 32 -> 64 (25) 293 -> 210,
//   40 -> 64 (32) 379 -> 418.  With a workgroup a CU at most, 16 x 14 x 14: 5 x 5, 32 -> 64 (25) 71 -> 60.
//   bf16, strides of 1: 3 x 3, 32 -> 64 (5) 40 -> 34, 64 -> 64 (9) 82 -> 66; 5 x 5, 32 -> 64 (13) 93 -> 111, 64 -> 64 (25) 135 -> 327; 4 x 4, 32 -> 64 (8)
//   60 -> 85, 2 x 2, 64 -> 64 (4) 28 -> 31 (rows of 8, 16 or 32 bytes fall on fewer of the L1's sets).  Strides of 2: 3 x 3, 64 -> 64 95 -> 72; 5 x 5, 32 ->
//   64 (13) 189 -> 118, 64 -> 64 (25) 204 -> 331.
// The same in bf16 by 64 x 128, mixed and whole: 3 x 3, 64 -> 64 60 and 49, 64 -> 16 30 -> 29 (whole 31 -> 29); 5 x 5, 64 -> 64 126 and 186, strides of 2 210 and
// 192; 1 x 1, 64 -> 32 18.8 -> 19.4 (whole 18.6 -> 17.1), 64 -> 8 15.8 -> 18.5.  Fewer pixels, 32 x 32 x 32 (512 tiles of 64 x 64), whole: 1 x 1, 64 -> 64
// 7.4 -> 8.2, 3 x 3, 64 -> 64 21.6 -> 20; 20 x 30 x 30 (282): 7.4 -> 8.2 and 20.6 -> 19.6.
struct DgradForm {
  bool whole, wider;
};
template <typename T>
static DgradForm dgrad_form(const ConvArgs<T>& a) {
  constexpr bool kBf16 = sizeof(T) == 2;
  const bool unit = a.g.sh == 1 && a.g.sw == 1, shallow = a.M <= 32;
  const long co = a.K / a.khkw, padded = ceil_div(co, kConvSlab) * kConvSlab;
  const bool full = 8 * padded <= 9 * co, most = 3 * padded <= 4 * co, half = 5 * padded <= 8 * co;  // slabs that are filled
  const long rows = std::min(a.M, 64), lines = std::min<long>(rows, ceil_div(rows * a.khkw * (long)sizeof(T), 128));
  const long tiles = ceil_div(a.M, 64) * ceil_div(a.N, 64);  // of 64 x 64
  const int share = (shallow ? ceil_div(a.N, 128) : tiles) <= 256 ? 2 : 1;
  const bool many = kBf16 && !shallow && tiles > 512, some = kBf16 && !shallow && tiles > 256 && a.khkw >= 9 && co >= 64;
  DgradForm f;
  if (a.khkw == 1)
    f.whole = !unit || shallow || co >= (many ? 32 : 64);
  else if (unit && shallow)
    f.whole = (full || (kBf16 && a.khkw <= 9 && most)) && lines <= (kBf16 ? a.khkw % 4 == 0 ? 3 : 9 : 13) * share;
  else if (unit && a.khkw % 2 == 0)
    f.whole = full && many && co >= 64 && lines <= 4;
  else if (unit)
    f.whole = (full || (kBf16 && most)) && lines <= (kBf16 ? 9 : 12 * share);
  else if (shallow)
    f.whole = half && lines <= (kBf16 ? 25 : 32);
  else
    f.whole = (most && lines <= (many || some ? 25 : kBf16 ? 10 * share : 20 * share)) || (kBf16 && half && lines <= 9);
  f.wider = f.whole ? many || some : many && unit && (a.khkw == 1 ? co >= 96 : a.khkw % 2 != 0 && a.khkw >= 9 && a.khkw <= 25 && co >= 16);
  return f;
}

template <typename T, ConvPass PASS, int BM, int BN>
static void launch_tile(hipStream_t st, const ConvArgs<T>& a, dim3 grid, bool whole) {
  const ConvGeom& g = a.g;
  const bool simple = PASS == kConvDgrad ? g.sh == 1 && g.sw == 1 : g.ph == 0 && g.pw == 0;
  // the furthest element of each operand, in bytes from its base
  auto reach = [](const Strides& s, long n, long c, long h, long w) {
    return (double)(n - 1) * s.n + (double)(c - 1) * s.c + (double)(h - 1) * s.h + (double)(w - 1) * s.w;
  };
  const long co = PASS == kConvDgrad ? a.K / a.khkw : a.M;
  double far = (double)ceil_div(co, a.n_s) * a.numel;
  far = std::max(far, PASS == kConvDgrad ? reach(a.s, g.n, co, g.ho, g.wo) : reach(a.s, g.n, g.c, g.h, g.w));
  if (PASS == kConvWgrad) far = std::max(far, reach(a.sd, g.n, co, g.ho, g.wo));
  const bool wide = (far + 1.0) * sizeof(T) >= (double)kBeyond;
#define RTP_CONV(SIMPLE, WIDE) hipLaunchKernelGGL((conv_igemm_kernel<T, PASS, BM, BN, SIMPLE, WIDE>), grid, dim3(256), 0, st, a)
  if constexpr (PASS == kConvDgrad)
    if (!wide && whole) {
      ConvArgs<T> b = a;
      b.co = (int)co, b.K = b.kchunk = (int)(ceil_div(co, kConvSlab) * kConvSlab) * a.khkw;
      if (simple)
        hipLaunchKernelGGL((conv_igemm_kernel<T, PASS, BM, BN, true, false, true>), grid, dim3(256), 0, st, b);
      else
        hipLaunchKernelGGL((conv_igemm_kernel<T, PASS, BM, BN, false, false, true>), grid, dim3(256), 0, st, b);
      return;
    }
  if constexpr (PASS == kConvWgrad && BM == 64) {  // dy contiguous, and planes and images whole aligned runs
    constexpr int NA = BM * kConvSlab / 256;
    if (!wide && a.sd.w == 1 && a.sd.h == g.wo && (long)g.ho * g.wo % NA == 0 && a.sd.n % NA == 0 && a.sd.c % NA == 0 &&
        reinterpret_cast<uintptr_t>(a.dy) % std::min<size_t>(16, NA * sizeof(T)) == 0) {
      if (simple)
        hipLaunchKernelGGL((conv_igemm_kernel<T, PASS, BM, BN, true, false, true>), grid, dim3(256), 0, st, a);
      else
        hipLaunchKernelGGL((conv_igemm_kernel<T, PASS, BM, BN, false, false, true>), grid, dim3(256), 0, st, a);
      return;
    }
  }
  if (wide)
    RTP_CONV(false, true);
  else if (simple)
    RTP_CONV(true, false);
  else
    RTP_CONV(false, false);
#undef RTP_CONV
}

// Products of at most 32 rows (few channels) take the 32-row tile.
static int tile_rows(long M) { return M <= 32 ? 32 : 64; }

template <typename T, ConvPass PASS>
static int launch_igemm(hipStream_t st, const char* name, ConvArgs<T>& a, double bytes) {
  constexpr bool WIDER = PASS == kConvDgrad && sizeof(T) == 2;
  const DgradForm form = PASS == kConvDgrad ? dgrad_form(a) : DgradForm{};
  const int bm = tile_rows(a.M), bn = form.wider ? 128 : 4096 / bm;
  const long tm = ceil_div(a.M, bm), tn = ceil_div(a.N, bn);
  RTP_REQUIRE(tn < (1l << 31) && tm < 65536 && a.splits < 65536, "%s: grid %ld x %ld x %d too large", name, tn, tm, a.splits);
  if (a.splits == 1) a.kchunk = (int)(ceil_div(a.K, kConvSlab) * kConvSlab);
  ProfileScope prof(st, name, 2.0 * (double)a.M * (double)a.N * (double)a.K, bytes);
  const dim3 grid((unsigned)tn, (unsigned)tm, (unsigned)a.splits);
  if (bm == 32)
    launch_tile<T, PASS, 32, 128>(st, a, grid, form.whole);
  else if (form.wider)
    launch_tile<T, PASS, 64, WIDER ? 128 : 64>(st, a, grid, form.whole);
  else
    launch_tile<T, PASS, 64, 64>(st, a, grid, form.whole);
  RTP_LAUNCH_CHECK();
  return RTP_OK;
}

// What the three passes share.  pix_h x pix_w: the pixel grid (output pixels, or input pixels for the input gradient).
template <typename T>
static ConvArgs<T> common_args(const ConvGeom& g, int64_t numel, int64_t n_s, int pix_h, int pix_w) {
  ConvArgs<T> a{};
  a.g = g;
  a.khkw = g.kh * g.kw, a.kp = g.c * a.khkw, a.n_s = (int)n_s, a.numel = numel;
  a.d_pix_img = make_fastdiv((unsigned)(pix_h * pix_w)), a.d_pix_row = make_fastdiv((unsigned)pix_w);
  a.d_khkw = make_fastdiv((unsigned)a.khkw), a.d_kw = make_fastdiv((unsigned)g.kw), a.d_ns = make_fastdiv((unsigned)n_s);
  a.d_sh = make_fastdiv((unsigned)g.sh), a.d_sw = make_fastdiv((unsigned)g.sw);
  a.splits = 1;
  return a;
}
static Strides strides_of(const int64_t* s) { return Strides{(long)s[0], (long)s[1], (long)s[2], (long)s[3]}; }

template <typename T>
static int conv_fwd(hipStream_t st, const void* x, const int64_t* sx, const ConvGeom& g, const void* w, int64_t numel,
                    int64_t shards, int64_t w_off, int64_t bias_off, int64_t n_s, void* y, int64_t co_first,
                    int64_t co_total) {
  ConvArgs<T> a = common_args<T>(g, numel, n_s, g.ho, g.wo);
  const long pix = (long)g.n * g.ho * g.wo;
  const T* wt = reinterpret_cast<const T*>(w);
  a.M = (int)(shards * n_s), a.N = (int)pix, a.K = a.kp;
  a.act = reinterpret_cast<const T*>(x), a.s = strides_of(sx);
  a.w = wt + w_off, a.bias = bias_off >= 0 ? wt + bias_off : nullptr;
  a.y = reinterpret_cast<T*>(y) + co_first * g.ho * g.wo, a.co_total = (int)co_total;
  const double bytes = sizeof(T) * ((double)g.n * g.c * g.h * g.w + (double)shards * n_s * ((double)a.kp + pix));
  return launch_igemm<T, kConvFwd>(st, "conv2d_fwd", a, bytes);
}

// The weight gradient contracts over all pixels of the batch and has few outputs: the contraction is dealt over
// `splits` workgroups per output tile (about three workgroups per CU in all, at least 4 slabs each).
struct WgradSplit {
  long splits, kchunk;
  size_t workspace;
};
static WgradSplit wgrad_split(const ConvGeom& g, int64_t shards, int64_t n_s) {
  const long kp = (long)g.c * g.kh * g.kw, pix = (long)g.n * g.ho * g.wo, M = shards * n_s;
  const int bm = tile_rows(M), bn = 4096 / bm;
  const long tiles = ceil_div(M, bm) * ceil_div(kp, bn), slabs = ceil_div(pix, kConvSlab);
  long want = std::min<long>(ceil_div(768, tiles), std::max<long>(1, slabs / 4));
  want = std::max<long>(1, std::min<long>(want, 65535));
  WgradSplit r;
  r.kchunk = ceil_div(slabs, want) * kConvSlab;
  r.splits = ceil_div(pix, r.kchunk);
  r.workspace = r.splits > 1 ? (size_t)r.splits * M * (kp + 1) * sizeof(float) : 0;
  return r;
}

template <typename T>
static int conv_wgrad(hipStream_t st, const void* dy, const int64_t* sdy, const void* x, const int64_t* sx,
                      const ConvGeom& g, void* grads, int64_t numel, int64_t shards, int64_t w_off, int64_t bias_off,
                      int64_t n_s, int64_t co_first, int accumulate, void* workspace, size_t workspace_bytes) {
  ConvArgs<T> a = common_args<T>(g, numel, n_s, g.ho, g.wo);
  const long pix = (long)g.n * g.ho * g.wo;
  const WgradSplit sp = wgrad_split(g, shards, n_s);
  if (workspace_bytes < sp.workspace || (sp.workspace && workspace == nullptr))
    return fail(RTP_ERR_WORKSPACE, "rtp_conv2d_wgrad: workspace %zu < required %zu", workspace_bytes, sp.workspace);
  a.M = (int)(shards * n_s), a.N = a.kp, a.K = (int)pix;
  RTP_REQUIRE((long)a.M * (a.kp + 1) < (1l << 31), "rtp_conv2d_wgrad: weight gradient of %d x %d entries too large", a.M, a.kp);
  a.splits = (int)sp.splits, a.kchunk = (int)sp.kchunk;
  a.act = reinterpret_cast<const T*>(x), a.s = strides_of(sx);
  a.sd = strides_of(sdy), a.dy = reinterpret_cast<const T*>(dy) + co_first * a.sd.c;
  a.grads = reinterpret_cast<T*>(grads), a.w_off = w_off, a.b_off = bias_off, a.accumulate = accumulate;
  a.part = sp.splits > 1 ? reinterpret_cast<float*>(workspace) : nullptr;
  const double bytes = sizeof(T) * ((double)g.n * g.c * g.h * g.w + (double)shards * n_s * ((double)a.kp + pix));
  if (int rc = launch_igemm<T, kConvWgrad>(st, "conv2d_wgrad", a, bytes)) return rc;
  if (sp.splits > 1) {
    const long total = (long)a.M * (a.kp + 1);
    ProfileScope prof(st, "conv2d_wgrad_reduce", 0.0, (double)sp.workspace + (double)total * sizeof(T));
    hipLaunchKernelGGL(wgrad_reduce_kernel<T>, dim3((unsigned)ceil_div(total, 256)), dim3(256), 0, st, a);
    RTP_LAUNCH_CHECK();
  }
  return RTP_OK;
}

template <typename T>
static int conv_dgrad(hipStream_t st, const void* dy, const int64_t* sdy, const ConvGeom& g, const void* w,
                      int64_t numel, int64_t shards, int64_t w_off, int64_t n_s, int64_t co_first, void* dx, int dx_f32,
                      const void* addend, int addend_f32) {
  ConvArgs<T> a = common_args<T>(g, numel, n_s, g.h, g.w);
  a.M = g.c, a.N = g.n * g.h * g.w, a.K = (int)(shards * n_s * a.khkw);
  a.s = strides_of(sdy), a.act = reinterpret_cast<const T*>(dy) + co_first * a.s.c;
  a.w = reinterpret_cast<const T*>(w) + w_off;
  a.dx = dx, a.addend = addend, a.dx_f32 = dx_f32, a.addend_f32 = addend_f32;
  const double bytes = sizeof(T) * ((double)g.n * g.c * g.h * g.w +
                                    (double)shards * n_s * ((double)g.c * a.khkw + (double)g.n * g.ho * g.wo));
  return launch_igemm<T, kConvDgrad>(st, "conv2d_dgrad", a, bytes);
}

}  // namespace rtp

using namespace rtp;

extern "C" int rtp_conv2d_fwd(void* stream, int dtype, const void* x, int64_t sx_n, int64_t sx_c, int64_t sx_h,
                              int64_t sx_w, const rtp_conv_geom* geom, const void* w, int64_t numel, int64_t shards,
                              int64_t w_off, int64_t bias_off, int64_t n_s, void* y, int64_t co_first,
                              int64_t co_total) {
  ConvGeom g;
  if (int rc = check_geom("rtp_conv2d_fwd", geom, g)) return rc;
  if (int rc = check_run("rtp_conv2d_fwd", dtype, numel, shards, w_off, bias_off, n_s, g)) return rc;
  RTP_REQUIRE(x && w && y, "rtp_conv2d_fwd: null pointer");
  RTP_REQUIRE(co_first >= 0 && co_first + shards * n_s <= co_total, "rtp_conv2d_fwd: channels %lld .. %lld of %lld",
              (long long)co_first, (long long)(co_first + shards * n_s), (long long)co_total);
  const int64_t sx[4] = {sx_n, sx_c, sx_h, sx_w};
  hipStream_t st = (hipStream_t)stream;
  if (dtype == RTP_F32)
    return conv_fwd<float>(st, x, sx, g, w, numel, shards, w_off, bias_off, n_s, y, co_first, co_total);
  return conv_fwd<bf16_t>(st, x, sx, g, w, numel, shards, w_off, bias_off, n_s, y, co_first, co_total);
}

extern "C" int rtp_conv2d_wgrad(void* stream, int dtype, const void* dy, int64_t sdy_n, int64_t sdy_c, int64_t sdy_h,
                                int64_t sdy_w, const void* x, int64_t sx_n, int64_t sx_c, int64_t sx_h, int64_t sx_w,
                                const rtp_conv_geom* geom, void* grads, int64_t numel, int64_t shards, int64_t w_off,
                                int64_t bias_off, int64_t n_s, int64_t co_first, int accumulate, void* workspace,
                                size_t workspace_bytes) {
  ConvGeom g;
  if (int rc = check_geom("rtp_conv2d_wgrad", geom, g)) return rc;
  if (int rc = check_run("rtp_conv2d_wgrad", dtype, numel, shards, w_off, bias_off, n_s, g)) return rc;
  RTP_REQUIRE(dy && x && grads && co_first >= 0, "rtp_conv2d_wgrad: null pointer or negative channel offset");
  const int64_t sdy[4] = {sdy_n, sdy_c, sdy_h, sdy_w}, sx[4] = {sx_n, sx_c, sx_h, sx_w};
  hipStream_t st = (hipStream_t)stream;
  if (dtype == RTP_F32)
    return conv_wgrad<float>(st, dy, sdy, x, sx, g, grads, numel, shards, w_off, bias_off, n_s, co_first, accumulate,
                             workspace, workspace_bytes);
  return conv_wgrad<bf16_t>(st, dy, sdy, x, sx, g, grads, numel, shards, w_off, bias_off, n_s, co_first, accumulate,
                            workspace, workspace_bytes);
}

extern "C" size_t rtp_conv2d_wgrad_workspace_bytes(const rtp_conv_geom* geom, int64_t shards, int64_t n_s) {
  ConvGeom g;
  if (check_geom("rtp_conv2d_wgrad_workspace_bytes", geom, g) != RTP_OK || shards < 1 || shards >= 65536 || n_s < 1)
    return 0;
  return wgrad_split(g, shards, n_s).workspace;
}

extern "C" int rtp_conv2d_dgrad(void* stream, int dtype, const void* dy, int64_t sdy_n, int64_t sdy_c, int64_t sdy_h,
                                int64_t sdy_w, const rtp_conv_geom* geom, const void* w, int64_t numel, int64_t shards,
                                int64_t w_off, int64_t n_s, int64_t co_first, void* dx, int dx_f32, const void* addend,
                                int addend_f32) {
  ConvGeom g;
  if (int rc = check_geom("rtp_conv2d_dgrad", geom, g)) return rc;
  if (int rc = check_run("rtp_conv2d_dgrad", dtype, numel, shards, w_off, -1, n_s, g)) return rc;
  RTP_REQUIRE(dy && w && dx && co_first >= 0, "rtp_conv2d_dgrad: null pointer or negative channel offset");
  const int64_t sdy[4] = {sdy_n, sdy_c, sdy_h, sdy_w};
  hipStream_t st = (hipStream_t)stream;
  if (dtype == RTP_F32)
    return conv_dgrad<float>(st, dy, sdy, g, w, numel, shards, w_off, n_s, co_first, dx, 1, addend, 1);
  return conv_dgrad<bf16_t>(st, dy, sdy, g, w, numel, shards, w_off, n_s, co_first, dx, dx_f32, addend, addend_f32);
}
