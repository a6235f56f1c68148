// Aligned copies of a product's operands.
#include "gemm_tile.h"

namespace rtp {

// The register loaders for unaligned operands take up to twice the time of direct-to-LDS loads in every slab of every tile, and an
// operand's rows are read once per tile column; a copy reads them once.  Bound by memory: a wave writes 1 KiB of consecutive vectors, a
// thread has kPackPer loads in flight.  Alone, out of the caches: 1250 x 18180 in two shards 14.4 us, 8 of 482 x 6400 19.3, 6546 x 3856
// in eight shards 22.0 (4.6 - 6.3 TB/s read and written); 4096 x 1023 6.0, of which 4 - 5 are a launch's.
constexpr int kPackPer = 4;
struct PackArgs {
  const char* src;
  char* dst;
  long ld, seg, copy;
  FastDiv d_line, d_lines, d_segs;  // vectors a line, lines a matrix, segments a copy
  int len;
  unsigned total;
};
__global__ __launch_bounds__(256) void gemm_pack_kernel(PackArgs p) {
  typedef unsigned short u16x8 __attribute__((ext_vector_type(8), aligned(2)));
  typedef unsigned short u16x8a __attribute__((ext_vector_type(8)));
  const unsigned first = blockIdx.x * (256u * kPackPer) + threadIdx.x;
  u16x8a v[kPackPer];
#pragma unroll
  for (int i = 0; i < kPackPer; ++i) {
    const unsigned at = min(first + i * 256u, p.total - 1);
    const unsigned row = fast_div(at, p.d_line), chunk = at - row * p.d_line.d;
    const unsigned z = fast_div(row, p.d_lines), line = row - z * p.d_lines.d;
    const unsigned c = fast_div(z, p.d_segs), g = z - c * p.d_segs.d;
    const unsigned short* src = reinterpret_cast<const unsigned short*>(p.src) + c * p.copy + g * p.seg + line * p.ld + chunk * 8;
    const int live = p.len - (int)chunk * 8;
    if (live >= 8) {
      v[i] = *reinterpret_cast<const u16x8*>(src);
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) v[i][e] = e < live ? src[e] : (unsigned short)0;
    }
  }
#pragma unroll
  for (int i = 0; i < kPackPer; ++i) {
    const unsigned at = first + i * 256u;
    if (at < p.total) reinterpret_cast<u16x8a*>(p.dst)[at] = v[i];
  }
}

int launch_pack(hipStream_t s, const PackShape& q, char* dst) {
  const int64_t total = q.vectors();
  RTP_REQUIRE(total >= 1 && total < (1ll << 31), "gemm: %lld vectors to pack", (long long)total);
  PackArgs p;
  p.src = q.src, p.dst = dst, p.ld = q.ld, p.seg = q.seg, p.copy = q.copy, p.len = (int)q.len, p.total = (unsigned)total;
  p.d_line = make_fastdiv((unsigned)((q.len + 7) / 8)), p.d_lines = make_fastdiv((unsigned)q.lines), p.d_segs = make_fastdiv((unsigned)q.segs);
  ProfileScope prof(s, "gemm_pack", 0.0, (double)(q.copies * q.segs * q.lines) * (double)q.len * 4.0);
  hipLaunchKernelGGL(gemm_pack_kernel, dim3((unsigned)ceil_div(total, 256 * kPackPer)), dim3(256), 0, s, p);
  RTP_LAUNCH_CHECK();
  return RTP_OK;
}

}  // namespace rtp
