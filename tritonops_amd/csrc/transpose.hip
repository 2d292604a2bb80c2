// Transposition of a matrix of 16-bit elements for gfx950.
//
// The gradient products of the fused cross-entropy sum over the vocabulary and
// over the tokens, along which w and x are not contiguous.  The library's
// kernels run at 1.55 to 1.6 PFLOP/s where both operands are contiguous along
// the summed index and at 1.17 to 1.36 otherwise, so that a transposed copy,
// 4 bytes per element through memory, pays where the other dimension of the
// product is large.
//
// HBM-bound.  A wavefront turns 64 x 64 elements without LDS: a lane reads the
// eight 16-byte pieces of an 8 x 8 block (eight lanes make 128 bytes of a row),
// turns the block with byte permutes in its registers and writes eight pieces
// (eight lanes make 128 bytes again).
#include "kernels.h"
#include "tile_core.h"

namespace mi {
namespace {

struct TransposeParams {
  const uint16_t* src;
  uint16_t* dst;
  int64_t ld_src, ld_dst, rows, cols;
  int32_t tiles_r, tiles_c;
};

__global__ void __launch_bounds__(256) transpose16_kernel(const TransposeParams p) {
  const int lane = threadIdx.x & 63;
  // four wavefronts take four neighbouring row blocks of one column block: 512 bytes of a row of dst
  const int64_t g = blockIdx.x;
  const int groups_r = (p.tiles_r + 3) / 4;
  const int64_t tile_c = g / groups_r;
  const int64_t tile_r = (g % groups_r) * 4 + (threadIdx.x >> 6);
  if (tile_r >= p.tiles_r) return;
  const int64_t c0 = tile_c * 64, r0 = tile_r * 64;
  i32x4 in[8], out[8];
  {
    const int64_t c = c0 + 8 * (lane & 7), r = r0 + 8 * (lane >> 3);
#pragma unroll
    for (int i = 0; i < 8; ++i)
      in[i] = (r + i < p.rows && c < p.cols)
                  ? __builtin_nontemporal_load(reinterpret_cast<const i32x4*>(p.src + (r + i) * p.ld_src + c))
                  : (i32x4){0, 0, 0, 0};
  }
  transpose8x8(in, out);
  const int64_t c = c0 + 8 * (lane & 7), r = r0 + 8 * (lane >> 3);
#pragma unroll
  for (int j = 0; j < 8; ++j)
    if (c + j < p.cols) *reinterpret_cast<i32x4*>(p.dst + (c + j) * p.ld_dst + r) = out[j];
}

}  // namespace

int launch_transpose16(const void* src, int64_t rows, int64_t cols, int64_t ld_src, void* dst, int64_t ld_dst, hipStream_t s) {
  TransposeParams p;
  p.src = static_cast<const uint16_t*>(src);
  p.dst = static_cast<uint16_t*>(dst);
  p.ld_src = ld_src; p.ld_dst = ld_dst; p.rows = rows; p.cols = cols;
  p.tiles_r = (int)((rows + 63) / 64);
  p.tiles_c = (int)((cols + 63) / 64);
  const long long grid = (long long)((p.tiles_r + 3) / 4) * p.tiles_c;   // the C entry bounds it
  hipLaunchKernelGGL(transpose16_kernel, dim3((unsigned)grid), dim3(256), 0, s, p);
  return (int)hipGetLastError();
}

}  // namespace mi
