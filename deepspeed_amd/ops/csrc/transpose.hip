// bf16 matrix transposes for MI355X (gfx950).
//
// transpose_2d: one matrix of any size, the operands of a linear layer's
// backward (ops/linear.py).
//
// transpose_bf16: a batch of matrices out of [B, H, R, C] or [B, R, H, C]
// through LDS tiles of 64 x 64 (padded), 16-byte accesses both ways. A general
// layout helper: attention reads its operands transposed by itself. For batch
// index bh the source matrix [R, C] starts at
//   src + (bh / inner) * outer_stride + (bh % inner) * inner_stride
// with row stride row_stride (elements); the destination is [bh][C][R].

#include "ds_kernels.h"

namespace {

constexpr int TILE = 64;

__global__ void transpose_bf16_kernel(const short* __restrict__ src,
                                      short* __restrict__ dst,
                                      const int R, const int C,
                                      const long long row_stride,
                                      const int inner,
                                      const long long inner_stride,
                                      const long long outer_stride) {
  // +8 shorts padding per row: byte stride 136*... keeps the column reads
  // off a single bank without breaking 16 B alignment of rows
  __shared__ short tile[TILE][TILE + 8];

  const int bh = blockIdx.z;
  const long long sbase = (long long)(bh / inner) * outer_stride +
                          (long long)(bh % inner) * inner_stride;
  const long long dbase = (long long)bh * R * C;
  const int r0 = blockIdx.y * TILE;
  const int c0 = blockIdx.x * TILE;

  // 256 threads: read 64 rows x 64 cols, 16B per thread -> 8 rows/pass
  const int tid = threadIdx.x;
  const int rlane = tid & 7;          // 8 lanes x 8 shorts = 64 cols
  const int rrow = tid >> 3;          // 32 rows per pass
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    const int r = r0 + rrow + p * 32;
    if (r < R && c0 + rlane * 8 < C) {
      const short* s = src + sbase + (long long)r * row_stride + c0 +
                       rlane * 8;
      *(ds::bf16x8*)&tile[rrow + p * 32][rlane * 8] =
          *(const ds::bf16x8*)s;
    }
  }
  __syncthreads();

  // write transposed: thread writes 8 consecutive R-elements of one C-row
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    const int c = c0 + rrow + p * 32;           // output row = source col
    const int r = r0 + rlane * 8;               // output col = source row
    if (c < C && r < R) {
      ds::bf16x8 v;
#pragma unroll
      for (int i = 0; i < 8; ++i)
        v.v[i] = *(ds::bf16*)&tile[rlane * 8 + i][rrow + p * 32];
      // r is a multiple of 8 and R a multiple of 8 -> 16 B aligned store
      *(ds::bf16x8*)(dst + dbase + (long long)c * R + r) = v;
    }
  }
}

// One matrix [R, C] of any size into [C, ld] (ld >= R, a multiple of 8; the
// pad is left as it is): the operands of a linear layer's backward, whose
// products read both operands along their contiguous axis. Bound by the two
// streams: a lane turns a block of 8 x 8 in its registers (one byte permute a
// pair of values, no LDS), a wave 64 x 64, so that its loads and its stores
// cover whole lines of 128 bytes. 8192 x
// 4096: 22 us (6.2 TB/s), 8192 x 14336: 114 us (4.1), 128256 x 4096: 416 us
// (5.1); the LDS tile of the kernel above takes 26, 113 and 427.
template <bool VEC>   // rows of src start on 16 bytes
__global__ __launch_bounds__(256) void transpose_2d_kernel(
    const short* __restrict__ src, short* __restrict__ dst, const int R,
    const int C, const int ld) {
  const int lane = threadIdx.x & 63;
  const int r0 = blockIdx.x * 64 + 8 * (lane >> 3);
  const int c0 = (blockIdx.y * 4 + (threadIdx.x >> 6)) * 64 + 8 * (lane & 7);
  if (r0 >= R || c0 >= C) return;
  union Row {
    ds::bf16x8 v;
    unsigned w[4];
    short e[8];
  } a[8], o;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const short* s = src + (long long)min(r0 + i, R - 1) * C + c0;
    if (VEC && c0 + 8 <= C) {
      a[i].v = *(const ds::bf16x8*)s;
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) a[i].e[e] = c0 + e < C ? s[e] : 0;
    }
  }
#pragma unroll
  for (int c = 0; c < 8; ++c) {
    if (c0 + c >= C) break;
#pragma unroll
    for (int k = 0; k < 4; ++k)
      o.w[k] = __builtin_amdgcn_perm(a[2 * k + 1].w[c / 2], a[2 * k].w[c / 2],
                                     c & 1 ? 0x07060302u : 0x05040100u);
    short* d = dst + (long long)(c0 + c) * ld + r0;
    if (r0 + 8 <= R) {
      *(ds::bf16x8*)d = o.v;
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (r0 + e < R) d[e] = o.e[e];
    }
  }
}

}  // namespace

extern "C" void ds_transpose_2d(const void* src, void* dst, int R, int C,
                                int ld, void* stream) {
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const dim3 grid((R + 63) / 64, (C + 255) / 256);
  if (C % 8 == 0 && ((uintptr_t)src & 15) == 0)
    hipLaunchKernelGGL((transpose_2d_kernel<true>), grid, dim3(256), 0, st,
                       (const short*)src, (short*)dst, R, C, ld);
  else
    hipLaunchKernelGGL((transpose_2d_kernel<false>), grid, dim3(256), 0, st,
                       (const short*)src, (short*)dst, R, C, ld);
}

extern "C" void ds_transpose_bf16(const void* src, void* dst, int n_batch,
                                  int R, int C, long long row_stride,
                                  int inner, long long inner_stride,
                                  long long outer_stride, void* stream) {
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  dim3 grid((C + TILE - 1) / TILE, (R + TILE - 1) / TILE, n_batch);
  hipLaunchKernelGGL(transpose_bf16_kernel, grid, dim3(256), 0, st,
                     (const short*)src, (short*)dst, R, C, row_stride, inner,
                     inner_stride, outer_stride);
}
