// Linear layers of a batch of rows for MI355X (gfx950): y = x W^T, x [M, K]
// bf16, W [N, K] bf16, M past what rows_linear.hip takes and small enough that
// reading W bounds it: decoding for many requests, short portions of prompts.
//
// Reference analogue: the GEMMs of inference/v2/kernels/core_ops/blas_kernels.
//
// A workgroup of four waves owns 128 features and up to 128 rows of x over a
// range of inputs. A wave's W goes from memory straight into the A operands of
// mfma_f32_16x16x32_bf16, two chunks of 128 inputs ahead; each of its elements
// is read by one wave, so LDS would only cost a copy. x is shared by the four
// waves: through registers into one of two LDS buffers, chunks of 16 bytes
// swizzled by the row (no bank conflicts), one barrier a chunk. Workgroups of
// the same W and other rows of x run on the same XCD, whose L2 then holds W for
// the second. Several layers on one input (q, k, v) are one launch; what leaves
// CUs idle is split along K, the partial sums stay fp32 and are added in their
// order by a second kernel.
//
//   * Waits on loads: a chunk's 32 KB of W are in flight a workgroup, one
//     workgroup a CU. Chunks of 64 inputs took 10 to 20% longer, x loaded one
//     chunk further ahead the same.
//   * N 4096 + 1024 + 1024, K 4096, three library products and this, us: 48 rows
//     42 / 19, 128 rows 48 / 26, 224 rows 47 / 36. N 4096, K 14336: 64 rows
//     40 / 34, 128 rows 76 / 44, 224 rows 62 / 59.

#include "ds_kernels.h"

namespace {

typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 b16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int NW = 4;       // waves a workgroup
constexpr int MAXL = 3;     // layers a launch
constexpr int KC = 128;     // inputs a chunk

struct Args {
  const short* w[MAXL];
  const short* bias[MAXL];
  short* out[MAXL];
  int n[MAXL];          // features, multiples of four
  int tile_end[MAXL];   // workgroups' tiles up to and with a layer
  int n_end[MAXL];      // features up to and with a layer
  const short* x;
  float* part;          // [splits, M, all features], splits > 1
  int M, K, layers, tiles, splits, mblocks;
};

__device__ __forceinline__ f32x4 mfma(s16x8 a, s16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(
      __builtin_bit_cast(b16x8, a), __builtin_bit_cast(b16x8, b), c, 0, 0, 0);
}
__device__ __forceinline__ short bits(float x) {
  return __builtin_bit_cast(short, (__bf16)x);
}
__device__ __forceinline__ float value(short x) {
  return __builtin_bit_cast(float, (unsigned)(unsigned short)x << 16);
}
__device__ __forceinline__ f32x4 add_bias(f32x4 y, const short* bias, int n) {
  if (bias)
#pragma unroll
    for (int e = 0; e < 4; ++e) y[e] += value(bias[n + e]);
  return y;
}
__device__ __forceinline__ void put(short* p, f32x4 y) {
  *(s16x4*)p = s16x4{bits(y[0]), bits(y[1]), bits(y[2]), bits(y[3])};
}

template <int MT>
__global__ __launch_bounds__(NW * 64, 2) void batch_linear_kernel(
    const Args a) {
  constexpr int ROWS = MT * 16;
  constexpr int XV = MT;      // vectors of x a thread
  __shared__ __attribute__((aligned(16))) short lds[2][ROWS * KC];

  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int col = lane & 15, g = lane >> 4;
  // 8 units, one an XCD, then the same ones for the next rows
  const int unit = blockIdx.x / (8 * a.mblocks) * 8 + blockIdx.x % 8;
  const int m0 = (blockIdx.x / 8) % a.mblocks * ROWS;
  if (unit >= a.tiles * a.splits) return;
  const int split = unit / a.tiles;
  int tile = unit % a.tiles, layer = 0;
  while (tile >= a.tile_end[layer]) ++layer;
  if (layer) tile -= a.tile_end[layer - 1];
  const int N = a.n[layer];
  // first feature of the wave's two tiles of 16
  int f0[2];
  const short* wp[2];
#pragma unroll
  for (int f = 0; f < 2; ++f) {
    f0[f] = tile * 128 + wid * 32 + 16 * f;
    wp[f] = a.w[layer] + (long long)min(f0[f] + col, N - 1) * a.K + 8 * g;
  }
  const int chunks = a.K / KC;
  const int c0 = (int)((long long)split * chunks / a.splits);
  const int c1 = (int)((long long)(split + 1) * chunks / a.splits);

  // x: thread t carries 16 bytes t & 15 of rows (t >> 4) + 16 i
  const int xc = threadIdx.x & 15;
  const short* xp[XV];
  int xl[XV];
#pragma unroll
  for (int i = 0; i < XV; ++i) {
    const int r = (threadIdx.x >> 4) + 16 * i;
    xp[i] = a.x + (long long)min(m0 + r, a.M - 1) * a.K + 8 * xc;
    xl[i] = r * KC + ((xc ^ (r & 7)) << 3);
  }
  // rows of W lie a multiple of the memory channels' interleave apart: the
  // workgroups begin at different chunks and go round
  const int count = c1 - c0, turn = unit % count;
  auto input = [&](int c) {
    c = min(c, count - 1) + turn;
    return (c0 + (c < count ? c : c - count)) * KC;
  };
  s16x8 xs[XV];
  auto load_x = [&](int c) {
    const int k = input(c);
#pragma unroll
    for (int i = 0; i < XV; ++i) xs[i] = *(const s16x8*)(xp[i] + k);
  };
  auto store_x = [&](int b) {
#pragma unroll
    for (int i = 0; i < XV; ++i)
      *(s16x8*)(&lds[b][xl[i]]) = xs[i];
  };

  f32x4 acc[2][MT];
#pragma unroll
  for (int f = 0; f < 2; ++f)
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[f][m] = f32x4{0.f, 0.f, 0.f, 0.f};

  s16x8 w[2][2][KC / 32];     // [buffer][tile of features][32 inputs]
  auto load_w = [&](int b, int c) {
    const int k = input(c);
#pragma unroll
    for (int f = 0; f < 2; ++f)
#pragma unroll
      for (int h = 0; h < KC / 32; ++h)
        w[b][f][h] = *(const s16x8*)(wp[f] + k + 32 * h);
  };
  load_x(0);
  load_w(0, 0);
  load_w(1, 1);
  store_x(0);
  load_x(1);

  auto step = [&](int b, int c) {
    __syncthreads();    // buffer b holds chunk c; the other one has been read
    store_x(b ^ 1);
    load_x(c + 2);
#pragma unroll
    for (int h = 0; h < KC / 32; ++h)
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        const int r = 16 * m + col;
        const s16x8 xb =
            *(const s16x8*)(&lds[b][r * KC + (((4 * h + g) ^ (r & 7)) << 3)]);
#pragma unroll
        for (int f = 0; f < 2; ++f)
          acc[f][m] = mfma(w[b][f][h], xb, acc[f][m]);
      }
    load_w(b, c + 2);
  };
  int c = 0;
  for (; c + 1 < count; c += 2) {
    step(0, c);
    step(1, c + 1);
  }
  if (c < count) step(0, c);

  // lane: row col of a tile of x, features 4 g + r of a tile of W
  const int all = a.n_end[a.layers - 1];
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    const int r = m0 + 16 * m + col;
    if (r >= a.M) continue;
#pragma unroll
    for (int f = 0; f < 2; ++f) {
      const int n = f0[f] + 4 * g;
      if (n >= N) continue;
      if (a.splits > 1)
        *(f32x4*)(a.part + ((long long)split * a.M + r) * all +
                  (layer ? a.n_end[layer - 1] : 0) + n) = acc[f][m];
      else
        put(a.out[layer] + (long long)r * N + n,
            add_bias(acc[f][m], a.bias[layer], n));
    }
  }
}

// Adds the splits up: four features of a row a thread.
__global__ __launch_bounds__(256) void batch_merge_kernel(const Args a) {
  const int all = a.n_end[a.layers - 1];
  const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  if (i >= (long long)a.M * (all / 4)) return;
  const int r = (int)(i / (all / 4)), n = (int)(i % (all / 4)) * 4;
  f32x4 y = {0.f, 0.f, 0.f, 0.f};
  const float* p = a.part + (long long)r * all + n;
#pragma unroll 4
  for (int s = 0; s < a.splits; ++s)
    y += *(const f32x4*)(p + (long long)s * a.M * all);
  int l = 0;
  while (n >= a.n_end[l]) ++l;
  const int at = n - (l ? a.n_end[l - 1] : 0);
  put(a.out[l] + (long long)r * a.n[l] + at, add_bias(y, a.bias[l], at));
}

template <int MT>
void launch(const Args& a, hipStream_t st) {
  const int units = a.tiles * a.splits;
  hipLaunchKernelGGL((batch_linear_kernel<MT>),
                     dim3((units + 7) / 8 * 8 * a.mblocks), dim3(NW * 64), 0,
                     st, a);
  if (a.splits == 1) return;
  const long long q = (long long)a.M * (a.n_end[a.layers - 1] / 4);
  hipLaunchKernelGGL(batch_merge_kernel, dim3((unsigned)((q + 255) / 256)),
                     dim3(256), 0, st, a);
}

}  // namespace

// Splits along K: one workgroup a CU (two: 10 to 30% slower), two chunks to fill
// the pipeline, and partial sums, 4 bytes each written and read, no more than
// W's own bytes.
extern "C" int ds_batch_linear_splits(const int* n, int layers, int M, int K) {
  int blocks = 0;
  for (int i = 0; i < layers; ++i) blocks += (n[i] + 127) / 128;
  blocks *= (M + 127) / 128;
  int s = 256 / blocks;
  if (s > K / (4 * M)) s = K / (4 * M);
  if (s > K / KC / 2) s = K / KC / 2;
  return s < 1 ? 1 : s;
}

// 1..3 weights on one input, M up to 256. K is a multiple of 128, every n of
// four. part: splits * M * all features, null for one split.
extern "C" void ds_batch_linear(const void* x, int layers,
                                const void* const* w, const void* const* bias,
                                void* const* out, const int* n, int M, int K,
                                int splits, float* part, void* stream) {
  Args a = {};
  int total = 0, tiles = 0;
  for (int i = 0; i < layers; ++i) {
    a.w[i] = (const short*)w[i];
    a.bias[i] = (const short*)bias[i];
    a.out[i] = (short*)out[i];
    a.n[i] = n[i];
    a.n_end[i] = total += n[i];
    a.tile_end[i] = tiles += (n[i] + 127) / 128;
  }
  a.x = (const short*)x;
  a.part = part;
  a.M = M; a.K = K; a.layers = layers; a.splits = splits;
  a.tiles = tiles;
  a.mblocks = (M + 127) / 128;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  // 16-row tiles a workgroup: even shares of the rows
  switch ((M + 16 * a.mblocks - 1) / (16 * a.mblocks)) {
    case 1: case 2: case 3: launch<3>(a, st); break;
    case 4: launch<4>(a, st); break;
    case 5: launch<5>(a, st); break;
    case 6: launch<6>(a, st); break;
    case 7: launch<7>(a, st); break;
    default: launch<8>(a, st); break;
  }
}
