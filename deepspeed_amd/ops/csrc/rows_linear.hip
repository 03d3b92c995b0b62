// Linear layers of a few rows for MI355X (gfx950): y = x W^T, x [M, K] bf16,
// W [N, K] bf16 (M up to 32) or groupwise int8 (M up to 64).
//
// Decoding reads every weight once for a handful of tokens, so a layer is as
// fast as its weights stream in. Reference analogues: the GEMV-shaped GEMMs of
// csrc/transformer/inference and the weight-only quantized linears of
// inference/v2/kernels/core_ops (cuda_linear).
//
// A workgroup of 8 waves owns 16 FT output features; the waves take every
// eighth chunk of inputs and add up through LDS, so that the 256 CUs have work
// at N = 4096 and each wave has a chunk's loads in flight while it computes the
// one before. W goes from memory straight into the A operand of
// mfma_f32_16x16x32_bf16 (16 features by 64 or, int8, 64 contiguous bytes an
// instruction), x into B (columns past M repeat the last row).
//
//   * Bound by the stream of W at few rows (N 128256, K 4096, M 1: 169 us, 6.2
//     TB/s; the library's product 187 us) and by x out of L2 at many; at 32
//     rows the library's GPU time is 5 to 30% less (N 14336 25.2 to 29.6 us, N
//     4096 12.5 to 15.7), but its calls cost the host 20 us each, which a step
//     of one layer's seven calls cannot hide, against 5 us here.
//   * int8: a lane's 16 bytes are 16 inputs, split over two products; the order
//     of the inputs inside a product is free, x is read in the same order. The
//     bytes become bf16 exactly (8 bits), are summed in fp32 and multiplied by
//     their group's scale in fp32: nothing is rounded before the output, and
//     the weight is not written out as bf16 and read again. N 14336, K 4096, M
//     8: 21.8 us; dequantizing takes 28 us and the product 28.
//   * Several layers on one input (q, k, v; gate and up) are one launch, and
//     the epilogue takes the gate's activation and the bias with it: four
//     launches a decoder layer instead of eight.

#include "ds_kernels.h"

namespace {

typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 b16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

constexpr int NW = 8;       // waves a workgroup
constexpr int MAXL = 3;     // layers a launch

enum { PLAIN = 0, SWIGLU = 1 };

struct Args {
  const void* w[MAXL];
  const float* scales[MAXL];
  const short* bias[MAXL];
  short* out[MAXL];
  int n[MAXL], tile_end[MAXL];
  const short* x;
  int M, K, group;
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

// four signed bytes to four bf16, exactly: u = b + 128 is 0..255
__device__ __forceinline__ void widen(unsigned b, unsigned& lo, unsigned& hi) {
  b ^= 0x80808080u;
  const float f0 = (float)(b & 255u) - 128.f;
  const float f1 = (float)((b >> 8) & 255u) - 128.f;
  const float f2 = (float)((b >> 16) & 255u) - 128.f;
  const float f3 = (float)(b >> 24) - 128.f;
  lo = __builtin_amdgcn_perm(__builtin_bit_cast(unsigned, f1),
                             __builtin_bit_cast(unsigned, f0), 0x07060302u);
  hi = __builtin_amdgcn_perm(__builtin_bit_cast(unsigned, f3),
                             __builtin_bit_cast(unsigned, f2), 0x07060302u);
}

// CH inputs of 16 features: CH / 32 A operands.
template <bool I8, int CH>
struct Weights {
  u32x4 r[I8 ? CH / 64 : CH / 32];

  // at: the lane's feature row and first input
  __device__ __forceinline__ void load(const void* w, long long at, int g) {
    if (I8) {
      const signed char* p = (const signed char*)w + at + 16 * g;
#pragma unroll
      for (int i = 0; i < CH / 64; ++i) r[i] = *(const u32x4*)(p + 64 * i);
    } else {
      const short* p = (const short*)w + at + 8 * g;
#pragma unroll
      for (int i = 0; i < CH / 32; ++i) r[i] = *(const u32x4*)(p + 32 * i);
    }
  }
  __device__ __forceinline__ s16x8 operand(int i) const {
    if (I8) {
      unsigned o[4];
      widen(r[i >> 1][2 * (i & 1)], o[0], o[1]);
      widen(r[i >> 1][2 * (i & 1) + 1], o[2], o[3]);
      return __builtin_bit_cast(s16x8, u32x4{o[0], o[1], o[2], o[3]});
    }
    return __builtin_bit_cast(s16x8, r[i]);
  }
};

// Input of operand i: bf16 takes 32 i + 8 g.., int8 64 (i/2) + 16 g + 8 (i%2)..
template <bool I8>
__device__ __forceinline__ int input_at(int i, int g) {
  return I8 ? 64 * (i >> 1) + 16 * g + 8 * (i & 1) : 32 * i + 8 * g;
}

template <bool I8, int MT, int MODE, int FT>
__global__ __launch_bounds__(NW * 64) void rows_linear_kernel(const Args a) {
  constexpr int CH = MT == 1 ? 256 : 128;     // inputs a chunk
  constexpr int L = MODE == SWIGLU ? 2 : 1;   // weight streams a workgroup
  constexpr int S = L * FT;                   // tiles of 16 features a wave
  __shared__ float lds[NW][S][256];

  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int col = lane & 15, g = lane >> 4;
  int layer = 0, tile = blockIdx.x;
  if (MODE == PLAIN) {
    while (tile >= a.tile_end[layer]) ++layer;
    if (layer) tile -= a.tile_end[layer - 1];
  }
  const int N = a.n[layer];
  const int n0 = tile * 16 * FT;

  const short* xp[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m)
    xp[m] = a.x + (long long)min(16 * m + col, a.M - 1) * a.K;
  long long row[FT];
#pragma unroll
  for (int f = 0; f < FT; ++f)
    row[f] = (long long)min(n0 + 16 * f + col, N - 1) * a.K;

  f32x4 acc[S][MT];
#pragma unroll
  for (int s = 0; s < S; ++s)
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[s][m] = f32x4{0.f, 0.f, 0.f, 0.f};

  const int chunks = a.K / CH;
  Weights<I8, CH> w[S];
  int c = wid;
  if (c < chunks)
#pragma unroll
    for (int s = 0; s < S; ++s)
      w[s].load(a.w[layer + s / FT], row[s % FT] + c * CH, g);
  for (; c < chunks; c += NW) {
    s16x8 xb[MT][CH / 32];
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int i = 0; i < CH / 32; ++i)
        xb[m][i] = *(const s16x8*)(xp[m] + c * CH + input_at<I8>(i, g));
    float sc[S][4];
    if (I8)     // of the rows 4 g + r that the lane holds the sums of
#pragma unroll
      for (int s = 0; s < S; ++s)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          sc[s][r] = a.scales[layer + s / FT][
              ((long long)min(n0 + 16 * (s % FT) + 4 * g + r, N - 1) * a.K +
               c * CH) / a.group];
    Weights<I8, CH> cur[S];
#pragma unroll
    for (int s = 0; s < S; ++s) cur[s] = w[s];
    if (c + NW < chunks)
#pragma unroll
      for (int s = 0; s < S; ++s)
        w[s].load(a.w[layer + s / FT], row[s % FT] + (c + NW) * CH, g);
#pragma unroll
    for (int s = 0; s < S; ++s) {
      f32x4 part[MT];
#pragma unroll
      for (int m = 0; m < MT; ++m)
        part[m] = I8 ? f32x4{0.f, 0.f, 0.f, 0.f} : acc[s][m];
#pragma unroll
      for (int i = 0; i < CH / 32; ++i) {
        const s16x8 wa = cur[s].operand(i);
#pragma unroll
        for (int m = 0; m < MT; ++m) part[m] = mfma(wa, xb[m][i], part[m]);
      }
#pragma unroll
      for (int m = 0; m < MT; ++m)
        if (I8)
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[s][m][r] += part[m][r] * sc[s][r];
        else
          acc[s][m] = part[m];
    }
  }

  // ---- add the waves up, 16 rows of x at a time; features 4 g + r of a
  // column lie side by side
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    if (16 * m >= a.M) break;
    if (m) __syncthreads();
#pragma unroll
    for (int s = 0; s < S; ++s)
      *(f32x4*)(&lds[wid][s][col * 16 + 4 * g]) = acc[s][m];
    __syncthreads();
    for (int e = threadIdx.x; e < FT * 256; e += NW * 64) {
      const int f = e >> 8, at = e & 255;
      const int r = 16 * m + (at >> 4), n = n0 + 16 * f + (at & 15);
      if (r >= a.M || n >= N) continue;
      float y[L];
#pragma unroll
      for (int s = 0; s < L; ++s) {
        float t = 0.f;
#pragma unroll
        for (int w_ = 0; w_ < NW; ++w_) t += lds[w_][s * FT + f][at];
        if (a.bias[layer + s]) t += value(a.bias[layer + s][n]);
        y[s] = t;
      }
      float o = y[0];
      if (MODE == SWIGLU) o = y[0] / (1.f + expf(-y[0])) * y[L - 1];
      const long long to = (long long)r * N + n;
      a.out[layer][to] = bits(o);
    }
  }
}

template <bool I8, int MT, int MODE, int FT>
void launch(Args a, int layers, hipStream_t st) {
  int tiles = 0;
  for (int i = 0; i < (MODE == SWIGLU ? 1 : layers); ++i)
    a.tile_end[i] = tiles += (a.n[i] + 16 * FT - 1) / (16 * FT);
  hipLaunchKernelGGL((rows_linear_kernel<I8, MT, MODE, FT>), dim3(tiles),
                     dim3(NW * 64), 0, st, a);
}

// Tiles of features a wave. Every workgroup reads all of x, which costs M rows
// out of L2 for 16 FT features of W: with more rows FT has to grow, but half
// the workgroups leave CUs idle where the layer is small. Measured (us, bf16,
// FT 1 / 2 / 4): M 8: N 4096 10.8 / 13.8 / 37, N 14336 29.2 / 29.2 / 51;
// M 16: N 6144 19.5 / 17.0 / 40, N 14336 35.7 / 31.5 / 52; M 32: N 4096 15.7 /
// 18.6 / 25, N 6144 26.1 / 20.3 / 25.5, N 14336 48 / 36.5 / 29.6. Gate and up
// (two streams share x): M 16 52.6 / 92, M 32 61.9 / 55.1. int8, for which x
// weighs twice as much, is within a tenth of its best by the same rule: M 8: N
// 4096 8.3 / 10.8 / 18, N 6144 13.0 / 11.8 / 19, N 14336 20.7 / 20.9 / 20.1; M
// 16: N 6144 15.4 / 12.8 / 20, N 14336 25.9 / 23.0 / 20.8, N 128256 176 / 163 /
// 152; M 32: N 6144 23 / 16.3 / 23, N 14336 40 / 29.7 / 24.0; M 64: N 4096 21.1 /
// 23.8 / 44, N 14336 74 / 46 / 51; gate and up M 8 35.9 / 34.8, M 16 39.5 / 37.2,
// M 32 53.8 / 42.6, M 64 88 / 67.
template <bool I8>
void launch_rows(const Args& a, int layers, int mode, hipStream_t st) {
  int tiles = 0;
  for (int i = 0; i < layers; ++i) tiles += (a.n[i] + 15) / 16;
  const bool big = tiles >= 384, huge = tiles >= 896;
  if (mode == SWIGLU) {
    if (a.M <= 16) launch<I8, 1, SWIGLU, 1>(a, layers, st);
    else if (a.M <= 32) launch<I8, 2, SWIGLU, 2>(a, layers, st);
    else if (I8) launch<true, 4, SWIGLU, 2>(a, layers, st);
  } else if (a.M <= 16) {
    if (a.M > 8 && big) launch<I8, 1, PLAIN, 2>(a, layers, st);
    else launch<I8, 1, PLAIN, 1>(a, layers, st);
  } else if (a.M <= 32) {
    if (huge) launch<I8, 2, PLAIN, 4>(a, layers, st);
    else if (big) launch<I8, 2, PLAIN, 2>(a, layers, st);
    else launch<I8, 2, PLAIN, 1>(a, layers, st);
  } else if (I8) {
    if (big) launch<true, 4, PLAIN, 2>(a, layers, st);
    else launch<true, 4, PLAIN, 1>(a, layers, st);
  }
}

}  // namespace

// layers: 1..3 weights on one input; mode 1: silu(layer 0) * layer 1. K and,
// int8, the group are multiples of 256: a chunk of a feature has one scale.
extern "C" void ds_rows_linear(const void* x, int layers, const void* const* w,
                               const float* const* scales,
                               const void* const* bias, void* const* out,
                               const int* n, int M,
                               int K, int group, int mode,
                               void* stream) {
  Args a = {};
  for (int i = 0; i < layers; ++i) {
    a.w[i] = w[i];
    a.scales[i] = scales ? scales[i] : nullptr;
    a.bias[i] = (const short*)bias[i];
    a.out[i] = (short*)out[i];
    a.n[i] = n[i];
  }
  a.x = (const short*)x;
  a.M = M; a.K = K; a.group = group;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  if (scales) launch_rows<true>(a, layers, mode, st);
  else launch_rows<false>(a, layers, mode, st);
}
