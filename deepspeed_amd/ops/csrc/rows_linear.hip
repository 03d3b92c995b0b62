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
// at N = 4096. W goes from memory straight into the A operand of
// mfma_f32_16x16x32_bf16 (16 features by 64 contiguous bytes an instruction), x
// into B (columns past M repeat the last row).
//
//   * Up to 16 rows, few_rows_kernel: W and x are loaded D chunks of 128 inputs
// ahead, so that a wave waits for neither, and the scales lie in LDS. Bound by
// the stream of W in large layers, by launch and first loads in small ones. us
// at 8 rows, before (chunks of 256, x loaded where it is used) and now: gate and
// up 14336, K 4096 bf16 50.7 / 45.8, int8 36.6 / 32.8; q, k, v 4096 + 2 x 1024,
// K 4096 16.0 / 13.3 and 12.2 / 10.8; N 128256 199 / 192 and 140 / 121; N 4096,
// K 14336 27.7 / 27.3 and 19.7 / 18.9; N 4096, K 4096 10.2 / 10.1 and 8.2 / 8.6.
// Three to six chunks ahead gained nothing more. Most layers of K 2048 to 4096 go
// on to going_rows_kernel, which was measured against this.
//   * More rows, rows_linear_kernel: bound by x out of L2. Only int8 weights, small
// layers and numbers of features that tile_linear.hip does not take come here.
//   * int8: a lane's 16 bytes are 16 inputs, split over two products; the order
//     of the inputs inside a product is free, x is read in the same order. The
//     bytes become bf16 exactly (8 bits), are summed in fp32 and multiplied by
//     their group's scale in fp32: nothing is rounded before the output, and
//     the weight is not written out as bf16 and read again.
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
constexpr int CH = 128;     // inputs a chunk

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

// four signed bytes to four bf16, exactly: signed, an instruction a byte and one a
// pair, or by way of b + 128 = 0..255, two a byte, which is faster where four tiles
// of rows are multiplied by two streams (gate and up 14336, K 4096, us by either:
// 17 rows 39.5 / 42.8, 33 rows 61.0 / 56.1, 48 rows 63.4 / 59.5)
template <bool SIGNED>
__device__ __forceinline__ void widen(unsigned b, unsigned& lo, unsigned& hi) {
  float f0, f1, f2, f3;
  if (SIGNED) {
    f0 = (float)(int)(signed char)b;
    f1 = (float)(int)(signed char)(b >> 8);
    f2 = (float)(int)(signed char)(b >> 16);
    f3 = (float)(int)(signed char)(b >> 24);
  } else {
    b ^= 0x80808080u;
    f0 = (float)(b & 255u) - 128.f;
    f1 = (float)((b >> 8) & 255u) - 128.f;
    f2 = (float)((b >> 16) & 255u) - 128.f;
    f3 = (float)(b >> 24) - 128.f;
  }
  lo = __builtin_amdgcn_perm(__builtin_bit_cast(unsigned, f1),
                             __builtin_bit_cast(unsigned, f0), 0x07060302u);
  hi = __builtin_amdgcn_perm(__builtin_bit_cast(unsigned, f3),
                             __builtin_bit_cast(unsigned, f2), 0x07060302u);
}

// CH inputs of 16 features: CH / 32 A operands.
template <bool I8>
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
  template <bool SIGNED = true>
  __device__ __forceinline__ s16x8 operand(int i) const {
    if (I8) {
      unsigned o[4];
      widen<SIGNED>(r[i >> 1][2 * (i & 1)], o[0], o[1]);
      widen<SIGNED>(r[i >> 1][2 * (i & 1) + 1], o[2], o[3]);
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
  Weights<I8> w[S];
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
    Weights<I8> cur[S];
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
        const s16x8 wa =
            cur[s].template operand<MT != 4 || MODE != SWIGLU>(i);
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

// EVEN: every wave's chunks are a multiple of D, so that no load runs ahead of the
// last one. Otherwise each is asked for by itself, and costs a branch (K 4096, q, k
// and v of 4096 + 2 x 1024, 8 rows 13.6 / 15.1). us at 8 rows, loads past the end
// repeating the last chunk and now: N 32000, K 1024 41.6 / 14.4; 3 of 3072, K 3072
// 22.2 / 16.6; gate and up 2816, K 1024 7.3 / 5.1; 8192, K 3072 24.3 / 20.1; 3584, K
// 18944 35.1 / 32.2.
template <bool I8, int MODE, int FT, int D, int OCC, bool EVEN>
__global__ __launch_bounds__(NW * 64, OCC) void few_rows_kernel(const Args a) {
  constexpr int L = MODE == SWIGLU ? 2 : 1;   // weight streams a workgroup
  constexpr int S = L * FT;                   // tiles of 16 features a wave
  // [waves][S][256] sums, then int8's scales [chunks][S][16]
  extern __shared__ __attribute__((aligned(16))) float lds[];
  float* const sums = lds;
  float* const scales = lds + NW * S * 256;

  const int lane = threadIdx.x & 63;
  const int wid = EVEN ? threadIdx.x >> 6
                       : __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, g = lane >> 4;
  int layer = 0, tile = blockIdx.x;
  if (MODE == PLAIN) {
    while (tile >= a.tile_end[layer]) ++layer;
    if (layer) tile -= a.tile_end[layer - 1];
  }
  const int N = a.n[layer], n0 = tile * 16 * FT;
  const short* xp = a.x + (long long)min(col, a.M - 1) * a.K;
  long long row[FT];
#pragma unroll
  for (int f = 0; f < FT; ++f)
    row[f] = (long long)min(n0 + 16 * f + col, N - 1) * a.K;

  const int chunks = a.K / CH;
  const int mine = (chunks - wid + NW - 1) / NW;    // wid, wid + NW, ..
  Weights<I8> w[D][S];
  s16x8 x[D][CH / 32];
  // Workgroups that all begin at the rows' beginnings read the same few memory
  // channels at a time where rows are whole multiples of 16 KB (int8: 4 KB) apart; each
  // begins elsewhere there (us, 8 rows, before / now: bf16 8192, K 8192 31.6 / 25.0,
  // 28672 x 2, K 8192 165 / 156; int8 14336 x 2, K 4096 33.8 / 30.8, 4096 8.6 / 7.8,
  // 128256 117 / 113, of 1 row 109 / 97; but apart by 6 KB, 8192 x 2, K 3072 bf16 19.7 /
  // 20.4, by 28, 4096, K 14336 of 1 row 22.7 / 23.9, by 8, 128256, K 4096 185 / 189).
  const int turn = a.K % (I8 ? 4096 : 8192) ? 0
      : __builtin_amdgcn_readfirstlane(
            (blockIdx.x / 8 * 13 + blockIdx.x % 8 * 7) % 32 * chunks / 32);
  auto chunk = [&](int i) __attribute__((always_inline)) {
    const int c = wid + i * NW + turn;
    return c < chunks ? c : c - chunks;
  };
  auto load = [&](int d, int i) __attribute__((always_inline)) {
    const int at = chunk(EVEN ? min(i, mine - 1) : i) * CH;
#pragma unroll
    for (int s = 0; s < S; ++s)
      w[d][s].load(a.w[layer + s / FT], row[s % FT] + at, g);
#pragma unroll
    for (int k = 0; k < CH / 32; ++k)
      x[d][k] = *(const s16x8*)(xp + at + input_at<I8>(k, g));
  };
  f32x4 acc[S];
#pragma unroll
  for (int s = 0; s < S; ++s) acc[s] = f32x4{0.f, 0.f, 0.f, 0.f};
  if (!EVEN || mine > 0)
#pragma unroll
    for (int d = 0; d < D; ++d)
      if (EVEN || d < mine) load(d, d);
  if (I8) {
    for (int e = threadIdx.x; e < chunks * S * 16; e += NW * 64) {
      const int c = e / (S * 16), f = e % (S * 16);
      const long long r = min(n0 + f % (16 * FT), N - 1);
      scales[e] = a.scales[layer + f / (16 * FT)][(r * a.K + c * CH) / a.group];
    }
    // the scales have arrived, and with them the loads above, which were first
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  }
  auto use = [&](int d, int i) __attribute__((always_inline)) {
#pragma unroll
    for (int s = 0; s < S; ++s) {
      f32x4 part = I8 ? f32x4{0.f, 0.f, 0.f, 0.f} : acc[s];
#pragma unroll
      for (int k = 0; k < CH / 32; ++k)
        part = mfma(w[d][s].operand(k), x[d][k], part);
      if (I8) {     // of the rows 4 g + r that the lane holds the sums of
        const f32x4 sc = *(const f32x4*)(
            scales + (chunk(i) * S + s) * 16 + 4 * g);
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[s][r] += part[r] * sc[r];
      } else {
        acc[s] = part;
      }
    }
  };
  if (mine > 0) {
    int i = 0;
    for (; i + D < mine; i += D)
#pragma unroll
      for (int d = 0; d < D; ++d) {
        use(d, i + d);
        if (EVEN || i + d + D < mine) load(d, i + d + D);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
    for (int d = 0; d < D; ++d)
      if (i + d < mine) use(d, i + d);
  }

  // ---- add the waves up; features 4 g + r of a column lie side by side
#pragma unroll
  for (int s = 0; s < S; ++s)
    *(f32x4*)(sums + (wid * S + s) * 256 + col * 16 + 4 * g) = acc[s];
  __syncthreads();
  for (int e = threadIdx.x; e < FT * 256; e += NW * 64) {
    const int f = e >> 8, at = e & 255;
    const int r = at >> 4, n = n0 + 16 * f + (at & 15);
    if (r >= a.M || n >= N) continue;
    float y[L];
#pragma unroll
    for (int s = 0; s < L; ++s) {
      float t = 0.f;
#pragma unroll
      for (int w_ = 0; w_ < NW; ++w_)
        t += sums[(w_ * S + s * FT + f) * 256 + at];
      if (a.bias[layer + s]) t += value(a.bias[layer + s][n]);
      y[s] = t;
    }
    float o = y[0];
    if (MODE == SWIGLU) o = y[0] / (1.f + expf(-y[0])) * y[L - 1];
    a.out[layer][(long long)r * N + n] = bits(o);
  }
}

// The same over contractions of X chunks a wave, for which x stays in registers: one
// workgroup a CU that goes on from tile to tile, with all chunks of the next tile on
// their way while this one's are multiplied and added up (sums and int8's scales
// have two places in LDS, and a tile one barrier). Reading x again for each tile
// takes the more of the time the more rows there are, and first loads and the last
// round's end are a quarter of a workgroup's life that reads one tile. As many
// workgroups as fill every round alike. us, few_rows_kernel / here, at 1, 8 and 16
// rows: gate and up 14336, K 4096 bf16 44.0 / 40.9, 46.0 / 42.1, 51.1 / 43.9, int8 at 8
// and 16 30.6 / 28.1, 35.4 / 29.7; 128256, K 4096 bf16 163 / 164, 186 / 174, 208 /
// 181, int8 96 / 87, 112 / 92, 134 / 99; 9216, K 3072 bf16 14.3 / 12.8, 16.7 / 13.6, 18.2
// (12 rows) / 14.2. Now 5.2 to 6.3 TB/s of W where it is large.
//
// A workgroup's tiles are fixed at the launch and it takes a CU whole: where another
// stream's kernel holds CUs and the workgroups are more than those left, some begin when
// the first others end (us, few_rows_kernel / here, 8 rows, weights from memory, alone
// and with 8 CUs held: 128256, K 4096 bf16 190 / 174 and 210 / 274, int8 128 / 97 and 132
// / 152; 28672 bf16 51 / 42 and 54 / 65; but gate and up 14336, 224 workgroups, 45 / 42
// and 46 / 41). Of the framework only ZeRO-3's gathers run beside such layers, and are
// many times as long; a serving step's collectives wait for it and it for them. With
// workgroups for 224 CUs nothing is lost where 8 are held, but alone 0 to 17% (int8
// 32000, K 4096 28.4 / 32.3, 16384 16.6 / 19.5, bf16 12288 20.0 / 21.9, 128256 none).
template <bool I8, int MODE, int FT, int X>
__global__ __launch_bounds__(NW * 64, 2) void going_rows_kernel(const Args a,
                                                                int tiles) {
  constexpr int L = MODE == SWIGLU ? 2 : 1;   // weight streams a workgroup
  constexpr int S = L * FT;                   // tiles of 16 features a wave
  constexpr int C = X * NW, R = I8 ? (C * S * 16 + NW * 64 - 1) / (NW * 64) : 1;
  __shared__ float sums[2][NW * S * 256];
  __shared__ __attribute__((aligned(16)))
  float scales[I8 ? 2 : 1][I8 ? C * S * 16 : 4];

  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, g = lane >> 4;
  const int turn = !I8 || a.K % 4096 ? 0      // as above
      : __builtin_amdgcn_readfirstlane(
            (blockIdx.x / 8 * 13 + blockIdx.x % 8 * 7) % 32 * C / 32);
  auto chunk = [&](int i) __attribute__((always_inline)) {
    const int c = wid + i * NW + turn;
    return c < C ? c : c - C;
  };
  struct Place { int layer, n0; };
  auto locate = [&](int tile) __attribute__((always_inline)) {
    int l = 0;
    if (MODE == PLAIN) {
      while (tile >= a.tile_end[l]) ++l;
      if (l) tile -= a.tile_end[l - 1];
    }
    return Place{l, tile * 16 * FT};
  };
  int tile = blockIdx.x;
  Place at = locate(tile);
  Weights<I8> w[X][S];
  long long row[FT];
  Place from = at;
  auto rows_of = [&](Place p) __attribute__((always_inline)) {
    from = p;
#pragma unroll
    for (int f = 0; f < FT; ++f)
      row[f] = (long long)min(p.n0 + 16 * f + col, a.n[p.layer] - 1) * a.K;
  };
  auto load = [&](int i) __attribute__((always_inline)) {
#pragma unroll
    for (int s = 0; s < S; ++s)
      w[i][s].load(a.w[from.layer + s / FT], row[s % FT] + chunk(i) * CH, g);
  };
  // int8's scales of a tile [chunks][S][16], by way of registers
  float sc[R];
  auto load_scales = [&](Place p) __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int e = min((int)threadIdx.x + r * NW * 64, C * S * 16 - 1);
      const int c = e / (S * 16), f = e % (S * 16);
      const long long n = min(p.n0 + f % (16 * FT), a.n[p.layer] - 1);
      sc[r] = a.scales[p.layer + f / (16 * FT)][(n * a.K + c * CH) / a.group];
    }
  };
  auto put_scales = [&](int b) __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int e = threadIdx.x + r * NW * 64;
      if (e < C * S * 16) scales[I8 ? b : 0][e] = sc[r];
    }
  };
  if (I8) load_scales(at);
  rows_of(at);
#pragma unroll
  for (int i = 0; i < X; ++i) load(i);
  s16x8 x[X][CH / 32];
  const short* xp = a.x + (long long)min(col, a.M - 1) * a.K;
#pragma unroll
  for (int i = 0; i < X; ++i)
#pragma unroll
    for (int k = 0; k < CH / 32; ++k)
      x[i][k] = *(const s16x8*)(xp + chunk(i) * CH + input_at<I8>(k, g));
  if (I8) {
    put_scales(0);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  }
  int b = 0;
  while (true) {
    const int then = tile + gridDim.x;
    const bool more = then < tiles;
    const Place next = more ? locate(then) : at;
    if (I8 && more) load_scales(next);
    f32x4 acc[S];
#pragma unroll
    for (int s = 0; s < S; ++s) acc[s] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < X; ++i) {
#pragma unroll
      for (int s = 0; s < S; ++s) {
        f32x4 part = I8 ? f32x4{0.f, 0.f, 0.f, 0.f} : acc[s];
#pragma unroll
        for (int k = 0; k < CH / 32; ++k)
          part = mfma(w[i][s].operand(k), x[i][k], part);
        if (I8) {     // of the rows 4 g + r that the lane holds the sums of
          const f32x4 v = *(const f32x4*)(
              &scales[I8 ? b : 0][(chunk(i) * S + s) * 16 + 4 * g]);
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[s][r] += part[r] * v[r];
        } else {
          acc[s] = part;
        }
      }
      if (i == 0) rows_of(next);
      if (more) load(i);
      __builtin_amdgcn_sched_barrier(0);
    }
    float* const sum = sums[b];
#pragma unroll
    for (int s = 0; s < S; ++s)
      *(f32x4*)(sum + (wid * S + s) * 256 + col * 16 + 4 * g) = acc[s];
    if (I8 && more) put_scales(b ^ 1);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    const int N = a.n[at.layer];
    for (int e = threadIdx.x; e < FT * 256; e += NW * 64) {
      const int f = e >> 8, o_ = e & 255;
      const int r = o_ >> 4, n = at.n0 + 16 * f + (o_ & 15);
      if (r >= a.M || n >= N) continue;
      float y[L];
#pragma unroll
      for (int s = 0; s < L; ++s) {
        float t = 0.f;
#pragma unroll
        for (int w_ = 0; w_ < NW; ++w_)
          t += sum[(w_ * S + s * FT + f) * 256 + o_];
        if (a.bias[at.layer + s]) t += value(a.bias[at.layer + s][n]);
        y[s] = t;
      }
      float o = y[0];
      if (MODE == SWIGLU) o = y[0] / (1.f + expf(-y[0])) * y[L - 1];
      a.out[at.layer][(long long)r * N + n] = bits(o);
    }
    if (!more) break;
    tile = then;
    at = next;
    b ^= 1;
  }
}

template <bool I8, int MODE, int X>
int launch_going(Args a, int layers, hipStream_t st) {
  constexpr int FT = I8 && MODE == PLAIN ? 2 : 1, CUS = 256;
  int tiles = 0;
  for (int i = 0; i < (MODE == SWIGLU ? 1 : layers); ++i)
    a.tile_end[i] = tiles += (a.n[i] + 16 * FT - 1) / (16 * FT);
  const int rounds = (tiles + CUS - 1) / CUS;
  hipLaunchKernelGGL((going_rows_kernel<I8, MODE, FT, X>),
                     dim3((tiles + rounds - 1) / rounds), dim3(NW * 64), 0, st,
                     a, tiles);
  return (int)hipGetLastError();
}

// Where they go on, for tiles of 16 features (us, few_rows_kernel / going on, K 4096
// unless said): not a single round (bf16 4096 of 1 row 8.8 / 8.9, int8 6.9 / 9.1). Gates
// whose rounds are whole from 9 rows on only (8192 of 1 row 25.2 / 25.9, 12288 35.1 /
// 36.0, of 16 rows 29.1 / 27.9; 8448 of 1 row 31.6 / 28.3), int8's from 5 on unless
// they are short (14336, K 3072 of 1 row 20.6 / 21.8, of 8 24.2 / 22.7; K 2048 of 1
// 15.7 / 14.8). bf16 of one or two rows up to 4096 tiles (50304 67.9 / 65.9, 128256 163
// / 164, K 3072 123 / 125). int8 of up to four rows not where the last round, of
// tiles of 32, is filled (13824, K 3072 11.9 / 12.2, 16384 15.2 / 16.0; 12288 14.6 /
// 14.1, 16640 20.2 / 18.7).
// K 2048 bf16, where a wave has two chunks on their way, stays (14336 x 2 of 1 row
// 23.9 / 26.4, 32000 of 8 25.2 / 27.2), as do 5 and more chunks a wave, for which the
// registers do not reach, and contractions that are not whole chunks of eight waves.
template <bool I8>
bool goes_on(const Args& a, int mode, int tiles) {
  const int X = a.K % (CH * NW) ? 0 : a.K / (CH * NW), pairs = tiles / 2;
  if (X < (I8 ? 2 : 3) || X > 4) return false;
  if (mode == SWIGLU)
    return pairs > 256 && (a.M > 8 || pairs % 256) &&
           (!I8 || a.M > 4 || X == 2);
  if (!I8) return tiles > 256 && (a.M > 2 || tiles < 4096);
  return a.M > 4 ? tiles > 256 : pairs > 512 || (pairs > 256 && pairs <= 384);
}

// D of chunks ahead, and the waves a SIMD that its registers leave.
template <bool I8, int MODE, int FT, int D, int OCC>
int launch_few(Args a, int layers, hipStream_t st) {
  int tiles = 0;
  for (int i = 0; i < (MODE == SWIGLU ? 1 : layers); ++i)
    a.tile_end[i] = tiles += (a.n[i] + 16 * FT - 1) / (16 * FT);
  constexpr int S = (MODE == SWIGLU ? 2 : 1) * FT;
  const int lds = NW * S * 1024 + (I8 ? a.K / CH * S * 64 : 0);
  auto kernel = a.K / CH % (NW * D) == 0
      ? few_rows_kernel<I8, MODE, FT, D, OCC, true>
      : few_rows_kernel<I8, MODE, FT, D, OCC, false>;
  if (lds > 64 * 1024) {
    const hipError_t e = hipFuncSetAttribute(
        (const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e != hipSuccess) return (int)e;
  }
  hipLaunchKernelGGL(kernel, dim3(tiles), dim3(NW * 64), lds, st, a);
  return (int)hipGetLastError();
}

template <bool I8, int MT, int MODE, int FT>
int launch(Args a, int layers, hipStream_t st) {
  int tiles = 0;
  for (int i = 0; i < (MODE == SWIGLU ? 1 : layers); ++i)
    a.tile_end[i] = tiles += (a.n[i] + 16 * FT - 1) / (16 * FT);
  hipLaunchKernelGGL((rows_linear_kernel<I8, MT, MODE, FT>), dim3(tiles),
                     dim3(NW * 64), 0, st, a);
  return (int)hipGetLastError();
}

// Tiles of features a wave, where workgroups have one tile. Every workgroup reads
// all of x, which costs M rows
// out of L2 for 16 FT features of W; half the workgroups leave CUs idle where the
// layer is small. Up to 16 rows (us, FT 1 / 2): N 4096 bf16 9.6 / 13, int8 8.6 /
// 10.4; N 6144 15.7 / 13.3 and 12.3 / 10.8; N 128256 8 rows 205 / 192 and 148 /
// 121, 16 rows 250 / 209 and 178 / 139, but bf16 1 row 168 / 178; gate and up,
// whose two streams share x, 45.8 / 50.7 and 32.8 / 34.1. With two tiles bf16
// has four chunks ahead where these are a wave's whole parts (N 6144 13.3, two
// 14.5; N 32000, K 1024 two 14.4, four 17.7), int8 two (10.8, four 11.5).
// Two tiles take two rounds of the CUs' time: not where the rounds grow by it (8
// rows, FT 1 / 2, bf16: N 9216, K 4096 20.7 / 25.0; 12288 22.8 / 26.2; 10240, K 8192
// 46 / 51; int8 of long layers and few rows: 10240, K 8192 28.0 / 31.3, but 12288, K
// 4096 17.8 / 17.0), nor, there, where it leaves a CU one workgroup (8192, K 8192, 1
// row 16.5 / 20.9).
// More rows, int8 (FT 1 / 2 / 4): M 32: N 4096 11 / 14 / 20, N 6144 23 / 16.3 /
// 23, N 14336 40 / 29.7 / 24.0; M 64: N 4096 21.1 / 23.8 / 44, N 14336 74 / 46 /
// 51; gate and up M 32 53.8 / 42.6, M 64 88 / 67.
template <bool I8>
int launch_rows(const Args& a, int layers, int mode, hipStream_t st) {
  int tiles = 0;
  for (int i = 0; i < layers; ++i) tiles += (a.n[i] + 15) / 16;
  const bool big = tiles >= 384, huge = tiles >= 896;
  // int8's scales in LDS: beside the sums 64 bytes a chunk and stream
  if (a.M <= 16 && goes_on<I8>(a, mode, tiles)) {
#define GO(X)                                                             \
  if (a.K == X * CH * NW)                                                 \
    return mode == SWIGLU ? launch_going<I8, SWIGLU, X>(a, layers, st)    \
                          : launch_going<I8, PLAIN, X>(a, layers, st);
    GO(4)
    GO(3)
    if constexpr (I8) { GO(2) }
#undef GO
  }
  if (a.M <= 16 && (!I8 || a.K <= 1 << 16)) {
    if (mode == SWIGLU) return launch_few<I8, SWIGLU, 1, 2, 4>(a, layers, st);
    const bool rounds = 2 * ((tiles + 511) / 512) <= (tiles + 255) / 256;
    const bool full = tiles > 448 && tiles <= 512;
    if (!big || (I8 ? a.M <= 8 && a.K > 4096 && (!rounds || full)
                    : !rounds || (a.M <= 4 && tiles >= 2048)))
      return launch_few<I8, PLAIN, 1, 2, 4>(a, layers, st);
    if (!I8 && a.K / CH % (4 * NW) == 0)
      return launch_few<I8, PLAIN, 2, 4, 2>(a, layers, st);
    return launch_few<I8, PLAIN, 2, 2, 4>(a, layers, st);
  }
  if (mode == SWIGLU) {
    if (a.M <= 32) return launch<I8, 2, SWIGLU, 2>(a, layers, st);
    return launch<true, 4, SWIGLU, 2>(a, layers, st);
  }
  if (a.M <= 32) {
    if (huge) return launch<I8, 2, PLAIN, 4>(a, layers, st);
    if (big) return launch<I8, 2, PLAIN, 2>(a, layers, st);
    return launch<I8, 2, PLAIN, 1>(a, layers, st);
  }
  if (big) return launch<true, 4, PLAIN, 2>(a, layers, st);
  return launch<true, 4, PLAIN, 1>(a, layers, st);
}

}  // namespace

// layers: 1..3 weights on one input; mode 1: silu(layer 0) * layer 1. K and,
// int8, the group are multiples of 256: a chunk of a feature has one scale.
// M up to 32, int8 64. Returns a hipError_t.
extern "C" int ds_rows_linear(const void* x, int layers, const void* const* w,
                              const float* const* scales,
                              const void* const* bias, void* const* out,
                              const int* n, int M, int K, int group, int mode,
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
  return scales ? launch_rows<true>(a, layers, mode, st)
                : launch_rows<false>(a, layers, mode, st);
}
