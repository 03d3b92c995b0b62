// Linear layers of a few rows for MI355X (gfx950): y = x W^T, x [M, K] bf16,
// W [N, K] bf16 (M up to 32) or groupwise int8 (M up to 64).
//
// Decoding reads every weight once for a handful of tokens, so a layer is as
// fast as its weights stream in. Reference analogues: the GEMV-shaped GEMMs of
// csrc/transformer/inference and the weight-only quantized linears of
// inference/v2/kernels/core_ops (cuda_linear).
//
// W is the A operand of mfma_f32_16x16x32_bf16 (16 features), x the B operand
// (columns past M are not stored); the waves of a workgroup have parts of the
// contraction and add up through LDS.
//
//   * Up to 16 rows, and up to 32 where the weights are int8 or the layer is small:
// stream_rows_kernel, in which every load goes to LDS, 128 bytes of 8 rows an
// instruction. Bound by the stream of W from memory, 6 to 7 TB/s where it is large,
// by launch and first loads where it is small.
//   * More rows of int8, and more than 2^22 inputs, rows_linear_kernel: W and x straight
// into registers, bound by x out of L2. bf16 layers of more rows are tile_linear.hip's.
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

constexpr int NW = 8;       // waves a workgroup, there
constexpr int MAXL = 3;     // layers a launch
constexpr int CH = 128;     // inputs a chunk of rows_linear_kernel

// QKV: three layers of heads of 128 features
enum { PLAIN = 0, SWIGLU = 1, QKV = 2 };

// With `dst`, where q, k and v go: q turned to out[0], k turned and v to rows dst of the
// paged pool [blocks, heads, BS, 128].
struct Append {
  const float *cs, *sn;     // [positions, 64]
  const int* positions;     // [M], or null: row % S
  const int* dst;
  short *kpool, *vpool;
  int S, heads, BS;
};

struct Args {
  const void* w[MAXL];
  const float* scales[MAXL];
  const short* bias[MAXL];
  short* out[MAXL];
  int n[MAXL], tile_end[MAXL];
  const short* x;
  int M, K, group;
  bool heads;               // PLAIN: workgroups begin as QKV's with their tiles do
  Append to;
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

template <int N>
__device__ __forceinline__ void wait_loads() {  // but for the N youngest
  static_assert(N < 64, "vmcnt has six bits");
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
__device__ __forceinline__ void barrier() {   // and what was read from LDS
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}
__device__ __forceinline__ int uni(int x) {
  return __builtin_amdgcn_readfirstlane(x);
}
// Loads past `left` bytes from `base` on bring zeros.
__device__ __forceinline__ u32x4 descriptor(const void* base, long long left) {
  const unsigned long long b = (unsigned long long)(uintptr_t)base;
  u32x4 d;
  d[0] = uni((unsigned)b);
  d[1] = uni((unsigned)(b >> 32) & 0xffffu);
  d[2] = uni(left > 0xffffffffll ? 0xffffffffu : (unsigned)left);
  d[3] = 0x00020000u;
  return d;
}
// 16 bytes a lane from descriptor + off + soff to LDS, lane after lane from `lds` on;
// ONCE: read by nobody else, past the caches.
template <bool ONCE>
__device__ __forceinline__ void load(u32x4 from, unsigned off, int soff, int lds) {
  if (ONCE)
    asm volatile("s_mov_b32 m0, %3\n\ts_nop 0\n\t"
                 "buffer_load_dwordx4 %0, %1, %2 offen nt lds"
                 :: "v"(off), "s"(from), "s"(soff), "s"(lds) : "memory", "m0");
  else
    asm volatile("s_mov_b32 m0, %3\n\ts_nop 0\n\t"
                 "buffer_load_dwordx4 %0, %1, %2 offen lds"
                 :: "v"(off), "s"(from), "s"(soff), "s"(lds) : "memory", "m0");
}
__device__ __forceinline__ void load_scales(const float* from, unsigned off, int lds) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\t"
               "global_load_lds_dword %0, %1"
               :: "v"(off), "s"(from), "s"(lds) : "memory", "m0");
}

// Each wave has a ring of its own in LDS, of D slots of 128 bytes of W's rows and what
// belongs to them of x and of int8's scales; it goes on from tile to tile, and waits for
// nobody before a tile's sums are added up. The ring is full meanwhile; but loads come
// back in their order, so threads that then fetch a bias or, with several tiles of q and
// k a workgroup, angles wait for what is in it.
//
//   * Loads to LDS, not to registers: as operands of the products lanes next to each
// other have different rows, and a load of 16 rows by 64 bytes takes the address unit
// four times as long as one of 8 by 128 (out of L2 9.7 and 30 TB/s). W in that form is
// a third of the unit's time at the memory's rate, x as much for every tile of 16
// features and twice that for int8: with either straight in registers, several chunks
// ahead, 8 rows took (us, K 4096 unless said, before / now): gate and up 14336 bf16
// 41.5 / 35.0, int8 28.2 / 21.7; q, k, v 4096 + 2 x 1024 13.2 / 10.2 and 10.3 / 7.9; N
// 4096 9.6 / 7.3 and 7.9 / 5.9; N 4096, K 14336 26.3 / 19.5 and 18.5 / 13.5; N 128256 175
// / 152 and 92.4 / 81.2; N 3584, K 18944 31.9 / 23.6 and 23.1 / 16.5; 2048, K 2048 6.0 /
// 4.6 and 5.1 / 4.2. 1 row and 16: 4096 8.6 / 7.2 and 10.9 / 8.0, N 128256 162 / 149 and
// 183 / 153; int8 24 rows 4096, K 14336 31.0 / 21.3. A read of as many bytes alone takes
// 6.4 (4096), 9.0 (6144) and 35 (28672 of K 4096 bf16).
//   * W, which nobody else reads, passes the caches by: 3 to 12%.
//   * Rows past M and features past N lie past their descriptors or repeat the last.
//
// A workgroup's tiles are fixed at the launch: where another stream's kernel holds CUs
// and the workgroups are more than those left, some begin when the first others end.

// A stream's place in LDS: W, x, int8's scales of the rows of a slot.
template <bool I8, int XR, int S, int MODE>
struct Slot {
  static constexpr int XROW = I8 ? 256 : 128;       // bytes of x a row
  static constexpr int X = S * 2048, SC = X + XR * XROW;
  static constexpr int SCL = !I8 ? 0 : MODE == PLAIN ? 1 : 2;
  static constexpr int BYTES = SC + SCL * 256;
  static constexpr int XL = XR * XROW / 1024, LOADS = 2 * S + XL + SCL;
};

// XR: rows of x that are loaded, 8 or 16 MT; S: tiles of 16 features a wave, with
// SWIGLU half of them of the gate; D: slots of a wave's ring.
//
// QKV: half of the tiles lie 64 features behind the others, so that the threads that add
// a pair up turn it and write it where attention reads it. What that asks for (positions,
// rows of the pool, angles) is fetched before the weights are waited for. A launch and 3
// us a layer less: steps of four layers, one request of 500 532 -> 525 us, 8 of 16000 873
// -> 857, int8 8 of 1000, where the host is as long, 402 -> 381. q, k and v that are only
// wanted as they are have the same sums: by the same tiles or, where these leave half of
// the CUs idle, by PLAIN's of 16 features, whose workgroups begin alike (`heads`).
template <bool I8, int XR, int S, int NW, int D, int MODE>
__global__ __launch_bounds__(NW * 64) void stream_rows_kernel(const Args a,
                                                              const int tiles) {
  using P = Slot<I8, XR, S, MODE>;
  constexpr int MT = (XR + 15) / 16, L = MODE == PLAIN ? 1 : 2, FT = S / L;
  constexpr int IN = I8 ? 128 : 64;     // inputs a chunk, 128 bytes of W's rows
  constexpr int RING = D * P::BYTES;
  extern __shared__ __attribute__((aligned(16))) char lds[];
  float* const sums = (float*)(lds + NW * RING);

  const int lane = threadIdx.x & 63, wid = uni(threadIdx.x >> 6);
  const int col = lane & 15, g = lane >> 4;
  const int KB = a.K * (I8 ? 1 : 2), chunks = a.K / IN;
  const int n = (chunks - wid + NW - 1) / NW;       // wid, wid + NW, ..
  // Each workgroup begins elsewhere in its rows, over an XCD and over the XCDs: rows
  // that are multiples of 4 KB apart lie in few memory channels.
  const unsigned begin = MODE == PLAIN && a.heads ? blockIdx.x / 8 * 4 + blockIdx.x % 4
                                                  : blockIdx.x;
  const int turn = uni((begin / 8 * 13 + begin % 8 * 7) % 32 * chunks / 32);
  auto chunk = [&](int i) __attribute__((always_inline)) {
    const int c = wid + i * NW + turn;
    return uni(c < chunks ? c : c - chunks);
  };
  struct Place { int layer, n0; };
  auto locate = [&](int tile) __attribute__((always_inline)) {
    int l = 0;
    if (MODE != SWIGLU) {
      while (tile >= a.tile_end[l]) ++l;
      if (l) tile -= a.tile_end[l - 1];
    }
    return Place{uni(l), uni(tile * 16 * FT)};
  };
  // QKV: n0 counts in the halves of heads
  auto feature = [&](int n) __attribute__((always_inline)) {
    return MODE == QKV ? (n >> 6) * 128 + (n & 63) : n;
  };

  // ---- loads. 16-byte chunk c of a row lies at c ^ (row & 7), so that 16 rows are
  // read without bank conflicts.
  const unsigned w0 = (lane >> 3) * (unsigned)KB + (((lane & 7) ^ (lane >> 3)) << 4);
  const unsigned w1 = w0 + 8 * (unsigned)KB;
  unsigned x0[P::XL];
#pragma unroll
  for (int j = 0; j < P::XL; ++j) {
    const int r = I8 ? 4 * j + (lane >> 4) : 8 * j + (lane >> 3);
    x0[j] = r * (unsigned)a.K * 2 + ((I8 ? (lane & 15) ^ (r & 7)
                                         : (lane & 7) ^ (r & 7)) << 4);
  }
  const u32x4 xfrom = descriptor(a.x, (long long)a.M * a.K * 2);
  const int put = uni((int)(uintptr_t)(__attribute__((address_space(3))) char*)lds +
                      wid * RING);
  int next = blockIdx.x, next_i = 0, at = 0;    // tile and chunk that come next
  bool more = n > 0;
  Place to;
  u32x4 wfrom[S];
  auto aim = [&]() __attribute__((always_inline)) {
    to = locate(next);
#pragma unroll
    for (int s = 0; s < S; ++s) {   // a tile past the end is the last row's
      const int l = MODE == SWIGLU ? s / FT : to.layer;
      const int f = min(feature(to.n0 + 16 * (s % FT)) +
                        (MODE == QKV ? s / FT * 64 : 0), a.n[l] - 1);
      wfrom[s] = descriptor((const char*)a.w[l] + (long long)f * KB,
                            (long long)(a.n[l] - f) * KB);
    }
  };
  auto fill = [&]() __attribute__((always_inline)) {
    if (next_i == 0) aim();
    const int c = chunk(next_i), b = put + at;
#pragma unroll
    for (int s = 0; s < S; ++s) {
      load<true>(wfrom[s], w0, c * 128, b + s * 2048);
      load<true>(wfrom[s], w1, c * 128, b + s * 2048 + 1024);
    }
#pragma unroll
    for (int j = 0; j < P::XL; ++j)
      load<false>(xfrom, x0[j], c * P::XROW, b + P::X + j * 1024);
    if constexpr (I8) {
      // lane: row; the group of its chunk, both in 256s of inputs
      const int f = feature(to.n0 + (lane & (16 * FT - 1)));
#pragma unroll
      for (int l = 0; l < P::SCL; ++l) {
        const int r = min(f + (MODE == QKV ? 64 * l : 0), a.n[to.layer] - 1);
        const unsigned i = ((unsigned)r * (unsigned)(a.K / 256) + c / 2) /
            (unsigned)(a.group / 256);
        load_scales(a.scales[MODE == SWIGLU ? l : to.layer], i * 4,
                    b + P::SC + l * 256);
      }
    }
    at = at + P::BYTES == RING ? 0 : at + P::BYTES;
    if (++next_i == n) {
      next_i = 0;
      next += gridDim.x;
      more = next < tiles;
    }
  };
  // A thread adds up elements threadIdx.x + k NW 64 of a tile, of one row or MT.
  constexpr int E = (FT * MT * 256 + NW * 64 - 1) / (NW * 64);
  auto row_of = [&](int k) __attribute__((always_inline)) {
    return min((int)((threadIdx.x + k * NW * 64) % (MT * 256)) >> 4, a.M - 1);
  };
  const bool turned = MODE == QKV && a.to.dst != nullptr;
  int position[MT], row[MT];
  if (turned)
#pragma unroll
    for (int k = 0; k < MT && k < E; ++k) {
      const int r = row_of(k);
      position[k] = a.to.positions ? a.to.positions[r] : r % a.to.S;
      row[k] = a.to.dst[r];
    }
  int filled = 0;
#pragma unroll 1      // short layers wait for the kernel's instructions
  for (; more && filled < D; ++filled) fill();

  const char* const get = lds + wid * RING;
  const int o0 = (g ^ (col & 7)) << 4;
  const int xr = XR == 8 ? col & 7 : col;
  int from = 0;
  for (int tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
    float angle[E][2];
    if (turned) {
      const Place p = locate(tile);
      if (p.layer < 2)
#pragma unroll
        for (int k = 0; k < E; ++k) {
          const int e = threadIdx.x + k * NW * 64;
          const int j = (p.n0 + e / (MT * 256) * 16 + (e & 15)) & 63;
          const long long at = (long long)position[k % MT] * 64 + j;
          angle[k][0] = a.to.cs[at];
          angle[k][1] = a.to.sn[at];
        }
    }
    f32x4 acc[S][MT];
#pragma unroll
    for (int s = 0; s < S; ++s)
#pragma unroll
      for (int m = 0; m < MT; ++m) acc[s][m] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int i = 0; i < n; ++i) {
      if (filled == D) wait_loads<(D - 1) * P::LOADS>();
      else wait_loads<0>();
      const char* const b = get + from;
      // the lane's 16 inputs of an int8 row are two operands'
      constexpr int Q = I8 ? 4 : 2;
      u32x4 w[S][2];
      s16x8 x[MT][Q];
      f32x4 sc[S];
#pragma unroll
      for (int s = 0; s < S; ++s)
#pragma unroll
        for (int h = 0; h < 2; ++h)
          w[s][h] = *(const u32x4*)(b + s * 2048 + col * 128 + (o0 ^ (64 * h)));
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int q = 0; q < Q; ++q) {
          const int c = I8 ? (2 * g + 8 * (q >> 1) + (q & 1)) ^ (col & 7) : 0;
          x[m][q] = *(const s16x8*)(b + P::X + (16 * m + xr) * P::XROW +
                                    (I8 ? c << 4 : o0 ^ (64 * q)));
        }
      if (I8)     // of the rows 4 g + r that the lane holds the sums of
#pragma unroll
        for (int s = 0; s < S; ++s)
          sc[s] = *(const f32x4*)(b + P::SC + s / FT * 256 + s % FT * 64 + 16 * g);
      // what was in the slot is in registers
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
      if (more) fill();
      else --filled;
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int s = 0; s < S; ++s) {
        f32x4 part[MT];
#pragma unroll
        for (int m = 0; m < MT; ++m)
          part[m] = I8 ? f32x4{0.f, 0.f, 0.f, 0.f} : acc[s][m];
#pragma unroll
        for (int q = 0; q < Q; ++q) {
          u32x4 o = w[s][I8 ? q >> 1 : q];
          if constexpr (I8) {
            const unsigned lo = o[2 * (q & 1)], hi = o[2 * (q & 1) + 1];
            unsigned v[4];
            widen<true>(lo, v[0], v[1]);
            widen<true>(hi, v[2], v[3]);
            o = u32x4{v[0], v[1], v[2], v[3]};
          }
#pragma unroll
          for (int m = 0; m < MT; ++m)
            part[m] = mfma(__builtin_bit_cast(s16x8, o), x[m][q], part[m]);
        }
#pragma unroll
        for (int m = 0; m < MT; ++m)
          if (I8)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[s][m][r] += part[m][r] * sc[s][r];
          else
            acc[s][m] = part[m];
      }
      from = from + P::BYTES == RING ? 0 : from + P::BYTES;
    }

    // ---- add the waves up; features 4 g + r of a column lie side by side
    if (tile != blockIdx.x) barrier();      // the last tile's are read
#pragma unroll
    for (int s = 0; s < S; ++s)
#pragma unroll
      for (int m = 0; m < MT; ++m)
        *(f32x4*)(sums + ((wid * S + s) * MT + m) * 256 + col * 16 + 4 * g) =
            acc[s][m];
    barrier();
    const Place p = locate(tile);
    const int N = a.n[p.layer];
#pragma unroll
    for (int k = 0; k < E; ++k) {
      const int e = threadIdx.x + k * NW * 64;
      const int f = e / (MT * 256), o_ = e % (MT * 256);
      const int r = o_ >> 4, c = feature(p.n0 + 16 * f + (o_ & 15));
      if (e >= FT * MT * 256 || r >= a.M || c >= N) continue;
      float y[L];
#pragma unroll
      for (int l = 0; l < L; ++l) {
        float t = 0.f;
#pragma unroll
        for (int w_ = 0; w_ < NW; ++w_)
          t += sums[(w_ * S + l * FT + f) * MT * 256 + o_];
        if (MODE == QKV) {
          if (a.bias[p.layer]) t += value(a.bias[p.layer][c + 64 * l]);
        } else if (a.bias[p.layer + l]) {
          t += value(a.bias[p.layer + l][c]);
        }
        y[l] = t;
      }
      if constexpr (MODE == QKV) {
        short* to = a.out[p.layer] + (long long)r * N + c;
        short lo = bits(y[0]), hi = bits(y[1]);
        if (turned && p.layer < 2) {
          const ds::Turned t =
              ds::turn(value(lo), value(hi), angle[k][0], angle[k][1]);
          lo = bits(t.lo);
          hi = bits(t.hi);
        }
        if (turned && p.layer) {
          const int at = row[k % MT];
          to = (p.layer == 1 ? a.to.kpool : a.to.vpool) + c % 128 +
              (((long long)(at / a.to.BS) * a.to.heads + c / 128) * a.to.BS +
               at % a.to.BS) * 128;
        }
        to[0] = lo;
        to[64] = hi;
      } else {
        float o = y[0];
        if (MODE == SWIGLU) o = y[0] / (1.f + expf(-y[0])) * y[L - 1];
        a.out[p.layer][(long long)r * N + c] = bits(o);
      }
    }
  }
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

// ALL: a workgroup a tile; otherwise as many as the CUs hold at a time, evenly.
template <bool I8, int XR, int S, int NW, int D, int MODE>
int launch_stream(Args a, int layers, bool all, hipStream_t st) {
  constexpr int MT = (XR + 15) / 16, FT = MODE == PLAIN ? S : S / 2;
  constexpr int LDS = NW * (D * Slot<I8, XR, S, MODE>::BYTES + S * MT * 1024);
  static_assert(LDS <= 160 * 1024 && (!I8 || 16 * FT <= 64), "");
  constexpr int CUS = 256, HELD = CUS * (160 * 1024 / LDS);
  int tiles = 0;
  for (int i = 0; i < (MODE == SWIGLU ? 1 : layers); ++i)
    a.tile_end[i] = tiles +=
        (a.n[i] / (MODE == QKV ? 2 : 1) + 16 * FT - 1) / (16 * FT);
  const int rounds = all ? 1 : (tiles + HELD - 1) / HELD;
  auto kernel = stream_rows_kernel<I8, XR, S, NW, D, MODE>;
  const hipError_t e = hipFuncSetAttribute(
      (const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
  if (e != hipSuccess) return (int)e;
  hipLaunchKernelGGL(kernel, dim3((tiles + rounds - 1) / rounds), dim3(NW * 64),
                     LDS, st, a, tiles);
  return (int)hipGetLastError();
}

// Tiles a wave and waves by the layer's tiles of 16 features. us at 1, 8 and 16 rows,
// S x waves, bf16 unless said:
//   * A round of the CUs: one tile, so that all of them have work (256 tiles, K 4096:
// 1 x 8 7.2, 7.3, 8.0, 2 x 8 8.4, 9.2, 10.0). Two up to two rounds (384, K 4096: 9.9,
// 10.2, 10.8 and one 10.3, 11.2, 12.8; 512, K 28672: 69.8, 70.6, 74.3 and 69.2, 72.9,
// 84.8; int8 384: 7.5, 7.9, 8.8 and 7.9, 8.4; by four waves 8.1, 8.1, 8.5).
//   * More: x, which is read for each tile, is a third and half of what arrives at one
// tile a wave of up to 8 and 16 rows, a ninth and a fifth at four. But one tile, for
// which two workgroups fit a CU, evens out (576 tiles, K 3072: 11.8, 12.4, 14.4, four
// 12.7, 13.3, 14.1; 2004: 30.0, 30.4, 34 and 31.1, 30.9, 31.3; 8016, K 4096: 149, 152,
// 158 and 151, 151, 153); short ones go on from tile to tile (2000, K 1024 12.0 and
// 12.1, a workgroup a tile 13.2). int8 by four waves, whose tiles end half as often
// (2 x 4 / 4 x 4: 8016 78.6, 82.9, 97 / 79.6, 81.2, 87.7; 2004, K 3072 18.3, 18.9, 21.8 /
// 19.1, 19.2, 20.9; 2000, K 1024 8.9, 9.4, 10.3 / 10.0, 10.1, 10.9; one tile: 576 9.0, 9.7,
// 12.2, four 9.5, 9.9, 10.8; 1024 13.6 and two 13.4).
//   * Gate and up, one pair: 896 pairs, K 4096 2 x 4 35.2, 35.0, 36.7, 4 x 4 35.7, 35.8,
// 35.8; 352, K 2048 9.3, 9.9, 10.9 and 9.4, 9.7, 10.2; int8 21.2, 22.4, 25.5 and 21.4,
// 21.7, 23.6; 176, K 1024 2 x 8 4.3, 4.5, 4.7, 2 x 4 4.6, 4.7, 4.9.
//   * q, k and v, two or four: 384 tiles, K 4096 2 x 8 10.9, 10.8, 11.4, 4 x 4 14.7, 15.3,
// 16.2, int8 8.7, 8.8, 9.4 and 13.1, 13.4, 14.7; 640, K 8192 29.0, 30.9, 33.4 and 28.2,
// 28.6, 30.0; 768, K 4096 18.1, 18.9, 20.1 and 19.3, 19.5, 19.8; int8 of 640 2 x 8 / 2 x 4
// / 4 x 4 20.4, 22.7, 26.1 / 20.5, 22.2, 25.7 / 21.3, 22.0, 23.6, of 576, K 3072 11.1,
// 11.7, 13.1 / 10.8, 11.1, 12.3 / 11.7, 12.0, 12.9.
//   * 17 to 32 rows of int8: 256 tiles, K 4096 1 x 4 8.8, 2 x 4 10.6; 384 14.7 and 11.0.
template <bool I8, int XR>
int launch_streams(const Args& a, int layers, int mode, int tiles,
                   hipStream_t st) {
#define STREAM(S, NW, D, MODE, ALL) \
  return launch_stream<I8, XR, S, NW, D, MODE>(a, layers, ALL, st)
  const bool few = a.M <= (I8 ? 4 : 8);
  if constexpr (XR == 32) {
    if constexpr (I8) {
      if (mode == SWIGLU) STREAM(2, 4, 2, SWIGLU, false);
      if (mode == QKV) STREAM(2, 4, 2, QKV, false);
      if (tiles <= 256) STREAM(1, 4, 3, PLAIN, false);
      STREAM(2, 4, 2, PLAIN, false);
    } else {
      if (mode == SWIGLU) STREAM(2, 8, 2, SWIGLU, false);
      if (mode == QKV) STREAM(2, 8, 2, QKV, false);
      if (tiles <= 256) STREAM(1, 8, 2, PLAIN, false);
      STREAM(2, 8, 2, PLAIN, false);
    }
  } else if (mode == SWIGLU) {
    if constexpr (I8) {
      if (few || tiles <= 512) STREAM(2, 4, 2, SWIGLU, false);
    } else {
      if (tiles <= 512) STREAM(2, 8, 2, SWIGLU, false);
      if (few) STREAM(2, 4, 4, SWIGLU, false);
    }
    STREAM(4, 4, 2, SWIGLU, false);
  } else if (mode == QKV) {
    if (tiles <= 512 || (!I8 && a.M <= 4)) STREAM(2, 8, 2, QKV, false);
    if (I8 && a.M <= 8) STREAM(2, 4, 2, QKV, false);
    STREAM(4, 4, 2, QKV, false);
  } else {
    if (tiles <= 256) STREAM(1, 8, 2, PLAIN, false);
    if constexpr (I8) {
      if (tiles <= 512) {
        if (a.M <= 8) STREAM(2, 8, 2, PLAIN, false);
        STREAM(2, 4, 2, PLAIN, false);
      }
      if (few && tiles < 1024 && a.K >= 3072) STREAM(1, 8, 2, PLAIN, true);
      if (few || a.K < 2048) STREAM(2, 4, 2, PLAIN, false);
    } else {
      if (tiles <= 512) STREAM(2, 8, 2, PLAIN, false);
      if (few) STREAM(1, 8, 2, PLAIN, a.K >= 3072);
    }
    STREAM(4, 4, 2, PLAIN, false);
  }
#undef STREAM
}

// Queries, keys and values, or what has their form.
bool in_heads(const Args& a, int layers) {
  return layers == 3 && a.n[0] % 128 == 0 && a.n[1] % 128 == 0 &&
      a.n[2] % 128 == 0;
}

// Layers of less than a round of tiles whose contraction is a load or two a wave, to
// rows_linear_kernel: straight to registers is a hop less, and less code to fetch. us of
// the stream / so: bf16 K 256, N 2048 8 and 16 rows 3.16 / 2.89, 3.19 / 2.95, but 24 rows
// of N 1024 2.96 / 3.28, and K 512, N 256 2.82 / 3.13; int8 K 256 2.75 to 3.40 / 2.83 to
// 3.00, K 512, N 1024 1, 16 and 24 rows 3.39 / 3.04, 3.54 / 3.15, 3.77 / 3.71, but 32 rows
// 3.77 / 3.89, a whole round of tiles at 16 3.67 / 3.88, and K 768, N 2048 3.59 / 3.77.
// Not what has the form of q, k and v: its sums are those of the products that append.
template <bool I8>
bool brief(const Args& a, int layers, int mode, int tiles) {
  if (mode != PLAIN || tiles >= 256 || in_heads(a, layers)) return false;
  return I8 ? a.K <= (a.M <= 24 ? 512 : 256) : a.M <= 16 && a.K <= 256;
}

// What stream_rows_kernel takes: a lane's offsets in a tile and int8's places of scales
// are 32 bits, and x, which each workgroup reads at another place, stays in an XCD's
// L2. Of 17 to 32 rows int8 but for short gates (2 x 5632, K 2048 32 rows 12.8, by
// rows_linear_kernel 12.2), bf16 as ds_rows_linear is given them.
template <bool I8>
bool streams(const Args& a, int layers, int mode, int tiles) {
  if (brief<I8>(a, layers, mode, tiles)) return false;
  if (a.M > 32 || a.K > 1 << 22) return false;
  if (I8)
    for (int i = 0; i < layers; ++i)
      if ((long long)a.n[i] * a.K >= 1ll << 38) return false;
  return a.M <= 16 || !I8 || mode == PLAIN || tiles <= 512 || a.K > 2048;
}

// Tiles of features a wave of rows_linear_kernel. Every workgroup reads all of x, which
// costs M rows out of L2 for 16 FT features of W; half the workgroups leave CUs idle
// where the layer is small (int8 of 64 rows, us, FT 1 / 2: N 4096 21.1 / 23.8, N 14336 74
// / 46; gate and up 88 / 67, 32 rows 53.8 / 42.6). Up to 32 rows only what the streams
// do not take comes here: brief layers, gates of few inputs, more than 2^22 of them.
template <bool I8>
int launch_rows(Args a, int layers, int mode, hipStream_t st) {
  int tiles = 0;
  for (int i = 0; i < layers; ++i) tiles += (a.n[i] + 15) / 16;
  if (streams<I8>(a, layers, mode, tiles)) {
    // Up to 256 tiles a workgroup has one, by either. us by pairs of tiles, and one:
    // bf16 1664 + 2 x 1024, K 5120, 2 rows 13.2 / 8.8, 3 x 896, K 3584, 12 rows 9.5 / 7.9,
    // 768 + 2 x 128, K 256, 2 rows 3.6 / 3.2; int8 640 + 2 x 1408, K 8192, 2 rows 12.4 /
    // 8.7, 128 + 2 x 640, K 6656, 32 rows 16.3 / 12.0; 0.83 over 35 layers.
    if (mode == PLAIN && in_heads(a, layers)) {
      if (a.to.dst || tiles > 256) mode = QKV;
      else a.heads = true;
    }
    if (a.M <= 8) return launch_streams<I8, 8>(a, layers, mode, tiles, st);
    if (a.M <= 16) return launch_streams<I8, 16>(a, layers, mode, tiles, st);
    return launch_streams<I8, 32>(a, layers, mode, tiles, st);
  }
  if (mode == SWIGLU) {
    if (a.M <= 32) return launch<I8, 2, SWIGLU, 2>(a, layers, st);
    return launch<true, 4, SWIGLU, 2>(a, layers, st);
  }
  if (a.M <= 16) return launch<I8, 1, PLAIN, 1>(a, layers, st);
  if (a.M <= 32) return launch<I8, 2, PLAIN, 1>(a, layers, st);
  if (tiles >= 384) return launch<true, 4, PLAIN, 2>(a, layers, st);
  return launch<true, 4, PLAIN, 1>(a, layers, st);
}

Args arguments(const void* x, int layers, const void* const* w,
               const float* const* scales, const void* const* bias,
               void* const* out, const int* n, int M, int K, int group) {
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
  return a;
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
  const Args a = arguments(x, layers, w, scales, bias, out, n, M, K, group);
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  return scales ? launch_rows<true>(a, layers, mode, st)
                : launch_rows<false>(a, layers, mode, st);
}

// q [M, H, 128] turned and k and v into the paged pool, as the layers and then
// ds_paged_append would have it bit by bit: one launch for two. -1: not these.
extern "C" int ds_rows_append(const void* x, const void* const* w,
                              const float* const* scales,
                              const void* const* bias, void* q, const int* n,
                              int M, int K, int group, void* kpool,
                              void* vpool, const int* dst, const float* cs,
                              const float* sn, const int* positions, int S,
                              int BS, void* stream) {
  void* const out[] = {q, nullptr, nullptr};
  Args a = arguments(x, 3, w, scales, bias, out, n, M, K, group);
  const int tiles = (n[0] + n[1] + n[2]) / 16;
  if (!in_heads(a, 3) || !(scales ? streams<true>(a, 3, PLAIN, tiles)
                                  : streams<false>(a, 3, PLAIN, tiles)))
    return -1;
  a.to = {cs, sn, positions, dst, (short*)kpool, (short*)vpool, S, n[1] / 128,
          BS};
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  return scales ? launch_rows<true>(a, 3, PLAIN, st)
                : launch_rows<false>(a, 3, PLAIN, st);
}
