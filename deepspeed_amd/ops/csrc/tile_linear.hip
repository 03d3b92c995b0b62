// Linear layers of many rows for MI355X (gfx950): y = x W^T, x [M, K] bf16,
// W [N, K] bf16, M past what rows_linear.hip takes: decoding for many requests,
// portions of prompts, whole prompts; and both gradients of training.
//
// Reference analogue: the GEMMs of inference/v2/kernels/core_ops/blas_kernels
// and the gated ones of core_ops/gated_activations.
//
// A workgroup owns a tile of BM rows by BN features. Stages of 64 inputs of
// both go from memory straight into a ring of NS buffers in LDS
// (global_load_lds, 16 bytes a lane; 16-byte chunk c of a row lies at
// c ^ (row & 7), which the lanes' addresses bring about, since a wave's load
// fills 1 KB of LDS in lane order: no bank conflicts counted). Operands of the
// products are read into registers one phase ahead. A stage's inputs take four
// phases: the first half of the wave's rows over inputs 0-31 and 32-63, then
// the second half; so W and the first half of x are read out after a quarter of
// the stage, their buffer is loaded anew from there on, and loads have one and
// a half stages to arrive in with only two buffers.
//
//   * Loads are spread between the products, two in a phase of 16: a burst of
//     them stalls its wave behind the address units, and the products after it
//     wait (8192 x 8192 x 8192: 805 us with the loads at once, 747 spread;
//     without loads 655, loads alone 650; the library's product 690 to 750).
//   * Several layers on one input (q, k, v) are one launch, so that narrow ones
//     fill the chip together; with SWIGLU a tile holds gate and up, 16 features
//     of each in turn, and the activation is taken from the fp32 sums.
//   * Where tiles leave CUs idle, the contraction is split; partial sums stay
//     fp32 and are added in their order by a second kernel, or by the next one.

#include "ds_kernels.h"

#include <cmath>
#include <utility>

#pragma clang diagnostic ignored "-Winline-asm"     // m0 among the clobbers

namespace {

typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 b16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

constexpr int MAXL = 3;     // layers a launch
constexpr int BK = 64;      // inputs a stage
constexpr int ROW = BK * 2; // bytes of a row of a stage

// on lambdas: one that is not inlined takes what it captures to scratch memory
#define INLINE __attribute__((always_inline))

// y = x W^T, silu(x W0^T) * (x W1^T), and of y = x W^T the gradients of x, a sum
// over the layers, and of each W.
enum { PLAIN = 0, SWIGLU = 1, GRAD_X = 2, GRAD_W = 3 };

// Operands by their place in the kernel: "w" brings the columns of an output,
// "x" its rows. GRAD_X: w are the weights [n, K], x the gradients dy [M, n], and
// the contraction runs over the features of one layer after the other. GRAD_W: w
// is the layers' input [M, K], x the gradients, contracted over M.
struct Args {
  const short* w[MAXL];
  const short* x[MAXL];
  const short* bias[MAXL];
  short* out[MAXL];
  int n[MAXL];          // features
  int n_end[MAXL];      // up to and with a layer: features,
  int tile_end[MAXL];   // tiles of the outputs' columns, or GRAD_W of its rows,
  int step_end[MAXL];   // and GRAD_X: stages
  float* part;          // [splits, rows, columns] of all outputs, splits > 1
  int M, K, layers, tiles, mtiles, splits, steps;
  bool turn;            // each workgroup begins elsewhere in its contraction
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
__device__ __forceinline__ s16x4 packed(f32x4 y) {
  return s16x4{bits(y[0]), bits(y[1]), bits(y[2]), bits(y[3])};
}

__device__ __forceinline__ int uni(int x) {
  return __builtin_amdgcn_readfirstlane(x);
}
__device__ __forceinline__ const char* uni(const char* p) {
  const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)(uintptr_t)p);
  const unsigned hi =
      __builtin_amdgcn_readfirstlane((unsigned)((uintptr_t)p >> 32));
  return (const char*)(((uintptr_t)hi << 32) | lo);
}

// 16 bytes a lane from base + off to LDS, lane after lane from `lds` on. Not the
// builtin: behind that the compiler waits for all loads before it reads LDS. ONCE:
// read by nobody else, past the caches.
template <bool ONCE>
__device__ __forceinline__ void load_lds(const char* base, unsigned off,
                                         int lds) {
  if (ONCE)
    asm volatile("s_mov_b32 m0, %2\n\t"
                 "s_nop 0\n\t"
                 "global_load_lds_dwordx4 %0, %1 nt"
                 :: "v"(off), "s"(uni(base)), "s"(uni(lds)) : "memory", "m0");
  else
    asm volatile("s_mov_b32 m0, %2\n\t"
                 "s_nop 0\n\t"
                 "global_load_lds_dwordx4 %0, %1"
                 :: "v"(off), "s"(uni(base)), "s"(uni(lds)) : "memory", "m0");
}
template <int N>
__device__ __forceinline__ void wait_loads() {  // but for the N youngest
  static_assert(N < 64, "vmcnt has six bits");
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
__device__ __forceinline__ void barrier() {   // and what was read from LDS
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

__device__ __forceinline__ s16x4 tr_read(const char* p) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (__attribute__((address_space(3))) s16x4*)p);
}

// MT products with NR reads from LDS in their first half and ND loads spread
// over all of them.
template <int MT, int NR, int ND, typename Mul, typename Read, typename Load>
__device__ __forceinline__ void phase(Mul mul, Read read, Load load) {
  constexpr int HALF = MT / 2 > 0 ? MT / 2 : 1;
#pragma unroll
  for (int i = 0; i < MT; ++i) {
#pragma unroll
    for (int q = 0; q < NR; ++q)
      if (q * HALF / (NR > 0 ? NR : 1) == i) {
        read(q);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
    for (int q = 0; q < ND; ++q)
      if ((2 * q + 1) * MT / (ND > 0 ? 2 * ND : 1) == i) {
        load(q);
        __builtin_amdgcn_sched_barrier(0);
      }
    mul(i);
  }
  __builtin_amdgcn_sched_barrier(0);
}

// By value: choosing among a lambda's captures would keep them in memory.
template <typename T>
__device__ __forceinline__ T pick(int i, T a, T b, T c) {
  return i == 2 ? c : i == 1 ? b : a;
}

template <int I>
struct Int {
  static constexpr int value = I;
};
template <int R, typename F>
__device__ __forceinline__ void last_steps(F& step, int it, int buf) {
  buf = step(Int<R>{}, it, buf);
  if constexpr (R > 0) last_steps<R - 1>(step, it + 1, buf);
}

// ONCE: each of W is one workgroup's.
template <int BM, int BN, int WM, int WN, int NS, int MODE, bool ONCE>
__global__ __launch_bounds__(WM* WN * 64, WM * WN / 4) void tile_linear_kernel(
    const Args a) {
  constexpr bool GLU = MODE == SWIGLU;
  // operands that lie across the contraction
  constexpr bool WT = MODE == GRAD_X || MODE == GRAD_W, XT = MODE == GRAD_W;
  constexpr int NW = WM * WN;
  // 16-row tiles of a wave: features, rows of x, the halves of these
  constexpr int FN = BN / WN / 16, FM = BM / WM / 16;
  constexpr int H0 = FM / 2, H1 = FM - H0;
  constexpr int C0 = H0 * 16, C1 = H1 * 16;
  // A stage in LDS: W, the first halves of all waves' rows of x, the second
  constexpr int X0 = C0 * WM, X1 = C1 * WM;
  constexpr int AT_X0 = BN * ROW, AT_X1 = AT_X0 + X0 * ROW;
  constexpr int STAGE = (BN + BM) * ROW;
  // loads of 1 KB a wave: of W, of the first halves, of the second ones
  constexpr int PW = BN / 8 / NW, P0 = X0 / 8 / NW, P1 = X1 / 8 / NW;
  static_assert(PW * NW * 8 == BN && P0 * NW * 8 == X0 && P1 * NW * 8 == X1 &&
                H0 > 0 && NW % 4 == 0 && (!GLU || FN % 2 == 0) &&
                (!XT || (X0 % 64 == 0 && X1 % 64 == 0)), "");
  constexpr int PA = PW + P0, P = PA + P1;
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int lane = threadIdx.x & 63;
  const int wid = uni(threadIdx.x >> 6);
  const int col = lane & 15, g = lane >> 4;
  const int wm = wid / WN, wn = wid % WN;

  // Consecutive workgroups go to the 8 XCDs in turn: each XCD takes a run of
  // tiles, rows first in groups of 4 or 8, so that its L2 serves W and x to many
  // (8192 x 8192 x 8192: groups of 1 1149 us, 2 858, 4 824, 8 844, 32 1024).
  constexpr int GROUP = BM >= 192 ? 4 : 8;
  const int per = a.tiles * a.mtiles, total = per * a.splits;
  int id = blockIdx.x;
  {
    const int q = total / 8, r = total % 8, xcd = id % 8;
    id = xcd * q + min(xcd, r) + id / 8;
  }
  const int split = uni(id / per);
  id -= split * per;
  const int group = id / (GROUP * a.tiles);
  const int high = min(GROUP, a.mtiles - GROUP * group);
  id -= group * GROUP * a.tiles;
  int mt = uni(GROUP * group + id % high);
  int nt = uni(id / high);
  int layer = 0;
  if (MODE == PLAIN) {
    while (nt >= a.tile_end[layer]) ++layer;
    if (layer) nt -= a.tile_end[layer - 1];
  }
  if (MODE == GRAD_W) {
    while (mt >= a.tile_end[layer]) ++layer;
    if (layer) mt -= a.tile_end[layer - 1];
  }
  // rows and columns of the output, its tile's first ones
  const int K = a.K, N = WT ? K : a.n[layer];
  const int rows = MODE == GRAD_W ? a.n[layer] : a.M;
  const int n0 = nt * (GLU ? BN / 2 : BN), m0 = mt * BM;
  const int steps = MODE == GRAD_X ? a.steps
      : MODE == GRAD_W ? (a.M + BK - 1) / BK : K / BK;
  const int s0 = uni(split * steps / a.splits);
  const int n_it = uni((split + 1) * steps / a.splits) - s0;    // NS or more
  const int turn = MODE > SWIGLU || !a.turn ? 0
      : uni((blockIdx.x / 8 * 13 + blockIdx.x % 8 * 7) % 32 * n_it / 32);

  // The lane's place in each load, which fills 1 KB: 8 rows of 64 inputs, or
  // 8 inputs of 64 columns. Rows and columns past the end repeat the last ones;
  // what comes of them is not stored.
  //   Along the contraction: chunk c of row r lies at c ^ (r & 7).
  //   Across it: blocks of 64 columns, [64 inputs][8 chunks], chunk c of input k
  // at c ^ (2 bit 1 of k + 4 bit 3): a transposing read takes 4 inputs by 32
  // bytes from each of four groups of 8 inputs, half of which share no bank.
  unsigned off[P];
  const int lr = lane >> 3, lc = lane & 7;
#pragma unroll
  for (int j = 0; j < P; ++j) {
    const bool of_w = j < PW;
    const int piece = (of_w ? j : j < PA ? j - PW : j - PA) * NW + wid;
    const bool t = of_w ? WT : XT;
    const int h = 2 * ((lr >> 1) & 1) + 4 * (piece & 1);
    int r = t ? piece / 8 * 64 + 8 * (lc ^ h) : piece * 8 + lr;
    if (!of_w) {
      const int c = j < PA ? C0 : C1;
      r = r / c * (BM / WM) + r % c + (j < PA ? 0 : C0);
    } else if (GLU) {
      r = (r >> 5) * 16 + (r & 15);
    }
    const int last = (of_w ? N - n0 : rows - m0) - (t ? 8 : 1);
    r = min(r, last);
    if (t) off[j] = 2 * r;
    else if (MODE == GRAD_X) off[j] = r;    // its layer's stride comes later
    else off[j] = (unsigned)r * K * 2 + ((lc ^ lr) << 4);
  }
  const short* w = GLU ? (wid & 2 ? a.w[1] : a.w[0]) : a.w[MODE == PLAIN ? layer : 0];
  const char* wb = uni((const char*)(w + (WT ? n0 : (long long)n0 * K)));
  const char* xb = uni((const char*)(
      a.x[MODE == GRAD_W ? layer : 0] +
      (XT ? m0 : MODE == GRAD_X ? 0 : (long long)m0 * K)));
  const int lds0 =
      (int)(uintptr_t)(__attribute__((address_space(3))) char*)lds + wid * 1024;
  // GRAD_X: where the layers begin and what is theirs
  const int e0 = a.layers > 1 ? a.step_end[0] : 1 << 30;
  const int e1 = a.layers > 2 ? a.step_end[1] : 1 << 30;
  const int f0 = a.n[0], f1 = a.n[1], f2 = a.n[2];
  const short *w0 = a.w[0], *w1 = a.w[1], *w2 = a.w[2];
  const short *d0 = a.x[0], *d1 = a.x[1], *d2 = a.x[2];
  // load j of a stage: W, the first halves (A, j < PA), the second ones
  auto fetch = [&](int it, int buf, int j) INLINE {
    const int at = j < PW ? j * NW * 1024 : j < PA
        ? AT_X0 + (j - PW) * NW * 1024 : AT_X1 + (j - PA) * NW * 1024;
    const bool t = j < PW ? WT : XT;
    const char* p = j < PW ? wb : xb;
    unsigned o = off[j];
    int step = s0 + it, ld = j < PW ? K : rows;
    if (MODE <= SWIGLU) step += it + turn < n_it ? turn : turn - n_it;
    if (MODE == GRAD_X) {
      const int l = (step >= e0) + (step >= e1);
      step -= pick(l, 0, e0, e1);
      if (j < PW) {
        p = (const char*)(pick(l, w0, w1, w2) + n0);
      } else {
        ld = pick(l, f0, f1, f2);
        p = (const char*)(pick(l, d0, d1, d2) + (long long)m0 * ld);
      }
    }
    if (t) {
      int k = ((j < PW ? j : j < PA ? j - PW : j - PA) * NW + wid) % 8 * 8 + lr;
      if (MODE == GRAD_W) k = min(k, a.M - 1 - step * BK);
      p += (long long)step * BK * ld * 2;
      o += (unsigned)k * ld * 2;
    } else {
      if (MODE == GRAD_X) o = o * ld * 2 + ((lc ^ lr) << 4);
      p += (long long)step * ROW;
    }
    if (ONCE && j < PW) load_lds<true>(p, o, lds0 + buf + at);
    else load_lds<false>(p, o, lds0 + buf + at);
  };

  f32x4 acc[FN][FM];
#pragma unroll
  for (int f = 0; f < FN; ++f)
#pragma unroll
    for (int m = 0; m < FM; ++m) acc[f][m] = f32x4{0.f, 0.f, 0.f, 0.f};

#pragma unroll
  for (int i = 0; i < NS; ++i)
#pragma unroll
    for (int j = 0; j < (i < NS - 1 ? P : PA); ++j) fetch(i, i * STAGE, j);
  wait_loads<(NS - 1) * P>();
  barrier();

  // 16 rows (or columns) by the inputs 32 h + 8 g + j, from tile i of a part of
  // a stage on
  const int o0 = (g ^ (col & 7)) << 4, o1 = o0 ^ 64;
  const int tr0 = (8 * g + (col >> 2)) * 128 + (col & 3) * 8;
  const int trh = 32 * ((col >> 3) & 1) + 64 * (g & 1);
  auto read = [&](auto across, int part, int first, int i, int h) INLINE {
    if constexpr (decltype(across)::value) {
      const int c = first / 16 + i;
      const char* p = lds + part + c / 4 * 8192 + h * 4096 +
          (tr0 ^ trh ^ (c % 4 * 32));
      const s16x4 lo = tr_read(p), hi = tr_read(p + 512);
      return s16x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    } else {
      return *(const s16x8*)(lds + part + (first + col) * ROW +
                             (h ? o1 : o0) + i * 16 * ROW);
    }
  };
  const Int<WT> wt;
  const Int<XT> xt;
  s16x8 wa[2][FN], x0[2][H0], x1[2][H1];
  auto get_w = [&](int buf, int i, int h) INLINE {
    wa[h][i] = read(wt, buf, wn * (BN / WN), i, h);
  };
  auto get_x0 = [&](int buf, int i, int h) INLINE {
    x0[h][i] = read(xt, buf + AT_X0, wm * C0, i, h);
  };
  auto get_x1 = [&](int buf, int i, int h) INLINE {
    x1[h][i] = read(xt, buf + AT_X1, wm * C1, i, h);
  };
  // GRAD_W: inputs past the last one (of the last stage) count for nothing
  const int beyond = MODE == GRAD_W && split == a.splits - 1
      ? a.M - (steps - 1) * BK : BK;
  auto cut = [&](s16x8& v, int h) INLINE {
    u32x4 d = __builtin_bit_cast(u32x4, v);
    const int left = beyond - 32 * h - 8 * g;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      d[e] &= left > 2 * e + 1 ? ~0u : left > 2 * e ? 0xffffu : 0u;
    v = __builtin_bit_cast(s16x8, d);
  };
#pragma unroll
  for (int f = 0; f < FN; ++f) get_w(0, f, 0);
#pragma unroll
  for (int m = 0; m < H0; ++m) get_x0(0, m, 0);

  // Loads of A of stage it + NS in three parts behind the stage's first barrier
  // (by then all waves have read A), those of the second halves of it - 1 + NS
  // before it. R: stages left after this one, NS for "at least NS".
  constexpr int A1 = (PA + 2) / 3, A2 = A1 + (PA - A1 + 1) / 2;
  auto step = [&](auto left, int it, int buf) INLINE {
    constexpr int R = decltype(left)::value;
    auto cut_last = [&](auto& of_w, int nw, auto& of_x, int nx,
                        int h) INLINE {
      if constexpr (MODE == GRAD_W && R == 0) {
        for (int i = 0; i < nw; ++i) cut(of_w[i], h);
        for (int i = 0; i < nx; ++i) cut(of_x[i], h);
      }
    };
    const int prev = buf == 0 ? (NS - 1) * STAGE : buf - STAGE;
    const int next = buf == (NS - 1) * STAGE ? 0 : buf + STAGE;
    cut_last(wa[0], FN, x0[0], H0, 0);
    phase<H0 * FN, FN + H0, (R >= NS - 1 ? P1 : 0)>(
        [&](int i) INLINE {
          acc[i % FN][i / FN] =
              mfma(wa[0][i % FN], x0[0][i / FN], acc[i % FN][i / FN]);
        },
        [&](int q) INLINE {
          if (q < FN) get_w(buf, q, 1);
          else get_x0(buf, q - FN, 1);
        },
        [&](int q) INLINE { fetch(it - 1 + NS, prev, PA + q); });
    // the second halves of this stage have arrived
    wait_loads<(R < NS - 1 ? R : NS - 1) * P>();
    barrier();
    cut_last(wa[1], FN, x0[1], H0, 1);
    phase<H0 * FN, H1, (R >= NS ? A1 : 0)>(
        [&](int i) INLINE {
          acc[i % FN][i / FN] =
              mfma(wa[1][i % FN], x0[1][i / FN], acc[i % FN][i / FN]);
        },
        [&](int q) INLINE { get_x1(buf, q, 0); },
        [&](int q) INLINE { fetch(it + NS, buf, q); });
    cut_last(wa[0], 0, x1[0], H1, 0);
    phase<H1 * FN, H1, (R >= NS ? A2 - A1 : 0)>(
        [&](int i) INLINE {
          acc[i % FN][i / FN + H0] =
              mfma(wa[0][i % FN], x1[0][i / FN], acc[i % FN][i / FN + H0]);
        },
        [&](int q) INLINE { get_x1(buf, q, 1); },
        [&](int q) INLINE { fetch(it + NS, buf, A1 + q); });
    // A of the next stage has arrived
    if constexpr (R >= NS) wait_loads<(NS - 2) * P + P1 + A2>();
    else if constexpr (R > 0) wait_loads<(R - 1) * P + P1>();
    barrier();
    cut_last(wa[1], 0, x1[1], H1, 1);
    phase<H1 * FN, (R > 0 ? FN + H0 : 0), (R >= NS ? PA - A2 : 0)>(
        [&](int i) INLINE {
          acc[i % FN][i / FN + H0] =
              mfma(wa[1][i % FN], x1[1][i / FN], acc[i % FN][i / FN + H0]);
        },
        [&](int q) INLINE {
          if (q < FN) get_w(next, q, 0);
          else get_x0(next, q - FN, 0);
        },
        [&](int q) INLINE { fetch(it + NS, buf, A2 + q); });
    return next;
  };
  int it = 0, buf = 0;
  for (; it + NS < n_it; ++it) buf = step(Int<NS>{}, it, buf);
  last_steps<NS - 1>(step, it, buf);

  // lane: row col of a tile of x, features 4 g + r of a tile of W
  if constexpr (!GLU && BN >= 192) {
    // Through LDS, so that whole lines are stored (8192 x 8192 x 4096: 10 us
    // less; narrower tiles gain nothing).
    if (a.splits == 1 && N % 8 == 0) {
      constexpr int RB = BN * 2 + 16;               // bytes a row
      constexpr int PASS = (BM * RB + NS * STAGE - 1) / (NS * STAGE);
      constexpr int MP = (FM + PASS - 1) / PASS;    // tiles of a wave a pass
      constexpr int VPR = BN / 8;                   // vectors a row
      static_assert(WM * MP * 16 * RB <= NS * STAGE, "");
#pragma unroll
      for (int p = 0; p < PASS; ++p) {
        barrier();
#pragma unroll
        for (int i = 0; i < MP; ++i) {
          const int m = p * MP + i;
          if (m >= FM) break;
          char* row = lds + ((wm * MP + i) * 16 + col) * RB;
#pragma unroll
          for (int f = 0; f < FN; ++f) {
            const int n = (wn * FN + f) * 16 + 4 * g;
            f32x4 y = acc[f][m];
            if (n0 + n < N) y = add_bias(y, a.bias[layer], n0 + n);
            *(s16x4*)(row + n * 2) = packed(y);
          }
        }
        barrier();
        for (int i = threadIdx.x; i < WM * MP * 16 * VPR; i += NW * 64) {
          const int at = i / VPR, n = n0 + i % VPR * 8;
          const int mr = at % (MP * 16) + p * MP * 16;
          const int r = m0 + at / (MP * 16) * (BM / WM) + mr;
          if (mr >= FM * 16 || r >= rows || n >= N) continue;
          *(s16x8*)(a.out[layer] + (long long)r * N + n) =
              *(const s16x8*)(lds + at * RB + i % VPR * 16);
        }
      }
      return;
    }
  }
  // partial sums: rows and columns before this layer's
  const int before = layer ? a.n_end[layer - 1] : 0;
  const int all = WT ? K : a.n_end[a.layers - 1];
  const int all_rows = MODE == GRAD_W ? a.n_end[a.layers - 1] : a.M;
#pragma unroll
  for (int m = 0; m < FM; ++m) {
    const int r = m0 + wm * (BM / WM) + 16 * m + col;
    if (r >= rows) continue;
    if constexpr (GLU) {
#pragma unroll
      for (int f = 0; f < FN; f += 2) {
        const int n = n0 + (wn * FN + f) * 8 + 4 * g;
        if (n >= N) continue;
        const f32x4 y = add_bias(acc[f][m], a.bias[0], n);
        f32x4 o = add_bias(acc[f + 1][m], a.bias[1], n);
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] *= y[e] / (1.f + expf(-y[e]));
        *(s16x4*)(a.out[0] + (long long)r * N + n) = packed(o);
      }
    } else {
#pragma unroll
      for (int f = 0; f < FN; ++f) {
        const int n = n0 + (wn * FN + f) * 16 + 4 * g;
        if (n >= N) continue;
        if (a.splits > 1)
          *(f32x4*)(a.part + ((long long)split * all_rows + r +
                              (MODE == GRAD_W ? before : 0)) * all +
                    (MODE == GRAD_W ? 0 : before) + n) = acc[f][m];
        else
          *(s16x4*)(a.out[layer] + (long long)r * N + n) =
              packed(add_bias(acc[f][m], a.bias[layer], n));
      }
    }
  }
}

template <int... I, typename F>
__device__ __forceinline__ void each(std::integer_sequence<int, I...>, F& f) {
  (f(Int<I>{}), ...);
}

// One operand's descriptor: loads past `left` bytes from `base` on bring zeros,
// stores there are dropped.
__device__ __forceinline__ u32x4 descriptor(const char* base, long long left) {
  const unsigned long long b = (unsigned long long)(uintptr_t)base;
  u32x4 d;
  d[0] = __builtin_amdgcn_readfirstlane((unsigned)b);
  d[1] = __builtin_amdgcn_readfirstlane((unsigned)(b >> 32) & 0xffffu);
  d[2] = __builtin_amdgcn_readfirstlane(
      left > 0xffffffffll ? 0xffffffffu : left < 0 ? 0u : (unsigned)left);
  d[3] = 0x00020000u;
  return d;
}
// 16 bytes a lane from descriptor + off + soff to LDS at m0, lane after lane. In
// two parts: m0 has to be written an instruction ahead, which a product fills.
__device__ __forceinline__ void load_to(int lds, int n) {
  asm volatile("s_add_u32 m0, %0, %1" :: "s"(lds), "i"(n) : "memory", "m0", "scc");
}
template <bool ONCE>
__device__ __forceinline__ void load(u32x4 from, unsigned off, int soff) {
  if (ONCE)
    asm volatile("buffer_load_dwordx4 %0, %1, %2 offen nt lds"
                 :: "v"(off), "s"(from), "s"(soff) : "memory");
  else
    asm volatile("buffer_load_dwordx4 %0, %1, %2 offen lds"
                 :: "v"(off), "s"(from), "s"(soff) : "memory");
}
// The sums of a wave that has all 256 accumulation registers: four from R on. They
// are named, not variables: those the compiler moves to other registers and, as they
// run out, to memory. It has to have no use for these registers itself (nothing is
// spilled: 147 to 176 of 256 others are taken). Operands have to be written, and
// products made, some instructions before they are read. Each build looks through the
// compiler's assembly for all of this but the products (ops/named_registers.py).
__device__ __forceinline__ void take_sums() {
  asm volatile("" ::: "a0", "a255");
}
template <int R>
__device__ __forceinline__ void add_product(s16x8 a, s16x8 b) {
  asm volatile("v_mfma_f32_16x16x32_bf16 a[%2:%3], %0, %1, a[%2:%3]"
               :: "v"(a), "v"(b), "n"(R), "n"(R + 3));
}
template <int R>
__device__ __forceinline__ void first_product(s16x8 a, s16x8 b) {
  asm volatile("v_mfma_f32_16x16x32_bf16 a[%2:%3], %0, %1, 0"
               :: "v"(a), "v"(b), "n"(R), "n"(R + 3));
}
template <int R>
__device__ __forceinline__ float sum() {
  float x;
  asm volatile("v_accvgpr_read_b32 %0, a[%1:%1]" : "=v"(x) : "n"(R));
  return x;
}
__device__ __forceinline__ void wait_reads() {    // of LDS
  __builtin_amdgcn_s_waitcnt(0xc07f);
}
__device__ __forceinline__ s16x8 lds_read(int at) {
  return *(const __attribute__((address_space(3))) s16x8*)(uintptr_t)(unsigned)at;
}
__device__ __forceinline__ s16x4 lds_tr_read(int at) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (__attribute__((address_space(3))) s16x4*)(uintptr_t)(unsigned)at);
}
__device__ __forceinline__ unsigned packed2(float lo, float hi) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  typedef __bf16 b16x2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(unsigned,
                            __builtin_convertvector((f32x2{lo, hi}), b16x2));
}

// The largest tiles, 256 x 256, by four waves of 128 x 128, one a SIMD (FX, FW: tiles of
// 16 rows and columns a wave; with six of either 192): a wave's sums are its accumulation
// registers, and LDS is read for 64 products of a half stage by 16 operands (eight
// waves of 128 x 64: 12 for 32). The chip's power bounds these products, so reads that
// are not made become clock.
//
//   * A tile a workgroup. One that goes on from tile to tile, its ring filled across
// the border, gains up to 1.3% alone on the chip (2.5 at K 2048, 4.5 at 1024), but
// where another kernel holds some of the CUs, a collective above all, the tiles of
// the workgroups that wait for these are late together, and the collective waits for
// the whole product (us with 8 CUs held, eight waves / one tile / going on: 4096 rows
// 28672, K 4096 771 / 796 / 1105; 8192 x 8192 x 8192 894 / 923 / 1234; dx of 14336, K
// 4096, 8192 rows 988 / 1003 / 1187; with 32 held 840 / 787 / 1098, 978 / 914 / 1224,
// 1054 / 1000 / 1186).
//   * One barrier a stage, behind the reads of its second half: from there on the
// stage's places in the ring are free (x two stages, W three), and the next stage
// has arrived. A barrier costs some 70 of a stage's 2500 cycles, a load between two
// products 17 (of 2048 that are products), their arrival nothing.
//   * PLAIN and SWIGLU: x is the first operand of the products and a lane's tiles
// of W are neighbouring features (brought about by which row is loaded where), so
// that 16 lanes store 256 bytes of a row without a pass through LDS. The gradients,
// whose W lies across, exchange halves between rows of 16 lanes.
//
//   * A tile's first products write its sums, those of no bias are stored as they
// are, and outputs pass the caches by: 2 to 4%.
//
// us one after another, eight waves and now: 8192 x 8192 x 8192 764 / 720; 4096 rows,
// K 4096: 28672 696 / 648, 6144 166 / 159, gate and up 14336 712 / 680; gate and up
// 18944, K 3584, 2331 rows 536 / 503; dx of 14336, K 4096, 8192 rows 745 / 706; dW of
// that 789 / 727 (its transposing reads are two an operand).
template <int MODE, bool PARTS, bool ONCE, int FX = 8, int FW = 8>
__global__ __launch_bounds__(256, 1) void wide_linear_kernel(const Args a) {
  constexpr bool GLU = MODE == SWIGLU;
  constexpr bool WT = MODE == GRAD_X || MODE == GRAD_W, XT = MODE == GRAD_W;
  constexpr int BM = 32 * FX, BN = 32 * FW;
  constexpr int P = FX, PW = FW;    // loads of 1 KB a wave: of x, of W
  static_assert((FX == 8 && FW == 8) ||
                ((FX == 8 || FX == 6) && (FW == 8 || FW == 6) && !PARTS && !ONCE &&
                 (FW == 8 || !GLU)), "");
  constexpr int SW = BN * ROW, SX = BM * ROW, XAT = 3 * SW;
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int lane = threadIdx.x & 63;
  const int wid = uni(threadIdx.x >> 6);
  const int col = lane & 15, g = lane >> 4;
  const int wm = wid >> 1, wn = wid & 1;
  const int K = a.K;

  // Tiles in the order of the kernel above; an XCD's workgroups take its run in
  // turn, so that they work side by side.
  constexpr int GROUP = 4;
  const int per = a.tiles * a.mtiles, total = per * a.splits;
  const int xcd = blockIdx.x % 8;
  const int item = xcd * (total / 8) + min(xcd, total % 8) + blockIdx.x / 8;

  struct Place {
    int m0, n0, s0, n_it, layer, split;
  };
  auto locate = [&](int id) INLINE {
    Place p;
    p.split = uni(id / per);
    id -= p.split * per;
    const int group = id / (GROUP * a.tiles);
    const int high = min(GROUP, a.mtiles - GROUP * group);
    id -= group * GROUP * a.tiles;
    int mt = GROUP * group + id % high, nt = id / high, l = 0;
    if (MODE == PLAIN) {
      while (nt >= a.tile_end[l]) ++l;
      if (l) nt -= a.tile_end[l - 1];
    }
    if (MODE == GRAD_W) {
      while (mt >= a.tile_end[l]) ++l;
      if (l) mt -= a.tile_end[l - 1];
    }
    p.layer = uni(l);
    p.n0 = uni(nt * (GLU ? BN / 2 : BN));
    p.m0 = uni(mt * BM);
    const int steps = MODE == GRAD_X ? a.steps
        : MODE == GRAD_W ? (a.M + BK - 1) / BK : K / BK;
    p.s0 = uni(p.split * steps / a.splits);
    p.n_it = uni((p.split + 1) * steps / a.splits) - p.s0;
    return p;
  };
  const Place at = locate(item);

  // ---- loads: the lanes' places in the pieces of 1 KB, as above. Rows past the
  // end lie past the descriptor's; columns past the end are not stored.
  const int lr = lane >> 3, lc = lane & 7;
  auto place_w = [&](int j) INLINE {
    const int piece = j * 4 + wid;
    if (WT)
      return (unsigned)(piece % 8 * 8 + lr) * K * 2 +
          2 * (piece / 8 * 64 +
               8 * (lc ^ (2 * ((lr >> 1) & 1) + 4 * (wid & 1))));
    // tile f of a wave: features FW c + f, or gate and up of 4 c + f / 2
    const int half = piece / (2 * FW), f = piece / 2 % FW, c = piece % 2 * 8 + lr;
    const int r = GLU ? half * 64 + FW / 2 * c + (f >> 1)
                      : half * 16 * FW + FW * c + f;
    return (unsigned)r * K * 2 + ((lc ^ lr) << 4);
  };
  auto place_x = [&](int j, int ld) INLINE {
    const int piece = j * 4 + wid;
    if (XT)
      return (unsigned)(piece % 8 * 8 + lr) * ld * 2 +
          2 * (piece / 8 * 64 +
               8 * (lc ^ (2 * ((lr >> 1) & 1) + 4 * (wid & 1))));
    return (unsigned)(piece * 8 + lr) * ld * 2 + ((lc ^ lr) << 4);
  };
  unsigned woff[PW], xoff[P];
#pragma unroll
  for (int j = 0; j < PW; ++j) woff[j] = place_w(j);
#pragma unroll
  for (int j = 0; j < P; ++j) xoff[j] = place_x(j, K);
  // From contraction step `step` of a tile on: descriptor, bytes to its end (the
  // operands that lie across move it), stages that follow one another there.
  u32x4 wfrom, xfrom;
  const char *wbase, *xbase;
  long long wend, xend;
  int wsoff = 0, xsoff = 0, wrow = ROW, xrow = ROW, wleft, xleft;
  int wstep, xstep, wstop, xstop, xld = K;
  auto seek_w = [&](int n0, int layer, int step, int stop) INLINE {
    wstop = uni(stop);
    wleft = stop - step;
    if (MODE == GRAD_X) {
      int l = 0;
      while (step >= a.step_end[l]) ++l;
      const int k = (step - (l ? a.step_end[l - 1] : 0)) * BK;
      wbase = (const char*)(a.w[l] + (long long)k * K + n0);
      wend = ((long long)(a.n[l] - k) * K - n0) * 2;
      wleft = min(stop, a.step_end[l]) - step;
    } else if (MODE == GRAD_W) {
      wbase = (const char*)(a.w[0] + (long long)step * BK * K + n0);
      wend = ((long long)(a.M - step * BK) * K - n0) * 2;
    } else {
      const short* w = GLU ? (wid & 2 ? a.w[1] : a.w[0]) : a.w[layer];
      wbase = (const char*)(w + (long long)n0 * K);
      wend = (long long)(a.n[layer] - n0) * K * 2;
      wsoff = uni(step * ROW);
    }
    wstep = uni(step);
    wleft = uni(wleft);
    wfrom = descriptor(wbase, wend);
  };
  auto seek_x = [&](int m0, int layer, int step, int stop) INLINE {
    xstop = uni(stop);
    xleft = stop - step;
    if (MODE == GRAD_X) {
      int l = 0;
      while (step >= a.step_end[l]) ++l;
      xld = uni(a.n[l]);
      xbase = (const char*)(a.x[l] + (long long)m0 * xld);
      xend = (long long)(a.M - m0) * xld * 2;
      xsoff = uni((step - (l ? a.step_end[l - 1] : 0)) * ROW);
      xleft = min(stop, a.step_end[l]) - step;
    } else if (MODE == GRAD_W) {
      xld = uni(a.n[layer]);
      xbase = (const char*)(a.x[layer] + (long long)step * BK * xld + m0);
      xend = ((long long)(a.M - step * BK) * xld - m0) * 2;
    } else {
      xbase = (const char*)(a.x[0] + (long long)m0 * K);
      xend = (long long)(a.M - m0) * K * 2;
      xsoff = uni(step * ROW);
    }
    xstep = uni(step);
    xleft = uni(xleft);
    xfrom = descriptor(xbase, xend);
    if (MODE >= GRAD_X)
#pragma unroll
      for (int j = 0; j < P; ++j) xoff[j] = place_x(j, xld);
  };
  // Behind the last of these: the next layer, or nothing, which is a descriptor of no
  // bytes.
  auto turn_w = [&]() INLINE {
    if (MODE == GRAD_X && wstep + 1 < wstop) {
      seek_w(at.n0, 0, wstep + 1, wstop);
    } else {
      wfrom[2] = 0;
      wsoff = wrow = 0;
      wend = 0;
      wleft = 1 << 30;
    }
  };
  auto turn_x = [&]() INLINE {
    if (MODE == GRAD_X && xstep + 1 < xstop) {
      seek_x(at.m0, 0, xstep + 1, xstop);
    } else {
      xfrom[2] = 0;
      xsoff = xrow = 0;
      xend = 0;
      xleft = 1 << 30;
    }
  };
  auto move_w = [&]() INLINE {
    if (WT) {
      const long long d = wrow ? (long long)BK * K * 2 : 0;
      wbase += d;
      wend -= d;
      wfrom = descriptor(wbase, wend);
      if (MODE == GRAD_X) ++wstep;
    } else {
      wsoff += wrow;
    }
  };
  auto move_x = [&]() INLINE {
    if (XT) {
      const long long d = xrow ? (long long)BK * xld * 2 : 0;
      xbase += d;
      xend -= d;
      xfrom = descriptor(xbase, xend);
    } else {
      xsoff += xrow;
      if (MODE == GRAD_X) ++xstep;
    }
  };
  const int lds_at = (int)(uintptr_t)(__attribute__((address_space(3))) char*)lds;
  const int put = lds_at + wid * 1024;
  int wput = put, xput = put + XAT, wget = 0, xget = 0;
  auto next_w = [&](int b, int first) INLINE {
    return b == first + 2 * SW ? first : b + SW;
  };
  auto fill_w = [&]() INLINE {
#pragma unroll
    for (int j = 0; j < PW; ++j) {
      load_to(wput, j * 4096);
      asm volatile("s_nop 0");
      load<ONCE>(wfrom, woff[j], wsoff);
    }
    wput = next_w(wput, put);
    if (--wleft == 0) turn_w();
    else move_w();
  };
  auto fill_x = [&]() INLINE {
#pragma unroll
    for (int j = 0; j < P; ++j) {
      load_to(xput, j * 4096);
      asm volatile("s_nop 0");
      load<false>(xfrom, xoff[j], xsoff);
    }
    xput = xput == put + XAT ? xput + SX : put + XAT;
    if (--xleft == 0) turn_x();
    else move_x();
  };

  // ---- operands: 16 rows (or columns) by inputs 32 h + 8 g + j, at the lane's
  // addresses and constants. Across, tiles of 16 columns have four of them, or where
  // a wave does not begin with a block of 64 one each.
  const int tr = (8 * g + (col >> 2)) * 128 + (col & 3) * 8 +
      32 * ((col >> 3) & 1) + 64 * (g & 1);
  const int o0 = (g ^ (col & 7)) << 4;
  const int w0 = WT ? lds_at + wn * 16384 + tr
                    : lds_at + (wn * (BN / 2) + col) * ROW + o0;
  const int x0 = XAT + (XT ? lds_at + wm * 16384 + tr
                           : lds_at + (wm * (BM / 2) + col) * ROW + o0);
  constexpr int WA = !WT ? 1 : FW == 8 ? 4 : FW, XA = !XT ? 1 : FX == 8 ? 4 : FX;
  int wat[WA], xat[XA];
  auto aim = [&](int h) INLINE {    // at a half of the stage
    if (!WT || h == 0)
#pragma unroll
      for (int c = 0; c < WA; ++c) {
        const int t = wn * FW + c;
        if (WT && FW < 8) wat[c] = lds_at + t / 4 * 8192 + (tr ^ t % 4 * 32) + wget;
        else wat[c] = (w0 ^ (WT ? 32 * c : 64 * h)) + wget;
        asm volatile("" : "+v"(wat[c]));
      }
    if (!XT || h == 0)
#pragma unroll
      for (int c = 0; c < XA; ++c) {
        const int t = wm * FX + c;
        if (XT && FX < 8)
          xat[c] = lds_at + XAT + t / 4 * 8192 + (tr ^ t % 4 * 32) + xget;
        else xat[c] = (x0 ^ (XT ? 32 * c : 64 * h)) + xget;
        asm volatile("" : "+v"(xat[c]));
      }
  };
  s16x8 wa[2][FW], xa[2][FX];
  auto across = [&](int at, int i, int h) INLINE {
    const s16x4 lo = lds_tr_read(at + i / 4 * 8192 + h * 4096);
    const s16x4 hi = lds_tr_read(at + i / 4 * 8192 + h * 4096 + 512);
    return s16x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
  };
  auto get = [&](int q, int h) INLINE {
    if (q < FW)
      wa[h][q] = WT ? across(wat[q % WA], FW == 8 ? q : 0, h)
                    : lds_read(wat[0] + q * 16 * ROW);
    else
      xa[h][q - FW] = XT ? across(xat[(q - FW) % XA], FX == 8 ? q - FW : 0, h)
                         : lds_read(xat[0] + (q - FW) * 16 * ROW);
  };
  // sums of a tile of W and one of x
#define acc(f, m) (((f) * FX + (m)) * 4)
  take_sums();

  seek_w(at.n0, at.layer, at.s0, at.s0 + at.n_it);
  seek_x(at.m0, at.layer, at.s0, at.s0 + at.n_it);
  fill_w();
  fill_x();
  fill_w();
  fill_x();
  fill_w();
  wait_loads<2 * PW + P>();
  barrier();
  aim(0);
#pragma unroll
  for (int q = 0; q < FW + FX; ++q) get(q, 0);

  // A stage's 2 FX FW products. Reads of its second half lie between the first ones,
  // those of the next stage's first half behind the middle; x two stages ahead and
  // W three are loaded behind the barrier.
  constexpr int N1 = FX * FW, N2 = 2 * N1;
  constexpr int BARRIER = N1 == 64 ? 30 : N1 == 48 ? 24 : 20;
  // loads of x and of W: the first one's product, a step
  constexpr int X1 = BARRIER + 2, XN = N1 == 64 ? 6 : FX == 6 && FW == 8 ? 5 : 4;
  constexpr int W1 = N1 == 64 ? 82 : N1 == 36 ? 46 : FW == 8 ? 54 : 58;
  constexpr int WN = N1 == 64 ? 6 : N1 == 36 ? 4 : FW == 8 ? 5 : 6;
  static_assert((FW + FX - 1) * 3 / 2 < BARRIER && X1 + XN * (P - 1) < W1 &&
                W1 + WN * (PW - 1) < N2 && N1 + 2 + 3 * (FW + FX - 1) < N2, "");
  auto stage = [&](auto first) INLINE {
    constexpr bool FIRST = decltype(first)::value;
    __builtin_amdgcn_sched_barrier(0);
    wait_reads();
    aim(1);
    auto product = [&](auto at) INLINE {
      constexpr int i = decltype(at)::value, h = i / N1, m = i / FW % FX;
      constexpr int f = m % 2 ? FW - 1 - i % FW : i % FW;
      if constexpr (i == BARRIER) {
        wait_loads<PW>();
        wait_reads();
        __builtin_amdgcn_s_barrier();
        wget = next_w(wget, 0);
        xget ^= SX;
        aim(0);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        if (q < P && i == X1 + XN * q) load_to(xput, q * 4096);
        if (q < PW && i == W1 + WN * q) load_to(wput, q * 4096);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int q = 0; q < FW + FX; ++q) {
        if (i == q * 3 / 2) get(q, 1);
        if (i == N1 + 2 + 3 * q) get(q, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
      const s16x8 u = WT ? wa[h][f] : xa[h][m], v = WT ? xa[h][m] : wa[h][f];
      if constexpr (FIRST && h == 0) first_product<acc(f, m)>(u, v);
      else add_product<acc(f, m)>(u, v);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        if (q < P && i == X1 + XN * q) load<false>(xfrom, xoff[q % P], xsoff);
        if (q < PW && i == W1 + WN * q) load<ONCE>(wfrom, woff[q % PW], wsoff);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    each(std::make_integer_sequence<int, N2>{}, product);
    xput = xput == put + XAT ? xput + SX : put + XAT;
    wput = next_w(wput, put);
    --wleft;
    --xleft;
    if (min(wleft, xleft) > 0) {
      move_w();
      move_x();
    } else {
      if (wleft == 0) turn_w();
      else move_w();
      if (xleft == 0) turn_x();
      else move_x();
    }
  };
  stage(Int<1>{});
#pragma clang loop unroll(disable)
  for (int it = 1; it < at.n_it; ++it) stage(Int<0>{});

  asm volatile("s_nop 15");     // the last products
  // past the tile's rows or columns to nowhere
  const int N = WT ? K : a.n[at.layer];
  const int rows = MODE == GRAD_W ? a.n[at.layer] : a.M;
  const int m_of = uni(at.m0 + wm * (BM / 2));
  const int have = uni(max(0, min(rows - m_of, BM / 2)));
  constexpr unsigned NOWHERE = 0x80000000u;
  if constexpr (PARTS) {
    const int before = a.n_end[at.layer] - a.n[at.layer];
    const int all = WT ? K : a.n_end[a.layers - 1];
    const int all_rows = MODE == GRAD_W ? a.n_end[a.layers - 1] : a.M;
    const __amdgpu_buffer_rsrc_t to = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(a.part + ((long long)at.split * all_rows + m_of +
                          (MODE == GRAD_W ? before : 0)) * all +
                (MODE == PLAIN ? before : 0)),
        (short)0, (int)((unsigned)have * all * 4), 0x00020000);
    // gradients: row col, columns 4 g ..; otherwise rows 4 g + r, half of eight
    const int n1 = at.n0 + wn * (BN / 2) + (WT ? 4 * g : FX * col);
    const int r1 = WT ? col : 4 * g;
    auto store = [&](auto at) INLINE {
      constexpr int m = decltype(at)::value / FX, i = decltype(at)::value % FX;
      constexpr int f = 4 * (i & 1), r = i >> 1;
      f32x4 v;
      if constexpr (WT)
        v = f32x4{sum<acc(i, m)>(), sum<acc(i, m) + 1>(), sum<acc(i, m) + 2>(),
                  sum<acc(i, m) + 3>()};
      else
        v = f32x4{sum<acc(f, m) + r>(), sum<acc(f + 1, m) + r>(),
                  sum<acc(f + 2, m) + r>(), sum<acc(f + 3, m) + r>()};
      const int row = r1 + 16 * m + (WT ? 0 : r);
      const int n = n1 + (WT ? 16 * i : f);
      __builtin_amdgcn_raw_buffer_store_b128(
          __builtin_bit_cast(u32x4, v), to,
          n < N && row < have ? (unsigned)(row * all + n) * 4 : NOWHERE, 0, 0);
    };
    each(std::make_integer_sequence<int, FX * FX>{}, store);
  } else {
    // outputs pass the caches by, which hold what other tiles still read
    constexpr int STREAM = 2;
    // Not where rows are no whole 64 bytes: a store of 64 (gradients) or 192 and 256 bytes
    // of a row is then parts of lines, which have to meet in a cache (us, past the caches /
    // through them: the input's gradient of 576 features, K 2968, 6126 rows 48.6 / 31.7,
    // the weights' of 23936 x 2408, 244 rows 108 / 57; over 220 of the largest tile 0.87;
    // forward 9416, K 192, 6622 rows 57.4 / 42.5, 11608, K 192, 8682 rows 88.0 / 76.0; over
    // 100 of the largest tile 0.95). But forward outputs that no cache holds go past, and
    // gates, 128 bytes of a row and longer in the making, are even (32336, K 640, 8271 rows
    // 353 / 391).
    const bool whole = N % 32 == 0 || GLU ||
        (!WT && (long long)rows * N > 1ll << 27);
    short* out = a.out[MODE == GRAD_X || GLU ? 0 : at.layer];
    const __amdgpu_buffer_rsrc_t to = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(out + (long long)m_of * N), (short)0,
        (int)((unsigned)have * N * 2), 0x00020000);
    if constexpr (WT) {
      // columns 4 g .. of two tiles to 8 of one: odd rows of lanes of the first
      // change places with even ones of the second
      const int n1 = at.n0 + wn * (BN / 2) + (g & 1) * 16 + (g >> 1) * 8;
      auto store = [&](auto by, auto at) INLINE {
        constexpr int f = decltype(at)::value / FX * 2, m = decltype(at)::value % FX;
        constexpr int A = acc(f, m), B = acc(f + 1, m);
        const unsigned y0 = packed2(sum<A>(), sum<A + 1>());
        const unsigned y1 = packed2(sum<A + 2>(), sum<A + 3>());
        const unsigned z0 = packed2(sum<B>(), sum<B + 1>());
        const unsigned z1 = packed2(sum<B + 2>(), sum<B + 3>());
        const auto lo = __builtin_amdgcn_permlane16_swap(y0, z0, false, false);
        const auto hi = __builtin_amdgcn_permlane16_swap(y1, z1, false, false);
        const int n = n1 + 16 * f;
        __builtin_amdgcn_raw_buffer_store_b128(
            u32x4{lo[0], hi[0], lo[1], hi[1]}, to,
            n < N ? (unsigned)((16 * m + col) * N + n) * 2 : NOWHERE, 0,
            decltype(by)::value);
      };
      auto past = [&](auto at) INLINE { store(Int<STREAM>{}, at); };
      auto through = [&](auto at) INLINE { store(Int<0>{}, at); };
      if (whole) each(std::make_integer_sequence<int, FW / 2 * FX>{}, past);
      else each(std::make_integer_sequence<int, FW / 2 * FX>{}, through);
    } else {
      constexpr int W = GLU ? FW / 2 : FW;    // features a lane
      const int n = at.n0 + wn * (GLU ? BN / 4 : BN / 2) + W * col;
      const bool at_edge = at.n0 + BN > N;
      float b[GLU ? 2 : 1][W];
      const bool biased = a.bias[GLU ? 0 : at.layer] || (GLU && a.bias[1]);
      if (biased)
#pragma unroll
      for (int l = 0; l < (GLU ? 2 : 1); ++l) {
        const short* bias = a.bias[GLU ? l : at.layer];   // of none: zeros
        const __amdgpu_buffer_rsrc_t from = __builtin_amdgcn_make_buffer_rsrc(
            (void*)bias, (short)0, bias ? N * 2 : 0, 0x00020000);
#pragma unroll
        for (int e = 0; e < W; ++e)
          b[l][e] = value((short)__builtin_amdgcn_raw_buffer_load_b16(
              from, (n + e) * 2, 0, 0));
      }
      typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
      auto store = [&](auto bias, auto by, auto at) INLINE {
        constexpr bool B = decltype(bias)::value;
        constexpr int S = decltype(by)::value;
        constexpr int m = decltype(at)::value / 4, r = decltype(at)::value % 4;
        const unsigned o =
            n < N ? (unsigned)((4 * g + 16 * m + r) * N + n) * 2 : NOWHERE;
        auto one = [&](auto at) INLINE {
          constexpr int e = decltype(at)::value;
          if constexpr (GLU) {
            const float t = sum<acc(2 * e, m) + r>() + (B ? b[0][e] : 0.f);
            return t / (1.f + expf(-t)) *
                (sum<acc(2 * e + 1, m) + r>() + (B ? b[GLU][e] : 0.f));
          } else {
            return B ? sum<acc(e, m) + r>() + b[0][e] : sum<acc(e, m) + r>();
          }
        };
        const u32x2 v = {packed2(one(Int<0>{}), one(Int<1>{})),
                         packed2(one(Int<2>{}), one(Int<3>{}))};
        if constexpr (GLU) {
          __builtin_amdgcn_raw_buffer_store_b64(v, to, o, 0, S);
        } else if constexpr (FW == 6) {
          typedef unsigned u32x3 __attribute__((ext_vector_type(3)));
          const unsigned u = packed2(one(Int<4>{}), one(Int<5>{}));
          if (at_edge) {      // N is a multiple of four, six features may pass it
            __builtin_amdgcn_raw_buffer_store_b32(v[0], to, o, 0, S);
            __builtin_amdgcn_raw_buffer_store_b32(
                v[1], to, n + 2 < N ? o + 4 : NOWHERE, 0, S);
            __builtin_amdgcn_raw_buffer_store_b32(
                u, to, n + 4 < N ? o + 8 : NOWHERE, 0, S);
          } else {
            __builtin_amdgcn_raw_buffer_store_b96(u32x3{v[0], v[1], u}, to, o, 0,
                                                  S);
          }
        } else {
          const u32x2 u = {packed2(one(Int<4>{}), one(Int<5>{})),
                           packed2(one(Int<6>{}), one(Int<7>{}))};
          if (N % 8 == 0) {
            __builtin_amdgcn_raw_buffer_store_b128(u32x4{v[0], v[1], u[0], u[1]},
                                                   to, o, 0, S);
          } else {
            __builtin_amdgcn_raw_buffer_store_b64(v, to, o, 0, S);
            __builtin_amdgcn_raw_buffer_store_b64(
                u, to, n + 4 < N ? o + 8 : NOWHERE, 0, S);
          }
        }
      };
      auto all = [&](auto bias, auto by) INLINE {
        auto one = [&](auto at) INLINE { store(bias, by, at); };
        each(std::make_integer_sequence<int, 4 * FX>{}, one);
      };
      if (biased && whole) all(Int<1>{}, Int<STREAM>{});
      else if (biased) all(Int<1>{}, Int<0>{});
      else if (whole) all(Int<0>{}, Int<STREAM>{});
      else all(Int<0>{}, Int<0>{});
    }
  }
  wait_loads<0>();
}
#undef acc

// Adds the splits up: four columns of a row a thread.
template <int MODE>
__global__ __launch_bounds__(256) void tile_merge_kernel(const Args a,
                                                         const int rows,
                                                         const int all) {
  const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  if (i >= (long long)rows * (all / 4)) return;
  int r = (int)(i / (all / 4)), n = (int)(i % (all / 4)) * 4;
  f32x4 y = {0.f, 0.f, 0.f, 0.f};
  const float* p = a.part + (long long)r * all + n;
#pragma unroll 4
  for (int s = 0; s < a.splits; ++s)
    y += *(const f32x4*)(p + (long long)s * rows * all);
  int l = 0, ld = all;
  if (MODE == PLAIN) {
    while (n >= a.n_end[l]) ++l;
    if (l) n -= a.n_end[l - 1];
    ld = a.n[l];
  }
  if (MODE == GRAD_W) {
    while (r >= a.n_end[l]) ++l;
    if (l) r -= a.n_end[l - 1];
  }
  *(s16x4*)(a.out[l] + (long long)r * ld + n) =
      packed(add_bias(y, a.bias[l], n));
}

// Tiles and stages of a launch, before the kernel's own numbers of them.
template <int BM, int BN, int MODE>
int count(Args& a) {
  constexpr int bn = MODE == SWIGLU ? BN / 2 : BN;
  int sum = 0, steps = 0;
  for (int i = 0; i < a.layers; ++i) {
    if (MODE != SWIGLU || i == 0)
      sum += MODE == GRAD_W ? (a.n[i] + BM - 1) / BM : (a.n[i] + bn - 1) / bn;
    a.tile_end[i] = sum;
    a.step_end[i] = steps += a.n[i] / BK;
  }
  a.steps = steps;
  a.tiles = MODE >= GRAD_X ? (a.K + bn - 1) / bn : sum;
  a.mtiles = MODE == GRAD_W ? sum : (a.M + BM - 1) / BM;
  return a.tiles * a.mtiles * a.splits;
}

template <int MODE>
int merge_splits(const Args& a, hipStream_t st) {
  const int n = a.n_end[a.layers - 1];
  const int rows = MODE == GRAD_W ? n : a.M, all = MODE >= GRAD_X ? a.K : n;
  const long long q = (long long)rows * (all / 4);
  hipLaunchKernelGGL(tile_merge_kernel<MODE>, dim3((unsigned)((q + 255) / 256)),
                     dim3(256), 0, st, a, rows, all);
  return (int)hipGetLastError();
}

// W past the caches, which are then x's: over one tile of rows (us, before / now, K 4096
// unless said: 224 rows 128256 247 / 216, gate and up 14336 63 / 60; 128 rows 128256 197 /
// 168, gate and up 50 / 47; 32 rows 128256 179 / 165, gate and up 43 / 38, 9216, K 3072
// 16.8 / 15.5). Not where the contraction is split (128 rows 4096, K 14336 in eight 34.0 /
// 36.4, 64 rows 4096 in four 12.7 / 13.4), nor over several tiles of rows, which share W
// (300 rows 128256 343 / 345, 2331 rows 3584, K 14336 245 / 251). Over 800 layers of 33 to
// 256 rows 0.95 of the time, 1.01 at most, from 16 MB on; smaller ones, 0.98 out of
// memory, may be found in the chip's cache of 256 MB as a whole model's (8 MB 1.08). So
// may larger ones of a small model: layers of 1024 and a head of 32000 in turn, 40 to 250
// rows, 1.01 of the time at 111 and 156 MB in all; but 0.98 at 246 MB, and layers of 2048,
// 672 MB, 0.97. A line at 64 MB would have these at 1.00 all four.
bool once(const Args& a) {
  return a.mtiles == 1 && a.splits == 1 &&
      (long long)a.n_end[a.layers - 1] * a.K >= 1 << 23;
}

template <int BM, int BN, int WM, int WN, int NS, int MODE>
int launch(Args a, bool merge, hipStream_t st) {
  constexpr int LDS = NS * (BM + BN) * ROW;
  static_assert(LDS <= 160 * 1024, "");
  const int items = count<BM, BN, MODE>(a);
  // One tile of rows reads W once, nothing of it is shared: tiles that all begin at
  // their rows' beginnings read the same few memory channels at a time where rows
  // are whole multiples of 4 KB apart. Begun apart over an XCD and over the XCDs (us,
  // before / now): 48 rows 16384, K 4096 31.5 / 25.2, 32000 60 / 47, 28672, K 8192 106 /
  // 82, gate and up 14336, K 4096 54.9 / 42.6, 11008 43.0 / 36.5; 128 rows 128256 222 /
  // 197, 32000 63 / 51; 224 rows 32000 73 / 69, gate and up 14336 65.2 / 64.4; even at
  // K 3072, 4608 and 5120. Other steps than 13 and 7 leave 18432, K 4096 at 43 to 52.
  // But each is at another place of x then, all of which has to stay in an XCD's 4 MB
  // of L2 beside W's stream. Of the time of beginning together, over 7000 layers with
  // weights from memory: x up to 1 MB 0.90, to 1.5 0.92, to 2 0.96, to 2.5 0.99, to 3
  // 1.02, to 4 1.07, to 6 1.15, more 1.22 (256 rows 32064, K 16384 255 / 459 us).
  a.turn = a.mtiles == 1 && a.splits == 1 && a.K * 2 % 4096 == 0 &&
      (long long)a.M * a.K <= 1 << 20;
  auto kernel = tile_linear_kernel<BM, BN, WM, WN, NS, MODE, false>;
  if constexpr (MODE <= SWIGLU)
    if (once(a)) kernel = tile_linear_kernel<BM, BN, WM, WN, NS, MODE, true>;
  const hipError_t e = hipFuncSetAttribute(
      (const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
  if (e != hipSuccess) return (int)e;
  hipLaunchKernelGGL(kernel, dim3(items), dim3(WM * WN * 64), LDS, st, a);
  if (a.splits > 1 && merge) return merge_splits<MODE>(a, st);
  return (int)hipGetLastError();
}

template <int MODE>
int launch_wide(Args a, bool merge, hipStream_t st) {
  constexpr int LDS = 160 * 1024;
  const int items = count<256, 256, MODE>(a);
  auto kernel = MODE != SWIGLU && a.splits > 1
      ? wide_linear_kernel<MODE, MODE != SWIGLU, false>
      : wide_linear_kernel<MODE, false, false>;
  if constexpr (MODE <= SWIGLU)
    if (once(a)) kernel = wide_linear_kernel<MODE, false, true>;
  const hipError_t e = hipFuncSetAttribute(
      (const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
  if (e != hipSuccess) return (int)e;
  hipLaunchKernelGGL(kernel, dim3(items), dim3(256), LDS, st, a);
  if (a.splits > 1 && merge) return merge_splits<MODE>(a, st);
  return (int)hipGetLastError();
}

// The next smaller tiles by four waves.
template <int BM, int BN, int MODE>
int launch_four(Args a, hipStream_t st) {
  constexpr int LDS = (3 * BN + 2 * BM) * ROW;
  const int items = count<BM, BN, MODE>(a);
  auto kernel = wide_linear_kernel<MODE, false, false, BM / 32, BN / 32>;
  const hipError_t e = hipFuncSetAttribute(
      (const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
  if (e != hipSuccess) return (int)e;
  hipLaunchKernelGGL(kernel, dim3(items), dim3(256), LDS, st, a);
  return (int)hipGetLastError();
}

// What the largest tile does not take: outputs are stored at 32-bit offsets in 128
// rows of ``columns`` sums, and the rows that GRAD_X reads lie behind a descriptor of
// less than 2^32 bytes, which 256 rows of 2^23 features fill.
bool past_wide(int mode, double columns, int most) {
  return columns >= 1 << 22 || (mode == GRAD_X && most >= 1 << 23);
}

// number, BM, BN, waves along rows and features, stages in LDS; us a stage and
// a tile of a chip full of them (fitted to 8000 calls in all four modes, of 33 to
// 8192 rows and 1024 x 1024 to 32000 x 18944; root mean square error 10%). The
// largest make the most products of what they load, the smaller ones fill the chip
// with fewer rows or features. 256 x 192 has waves of three tiles of features: no gates.
#define TILES(X)                           \
  X(0, 64, 64, 2, 2, 8, 0.305f, 1.2f)      \
  X(1, 64, 128, 2, 2, 6, 0.437f, 2.6f)     \
  X(2, 128, 64, 4, 2, 6, 0.365f, 2.6f)     \
  X(3, 128, 128, 4, 2, 5, 0.532f, 3.4f)    \
  X(4, 128, 256, 2, 4, 3, 0.759f, 4.9f)    \
  X(5, 192, 128, 4, 2, 4, 0.674f, 5.2f)    \
  X(6, 192, 256, 4, 2, 2, 1.047f, 6.3f)    \
  X(7, 256, 128, 4, 2, 3, 0.754f, 5.2f)    \
  X(8, 256, 192, 2, 4, 2, 1.023f, 6.3f)
// 192 x 256, 256 x 192 and (SQUARE) 192 x 192 are wide_linear_kernel's as well: by eight
// waves LDS bounds them (256 x 192: 1850 cycles of it for 1536 of products), by four of
// 128 x 96 it does not. Whole contractions of several tiles of rows; one tile of rows and
// splits, which memory bounds, keep the deeper ring. us by eight waves and four, forward
// 4000 rows 9216, K 3072 179 / 160, 171 / 159, 178 / 165, 2331 rows 3584, K 18944 290 /
// 259, 277 / 264, 256 / 239; gate and up 14336, K 4096, 4096 rows 766 / 710; the input's
// gradient of 4000 rows 9216, K 3072 185 / 159, 177 / 161, 284 / 235; the weights' 230 /
// 204, 220 / 204, 196 / 179.
constexpr int LOW = 6, NARROW = 8;
constexpr int WIDE = 9;
// 192 x 192, for what lies between the rounds of the others (us, the choice without it /
// this; over 500 layers that it is chosen for 0.94 of one's or several layers' forward,
// 0.88 of gate and up, 0.97 of the input's gradient and 0.93 of the weights', 22 of them
// more than 5% and at worst 20% slower, 185 rows of 32000 + 2 of 8000, K 16384, as
// other tiles' are that the estimate does not hold for; taken for a lead of 2.5% and
// more only, it would gain 0.2%): 2331 rows 3584, K 4096 62.4 / 57.7, K 18944 291 /
// 272; 573 rows 14336, K 3584 60.2 / 50.3, gate and up of 543, K 4096 128 / 111; 1524
// rows 11008, K 4096 127 / 109; 540 rows 32000, K 4096 157 / 132. The input's gradient,
// whose W is read across, takes a little more than its terms say (3000 rows, n 32000, K
// 3072 in three splits of 256 x 256 508, in this 549).
constexpr int SQUARE = 10;
#define BETWEEN(X) X(SQUARE, 192, 192, 4, 2, 3, 0.804f, 6.3f)
// Short contractions, as much first loads and stores, which eight waves make beside each
// other's products, stay as below. Of the time by eight waves, over 1200 weights and rows
// (192 x 256, 256 x 192, 192 x 192): the input's gradient 1.04, 1.07 and 0.99 at 4 stages,
// 0.98, 1.02 and 0.94 at 8, 0.95, 0.99 and 0.90 at 12 (4000 rows 256 features, K 14336 in
// 256 x 192 45 by eight / 56 us, 512, K 11008 57 / 62, 1024, K 3072 26.1 / 24.4); the
// weights' of more than 12288 columns that are no power of two up to 1.07 and 1.13 at 4,
// 0.99 and 1.06 at 8 and 0.89 at 4 for 192 x 192 (4608 x 18432, 256 rows in 256 x 192 74 /
// 82), of others 0.89, 0.93 and 0.84 at 4 already (3072 x 8192, 300 rows 29.3 / 23.8).
// Gradients of columns that are no whole 64 bytes, over 190: 256 x 192 1.03 up to 10
// stages (3072 x 3832, 216 rows 14.3 / 16.2; the input's of 576 features, K 4880, 4492
// rows 33.4 / 35.3), 0.97 from 12 on, the others 0.91 as all.
bool by_four(int tile, int M, int K, int steps, int splits, int mode) {
  if (tile != LOW && tile != NARROW && tile != SQUARE) return false;
  if (tile != LOW && mode == SWIGLU) return false;
  if (mode != GRAD_W && M <= (tile == NARROW ? 256 : 192)) return false;
  const bool across = K > 12288 && (K & (K - 1)), ragged = K % 32 != 0;
  int few = mode == SWIGLU ? 24 : 0;
  if (mode == GRAD_X) few = tile == SQUARE ? 4 : 8;
  if (mode == GRAD_W && across) few = tile == LOW ? 5 : tile == NARROW ? 8 : 0;
  if (mode >= GRAD_X && ragged && tile == NARROW) few = 12;
  return splits == 1 && steps > few;
}
// Of the time by eight waves, which the table's terms are fitted to: by mode. Less is
// gained over few stages.
float four_takes(int tile, int steps, int mode) {
  static const float of[3][4] = {
      {0.91f, 0.94f, 0.88f, 0.92f}, {0.95f, 1, 0.91f, 0.94f}, {0.935f, 1, 0.84f, 0.90f}};
  static const float most[3] = {0.853f, 0.905f, 0.815f};    // of the input's gradient
  const int i = tile == LOW ? 0 : tile == NARROW ? 1 : 2;
  if (mode == GRAD_X) return fmaxf(of[i][mode], most[i] + 1.f / steps);
  if (mode == GRAD_W && steps <= 8 && tile != SQUARE) return 0.96f;
  return of[i][mode];
}
// The largest tile by eight waves, two a SIMD: a short contraction is as much its first
// loads and its stores, which the waves make beside each other's products. In place of
// WIDE up to so many stages. Over 7000 layers, of the four waves' time: gate and up
// 0.98 at 8, 0.99 to 32, then even; the input's gradient 0.93 at 8, 0.98 at 16 and 1.02
// at 32; the weights', of 5120 and more columns, 0.89 to 4, 0.93 to 8, 0.97 to 12, 0.99
// to 16 and 1.02 from there. Gradients of fewer than 3072 columns are even or lose (K
// 1536 1.00, 2048 1.07), and of columns that are a power of two, whose rows' stores meet
// in the same memory channels (4096 1.05, 8192 1.02, 16384 0.99, but 3584 0.97). PLAIN,
// whose outputs go through LDS here, 1.10 at 8 and 1.06 from 24 on: never.
constexpr int EIGHT = 11;
bool short_contraction(int mode, int stages, int columns) {
  static const int most[] = {0, 24, 16, 12};    // by mode
  return stages <= most[mode] &&
      (mode == SWIGLU || (columns >= 3072 && (columns & (columns - 1))));
}

// A wave's gate and up tiles in pairs; halves of x in blocks of 64 columns.
#define GATES(BN, WN) (BN / WN / 16 % 2 == 0)
#define BLOCKS(BM, WM) (BM / WM / 32 * 16 * WM % 64 == 0)

struct Tile {
  int bm, bn, stages;
  bool gates, blocks;
  float stage, fixed;
  bool plain = true;
  bool takes(int mode) const {
    return (gates || mode != SWIGLU) && (blocks || mode != GRAD_W) &&
        (plain || mode != PLAIN);
  }
};
const Tile tiles_[] = {
#define X(I, BM, BN, WM, WN, NS, U, F) \
  {BM, BN, NS, GATES(BN, WN), BLOCKS(BM, WM), U, F},
    TILES(X)
    {256, 256, 2, true, true, 1.149f, 8.8f},    // WIDE
    BETWEEN(X)
    {256, 256, 2, true, true, 0, 0, false},     // EIGHT
#undef X
};

// us that a tile and a number of splits take: rounds of the 256 CUs (the last
// one, in part empty, runs faster: less power, less traffic) or W and x from
// memory, whichever is longer, then adding the splits up. Memory gives less to few
// workgroups (8192 x 8192, 64 rows: 128 of them 43.7 us, 256 36.1; but 11008 x 4096,
// 17 rows: 172 22.7, 344 25.5) and to W read across in columns of 64, 128 bytes a row
// (its gradient's input, 128 rows, 14336 x 14336: 128 x 64 133 us, 192 x 256 95; 64
// rows, 32000 x 18944 by 64 x 128 304, by 128 x 256 206).
float estimate(const Tile& t, double tiles, int steps, double rows,
               double columns, double bytes, int splits, int mode) {
  tiles *= splits;
  const double whole = (double)(long long)(tiles / 256);
  const double rest = tiles / 256 - whole;
  double us = (whole + (rest > 0 ? 0.82 + 0.18 * rest : 0)) *
      (steps / (double)splits * t.stage * (mode == GRAD_W ? 0.95 : 1) + t.fixed);
  double mem = bytes / (mode == GRAD_X && t.bn == 64 ? 4.3e6
                        : mode == PLAIN && tiles < 168 ? 4.0e6 : 5.7e6);
  us *= us * us;
  mem *= mem * mem;
  us = cbrt(sqrt(us * us + mem * mem));
  if (splits > 1) us += 2.65 + 0.276e-6 * splits * rows * columns * 4;
  return (float)us;
}

}  // namespace

// The tile for 1..3 weights on one input and the splits of the contraction, by
// ``estimate``: over those calls 0.6% over the fastest on average, 0.9% for the
// input's gradient (4.4% by an earlier fit). Each split needs the ring's stages. The
// addition of the splits is counted also where the next kernel makes it as it reads
// them. -1: no tile for this K.
extern "C" int ds_tile_linear_plan(const int* n, int layers, int M, int K,
                                   int mode, int* splits) {
  static const int some[] = {1, 2, 3, 4, 6, 8, 12, 16, 24, 32};
  double all = 0;
  int most = 0;
  for (int l = 0; l < layers; ++l) {
    all += n[l];
    most = n[l] > most ? n[l] : most;
  }
  const int steps = mode == GRAD_X ? (int)(all / BK)
      : mode == GRAD_W ? (M + BK - 1) / BK : K / BK;
  const double rows = mode == GRAD_W ? all : M;
  const double columns = mode >= GRAD_X ? K : all;
  const double bytes = 2 * (all * K + (double)M * (K + all));
  struct Choice {
    int tile = -1, splits = 1;
    float eight = 0, us = 0;
  };
  Choice best, old;       // by these terms, and with eight waves alone
  for (int i = 0; i < EIGHT; ++i) {
    const Tile& t = tiles_[i];
    if (!t.takes(mode) || (i == WIDE && past_wide(mode, columns, most)))
      continue;
    double tiles = 0;
    for (int l = 0; l < layers; ++l)    // SWIGLU: a gate and an up each
      tiles += mode == GRAD_W ? (n[l] + t.bm - 1) / t.bm
          : mode == SWIGLU ? 0.5 * ((2 * n[l] + t.bn - 1) / t.bn)
          : (n[l] + t.bn - 1) / t.bn;
    if (mode == GRAD_X) tiles = 1;
    tiles *= mode >= GRAD_X ? (K + t.bn - 1) / t.bn : 1;
    tiles *= mode == GRAD_W ? 1 : (M + t.bm - 1) / t.bm;
    for (int s : some) {
      if (s > 1 && (mode == SWIGLU || tiles * s > 520)) break;
      if (steps / s < t.stages) break;
      float us = estimate(t, tiles, steps, rows, columns, bytes, s, mode);
      if (i == SQUARE && mode == GRAD_X) us *= 1.04f;
      const bool least_by_eight = old.tile < 0 || us < old.eight;
      if (least_by_eight) old = {i, s, us, us};
      if (by_four(i, M, K, steps, s, mode)) us *= four_takes(i, steps, mode);
      if (least_by_eight) old.us = us;
      if (best.tile < 0 || us < best.us) best = {i, s, us, us};
    }
  }
  // The terms are off by a tenth: another tile for a lead only (3369 rows 32000, K 1024
  // 256 x 256 185, 192 x 256, which these terms have ahead by a little, 190). Short
  // gradients of the largest tile are EIGHT's.
  const bool eight = old.tile == WIDE && mode >= GRAD_X &&
      short_contraction(mode, steps / old.splits, K);
  if (best.us > (eight ? 0.9f : 0.96f) * old.us) best = old;
  *splits = best.splits;
  if (best.tile == WIDE && short_contraction(mode, steps / *splits, K)) return EIGHT;
  return best.tile;
}

// Stages of inputs that a split has to hold at least; 0: no such tile.
extern "C" int ds_tile_linear_stages(int tile, int mode) {
  if (tile < 0 || tile >= (int)(sizeof(tiles_) / sizeof(Tile))) return 0;
  return tiles_[tile].takes(mode) ? tiles_[tile].stages : 0;
}

// 1..3 weights [n, K] of layers on one input of M rows. PLAIN and SWIGLU: x[0]
// [M, K] to out [M, n], one each or one; K is a multiple of 64, n of four.
// GRAD_X: x are the gradients dy [M, n], out[0] [M, K]; n is a multiple of 64, K
// of eight. GRAD_W: w[0] is the input, x the gradients, out [n, K]; n and K are
// multiples of eight. K is at most 2^22 and the gradients' n 2^23: a lane's offset
// in a tile, up to 255 rows, is 32 bits. All operands at 16 bytes; bias only for the
// first two.
// tile and splits from the plan; part: splits * rows * columns of all outputs,
// null for one split; merge 0 leaves these for the next kernel to add up, in
// their order and with the bias (norms.hip, paged_attention.hip). Returns a
// hipError_t.
extern "C" int ds_tile_linear(const void* const* x, int layers,
                              const void* const* w, const void* const* bias,
                              void* const* out, const int* n, int M, int K,
                              int mode, int tile, int splits, float* part,
                              int merge, void* stream) {
  Args a = {};
  int total = 0, most = 0;
  for (int i = 0; i < layers; ++i) {
    most = n[i] > most ? n[i] : most;
    a.w[i] = (const short*)w[mode == GRAD_W ? 0 : i];
    a.x[i] = (const short*)x[mode >= GRAD_X ? i : 0];
    a.bias[i] = mode >= GRAD_X ? nullptr : (const short*)bias[i];
    a.out[i] = (short*)out[mode == GRAD_X || mode == SWIGLU ? 0 : i];
    a.n[i] = n[i];
    a.n_end[i] = total += n[i];
  }
  a.part = part;
  a.M = M; a.K = K; a.layers = layers; a.splits = splits;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  if (tile == WIDE && past_wide(mode, mode >= GRAD_X ? K : total, most))
    return (int)hipErrorInvalidValue;
  const int steps = mode == GRAD_X ? total / BK
      : mode == GRAD_W ? (M + BK - 1) / BK : K / BK;
  if (by_four(tile, M, K, steps, splits, mode) &&
      !past_wide(mode, mode >= GRAD_X ? K : total, most)) {
#define FOUR(BM, BN)                                                    \
  mode == GRAD_X ? launch_four<BM, BN, GRAD_X>(a, st)                   \
      : mode == GRAD_W ? launch_four<BM, BN, GRAD_W>(a, st)             \
      : launch_four<BM, BN, PLAIN>(a, st)
    if (tile == SQUARE) return FOUR(192, 192);
    if (tile == NARROW) return FOUR(256, 192);
    if (mode == SWIGLU) return launch_four<192, 256, SWIGLU>(a, st);
    return FOUR(192, 256);
#undef FOUR
  }
  switch (tile) {
#define X(I, BM, BN, WM, WN, NS, U, F)                                    \
  case I:                                                                 \
    if (mode == GRAD_X)                                                   \
      return launch<BM, BN, WM, WN, NS, GRAD_X>(a, merge, st);            \
    if (mode == GRAD_W)                                                   \
      return launch<BM, BN, WM, WN, NS,                                   \
                    BLOCKS(BM, WM) ? GRAD_W : PLAIN>(a, merge, st);       \
    if (mode == SWIGLU)                                                   \
      return launch<BM, BN, WM, WN, NS,                                   \
                    GATES(BN, WN) ? SWIGLU : PLAIN>(a, merge, st);        \
    return launch<BM, BN, WM, WN, NS, PLAIN>(a, merge, st);
    TILES(X)
    BETWEEN(X)
#undef X
  case EIGHT:
    if (mode == GRAD_X) return launch<256, 256, 2, 4, 2, GRAD_X>(a, merge, st);
    if (mode == GRAD_W) return launch<256, 256, 2, 4, 2, GRAD_W>(a, merge, st);
    if (mode == SWIGLU) return launch<256, 256, 2, 4, 2, SWIGLU>(a, merge, st);
    break;
  case WIDE:
    if (mode == GRAD_X) return launch_wide<GRAD_X>(a, merge, st);
    if (mode == GRAD_W) return launch_wide<GRAD_W>(a, merge, st);
    if (mode == SWIGLU) return launch_wide<SWIGLU>(a, merge, st);
    return launch_wide<PLAIN>(a, merge, st);
  }
  return (int)hipErrorInvalidValue;
}
