// Attention over the paged key/value pool for MI355X (gfx950).
//
// Reference analogue: inference/v2/kernels/ragged_ops/blocked_flash and
// linear_blocked_kv_rotary (rotary embedding fused with the cache write).
//
// A serving step is a list of RUNS: m new tokens of one request at the
// positions kv_len - m .. kv_len - 1. Three kernels serve every step, be it
// single-token decoding, a portion of a prompt or both packed together:
//
//   append   rotary embedding of the new queries and keys (optional) and the
//            new rows of keys and values written into their blocks, one launch
//            for the whole step: 3.4 us a layer at 32 requests, 7.5 us for a
//            portion of 1024 tokens. As two strided copies a token it took 159
//            us a layer (64 launches) and 5.2 ms (2051 launches).
//            Of a few rows the products of q, k and v write them themselves
//            (rows_linear.hip).
//   rows     the split-KV attention described below; for steps of long runs
//            block_kernel.
//   merge    log-sum-exp merge of the splits, only where there is more than
//            one.
//
// rows: a work item is (run, a tile of 16*NQ columns, a range of keys); a
// column is one query row of the group of H/Hkv heads that share a key head,
// token-major, so a decoding request with 4 heads a key head fills 4 of 16
// columns and reads its keys and values ONCE. The four waves of a workgroup
// take every fourth tile of 32 keys and merge through LDS at the end.
//
//   * Bound by the stream of K and V (decode): 16-byte loads, the next tile in
//     flight while the softmax and the second product of this one run, three
//     waves a SIMD. 48 us a layer at 32 requests of 2000 tokens and 8 key
//     heads (5.5 TB/s), 83 to 91 us at 8 of 16000 (5.8 to 6.3 TB/s; a large
//     read reaches 6.3, past the caches 7.0). One position a wave at a time
//     (2-byte loads, a six-step shuffle chain each) took 240 and 459 us.
//   * S^T = K Q^T on mfma_f32_16x16x32_bf16: K rows go from global memory
//     straight into A fragments (64 contiguous bytes a row and instruction).
//     Lane (g = lane >> 4) then holds the scores of keys 16 t + 4 g + r of
//     column lane & 15.
//   * O^T = V^T P^T needs eight consecutive keys a lane. The order of keys
//     inside a product is free, so key 16 (j >> 2) + 4 g + (j & 3) is made the
//     lane's j-th: the probabilities stay in the registers they were computed
//     in, and V is read from LDS with ds_read_b64_tr_b16, four keys of one
//     coordinate a lane. The LDS rows are swizzled (16-byte chunk ^ row), which
//     leaves neither the stores nor the transposing loads a bank conflict.
//   * Probabilities are fp32; the matrix core takes them as the sum of two
//     bf16 numbers (p = hi + lo, relative remainder 2^-18), which the matrix
//     cores have time for: against fp64 the result is off by its own rounding
//     to bf16 and no more (0.001668 of it at 32 requests of 2000, 0.001649 at 8
//     of 16000, with fp32 probabilities the same to six digits).
//
// Layouts: q [T, H, 128], pool [blocks, Hkv, BS, 128], out [T, H, 128], bf16.

#include "attention_tile.h"
#include "ds_kernels.h"

namespace {

using namespace attn;
using attn::mfma;

constexpr int D = 128;
constexpr int KT = 32;        // keys a tile
constexpr int NW = 4;         // waves a workgroup
constexpr int OSTR = D + 4;   // floats between columns of a merged tile

// runs[j] = {first row, rows, keys including the new ones, offset of the
// run's blocks in the table}; items[i] = {run, tile of columns, first key,
// end of keys}, the end negated where the item is its tile's only one.
struct Args {
  const short* q;
  const short* kpool;
  const short* vpool;
  const int* table;
  const int4* runs;     // null: one row a run, `lens` keys, `splits` items
  const int4* items;
  const int* lens;
  short* out;
  float* part;          // [items, Hkv, 16 NQ, 128]
  float* part_ml;       // [items, Hkv, 16 NQ, 2]
  int H, Hkv, BS, max_blocks, splits;
  float c;              // |scale| * log2(e)
  bool flip;            // scale < 0
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

// One tile of keys: ALIGNED blocks (BS a multiple of 32) hold it whole, the block `id`.
// ONCE, where no other columns read them: V, whole lines of it a load, passes the
// caches by (8 requests of 16000 105 -> 95 us; but 24 of 1000 beside a run of 200 rows,
// whose tiles share its keys, 40 -> 46); K's lines are four loads', which find them
// there.
template <bool ALIGNED, bool ONCE>
struct Keys {
  s16x8 k[2][4], v[8];

  __device__ __forceinline__ void load(const Args& a, const int* tab, int id,
                                       int hkv, int kb, int kv_len, int lane) {
    const int row = lane & 15, g = lane >> 4;
    if (ALIGNED) {
      const long long blk = id;
      const long long base = ((blk * a.Hkv + hkv) * a.BS + kb % a.BS) * D;
      const short* kp = a.kpool + base + row * D + 8 * g;
      const short* vp = a.vpool + base + g * D + 8 * row;
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int kk = 0; kk < 4; ++kk)
          k[t][kk] = *(const s16x8*)(kp + t * 16 * D + kk * 32);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const s16x8* p = (const s16x8*)(vp + i * 4 * D);
        v[i] = ONCE ? __builtin_nontemporal_load(p) : *p;
      }
    } else {
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const int key = min(kb + 16 * t + row, kv_len - 1);
        const long long at = (((long long)tab[key / a.BS] * a.Hkv + hkv) *
                                  a.BS + key % a.BS) * D + 8 * g;
#pragma unroll
        for (int kk = 0; kk < 4; ++kk)
          k[t][kk] = *(const s16x8*)(a.kpool + at + kk * 32);
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int key = min(kb + 4 * i + g, kv_len - 1);
        v[i] = *(const s16x8*)(a.vpool +
                               (((long long)tab[key / a.BS] * a.Hkv + hkv) *
                                    a.BS + key % a.BS) * D + 8 * row);
      }
    }
  }
};

template <int NQ, bool ALIGNED>
__global__ __launch_bounds__(NW * 64, NQ == 1 ? 3 : 2) void rows_kernel(const Args a) {
  __shared__ __attribute__((aligned(16))) float lds[NW][16 * OSTR];
  __shared__ float lds_ml[NW][NQ * 16][2];
  static_assert(16 * OSTR * 4 >= KT * D * 2, "the V tile fits");

  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, g = lane >> 4;
  const int hkv = blockIdx.y, G = a.H / a.Hkv;

  int row0, m, kv_len, tab_at, tile, key0, key1;
  bool sole;
  if (a.runs) {
    const int4 it = a.items[blockIdx.x];
    const int4 run = a.runs[it.x];
    row0 = run.x; m = run.y; kv_len = run.z; tab_at = run.w;
    tile = it.y; key0 = it.z; sole = it.w < 0; key1 = abs(it.w);
  } else {
    const int j = blockIdx.x / a.splits, s = blockIdx.x % a.splits;
    row0 = j; m = 1; kv_len = a.lens[j]; tab_at = j * a.max_blocks;
    tile = 0; sole = a.splits == 1;
    const int per = ((kv_len + a.splits - 1) / a.splits + KT - 1) / KT * KT;
    key0 = min(kv_len, s * per);
    key1 = min(kv_len, key0 + per);
  }
  const int* tab = a.table + tab_at;
  const int ncols = m * G;

  // ---- query fragments; a column past the last repeats the last
  s16x8 qf[NQ][4];
  int limit[NQ];          // the last key that the lane's column sees
#pragma unroll
  for (int n = 0; n < NQ; ++n) {
    const int rr = min((tile * NQ + n) * 16 + col, ncols - 1);
    const int tok = rr / G;
    const short* qp = a.q + ((long long)(row0 + tok) * a.H + hkv * G +
                             rr % G) * D + 8 * g;
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
      qf[n][kk] = *(const s16x8*)(qp + kk * 32);
      if (a.flip)   // a negative scale: the maxima below want c > 0
        qf[n][kk] ^= s16x8{-32768, -32768, -32768, -32768,
                           -32768, -32768, -32768, -32768};
    }
    limit[n] = kv_len - m + tok;
  }
  const int low = kv_len - m + (tile * NQ * 16) / G;  // the first column's

  float mx[NQ], l[NQ];
  f32x4 acc[NQ][8];
#pragma unroll
  for (int n = 0; n < NQ; ++n) {
    mx[n] = -1e30f;
    l[n] = 0.f;
#pragma unroll
    for (int d = 0; d < 8; ++d) acc[n][d] = f32x4{0.f, 0.f, 0.f, 0.f};
  }

  short* vt = (short*)lds[wid];
  // transposing read: lane s = lane & 15 of a group of 16 points at key s >> 2
  // and coordinates 4 (s & 3)..; swizzled by the row
  const int xr = 4 * g + (col >> 2);
  const int xc = (col & 3) >> 1, xe = (col & 1) * 4;

  Keys<ALIGNED, NQ == 1> x;
  int kb = key0 + wid * KT;
  // Blocks are looked up a tile ahead of the loads from them: a wave has one tile in
  // flight, and waited for the table's entry before each (8 requests of 16000 in 2 and
  // 12 splits 204 / 142 and 95 / 92 us, 32 of 2000 whole 58 / 48).
  auto find = [&](int k) __attribute__((always_inline)) {
    return ALIGNED ? tab[min(k, key1 - 1) / a.BS] : 0;
  };
  int id = 0;
  if (kb < key1) {
    x.load(a, tab, find(kb), hkv, kb, kv_len, lane);
    id = find(kb + NW * KT);
  }
  for (; kb < key1; kb += NW * KT) {
    // V into LDS (own region of the wave: its LDS operations keep their order)
    if (kb + KT > kv_len) {   // rows past the end: whatever the pool holds
#pragma unroll
      for (int i = 0; i < 8; ++i)
        if (kb + 4 * i + g >= kv_len) x.v[i] = s16x8{0, 0, 0, 0, 0, 0, 0, 0};
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int r = 4 * i + g;
      *(s16x8*)(vt + (r * 16 + (col ^ (r & 15))) * 8) = x.v[i];
    }
    // scores
    f32x4 s[NQ][2];
#pragma unroll
    for (int n = 0; n < NQ; ++n)
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        s[n][t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kk = 0; kk < 4; ++kk)
          s[n][t] = mfma(x.k[t][kk], qf[n][kk], s[n][t]);
      }
    // the next tile's loads run behind the rest of this one
    if (kb + NW * KT < key1) {
      x.load(a, tab, id, hkv, kb + NW * KT, kv_len, lane);
      id = find(kb + 2 * NW * KT);
    }

    const bool whole = kb + KT <= key1 && kb + KT - 1 <= low;
    s16x8 hi[NQ], lo[NQ];
#pragma unroll
    for (int n = 0; n < NQ; ++n) {
      const int last = min(limit[n], key1 - 1) - kb - 4 * g;
      float mt = -1e30f;
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          if (!whole && 16 * t + r > last) s[n][t][r] = -1e30f;
          mt = fmaxf(mt, s[n][t][r]);
        }
      mt = fmaxf(mt, __shfl_xor(mt, 16, 64));
      mt = fmaxf(mt, __shfl_xor(mt, 32, 64));
      if (__any(mt > mx[n])) {
        const float mn = fmaxf(mx[n], mt);
        const float alpha = __builtin_amdgcn_exp2f((mx[n] - mn) * a.c);
        mx[n] = mn;
        l[n] *= alpha;
#pragma unroll
        for (int d = 0; d < 8; ++d)
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[n][d][r] *= alpha;
      }
      const float mc = mx[n] * a.c;
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          float p = __builtin_amdgcn_exp2f(__builtin_fmaf(s[n][t][r], a.c,
                                                          -mc));
          if (!whole && 16 * t + r > last) p = 0.f;
          l[n] += p;
          const short h = bits(p);
          hi[n][4 * t + r] = h;
          lo[n][4 * t + r] = bits(p - value(h));
        }
    }
#pragma unroll
    for (int d = 0; d < 8; ++d) {
      const int at = (xr * 16 + ((2 * d + xc) ^ xr)) * 8 + xe;
      const s16x4 v0 = tr_read(vt + at), v1 = tr_read(vt + 16 * D + at);
      const s16x8 va = {v0[0], v0[1], v0[2], v0[3],
                        v1[0], v1[1], v1[2], v1[3]};
#pragma unroll
      for (int n = 0; n < NQ; ++n) {
        acc[n][d] = mfma(va, hi[n], acc[n][d]);
        acc[n][d] = mfma(va, lo[n], acc[n][d]);
      }
    }
  }

  // ---- merge the four waves, one tile of 16 columns at a time
#pragma unroll
  for (int n = 0; n < NQ; ++n) {
    l[n] += __shfl_xor(l[n], 16, 64);
    l[n] += __shfl_xor(l[n], 32, 64);
    if (g == 0) {
      lds_ml[wid][n * 16 + col][0] = mx[n];
      lds_ml[wid][n * 16 + col][1] = l[n];
    }
    __syncthreads();      // the V tiles, or the last columns, have been read
#pragma unroll
    for (int d = 0; d < 8; ++d)
      *(f32x4*)(&lds[wid][col * OSTR + 16 * d + 4 * g]) = acc[n][d];
    __syncthreads();
    const int c = threadIdx.x >> 4, d0 = (threadIdx.x & 15) * 8;
    const int rr = (tile * NQ + n) * 16 + c;
    if (rr < ncols) {
      float mg = -1e30f, lg = 0.f, o[8] = {};
#pragma unroll
      for (int w = 0; w < NW; ++w) mg = fmaxf(mg, lds_ml[w][n * 16 + c][0]);
#pragma unroll
      for (int w = 0; w < NW; ++w) {
        const float al = __builtin_amdgcn_exp2f(
            (lds_ml[w][n * 16 + c][0] - mg) * a.c);
        lg += lds_ml[w][n * 16 + c][1] * al;
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] += lds[w][c * OSTR + d0 + e] * al;
      }
      if (sole) {
        const float inv = lg > 0.f ? 1.f / lg : 0.f;
        s16x8 ob;
#pragma unroll
        for (int e = 0; e < 8; ++e) ob[e] = bits(o[e] * (lg != lg ? lg : inv));
        *(s16x8*)(a.out + ((long long)(row0 + rr / G) * a.H + hkv * G +
                           rr % G) * D + d0) = ob;
      } else {
        const long long at =
            ((long long)blockIdx.x * a.Hkv + hkv) * (16 * NQ) + n * 16 + c;
#pragma unroll
        for (int e = 0; e < 8; e += 4)
          *(f32x4*)(a.part + at * D + d0 + e) =
              f32x4{o[e], o[e + 1], o[e + 2], o[e + 3]};
        if (d0 == 0) {
          a.part_ml[at * 2] = mg;
          a.part_ml[at * 2 + 1] = lg;
        }
      }
    }
  }
}

// ---- runs of many columns

constexpr int BC = 128, BK = 128;     // columns and keys of a step
constexpr int BNW = 8;                // waves
constexpr int KROW = D * 2;           // bytes of a row in LDS
constexpr int HALF = BK * KROW;       // LDS: keys of two steps, then values
constexpr int VALUES = 2 * HALF;
constexpr int AHEAD = 2;              // operands read before their product

// on lambdas: one that is not inlined takes what it captures to scratch memory
#define INLINE __attribute__((always_inline))

__device__ __forceinline__ int uni(int x) {
  return __builtin_amdgcn_readfirstlane(x);
}
typedef int i32x4 __attribute__((ext_vector_type(4)));
struct True { static constexpr bool value = true; };
struct False { static constexpr bool value = false; };

// Registers 8 s + 2 i and the next as two bf16 numbers each, whose sum they are
// but for 2^-18.
__device__ __forceinline__ void split2(const f32x16& p, int s, int i,
                                       i32x4& hi, i32x4& lo) {
  const float a = p[8 * s + 2 * i], b = p[8 * s + 2 * i + 1];
  const int h = pack2(a, b);
  hi[i] = h;
  lo[i] = pack2(a - __builtin_bit_cast(float, h << 16),
                b - __builtin_bit_cast(float, (int)(h & 0xffff0000)));
}

// An item is (run, a tile of 128 columns, a range of keys). Four waves own 32
// columns each over the first 64 keys of a step, four over the last 64, and the
// two of a column are merged through LDS at the end: 256 items are a chip full
// of two waves a SIMD, where one wave a column would leave the half of it idle.
// K and V go from the pool's blocks straight into LDS behind the products of a
// step before. Bound by the vector unit beside the matrix cores, so the two work
// at once: the scores of the next step are made between the exponentials of this
// one, its probabilities split in two between the products of its values. A
// portion of 1024 tokens behind 1500, 32 on 8 heads, alone: 74 us (457 TFLOP/s,
// 685 with the second halves of the probabilities); without that order 82, on
// rows_kernel's tiles of 32 columns, which load a key four times as often, 104.
// Between the layers' products, at the clock that these leave, 100 and 123.
template <bool ALIGNED>
__global__ __launch_bounds__(BNW * 64) void block_kernel(const Args a) {
  using T = Tile<D>;
  constexpr int DB = D / 32, KK = D / 16;
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int lane = threadIdx.x & 63, wid = uni(threadIdx.x >> 6);
  const int col = lane & 31, half = lane >> 5;
  const int cg = wid & 3, kg = wid >> 2;
  const int hkv = uni(blockIdx.x % a.Hkv), item = uni(blockIdx.x / a.Hkv);
  const int G = a.H / a.Hkv;
  const int4 it4 = a.items[item];
  const int4 run = a.runs[it4.x];
  const int row0 = run.x, kv_len = run.z, first = kv_len - run.y;
  const int ncols = run.y * G, c0 = it4.y * BC + cg * 32;
  const int key0 = uni(it4.z), key1 = uni(abs(it4.w));
  const int* tab = a.table + run.w;

  const int rr = min(c0 + col, ncols - 1), tok = rr / G;
  const long long at = (long long)(row0 + tok) * a.H + hkv * G + rr % G;
  s16x8 qf[KK];
  {
    const short* qp = a.q + at * D + 8 * half;
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
      qf[kk] = *(const s16x8*)(qp + 16 * kk);
      if (a.flip)   // a negative scale: the maxima below want c > 0
        qf[kk] ^= s16x8{-32768, -32768, -32768, -32768,
                        -32768, -32768, -32768, -32768};
    }
  }
  // the last key that the column sees here, and that the wave's first one does
  const int limit = min(first + tok, key1 - 1);
  const int low = uni(min(first + min(c0, ncols - 1) / G, key1 - 1));
  const bool active = c0 < ncols;
  // a scale of 0, too, leaves the probability 0 to keys that are not seen, and
  // one that is no number gives none
  const float c = a.c < 1e-30f ? 1e-30f : a.c;

  // Rows i * 32 + 4 wid + lane / 16 of a step, chunks by the tile's swizzle; an
  // aligned block holds the four rows of a wave's load. Rows past the last key
  // repeat it.
  const int lr = 4 * wid + (lane >> 4);
  const int lds0 = lds_at(lds);
  int ids[2][4];      // blocks of the next values, of the next keys but one
  auto find = [&](int (&id)[4], int kb) INLINE {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      id[i] = tab[min(kb + i * 32 + (ALIGNED ? 4 * wid : lr), kv_len - 1) /
                  a.BS];
  };
  auto fetch = [&](const short* pool, const int (&id)[4], int kb, int buf)
      INLINE {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = i * 32 + lr, key = min(kb + r, kv_len - 1);
      const int in = ALIGNED
          ? key - min(kb + i * 32 + 4 * wid, kv_len - 1) / a.BS * a.BS
          : key % a.BS;
      const int blk = ALIGNED ? uni(id[i]) : id[i];
      const long long off =
          ((((long long)blk * a.Hkv + hkv) * a.BS + in) * D) +
          (((lane & 15) ^ T::turn(r)) << 3);
      load_lds(pool + off, lds0 + buf + (i * 32 + 4 * wid) * KROW);
    }
  };

  const int ra = T::rows_at(lane), ca = T::cols_at(lane);
  const char* own = lds + 64 * kg * KROW;     // the wave's half of a buffer
  float m = -1e30f, l = 0.f;
  f32x16 acc[DB] = {};
  // the maximum of the scores p of the keys from k0 on, past the last key none
  auto top = [&](f32x16 (&p)[2], int k0) INLINE {
    if (k0 + 63 > low) {
      const int last = limit - k0 - 4 * half;
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (32 * t + (r & 3) + 8 * (r >> 2) > last) p[t][r] = -3e38f;
    }
    float mt = -1e30f;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) mt = fmaxf(mt, p[t][r]);
    mt = fmaxf(mt, __shfl_xor(mt, 32, 64));
    // raised only where it grows by more than 2^8: most steps rescale nothing
    if (!__all((mt - m) * c <= 8.f)) {
      const float mn = fmaxf(m, mt);
      const float alpha = __builtin_amdgcn_exp2f((m - mn) * c);
      m = mn;
      l *= alpha;
#pragma unroll
      for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[db][r] *= alpha;
    }
  };
  // Product i of the 16 of a step's scores takes half kk = i / 2 of tile i % 2.
  auto key = [&](int buf, int i) INLINE {
    return T::rows((const short*)(own + buf), 32 * (i % 2), i / 2, ra);
  };
  // p: scores to probabilities; q: the scores of the keys in ``next``
  auto soften = [&](auto more, f32x16 (&p)[2], f32x16 (&q)[2], int next)
      INLINE {
    constexpr bool MORE = decltype(more)::value;
    const float mc = m * c;
    float l0 = 0.f, l1 = 0.f;
    s16x8 k[AHEAD + 1];
    if constexpr (MORE) {
      q[0] = q[1] = f32x16{};
#pragma unroll
      for (int i = 0; i < AHEAD; ++i) k[i] = key(next, i);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int t = i / 8, r = i % 8 * 2;
      if constexpr (MORE) {
        if (i + AHEAD < 16) k[(i + AHEAD) % (AHEAD + 1)] = key(next, i + AHEAD);
        q[i % 2] = mfma(k[i % (AHEAD + 1)], qf[i / 2], q[i % 2]);
      }
      p[t][r] = __builtin_amdgcn_exp2f(__builtin_fmaf(p[t][r], c, -mc));
      p[t][r + 1] =
          __builtin_amdgcn_exp2f(__builtin_fmaf(p[t][r + 1], c, -mc));
      l0 += p[t][r];
      l1 += p[t][r + 1];
      __builtin_amdgcn_sched_barrier(0);
    }
    l += l0 + l1;
  };
  // Products i and the next are of coordinates 32 (i % 4).. and of probabilities
  // 8 (i / 4)..
  auto values = [&](const f32x16 (&p)[2], int buf) INLINE {
    const short* vt = (const short*)(own + VALUES + buf);
    auto value = [&](int i) INLINE {
      return T::cols(vt, 16 * (i / 4), i % 4, ca);
    };
    s16x8 v[AHEAD + 1];
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) v[i] = value(i);
    i32x4 hi, lo, nhi, nlo;
#pragma unroll
    for (int i = 0; i < 4; ++i) split2(p[0], 0, i, hi, lo);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int g = i / 4 + 1;
      if (i + AHEAD < 16) v[(i + AHEAD) % (AHEAD + 1)] = value(i + AHEAD);
      const s16x8 x = v[i % (AHEAD + 1)];
      acc[i % 4] = mfma(x, __builtin_bit_cast(s16x8, hi), acc[i % 4]);
      if (g < 4) split2(p[g / 2], g % 2, i % 4, nhi, nlo);
      acc[i % 4] = mfma(x, __builtin_bit_cast(s16x8, lo), acc[i % 4]);
      if (i % 4 == 3) { hi = nhi; lo = nlo; }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // A step of the keys from kb on, whose scores are p; the next step's go to q.
  auto step = [&](f32x16 (&p)[2], f32x16 (&q)[2], int kb, int buf) INLINE {
    const int next = buf ^ HALF;
    if (kb + BK < key1) {
      fetch(a.vpool, ids[0], kb + BK, next + VALUES);
      if (kb + 2 * BK < key1) fetch(a.kpool, ids[1], kb + 2 * BK, buf);
#pragma unroll
      for (int i = 0; i < 4; ++i) ids[0][i] = ids[1][i];
      find(ids[1], kb + 3 * BK);
    }
    if (active) {
      top(p, kb + 64 * kg);
      if (kb + BK < key1) soften(True(), p, q, next);
      else soften(False(), p, q, next);
      values(p, buf);
    }
    arrive();
  };

  f32x16 p[2] = {}, q[2];
  find(ids[0], key0);
  fetch(a.kpool, ids[0], key0, 0);
  fetch(a.vpool, ids[0], key0, VALUES);
  find(ids[0], key0 + BK);
  fetch(a.kpool, ids[0], key0 + BK, HALF);
  find(ids[1], key0 + 2 * BK);
  arrive();
#pragma unroll
  for (int i = 0; i < 16; ++i)
    p[i % 2] = mfma(key(0, i), qf[i / 2], p[i % 2]);
  // all keys have been read where the next but one are loaded
  arrive();
  for (int kb = key0;; kb += 2 * BK) {
    step(p, q, kb, 0);
    if (kb + BK >= key1) break;
    step(q, p, kb + BK, HALF);
    if (kb + 2 * BK >= key1) break;
  }

  // ---- the two waves of a column
  l += __shfl_xor(l, 32, 64);
  f32x4* po = (f32x4*)(lds + cg * 16384) + lane;
  float2* pm = (float2*)(lds + 4 * 16384) + cg * 64 + lane;
  if (kg == 1) {
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        po[(4 * db + g) * 64] = f32x4{acc[db][4 * g], acc[db][4 * g + 1],
                                      acc[db][4 * g + 2], acc[db][4 * g + 3]};
    *pm = float2{m, l};
  }
  arrive();
  if (kg == 1 || c0 + col >= ncols) return;
  const float2 o = *pm;
  const float mg = fmaxf(m, o.x);
  const float a0 = __builtin_amdgcn_exp2f((m - mg) * c);
  const float a1 = __builtin_amdgcn_exp2f((o.x - mg) * c);
  const float lg = l * a0 + o.y * a1;
  const bool sole = it4.w < 0;
  const float inv = !sole ? 1.f : lg > 0.f ? 1.f / lg : lg != lg ? lg : 0.f;
  const long long pat = ((long long)item * a.Hkv + hkv) * BC + cg * 32 + col;
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const f32x4 y = po[(4 * db + g) * 64];
      const int d = 32 * db + 8 * g + 4 * half;
      f32x4 x;
#pragma unroll
      for (int e = 0; e < 4; ++e)
        x[e] = (acc[db][4 * g + e] * a0 + y[e] * a1) * inv;
      if (sole) {
        typedef int i32x2 __attribute__((ext_vector_type(2)));
        *(i32x2*)(a.out + at * D + d) =
            i32x2{pack2(x[0], x[1]), pack2(x[2], x[3])};
      } else {
        *(f32x4*)(a.part + pat * D + d) = x;
      }
    }
  if (!sole && half == 0) {
    a.part_ml[pat * 2] = mg;
    a.part_ml[pat * 2 + 1] = lg;
  }
}

// merges[i] = {first item, items}; NQ tiles of 16 columns an item, 32 threads a
// column. Waits on memory only: the maxima of 32 items in one load, four numbers
// of eight items in flight a thread (8 requests of 16000 9.5 -> 6.8 us, 24 of
// 1000 and a portion of 200 rows 9.0 -> 5.6, with a workgroup a column before).
template <int NQ>
__global__ __launch_bounds__(128) void merge_kernel(const Args a,
                                                    const int2* merges) {
  const int sub = threadIdx.x & 31;
  const int hkv = blockIdx.y, G = a.H / a.Hkv;
  const int c = blockIdx.z * 4 + (threadIdx.x >> 5);
  int first, n, row0, m, tile;
  if (a.runs) {
    first = merges[blockIdx.x].x;
    n = merges[blockIdx.x].y;
    const int4 it = a.items[first];
    const int4 run = a.runs[it.x];
    row0 = run.x; m = run.y; tile = it.y;
    if (it.w < 0) return;
  } else {
    first = blockIdx.x * a.splits;
    n = a.splits; row0 = blockIdx.x; m = 1; tile = 0;
  }
  const int rr = tile * NQ * 16 + c;
  if (rr >= m * G) return;      // the lanes of a column leave together
  const long long stride = (long long)a.Hkv * (16 * NQ);
  const long long at = ((long long)first * a.Hkv + hkv) * (16 * NQ) + c;
  float mg = -1e30f;
  for (int i = sub; i < n; i += 32)
    mg = fmaxf(mg, a.part_ml[(at + i * stride) * 2]);
#pragma unroll
  for (int off = 16; off > 0; off >>= 1)
    mg = fmaxf(mg, __shfl_xor(mg, off, 32));
  float lg = 0.f;
  f32x4 o = {0.f, 0.f, 0.f, 0.f};
  const float* p = a.part + at * D + sub * 4;
#pragma unroll 8
  for (int i = 0; i < n; ++i) {
    const float al = __builtin_amdgcn_exp2f(
        (a.part_ml[(at + i * stride) * 2] - mg) * a.c);
    lg += a.part_ml[(at + i * stride) * 2 + 1] * al;
    o += *(const f32x4*)(p + i * stride * D) * al;
  }
  const float inv = lg > 0.f ? 1.f / lg : lg != lg ? lg : 0.f;
  *(s16x4*)(a.out + ((long long)(row0 + rr / G) * a.H + hkv * G + rr % G) * D +
            sub * 4) = s16x4{bits(o[0] * inv), bits(o[1] * inv),
                             bits(o[2] * inv), bits(o[3] * inv)};
}

// Eight threads a head row of 128: coordinates j..j+7 and j+64..j+71 of it. With
// PARTS q, k and v are still in parts, part[splits][T][(H + 2 Hkv) 128], that
// tile_linear.hip's split contraction left, added up here in their order, with
// the bias and rounded as its merge would: a launch of 4 us at 32 requests less,
// for one more in this one.
template <bool PARTS>
__global__ __launch_bounds__(256) void append_kernel(
    const short* __restrict__ q, const short* __restrict__ k,
    const short* __restrict__ v,         // PARTS: the biases, or null
    const float* __restrict__ part, const int splits,
    short* __restrict__ qout,
    short* __restrict__ kpool, short* __restrict__ vpool,
    const int* __restrict__ dst,         // [T] block * BS + row in it
    const float* __restrict__ cs, const float* __restrict__ sn,  // or null
    const int* __restrict__ positions,   // [T] or null: t % S
    const int T, const int S, const int H, const int Hkv, const int BS) {
  const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  const int per = (cs ? H : 0) + 2 * Hkv;
  const long long u = i >> 3;
  if (u >= (long long)T * per) return;
  const int j = (int)(i & 7) * 8;
  const int t = (int)(u / per);
  int h = (int)(u % per);
  const int all = h;      // PARTS: the head among those of q, k and v
  const short* src;
  short* to;
  bool turn = cs != nullptr;
  if (cs && h < H) {
    src = PARTS ? (q ? q + h * D : nullptr) : q + ((long long)t * H + h) * D;
    to = qout + ((long long)t * H + h) * D;
  } else {
    if (cs) h -= H;
    const bool is_k = h < Hkv;
    if (!is_k) h -= Hkv;
    src = is_k ? k : v;
    if (PARTS) src = src ? src + h * D : nullptr;
    else src += ((long long)t * Hkv + h) * D;
    const int at = dst[t];
    to = (is_k ? kpool : vpool) +
         (((long long)(at / BS) * Hkv + h) * BS + at % BS) * D;
    turn = turn && is_k;
  }
  s16x8 x1, x2;
  if (PARTS) {
    f32x4 y[4] = {};
    const float* p = part + ((long long)t * per + all) * D + j;
#pragma unroll 4
    for (int s = 0; s < splits; ++s) {
      const float* ps = p + (long long)s * T * per * D;
#pragma unroll
      for (int e = 0; e < 4; ++e)
        y[e] += *(const f32x4*)(ps + (e >> 1) * 64 + (e & 1) * 4);
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      float a = y[e >> 2][e & 3], b = y[2 + (e >> 2)][e & 3];
      if (src) {
        a += value(src[j + e]);
        b += value(src[j + 64 + e]);
      }
      x1[e] = bits(a);
      x2[e] = bits(b);
    }
  } else {
    x1 = *(const s16x8*)(src + j);
    x2 = *(const s16x8*)(src + j + 64);
  }
  if (turn) {
    const int pos = positions ? positions[t] : t % S;
    const float* cp = cs + (long long)pos * 64 + j;
    const float* sp = sn + (long long)pos * 64 + j;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float a = value(x1[e]), b = value(x2[e]);
      const ds::Turned t = ds::turn(a, b, cp[e], sp[e]);
      x1[e] = bits(t.lo);
      x2[e] = bits(t.hi);
    }
  }
  *(s16x8*)(to + j) = x1;
  *(s16x8*)(to + j + 64) = x2;
}

template <bool ALIGNED>
int launch_block(const Args& a, int n_items, hipStream_t st) {
  const hipError_t e = hipFuncSetAttribute(
      (const void*)block_kernel<ALIGNED>,
      hipFuncAttributeMaxDynamicSharedMemorySize, 2 * VALUES);
  if (e != hipSuccess) return (int)e;
  hipLaunchKernelGGL(block_kernel<ALIGNED>, dim3((unsigned)n_items * a.Hkv),
                     dim3(BNW * 64), 2 * VALUES, st, a);
  return 0;
}

template <int NQ>
int launch_rows(const Args& a, const int2* merges, int n_items, int n_merges,
                bool any_merge, hipStream_t st) {
  const dim3 grid(n_items, a.Hkv);
  const bool aligned = a.BS % KT == 0;
  if constexpr (NQ * 16 == BC) {
    const int e = aligned ? launch_block<true>(a, n_items, st)
                          : launch_block<false>(a, n_items, st);
    if (e) return e;
  } else if (aligned) {
    hipLaunchKernelGGL((rows_kernel<NQ, true>), grid, dim3(NW * 64), 0, st, a);
  } else {
    hipLaunchKernelGGL((rows_kernel<NQ, false>), grid, dim3(NW * 64), 0, st,
                       a);
  }
  if (any_merge)
    hipLaunchKernelGGL((merge_kernel<NQ>), dim3(n_merges, a.Hkv, 4 * NQ),
                       dim3(128), 0, st, a, merges);
  return (int)hipGetLastError();
}

}  // namespace

// part: null, or q, k and v in parts (then these are their biases, or null, and
// there are tables).
extern "C" void ds_paged_append(const void* q, const void* k, const void* v,
                                const float* part, int splits, void* qout,
                                void* kpool, void* vpool, const int* dst,
                                const float* cs, const float* sn,
                                const int* positions, int T, int S, int H,
                                int Hkv, int BS, void* stream) {
  const long long threads = (long long)T * ((cs ? H : 0) + 2 * Hkv) * 8;
  auto kernel = part ? append_kernel<true> : append_kernel<false>;
  hipLaunchKernelGGL(kernel, dim3((unsigned)((threads + 255) / 256)),
                     dim3(256), 0, reinterpret_cast<hipStream_t>(stream),
                     (const short*)q, (const short*)k, (const short*)v, part,
                     splits, (short*)qout, (short*)kpool, (short*)vpool, dst,
                     cs, sn, positions, T, S, H, Hkv, BS);
}

// nq: tiles of 16 columns an item (1, 2 or 8). runs/items/merges null: `lens`
// and `splits` describe one row a run. Returns a hipError_t.
extern "C" int ds_paged_rows(const void* q, const void* kpool,
                              const void* vpool, const int* table,
                              const int* runs, const int* items,
                              const int* merges, const int* lens, void* out,
                              float* part, float* part_ml, int n_items,
                              int n_merges, int any_merge, int nq, int H,
                              int Hkv, int BS, int max_blocks, int splits,
                              float scale, void* stream) {
  Args a;
  a.q = (const short*)q;
  a.kpool = (const short*)kpool;
  a.vpool = (const short*)vpool;
  a.table = table;
  a.runs = (const int4*)runs;
  a.items = (const int4*)items;
  a.lens = lens;
  a.out = (short*)out;
  a.part = part;
  a.part_ml = part_ml;
  a.H = H; a.Hkv = Hkv; a.BS = BS; a.max_blocks = max_blocks;
  a.splits = splits;
  a.c = fabsf(scale) * 1.4426950408889634f;
  a.flip = scale < 0.f;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const int2* mg = (const int2*)merges;
  if (nq == 1) return launch_rows<1>(a, mg, n_items, n_merges, any_merge, st);
  if (nq == 2) return launch_rows<2>(a, mg, n_items, n_merges, any_merge, st);
  return launch_rows<8>(a, mg, n_items, n_merges, any_merge, st);
}
