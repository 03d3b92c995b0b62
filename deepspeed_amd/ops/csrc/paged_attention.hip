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
//   rows     the split-KV attention described below.
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
//     waves a SIMD. 55 us a layer at 32 requests of 2000 tokens and 8 key
//     heads (4.8 TB/s), 100 us at 8 of 16000 (5.2 TB/s; a large copy reaches
//     5.0). One position a wave at a time (2-byte loads, a six-step shuffle
//     chain each) took 240 and 459 us. A portion of 1024 tokens behind 1500
//     takes 123 us, on two tiles of columns an item.
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

#include "ds_kernels.h"

namespace {

typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 b16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

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

__device__ __forceinline__ s16x4 tr_read(const short* p) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (__attribute__((address_space(3))) s16x4*)p);
}

__device__ __forceinline__ short bits(float x) {
  return __builtin_bit_cast(short, (__bf16)x);
}
__device__ __forceinline__ float value(short x) {
  return __builtin_bit_cast(float, (unsigned)(unsigned short)x << 16);
}

// One tile of keys: ALIGNED blocks (BS a multiple of 32) hold it whole.
template <bool ALIGNED>
struct Tile {
  s16x8 k[2][4], v[8];

  __device__ __forceinline__ void load(const Args& a, const int* tab, int hkv,
                                       int kb, int kv_len, int lane) {
    const int row = lane & 15, g = lane >> 4;
    if (ALIGNED) {
      const long long blk = tab[kb / a.BS];
      const long long base = ((blk * a.Hkv + hkv) * a.BS + kb % a.BS) * D;
      const short* kp = a.kpool + base + row * D + 8 * g;
      const short* vp = a.vpool + base + g * D + 8 * row;
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int kk = 0; kk < 4; ++kk)
          k[t][kk] = *(const s16x8*)(kp + t * 16 * D + kk * 32);
#pragma unroll
      for (int i = 0; i < 8; ++i) v[i] = *(const s16x8*)(vp + i * 4 * D);
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

  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
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

  Tile<ALIGNED> x;
  int kb = key0 + wid * KT;
  if (kb < key1) x.load(a, tab, hkv, kb, kv_len, lane);
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
    if (kb + NW * KT < key1)
      x.load(a, tab, hkv, kb + NW * KT, kv_len, lane);

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

// merges[i] = {first item, items, 0, 0}; one workgroup a column. Waits on
// memory only: 128 threads read an item's 512 bytes, items unrolled by four.
template <int NQ>
__global__ __launch_bounds__(D) void merge_kernel(const Args a,
                                                  const int2* merges) {
  const int hkv = blockIdx.y, c = blockIdx.z, G = a.H / a.Hkv;
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
  if (rr >= m * G) return;
  const long long stride = (long long)a.Hkv * (16 * NQ);
  const long long at = ((long long)first * a.Hkv + hkv) * (16 * NQ) + c;
  float mg = -1e30f;
  for (int i = 0; i < n; ++i)
    mg = fmaxf(mg, a.part_ml[(at + i * stride) * 2]);
  float lg = 0.f, o = 0.f;
#pragma unroll 4
  for (int i = 0; i < n; ++i) {
    const float al = __builtin_amdgcn_exp2f(
        (a.part_ml[(at + i * stride) * 2] - mg) * a.c);
    lg += a.part_ml[(at + i * stride) * 2 + 1] * al;
    o += a.part[(at + i * stride) * D + threadIdx.x] * al;
  }
  const float inv = lg > 0.f ? 1.f / lg : 0.f;
  a.out[((long long)(row0 + rr / G) * a.H + hkv * G + rr % G) * D +
        threadIdx.x] = bits(o * (lg != lg ? lg : inv));
}

// Eight threads a head row of 128: coordinates j..j+7 and j+64..j+71 of it.
__global__ __launch_bounds__(256) void append_kernel(
    const short* __restrict__ q, const short* __restrict__ k,
    const short* __restrict__ v, short* __restrict__ qout,
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
  const short* src;
  short* to;
  bool turn = cs != nullptr;
  if (cs && h < H) {
    src = q + ((long long)t * H + h) * D;
    to = qout + ((long long)t * H + h) * D;
  } else {
    if (cs) h -= H;
    const bool is_k = h < Hkv;
    if (!is_k) h -= Hkv;
    src = (is_k ? k : v) + ((long long)t * Hkv + h) * D;
    const int at = dst[t];
    to = (is_k ? kpool : vpool) +
         (((long long)(at / BS) * Hkv + h) * BS + at % BS) * D;
    turn = turn && is_k;
  }
  s16x8 x1 = *(const s16x8*)(src + j), x2 = *(const s16x8*)(src + j + 64);
  if (turn) {
    const int pos = positions ? positions[t] : t % S;
    const float* cp = cs + (long long)pos * 64 + j;
    const float* sp = sn + (long long)pos * 64 + j;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float a = value(x1[e]), b = value(x2[e]);
      x1[e] = bits(a * cp[e] - b * sp[e]);
      x2[e] = bits(b * cp[e] + a * sp[e]);
    }
  }
  *(s16x8*)(to + j) = x1;
  *(s16x8*)(to + j + 64) = x2;
}

template <int NQ>
void launch_rows(const Args& a, const int2* merges, int n_items, int n_merges,
                 bool any_merge, hipStream_t st) {
  const dim3 grid(n_items, a.Hkv);
  if (a.BS % KT == 0)
    hipLaunchKernelGGL((rows_kernel<NQ, true>), grid, dim3(NW * 64), 0, st, a);
  else
    hipLaunchKernelGGL((rows_kernel<NQ, false>), grid, dim3(NW * 64), 0, st,
                       a);
  if (any_merge)
    hipLaunchKernelGGL((merge_kernel<NQ>), dim3(n_merges, a.Hkv, 16 * NQ),
                       dim3(D), 0, st, a, merges);
}

}  // namespace

extern "C" void ds_paged_append(const void* q, const void* k, const void* v,
                                void* qout, void* kpool, void* vpool,
                                const int* dst, const float* cs,
                                const float* sn, const int* positions, int T,
                                int S, int H, int Hkv, int BS, void* stream) {
  const long long threads = (long long)T * ((cs ? H : 0) + 2 * Hkv) * 8;
  hipLaunchKernelGGL(append_kernel, dim3((unsigned)((threads + 255) / 256)),
                     dim3(256), 0, reinterpret_cast<hipStream_t>(stream),
                     (const short*)q, (const short*)k, (const short*)v,
                     (short*)qout, (short*)kpool, (short*)vpool, dst, cs, sn,
                     positions, T, S, H, Hkv, BS);
}

// nq: tiles of 16 columns an item (1 or 2). runs/items/merges null: `lens`
// and `splits` describe one row a run.
extern "C" void ds_paged_rows(const void* q, const void* kpool,
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
  if (nq == 1)
    launch_rows<1>(a, (const int2*)merges, n_items, n_merges, any_merge, st);
  else
    launch_rows<2>(a, (const int2*)merges, n_items, n_merges, any_merge, st);
}
