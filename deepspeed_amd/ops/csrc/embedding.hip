// Gradient of an embedding's table for MI355X (gfx950), bf16: row v is the sum of
// the gradients of the tokens v, in their order, in fp32, rounded once. Rows of
// other tokens are left as they are (zero).
//
// Reference analogue: the sparse gradients of runtime/sparse_tensor.py, which
// also move only the rows that a batch touches.
//
// The rows are all the memory that has to move; what is in the way is to find the
// tokens of a row without a sort of the whole batch (ten launches in torch) and
// without sums in an order that the machine chooses. Two launches:
//
//   rank_kernel   256 tokens a workgroup, sorted by value and place by counting
//                 those before each (256 compares a thread out of LDS). A bit
//                 says that the block has the token, a table where.
//   sum_kernel    a wave per token and 512 columns; the first block's is the
//                 owner, goes through the blocks that have the token in order
//                 and adds up. From 32 rows on (frequent tokens, padding) the
//                 four waves of a workgroup share them and add up through LDS.
//
// us, into a table that is zero already; torch's, and with the addition to such a
// table: 1024 tokens of 32000 x 1024 16; 76, 101. 4000 of 32064 x 3072 25; 157, 278.
// 8192 of 128256 x 4096 41 (a new table's clearing included 214); 457, 990. 32768
// of these 201; 1268, 1797. Half of 8192 one token: 224; 455, 991.

#include "ds_kernels.h"

namespace {

typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int BLK = 256;      // tokens a block
constexpr int COLS = 512;     // columns a wave
constexpr int WAVES = 4;
constexpr int MANY = 32;      // rows that a workgroup shares
constexpr int AHEAD = 4;      // rows in flight a wave

__device__ __forceinline__ float value(short x) {
  return __builtin_bit_cast(float, (unsigned)(unsigned short)x << 16);
}
__device__ __forceinline__ short bits(float x) {
  return __builtin_bit_cast(short, (__bf16)x);
}

// order [T]: tokens' places, sorted inside each block; key [T]: their values;
// spans [V][blocks]: first place in the block's part of order, rows << 16;
// has [V][words]: blocks that have the value.
__global__ __launch_bounds__(BLK) void rank_kernel(
    const long long* __restrict__ ids, int* __restrict__ order,
    int* __restrict__ key, unsigned* __restrict__ has, int* __restrict__ spans,
    const int T, const int V, const long long padding, const int blocks,
    const int words) {
  __shared__ __attribute__((aligned(16))) int all[BLK];
  const int t = threadIdx.x, b = blockIdx.x, at = b * BLK + t;
  int mine = 0x7fffffff;        // past the end, and of no row: behind the others
  if (at < T) {
    const long long id = ids[at];
    if (id >= 0 && id < V && id != padding) mine = (int)id;
  }
  all[t] = mine;
  __syncthreads();
  int before = 0, same = 0, earlier = 0;
#pragma unroll 4
  for (int j = 0; j < BLK; j += 4) {
    const int4 x = *(const int4*)(all + j);
    const int e[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      before += e[i] < mine;
      same += e[i] == mine;
      earlier += e[i] == mine && j + i < t;
    }
  }
  // places past T lie behind: the last block holds T - b BLK of them in front
  const int to = b * BLK + before + earlier;
  if (to < T) {
    order[to] = at;
    key[to] = mine;
  }
  if (mine != 0x7fffffff && earlier == 0) {
    spans[(long long)mine * blocks + b] = before | same << 16;
    atomicOr(has + (long long)mine * words + b / 32, 1u << (b % 32));
  }
}

struct Rows {
  const short* grad;    // at the lane's columns
  const int* order;
  long long H;
  bool live;            // the lane has columns

  // rows first, first + step, .. of the n at order[at..]
  __device__ __forceinline__ void add(float (&sum)[8], int at, int n, int first,
                                      int step) const {
    for (int i = first; i < n; i += AHEAD * step) {
      s16x8 x[AHEAD];
#pragma unroll
      for (int a = 0; a < AHEAD; ++a) {
        const int j = i + a * step;
        x[a] = s16x8{0, 0, 0, 0, 0, 0, 0, 0};
        if (j < n && live) x[a] = *(const s16x8*)(grad + order[at + j] * H);
      }
#pragma unroll
      for (int a = 0; a < AHEAD; ++a)
#pragma unroll
        for (int e = 0; e < 8; ++e) sum[e] += value(x[a][e]);
    }
  }
};

__global__ __launch_bounds__(WAVES * 64) void sum_kernel(
    const short* __restrict__ grad, const int* __restrict__ order,
    const int* __restrict__ key, const unsigned* __restrict__ has,
    const int* __restrict__ spans, short* __restrict__ out, const int T,
    const int H, const int blocks, const int words) {
  __shared__ int shared_id[WAVES];
  __shared__ __attribute__((aligned(16))) float part[WAVES][COLS];
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int p = blockIdx.x * WAVES + wid;
  const int c = blockIdx.y * COLS + lane * 8;
  const bool live = c < H;
  const Rows rows = {grad + c, order, H, live};

  // each block that has the value, in order: f(place in order, rows)
  auto each = [&](int id, auto f) __attribute__((always_inline)) {
    for (int w = 0; w < words; ++w) {
      unsigned m = __builtin_amdgcn_readfirstlane(
          has[(long long)id * words + w]);
      int span = 0;
      if (lane < 32 && (m >> lane & 1))
        span = spans[(long long)id * blocks + w * 32 + lane];
      while (m) {
        const int i = __builtin_ctz(m);
        m &= m - 1;
        const int s = __builtin_amdgcn_readlane(span, i);
        f((w * 32 + i) * BLK + (s & 0xffff), s >> 16);
      }
    }
  };

  int id = -1, total = 0;       // the value that this wave owns, its rows
  if (p < T) {
    const int k = __builtin_amdgcn_readfirstlane(key[p]);
    if (k != 0x7fffffff && (p % BLK == 0 || key[p - 1] != k)) {
      int first = -1;
      each(k, [&](int at, int n) __attribute__((always_inline)) {
        if (first < 0) first = at;
        total += n;
      });
      if (first == p) id = k;
    }
  }
  id = __builtin_amdgcn_readfirstlane(id);
  total = __builtin_amdgcn_readfirstlane(total);
  auto store = [&](int v, const float (&s)[8]) __attribute__((always_inline)) {
    s16x8 y;
#pragma unroll
    for (int e = 0; e < 8; ++e) y[e] = bits(s[e]);
    if (live) *(s16x8*)(out + (long long)v * H + c) = y;
  };
  if (id >= 0 && total < MANY) {
    float sum[8] = {};
    each(id, [&](int at, int n) __attribute__((always_inline)) {
      rows.add(sum, at, n, 0, 1);
    });
    store(id, sum);
  }
  if (lane == 0) shared_id[wid] = total >= MANY ? id : -1;
  __syncthreads();
  for (int q = 0; q < WAVES; ++q) {
    const int v = __builtin_amdgcn_readfirstlane(shared_id[q]);
    if (v < 0) continue;        // the same for all waves
    float sum[8] = {};
    int turn = 0;               // rows so far: every fourth is the wave's
    each(v, [&](int at, int n) __attribute__((always_inline)) {
      rows.add(sum, at, n, (wid - turn) & (WAVES - 1), WAVES);
      turn += n;
    });
#pragma unroll
    for (int e = 0; e < 8; e += 4)
      *(f32x4*)&part[wid][lane * 8 + e] =
          f32x4{sum[e], sum[e + 1], sum[e + 2], sum[e + 3]};
    __syncthreads();
    if (wid == q) {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        float s = 0.f;
#pragma unroll
        for (int w = 0; w < WAVES; ++w) s += part[w][lane * 8 + e];
        sum[e] = s;
      }
      store(v, sum);
    }
    __syncthreads();
  }
}

}  // namespace

// ids [T], grad [T, H] bf16, H a multiple of eight, on 16 bytes, out [V, H]; rows
// of `padding` get nothing (-1: there is none). Workspaces: order, key [T], has [V
// * words] zeroed, words = ceil(blocks / 32), spans [V * blocks], blocks =
// ceil(T / 256).
extern "C" int ds_embedding_block() { return BLK; }
extern "C" void ds_embedding_bwd(const long long* ids, const void* grad,
                                 int* order, int* key, unsigned* has,
                                 int* spans, void* out, int T, int V, int H,
                                 long long padding, void* stream) {
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const int blocks = (T + BLK - 1) / BLK, words = (blocks + 31) / 32;
  hipLaunchKernelGGL(rank_kernel, dim3(blocks), dim3(BLK), 0, st, ids, order,
                     key, has, spans, T, V, padding, blocks, words);
  hipLaunchKernelGGL(sum_kernel,
                     dim3((T + WAVES - 1) / WAVES, (H + COLS - 1) / COLS),
                     dim3(WAVES * 64), 0, st, (const short*)grad, order, key,
                     has, spans, (short*)out, T, H, blocks, words);
}
