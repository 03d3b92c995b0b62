// Flash attention, forward and backward, for MI355X (gfx950) on the matrix
// cores: any sequence length, heads of 64, 96 and 128, grouped key heads,
// causal or full. q, o, do [B, S, H, D], k, v [B, S, Hkv, D] bf16 (any strides
// between tokens and heads, unit stride inside a head), lse fp32 [B, H, S].
//
// Reference analogue: the softmax and GEMM chain of csrc/transformer and the
// blocked flash attention of inference/v2.
//
// mfma_f32_32x32x16_bf16 lane maps (col = lane & 31, half = lane >> 5):
//   A: row = col, k = 8 half + j    B: col, k = 8 half + j   (j = 0..7)
//   C/D: col, row = (r & 3) + 8 (r >> 2) + 4 half            (r = 0..15)
//
// One idea runs through all kernels: the order of the contracted index is
// free. A product's result holds, for its column, the rows 16 s + 8 (j >> 2) +
// 4 half + (j & 3) in the registers 8 s + j; taken as the contracted index of
// the next product in just that order, those registers ARE its B operand. The
// other operand has to bring the same rows, transposed: ds_read_b64_tr_b16
// reads four consecutive rows of one column, which is a run of j & 3. So
// neither probabilities nor their gradients move between lanes or through
// LDS, and no operand is transposed in memory beforehand (the transposed
// copies of V, K, Q and dO that the earlier kernels took cost a pass each).
//
// LDS tiles are rows of 16-byte chunks, chunk c of row r stored at c ^ f(r),
// which spreads both the row-wise (b128) and the transposing reads over the
// banks. Heads of 96 use the layout of 128.

#include "attention_tile.h"
#include "ds_kernels.h"

namespace {

using namespace attn;

constexpr float LOG2E = 1.4426950408889634f;

struct View {             // element strides of [B, S, H, D]
  long long b, s, h;
};

// Workgroup -> (block of rows, batch * head): workgroups go round the eight
// XCDs, so each XCD takes an eighth of the heads (its L2 then holds their K
// and V, or Q and dO), and the blocks that see the most come first.
__device__ __forceinline__ void place(int id, int blocks, int heads, int& blk,
                                      int& bh) {
  if (heads % 8 == 0) {
    const int per = heads / 8, k = id >> 3;
    blk = k / per;
    bh = (id & 7) * per + k % per;
  } else {
    blk = id / heads;
    bh = id % heads;
  }
}

// ------------------------------------------------------------------ forward
//
// 8 waves of 32 query rows; 64 keys a step, K and V double-buffered, the next
// tile's direct loads in flight behind this one's products. Per key and row
// the vector unit does one multiply-add, one exp2, half a maximum, one add and
// half a conversion; the maximum is raised only where it grows by more than
// 2^8, so that most steps rescale nothing. Bound by the vector unit beside the
// matrix cores. 32 on 8 heads of 128, causal: 1 x 4096 170 us (810 TFLOP/s; 189
// beside a prompt's products), 2 x 4096 302 (911), 8 x 4096 1250 (879), 5% more while
// every step waited for the next one's loads; with V transposed beforehand, fp32
// scaling and conversions bit by bit 1 x 4096 took 350 us, torch's attention 389 and
// 2716 at 8 x 4096.

template <int D, bool CAUSAL>
__global__ __launch_bounds__(512) void fwd_kernel(
    const short* __restrict__ q, const short* __restrict__ k,
    const short* __restrict__ v, short* __restrict__ o,
    float* __restrict__ lse, const View vq, const View vk, const View vv,
    const View vo, const int S, const int H, const int Hkv, const float c,
    const int blocks, const int heads) {
  constexpr int KB = 64, DB = D / 32, KK = D / 16;
  using T = Tile<D>;
  __shared__ __attribute__((aligned(16))) short kt[2][KB * T::SC * 8];
  __shared__ __attribute__((aligned(16))) short vt[2][KB * T::SC * 8];

  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const int col = lane & 31, half = lane >> 5;
  const int ra = T::rows_at(lane), ca = T::cols_at(lane);
  int blk, bh;
  place(blockIdx.x, blocks, heads, blk, bh);
  blk = blocks - 1 - blk;
  const int b = bh / H, h = bh % H, hkv = h / (H / Hkv);
  const int q0b = blk * 256, q0 = q0b + wid * 32, row = q0 + col;

  const short* kp = k + b * vk.b + hkv * vk.h;
  const short* vp = v + b * vv.b + hkv * vv.h;

  s16x8 qf[KK];
  {
    const short* qp = q + b * vq.b + h * vq.h + min(row, S - 1) * vq.s;
#pragma unroll
    for (int kk = 0; kk < KK; ++kk)
      qf[kk] = *(const s16x8*)(qp + 16 * kk + 8 * half);
  }

  float m = -1e30f, l = 0.f;
  f32x16 acc[DB] = {};
  const int end_b = CAUSAL ? min(S, q0b + 256) : S;
  const int end_w = CAUSAL ? min(S, q0 + 32) : S;
  const int steps = (end_b + KB - 1) / KB;

  T::template fetch<KB, 512>(kp, (int)vk.s, S, kt[0], tid);
  T::template fetch<KB, 512>(vp, (int)vv.s, S, vt[0], tid);
  arrive();

  for (int it = 0; it < steps; ++it) {
    const int k0 = it * KB, cur = it & 1;
    if (it + 1 < steps) {
      T::template fetch<KB, 512>(kp + (k0 + KB) * vk.s, (int)vk.s, S - k0 - KB,
                                kt[cur ^ 1], tid);
      T::template fetch<KB, 512>(vp + (k0 + KB) * vv.s, (int)vv.s, S - k0 - KB,
                                vt[cur ^ 1], tid);
    }
    if (k0 < end_w) {
      f32x16 p[2] = {};
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int kk = 0; kk < KK; ++kk)
          p[t] = mfma(T::rows(kt[cur], 32 * t, kk, ra), qf[kk], p[t]);
      __builtin_amdgcn_s_setprio(0);

      if (k0 + KB > (CAUSAL ? min(S, q0 + 1) : S)) {
        const int last = (CAUSAL ? min(row, S - 1) : S - 1) - k0 - 4 * half;
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int r = 0; r < 16; ++r)
            if (32 * t + (r & 3) + 8 * (r >> 2) > last) p[t][r] = -1e30f;
      }
      float mt = -1e30f;
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) mt = fmaxf(mt, p[t][r]);
      mt = fmaxf(mt, __shfl_xor(mt, 32, 64));
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
      const float mc = m * c;
      float l0 = 0.f, l1 = 0.f;
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int r = 0; r < 16; r += 2) {
          p[t][r] = __builtin_amdgcn_exp2f(__builtin_fmaf(p[t][r], c, -mc));
          p[t][r + 1] =
              __builtin_amdgcn_exp2f(__builtin_fmaf(p[t][r + 1], c, -mc));
          l0 += p[t][r];
          l1 += p[t][r + 1];
        }
      l += l0 + l1;

      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          const s16x8 pb = operand(p[t], s);
#pragma unroll
          for (int db = 0; db < DB; ++db)
            acc[db] = mfma(T::cols(vt[cur], 32 * t + 16 * s, db, ca), pb, acc[db]);
        }
      __builtin_amdgcn_s_setprio(0);
    }
    arrive();
  }

  l += __shfl_xor(l, 32, 64);
  if (row >= S) return;
  const float inv = l > 0.f ? 1.f / l : (l != l ? l : 0.f);
  if (lse != nullptr && half == 0)
    lse[((long long)b * H + h) * S + row] =
        m * c * (1.f / LOG2E) + __logf(l);
  short* op = o + b * vo.b + h * vo.h + row * vo.s + 4 * half;
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      typedef int i32x2 __attribute__((ext_vector_type(2)));
      *(i32x2*)(op + 32 * db + 8 * g) =
          i32x2{pack2(acc[db][4 * g] * inv, acc[db][4 * g + 1] * inv),
                pack2(acc[db][4 * g + 2] * inv, acc[db][4 * g + 3] * inv)};
    }
}

// ----------------------------------------------------------------- backward
//
// stat[0][b, h, s] = lse * log2(e), stat[1][b, h, s] = sum(do * o): one wave
// four rows of a head; both passes below start from these two numbers a row.

template <int D>
__global__ __launch_bounds__(256) void stat_kernel(
    const short* __restrict__ dout, const short* __restrict__ o,
    const float* __restrict__ lse, float* __restrict__ stat, const View vd,
    const View vo, const int S, const int H, const long long rows) {
  const int sub = threadIdx.x & 15;
  const long long u = (long long)blockIdx.x * 16 + (threadIdx.x >> 4);
  if (u >= rows) return;               // u = (b S + s) H + h
  const int h = (int)(u % H);
  const long long bs = u / H;
  const int s = (int)(bs % S);
  const long long b = bs / S;
  float sum = 0.f;
  if (8 * sub < D) {
    const s16x8 x = *(const s16x8*)(dout + b * vd.b + s * vd.s + h * vd.h +
                                    8 * sub);
    const s16x8 y = *(const s16x8*)(o + b * vo.b + s * vo.s + h * vo.h +
                                    8 * sub);
#pragma unroll
    for (int e = 0; e < 8; ++e)
      sum += __builtin_bit_cast(float, (unsigned)(unsigned short)x[e] << 16) *
             __builtin_bit_cast(float, (unsigned)(unsigned short)y[e] << 16);
  }
#pragma unroll
  for (int off = 8; off > 0; off >>= 1) sum += __shfl_xor(sum, off, 64);
  if (sub == 0) {
    const long long at = (b * H + h) * S + s;
    stat[at] = lse[at] * LOG2E;
    stat[rows + at] = sum;
  }
}

// Both passes recompute S and dP: seven products where one pass with atomic
// sums of dQ would have five, but every sum is made in registers, in one order.
// Backward in all, 32 on 8 heads of 128, causal: 2 x 4096 1100 us (620
// TFLOP/s of the five), 8 x 4096 4205 us (654); torch's attention 3324 and
// 12151, the earlier kernels over transposed copies 15800 at 8 x 4096.
//
// dK and dV: a wave owns 32 key rows of one key head (K and V as B operands in
// registers) and walks the queries of the group's heads, 64 rows of Q and dO a
// step, double-buffered in LDS by direct loads. S = Q K^T and dP = dO V^T come
// out with a key a column; P and dS are then B operands of dV^T += dO^T P and
// dK^T += Q^T dS, and the same LDS tiles give dO^T and Q^T by transposing
// reads. 4 waves a workgroup, two workgroups a CU. Where that leaves CUs idle,
// the group's heads are split over more workgroups, whose fp32 sums add_kernel
// adds up.
template <int D, bool CAUSAL>
__global__ __launch_bounds__(256, 2) void dkdv_kernel(
    const short* __restrict__ q, const short* __restrict__ k,
    const short* __restrict__ v, const short* __restrict__ dout,
    const float* __restrict__ stat, short* __restrict__ dk,
    short* __restrict__ dv, const View vq, const View vk, const View vv,
    const View vd, const View vdk, const View vdv, const int S, const int H,
    const int Hkv, const float scale, const int blocks, const int heads,
    const long long rows, float* __restrict__ part) {
  constexpr int QB = 64, DB = D / 32, KK = D / 16;
  using T = Tile<D>;
  __shared__ __attribute__((aligned(16))) short qt[2][QB * T::SC * 8];
  __shared__ __attribute__((aligned(16))) short dt[2][QB * T::SC * 8];
  __shared__ __attribute__((aligned(16))) float st[2][2][QB];

  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const int col = lane & 31, half = lane >> 5;
  const int ra0 = T::rows_at(lane), ca0 = T::cols_at(lane);
  int blk, bh;
  place(blockIdx.x, blocks, heads, blk, bh);
  const int b = bh / Hkv, hkv = bh % Hkv, G = H / Hkv;
  const int k0b = blk * 128, k0 = k0b + wid * 32, key = k0 + col;
  const float c = scale * LOG2E;

  s16x8 kf[KK], vf[KK];
  {
    const short* kp = k + b * vk.b + hkv * vk.h + min(key, S - 1) * vk.s;
    const short* vp = v + b * vv.b + hkv * vv.h + min(key, S - 1) * vv.s;
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
      kf[kk] = *(const s16x8*)(kp + 16 * kk + 8 * half);
      vf[kk] = *(const s16x8*)(vp + 16 * kk + 8 * half);
    }
  }
  f32x16 dka[DB] = {}, dva[DB] = {};

  const int first = CAUSAL ? k0b : 0;       // a multiple of 64
  const int per = (S - first + QB - 1) / QB;
  // the group's heads of this split
  const int g0 = blockIdx.y * G / gridDim.y;
  const int steps = ((blockIdx.y + 1) * G / gridDim.y - g0) * per;

  auto fetch = [&](int h, int s0, int buf, int tid) {
    T::template fetch<QB, 256>(q + b * vq.b + h * vq.h + s0 * vq.s,
                               (int)vq.s, S - s0, qt[buf], tid);
    T::template fetch<QB, 256>(dout + b * vd.b + h * vd.h + s0 * vd.s,
                               (int)vd.s, S - s0, dt[buf], tid);
    if (wid < 2) {
      const float* p = stat + wid * rows + ((long long)b * H + h) * S + s0;
      load_lds<4>(p, 4u * min(lane, S - s0 - 1), lds_at(&st[buf][wid][0]));
    }
  };

  int h = hkv * G + g0, s0 = first;
  fetch(h, s0, 0, tid);
  arrive();
  for (int it = 0; it < steps; ++it) {
    const int cur = it & 1;
    int s1 = s0 + QB;
    if (s1 >= S) {
      s1 = first;
      ++h;
    }
    if (it + 1 < steps) {
      int tid_ = tid;
      asm("" : "+v"(tid_));
      fetch(h, s1, cur ^ 1, tid_);
    }
#pragma unroll 1
    for (int t = 0; t < 2; ++t) {
      const int r0 = s0 + 32 * t;
      if ((CAUSAL && r0 + 31 < k0) || r0 >= S) continue;
      // recomputed here: kept out of the loop they would take registers that
      // the loop needs
      int ra = ra0, ca = ca0;
      asm("" : "+v"(ra), "+v"(ca));
      f32x16 p = {}, dp = {};
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int kk = 0; kk < KK; ++kk)
        p = mfma(T::rows(qt[cur], 32 * t, kk, ra), kf[kk], p);
#pragma unroll
      for (int kk = 0; kk < KK; ++kk)
        dp = mfma(T::rows(dt[cur], 32 * t, kk, ra), vf[kk], dp);
      __builtin_amdgcn_s_setprio(0);
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const f32x4 ls = *(const f32x4*)&st[cur][0][32 * t + 8 * g + 4 * half];
        const f32x4 dl = *(const f32x4*)&st[cur][1][32 * t + 8 * g + 4 * half];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int r = 4 * g + e;
          p[r] = __builtin_amdgcn_exp2f(__builtin_fmaf(p[r], c, -ls[e]));
          dp[r] -= dl[e];
        }
      }
      if ((CAUSAL && r0 < k0 + 31) || r0 + 32 > S) {
        const int from = (CAUSAL ? key : 0) - r0 - 4 * half;
        const int to = S - r0 - 4 * half;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int at = (r & 3) + 8 * (r >> 2);
          if (at < from || at >= to) p[r] = 0.f;
        }
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) dp[r] *= p[r];
      if ((CAUSAL && r0 < k0 + 31) || r0 + 32 > S) {
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (p[r] == 0.f) dp[r] = 0.f;      // also where dP overflowed
      }
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const s16x8 pb = operand(p, s), sb = operand(dp, s);
#pragma unroll
        for (int db = 0; db < DB; ++db) {
          dva[db] = mfma(T::cols(dt[cur], 32 * t + 16 * s, db, ca), pb, dva[db]);
          dka[db] = mfma(T::cols(qt[cur], 32 * t + 16 * s, db, ca), sb, dka[db]);
        }
      }
      __builtin_amdgcn_s_setprio(0);
    }
    arrive();
    s0 = s1;
  }

  if (key >= S) return;
  if (part != nullptr) {     // added up by add_kernel
    const long long n = rows / H * Hkv * D;
    float* pp = part + 2 * n * blockIdx.y +
                (((long long)b * S + key) * Hkv + hkv) * D + 4 * half;
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        *(f32x4*)(pp + 32 * db + 8 * g) =
            f32x4{dka[db][4 * g], dka[db][4 * g + 1], dka[db][4 * g + 2],
                  dka[db][4 * g + 3]};
        *(f32x4*)(pp + n + 32 * db + 8 * g) =
            f32x4{dva[db][4 * g], dva[db][4 * g + 1], dva[db][4 * g + 2],
                  dva[db][4 * g + 3]};
      }
    return;
  }
  typedef int i32x2 __attribute__((ext_vector_type(2)));
  short* kp = dk + b * vdk.b + hkv * vdk.h + key * vdk.s + 4 * half;
  short* vp = dv + b * vdv.b + hkv * vdv.h + key * vdv.s + 4 * half;
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      *(i32x2*)(kp + 32 * db + 8 * g) = i32x2{
          pack2(dka[db][4 * g] * scale, dka[db][4 * g + 1] * scale),
          pack2(dka[db][4 * g + 2] * scale, dka[db][4 * g + 3] * scale)};
      *(i32x2*)(vp + 32 * db + 8 * g) =
          i32x2{pack2(dva[db][4 * g], dva[db][4 * g + 1]),
                pack2(dva[db][4 * g + 2], dva[db][4 * g + 3])};
    }
}

// dK and dV from the partial sums of the splits: part [splits][dk, dv][n].
__global__ __launch_bounds__(256) void add_kernel(
    const float* __restrict__ part, short* __restrict__ dk,
    short* __restrict__ dv, const long long n, const int splits,
    const float scale) {
  const long long i = ((long long)blockIdx.x * 256 + threadIdx.x) * 4;
  if (i >= 2 * n) return;
  f32x4 t = {0.f, 0.f, 0.f, 0.f};
  for (int s = 0; s < splits; ++s) t += *(const f32x4*)(part + 2 * n * s + i);
  const bool is_k = i < n;
  if (is_k) t *= scale;
  typedef int i32x2 __attribute__((ext_vector_type(2)));
  *(i32x2*)((is_k ? dk : dv - n) + i) =
      i32x2{pack2(t[0], t[1]), pack2(t[2], t[3])};
}

// dQ: a wave owns 32 query rows (Q and dO as B operands) and walks the keys, 64
// rows of K and V a step. S^T = K Q^T, dP^T = V dO^T, dQ^T += K^T dS^T.
template <int D, bool CAUSAL>
__global__ __launch_bounds__(256, 2) void dq_kernel(
    const short* __restrict__ q, const short* __restrict__ k,
    const short* __restrict__ v, const short* __restrict__ dout,
    const float* __restrict__ stat, short* __restrict__ dq, const View vq,
    const View vk, const View vv, const View vd, const View vdq, const int S,
    const int H, const int Hkv, const float scale, const int blocks,
    const int heads, const long long rows) {
  constexpr int KB = 64, DB = D / 32, KK = D / 16;
  using T = Tile<D>;
  __shared__ __attribute__((aligned(16))) short kt[2][KB * T::SC * 8];
  __shared__ __attribute__((aligned(16))) short vt[2][KB * T::SC * 8];

  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const int col = lane & 31, half = lane >> 5;
  const int ra = T::rows_at(lane), ca = T::cols_at(lane);
  int blk, bh;
  place(blockIdx.x, blocks, heads, blk, bh);
  blk = blocks - 1 - blk;
  const int b = bh / H, h = bh % H, hkv = h / (H / Hkv);
  const int q0b = blk * 128, q0 = q0b + wid * 32, row = q0 + col;
  const int at = min(row, S - 1);
  const float c = scale * LOG2E;
  const short* kp = k + b * vk.b + hkv * vk.h;
  const short* vp = v + b * vv.b + hkv * vv.h;

  s16x8 qf[KK], df[KK];
  {
    const short* qp = q + b * vq.b + h * vq.h + at * vq.s;
    const short* dp = dout + b * vd.b + h * vd.h + at * vd.s;
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
      qf[kk] = *(const s16x8*)(qp + 16 * kk + 8 * half);
      df[kk] = *(const s16x8*)(dp + 16 * kk + 8 * half);
    }
  }
  const long long sat = ((long long)b * H + h) * S + at;
  const float ls = stat[sat], dl = stat[rows + sat];
  f32x16 acc[DB] = {};

  const int end_b = CAUSAL ? min(S, q0b + 128) : S;
  const int end_w = CAUSAL ? min(S, q0 + 32) : S;
  const int steps = (end_b + KB - 1) / KB;
  T::template fetch<KB, 256>(kp, (int)vk.s, S, kt[0], tid);
  T::template fetch<KB, 256>(vp, (int)vv.s, S, vt[0], tid);
  arrive();
  for (int it = 0; it < steps; ++it) {
    const int k0 = it * KB, cur = it & 1;
    if (it + 1 < steps) {
      T::template fetch<KB, 256>(kp + (k0 + KB) * vk.s, (int)vk.s, S - k0 - KB,
                                kt[cur ^ 1], tid);
      T::template fetch<KB, 256>(vp + (k0 + KB) * vv.s, (int)vv.s, S - k0 - KB,
                                vt[cur ^ 1], tid);
    }
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const int key0 = k0 + 32 * t;
      if (key0 >= end_w) continue;
      f32x16 p = {}, dp = {};
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int kk = 0; kk < KK; ++kk)
        p = mfma(T::rows(kt[cur], 32 * t, kk, ra), qf[kk], p);
#pragma unroll
      for (int kk = 0; kk < KK; ++kk)
        dp = mfma(T::rows(vt[cur], 32 * t, kk, ra), df[kk], dp);
      __builtin_amdgcn_s_setprio(0);
#pragma unroll
      for (int r = 0; r < 16; ++r)
        dp[r] = __builtin_amdgcn_exp2f(__builtin_fmaf(p[r], c, -ls)) *
                (dp[r] - dl);
      if (key0 + 32 > (CAUSAL ? min(S, q0 + 1) : S)) {
        const int last = (CAUSAL ? at : S - 1) - key0 - 4 * half;
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if ((r & 3) + 8 * (r >> 2) > last) dp[r] = 0.f;
      }
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const s16x8 sb = operand(dp, s);
#pragma unroll
        for (int db = 0; db < DB; ++db)
          acc[db] = mfma(T::cols(kt[cur], 32 * t + 16 * s, db, ca), sb, acc[db]);
      }
      __builtin_amdgcn_s_setprio(0);
    }
    arrive();
  }
  if (row >= S) return;
  typedef int i32x2 __attribute__((ext_vector_type(2)));
  short* qp = dq + b * vdq.b + h * vdq.h + row * vdq.s + 4 * half;
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int g = 0; g < 4; ++g)
      *(i32x2*)(qp + 32 * db + 8 * g) = i32x2{
          pack2(acc[db][4 * g] * scale, acc[db][4 * g + 1] * scale),
          pack2(acc[db][4 * g + 2] * scale, acc[db][4 * g + 3] * scale)};
}

View view(const long long* s) { return View{s[0], s[1], s[2]}; }

template <int D>
void launch_fwd(const void* q, const void* k, const void* v, void* o,
                float* lse, const long long* st, int B, int S, int H, int Hkv,
                float scale, bool causal, hipStream_t s) {
  const int blocks = (S + 255) / 256, heads = B * H;
#define GO(C)                                                                \
  hipLaunchKernelGGL((fwd_kernel<D, C>), dim3((unsigned)blocks * heads),     \
                     dim3(512), 0, s, (const short*)q, (const short*)k,      \
                     (const short*)v, (short*)o, lse, view(st), view(st + 3),\
                     view(st + 6), view(st + 9), S, H, Hkv, scale * LOG2E,   \
                     blocks, heads)
  if (causal) GO(true);
  else GO(false);
#undef GO
}

template <int D>
void launch_bwd(const void* q, const void* k, const void* v, const void* o,
                const void* dout, const float* lse, float* stat, float* part,
                int splits, void* dq, void* dk, void* dv, const long long* st,
                int B, int S, int H, int Hkv, float scale, bool causal,
                hipStream_t s) {
  const long long rows = (long long)B * S * H;
  hipLaunchKernelGGL((stat_kernel<D>), dim3((unsigned)((rows + 15) / 16)),
                     dim3(256), 0, s, (const short*)dout, (const short*)o, lse,
                     stat, view(st + 12), view(st + 9), S, H, rows);
  const int blocks = (S + 127) / 128;
#define GO(C)                                                                 \
  hipLaunchKernelGGL((dkdv_kernel<D, C>),                                     \
                     dim3((unsigned)blocks * B * Hkv, splits), dim3(256), 0,  \
                     s, (const short*)q, (const short*)k, (const short*)v,    \
                     (const short*)dout, stat, (short*)dk, (short*)dv,        \
                     view(st), view(st + 3), view(st + 6), view(st + 12),     \
                     view(st + 18), view(st + 21), S, H, Hkv, scale, blocks,  \
                     B * Hkv, rows, splits > 1 ? part : nullptr);             \
  hipLaunchKernelGGL((dq_kernel<D, C>), dim3((unsigned)blocks * B * H),       \
                     dim3(256), 0, s, (const short*)q, (const short*)k,       \
                     (const short*)v, (const short*)dout, stat, (short*)dq,   \
                     view(st), view(st + 3), view(st + 6), view(st + 12),     \
                     view(st + 15), S, H, Hkv, scale, blocks, B * H, rows)
  if (causal) { GO(true); }
  else { GO(false); }
#undef GO
  if (splits > 1) {
    const long long n = (long long)B * S * Hkv * D;
    hipLaunchKernelGGL(add_kernel, dim3((unsigned)((2 * n / 4 + 255) / 256)),
                       dim3(256), 0, s, part, (short*)dk, (short*)dv, n,
                       splits, scale);
  }
}

}  // namespace

// strides: (batch, token, head) of q, k, v, o. scale > 0; lse may be null.
extern "C" void ds_flash_fwd(const void* q, const void* k, const void* v,
                             void* o, float* lse, const long long* strides,
                             int B, int S, int H, int Hkv, int D, float scale,
                             int causal, void* stream) {
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
#define GO(N) \
  launch_fwd<N>(q, k, v, o, lse, strides, B, S, H, Hkv, scale, causal, s)
  if (D == 64) GO(64);
  else if (D == 96) GO(96);
  else GO(128);
#undef GO
}

// Splits of a key head's group for dK and dV. 512 workgroups are resident and
// a causal one's work goes from nothing to the whole sequence: under 1024 some
// CUs are idle for a good part, and a divisor of the group (an uneven split
// leaves the longest as long) that makes 2048 of them pays. Backward, us, by
// splits 1 / 2 / 4: B 1 x 4096, 32 on 8 heads of 128 (256 workgroups) 995 /
// 723 / 647; B 2 1362 / 1129 / 1100; B 8 x 2048 (1024) 1236 / 1239 / 1317; 3 x
// 777, 28 on 4 heads (84), splits 1 / 7: 327 / 126.
extern "C" int ds_flash_bwd_splits(int B, int S, int H, int Hkv) {
  const long long wgs = (long long)((S + 127) / 128) * B * Hkv;
  const int G = H / Hkv;
  if (wgs >= 1024) return 1;
  int n = 1;
  while (n < G && (G % n || wgs * n < 2048)) ++n;
  return n;
}

// strides: (batch, token, head) of q, k, v, o, do, dq, dk, dv; dk and dv are
// contiguous. stat: 2 B H S floats of workspace, part: splits 2 B S Hkv D
// (splits > 1).
extern "C" void ds_flash_bwd(const void* q, const void* k, const void* v,
                             const void* o, const void* dout, const float* lse,
                             float* stat, float* part, int splits, void* dq,
                             void* dk, void* dv, const long long* strides,
                             int B, int S, int H, int Hkv, int D, float scale,
                             int causal, void* stream) {
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
#define GO(N)                                                              \
  launch_bwd<N>(q, k, v, o, dout, lse, stat, part, splits, dq, dk, dv,     \
                strides, B, S, H, Hkv, scale, causal, s)
  if (D == 64) GO(64);
  else if (D == 96) GO(96);
  else GO(128);
#undef GO
}
