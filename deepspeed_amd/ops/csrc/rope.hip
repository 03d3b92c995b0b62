// Rotary position embedding (RoPE) for MI355X (gfx950).
//
// Capability parity with the reference's apply_rotary_pos_emb.cu
// (csrc/transformer/inference/csrc/apply_rotary_pos_emb.cu:27, neox
// rotate-half style, GQA-aware), re-designed for CDNA4:
//  * cos/sin are a precomputed fp32 host table [max_seq, D/2] (per the CDNA4
//    guide, on-device sinf/cosf turns this memory-bound op VALU-bound)
//  * layout [B, S, Hh, D] (the natural attention-projection output; avoids
//    the reference's 0213 transpose kernels entirely)
//  * queries and keys of a layer in one launch, into new tensors or in place;
//    16-bit heads with D/2 a multiple of 8 move 16 bytes a lane. Queries and
//    keys of 8192 tokens, 32 and 8 heads of 128: 33 us (5.1 TB/s); a copy and
//    a pair-at-a-time rotation of the copy, each tensor by itself, took 108.
//  * backward = inverse rotation (negated sin), same kernel.

#include "ds_kernels.h"

namespace {

struct Pair {
  const void* x[2];
  void* y[2];       // may be x
  int heads[2];     // heads[1] == 0: one tensor
};

// VEC coordinates j.. and j + D/2.. of one head a thread.
template <typename T, int VEC>
__global__ __launch_bounds__(256) void rope_kernel(
    const Pair p, const float* __restrict__ cs,  // [max_seq, D/2] cos
    const float* __restrict__ sn, const int* __restrict__ positions,  // or null
    const float sign, const long long total, const int S, const int D) {
  const int half = D / 2, parts = half / VEC;
  const int heads = p.heads[0] + p.heads[1];
  const long long stride = (long long)gridDim.x * blockDim.x;
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
       i < total; i += stride) {
    const int j = (int)(i % parts) * VEC;
    const long long u = i / parts;
    int h = (int)(u % heads);
    const long long bs = u / heads;             // b * S + s
    const int which = h >= p.heads[0];
    if (which) h -= p.heads[0];
    const int pos = positions ? positions[bs] : (int)(bs % S);
    const long long at = (bs * p.heads[which] + h) * D + j;
    const T* x = reinterpret_cast<const T*>(p.x[which]) + at;
    T* y = reinterpret_cast<T*>(p.y[which]) + at;
    const float* c = cs + (long long)pos * half + j;
    const float* s = sn + (long long)pos * half + j;
    struct alignas(sizeof(T) * VEC) Vec {
      T v[VEC];
    } a = *reinterpret_cast<const Vec*>(x),
      b = *reinterpret_cast<const Vec*>(x + half);
#pragma unroll
    for (int e = 0; e < VEC; ++e) {
      const float x1 = ds::to_f32(a.v[e]), x2 = ds::to_f32(b.v[e]);
      const float ce = c[e], se = sign * s[e];
      a.v[e] = ds::from_f32<T>(x1 * ce - x2 * se);
      b.v[e] = ds::from_f32<T>(x2 * ce + x1 * se);
    }
    *reinterpret_cast<Vec*>(y) = a;
    *reinterpret_cast<Vec*>(y + half) = b;
  }
}

template <typename T, int VEC>
void launch(const Pair& p, const float* cs, const float* sn,
            const int* positions, long long tokens, int S, int D, bool bwd,
            hipStream_t s) {
  const long long total =
      tokens * (p.heads[0] + p.heads[1]) * (D / 2 / VEC);
  long long blocks = (total + 255) / 256;
  if (blocks > 65536) blocks = 65536;
  if (total)
    hipLaunchKernelGGL((rope_kernel<T, VEC>), dim3((unsigned)blocks),
                       dim3(256), 0, s, p, cs, sn, positions,
                       bwd ? -1.f : 1.f, total, S, D);
}

}  // namespace

// x2 == null: one tensor. y may be x.
extern "C" void ds_rope(const void* x1, void* y1, int heads1, const void* x2,
                        void* y2, int heads2, const float* cos_table,
                        const float* sin_table, const int* positions,
                        long long batch, long long seq, long long dim, int bwd,
                        int dtype, void* stream) {
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const Pair p = {{x1, x2}, {y1, y2}, {heads1, x2 ? heads2 : 0}};
  const long long n = batch * seq;
  const int S = (int)seq, D = (int)dim;
  bool vec = dim % 16 == 0;
  for (const void* q : {x1, (const void*)y1, x2, (const void*)y2})
    vec = vec && reinterpret_cast<uintptr_t>(q) % 16 == 0;
#define GO(T, V) \
  launch<T, V>(p, cos_table, sin_table, positions, n, S, D, bwd != 0, s)
  if (dtype == 1) {
    if (vec) GO(ds::bf16, 8);
    else GO(ds::bf16, 1);
  } else if (dtype == 2) {
    if (vec) GO(ds::f16, 8);
    else GO(ds::f16, 1);
  } else {
    GO(float, 1);
  }
#undef GO
}
