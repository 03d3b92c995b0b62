// Fused Adam/AdamW for MI355X (gfx950).
//
// MI355X-first design: the ZeRO optimizers in this framework keep the
// fp32 master weights, optimizer state and 16-bit gradients as single
// contiguous flat shards, so the hot path is ONE memory-bound
// kernel over flat buffers — no multi-tensor-apply chunk harness (the
// reference needs one because it steps thousands of separate tensors:
// csrc/adam/multi_tensor_adam.cu:129). Optionally writes the updated
// bf16 param shard in the same pass (saves the separate master->bf16 cast
// copy: one fewer full read+write of the shard at 8 TB/s HBM3E).
//
// Memory-bound: 4 streams read (p, g, m, v) + 3-4 written per element, 28 bytes
// with bf16 gradients and mirror. A thread takes two vectors half an array
// apart, one launch's worth of workgroups runs over the array once, and large
// arrays go past the caches (nontemporal): 525M elements 2550 us (5.8 TB/s).
// 2048 workgroups striding over it took 3300 (4.45 TB/s), without the
// nontemporal hints 2780; 16M elements, which the last-level cache holds, 56
// with plain accesses and 71 with nontemporal ones.

#include "ds_kernels.h"

namespace {

struct Hyper {
  float lr, beta1, beta2, eps, weight_decay, bias_corr1, bias_corr2_sqrt,
      inv_scale;
};

template <bool ADAMW>
__device__ __forceinline__ void adam_one(float& p, float& m, float& v,
                                         float grad, const Hyper& h) {
  grad *= h.inv_scale;
  if (!ADAMW && h.weight_decay != 0.f) grad += h.weight_decay * p;
  m = h.beta1 * m + (1.f - h.beta1) * grad;
  v = h.beta2 * v + (1.f - h.beta2) * grad * grad;
  const float mhat = m / h.bias_corr1;
  const float denom = sqrtf(v) / h.bias_corr2_sqrt + h.eps;
  float update = mhat / denom;
  if (ADAMW && h.weight_decay != 0.f) update += h.weight_decay * p;
  p -= h.lr * update;
}

typedef float vec4 __attribute__((ext_vector_type(4)));

template <bool NT, typename V>
__device__ __forceinline__ V load(const V* p) {
  return NT ? __builtin_nontemporal_load(p) : *p;
}
template <bool NT, typename V>
__device__ __forceinline__ void store(V x, V* p) {
  if (NT) __builtin_nontemporal_store(x, p);
  else *p = x;
}

// n4 vectors of four, all streams aligned to them. Thread i takes vectors i
// and i + half.
template <typename grad_t, bool ADAMW, bool WRITE_BF16, bool NT>
__global__ __launch_bounds__(256) void fused_adam_vec_kernel(
    float* __restrict__ p, const grad_t* __restrict__ g,
    float* __restrict__ m, float* __restrict__ v, ds::bf16* __restrict__ p16,
    const long long n4, const long long half, const Hyper h) {
  typedef short gvec __attribute__((ext_vector_type(2 * sizeof(grad_t))));
  typedef short ovec __attribute__((ext_vector_type(4)));
  const long long i0 = (long long)blockIdx.x * 256 + threadIdx.x;
  vec4 pv[2], mv[2], vv[2];
  gvec gv[2];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const long long i = i0 + u * half;
    if (i0 < half && i < n4) {
      pv[u] = load<NT>((const vec4*)p + i);
      mv[u] = load<NT>((const vec4*)m + i);
      vv[u] = load<NT>((const vec4*)v + i);
      gv[u] = load<NT>((const gvec*)g + i);
    }
  }
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const long long i = i0 + u * half;
    if (i0 >= half || i >= n4) continue;
    ovec o;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float pe = pv[u][e], me = mv[u][e], ve = vv[u][e];
      adam_one<ADAMW>(pe, me, ve,
                      ds::to_f32(reinterpret_cast<const grad_t*>(&gv[u])[e]),
                      h);
      pv[u][e] = pe; mv[u][e] = me; vv[u][e] = ve;
      if (WRITE_BF16) o[e] = __builtin_bit_cast(short, (__bf16)pe);
    }
    store<NT>(pv[u], (vec4*)p + i);
    store<NT>(mv[u], (vec4*)m + i);
    store<NT>(vv[u], (vec4*)v + i);
    if (WRITE_BF16) store<NT>(o, (ovec*)p16 + i);
  }
}

// Unaligned streams, and the last elements of the others.
template <typename grad_t, bool ADAMW, bool WRITE_BF16>
__global__ __launch_bounds__(256) void fused_adam_flat_kernel(
    float* __restrict__ p, const grad_t* __restrict__ g,
    float* __restrict__ m, float* __restrict__ v, ds::bf16* __restrict__ p16,
    const long long n, const Hyper h) {
  const long long stride = (long long)gridDim.x * 256;
  for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < n;
       i += stride) {
    float pe = p[i], me = m[i], ve = v[i];
    adam_one<ADAMW>(pe, me, ve, ds::to_f32(g[i]), h);
    p[i] = pe; m[i] = me; v[i] = ve;
    if (WRITE_BF16) p16[i] = ds::from_f32<ds::bf16>(pe);
  }
}

template <typename grad_t, bool ADAMW, bool WRITE_BF16>
void launch_kernels(float* p, const grad_t* g, float* m, float* v,
                    ds::bf16* p16, long long n, const Hyper& h,
                    hipStream_t s) {
  const uintptr_t wide = (uintptr_t)p | (uintptr_t)m | (uintptr_t)v;
  const bool vec = wide % 16 == 0 &&
                   (uintptr_t)g % (4 * sizeof(grad_t)) == 0 &&
                   (uintptr_t)p16 % 8 == 0;
  const long long n4 = vec ? n / 4 : 0;
  if (n4) {
    const long long half = (n4 + 1) / 2;
    const dim3 grid((unsigned)((half + 255) / 256));
    // past the last-level cache (256 MB) by some
    if (n > (1ll << 25))
      hipLaunchKernelGGL((fused_adam_vec_kernel<grad_t, ADAMW, WRITE_BF16,
                                                true>),
                         grid, dim3(256), 0, s, p, g, m, v, p16, n4, half, h);
    else
      hipLaunchKernelGGL((fused_adam_vec_kernel<grad_t, ADAMW, WRITE_BF16,
                                                false>),
                         grid, dim3(256), 0, s, p, g, m, v, p16, n4, half, h);
  }
  const long long at = 4 * n4;
  if (at < n)
    hipLaunchKernelGGL((fused_adam_flat_kernel<grad_t, ADAMW, WRITE_BF16>),
                       dim3(ds::ds_num_blocks(n - at, 256)), dim3(256), 0, s,
                       p + at, g + at, m + at, v + at,
                       WRITE_BF16 ? p16 + at : nullptr, n - at, h);
}

template <typename grad_t>
void launch_typed(float* p, const grad_t* g, float* m, float* v,
                  ds::bf16* p16, long long n, const Hyper& h, bool adamw,
                  hipStream_t s) {
  if (adamw) {
    if (p16) launch_kernels<grad_t, true, true>(p, g, m, v, p16, n, h, s);
    else launch_kernels<grad_t, true, false>(p, g, m, v, p16, n, h, s);
  } else {
    if (p16) launch_kernels<grad_t, false, true>(p, g, m, v, p16, n, h, s);
    else launch_kernels<grad_t, false, false>(p, g, m, v, p16, n, h, s);
  }
}

}  // namespace

extern "C" void ds_fused_adam_flat(float* p, const void* g, int grad_dtype,
                                   float* m, float* v, void* p16, long long n,
                                   float lr, float beta1, float beta2, float eps,
                                   float weight_decay, int step, float inv_scale,
                                   int adamw, void* stream) {
  const float bc1 = 1.f - powf(beta1, (float)step);
  const float bc2s = sqrtf(1.f - powf(beta2, (float)step));
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  ds::bf16* p16t = reinterpret_cast<ds::bf16*>(p16);
  const Hyper h = {lr, beta1, beta2, eps, weight_decay, bc1, bc2s, inv_scale};
  switch (grad_dtype) {
    case 0:  // fp32
      launch_typed(p, reinterpret_cast<const float*>(g), m, v, p16t, n, h,
                   adamw != 0, s);
      break;
    case 1:  // bf16
      launch_typed(p, reinterpret_cast<const ds::bf16*>(g), m, v, p16t, n, h,
                   adamw != 0, s);
      break;
    case 2:  // fp16
      launch_typed(p, reinterpret_cast<const ds::f16*>(g), m, v, p16t, n, h,
                   adamw != 0, s);
      break;
  }
}
