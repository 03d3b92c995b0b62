// Fused RMSNorm / LayerNorm forward+backward for MI355X (gfx950).
//
// Capability parity with the reference's normalization kernels
// (csrc/transformer/inference/csrc/rms_norm.cu, layer_norm.cu and the
// training-side normalize_kernels.cu), re-derived for CDNA4:
//  * wave64 shuffle reductions (not 32-wide warp ladders)
//  * 16 B/lane vectorized bf16 loads (bf16x8)
//  * forward caches the row in registers when H <= 16384 (one HBM read)
//  * the residual stream's add belongs to the norm: the forward reads the
//    sublayer's output and the stream, writes their sum and its norm (taken
//    from the fp32 sum, not from its rounding, which is what the backward reads
//    again, with the fp32 sum's 1/rms); the backward adds the stream's
//    gradient before it rounds. An add kernel each way moved three more
//    tensors and rounded once more.
//  * backward: a row in registers (one read), the weight's gradient in
//    registers over a block's rows, then one row of partial sums a block and
//    a second kernel that adds them up in a fixed order. 8192 x 4096 with the
//    stream's gradient: 48 us (5.6 TB/s); element-wise loads, two reads of the
//    row and an atomic a column and block took 120 us, 30 us at 1024 x 1024
//    (now 8), and the stream's add 40 us more.
//
// Memory-bound ops: target is the ~6.3 TB/s achievable HBM3E bandwidth.

#include <initializer_list>

#include "ds_kernels.h"

namespace {

constexpr int BLOCK = 256;
constexpr int VEC = 8;  // bf16 per 16B load

// ---------------------------------------------------------------------------
// Forward. One block per row (grid-stride). RMS: invrms = rsqrt(mean(x^2)+eps)
// LN: also subtract mean. Saves fp32 invrms (and mean for LN) for backward.
// ---------------------------------------------------------------------------

// A row whose elements c.. c + VEC - 1 `load` brings. The weight is read with
// the row, not behind the reduction: one wait for memory instead of two.
template <typename T, bool LN, int ITERS, bool RES, typename Load>
__device__ __forceinline__ void norm_row(Load load, const long long at,
                                         const T* res, T* sum_out, const T* w,
                                         const T* b, T* y, float* invrms_out,
                                         float* mean_out, const int row,
                                         const int H, const float eps,
                                         float* red) {
  using VecT = ds::bf16x8;  // same layout for f16 via reinterpret of 16B
  const bool mine = threadIdx.x < BLOCK;
  const bool vec = (reinterpret_cast<uintptr_t>(w) & 15) == 0;
  float xv[ITERS][VEC];
  T wv[ITERS][VEC];
  float sum = 0.f, sumsq = 0.f;
#pragma unroll
  for (int it = 0; it < ITERS; ++it) {
    const int c = (it * BLOCK + threadIdx.x) * VEC;
    if (mine && c < H) {
      if (vec)
        *reinterpret_cast<VecT*>(wv[it]) =
            *reinterpret_cast<const VecT*>(w + c);
      else
#pragma unroll
        for (int j = 0; j < VEC; ++j) wv[it][j] = w[c + j];
      T v[VEC], r[VEC];
      if (RES)
        *reinterpret_cast<VecT*>(r) =
            *reinterpret_cast<const VecT*>(res + at + c);
      load(c, v);
#pragma unroll
      for (int j = 0; j < VEC; ++j) {
        float f = ds::to_f32(v[j]);
        if (RES) {
          f += ds::to_f32(r[j]);
          r[j] = ds::from_f32<T>(f);
        }
        xv[it][j] = f;
        if (LN) sum += f;
        sumsq += f * f;
      }
      if (RES)
        *reinterpret_cast<VecT*>(sum_out + at + c) =
            *reinterpret_cast<const VecT*>(r);
    }
  }
  float mean = 0.f;
  if (LN) {
    mean = ds::block_reduce_sum<BLOCK>(sum, red) / H;
    __syncthreads();
  }
  float var = ds::block_reduce_sum<BLOCK>(sumsq, red) / H;
  if (LN) var -= mean * mean;
  const float inv = rsqrtf(var + eps);
  if (threadIdx.x == 0) {
    if (invrms_out != nullptr) invrms_out[row] = inv;
    if (LN) mean_out[row] = mean;
  }
#pragma unroll
  for (int it = 0; it < ITERS; ++it) {
    const int c = (it * BLOCK + threadIdx.x) * VEC;
    if (mine && c < H) {
      T out[VEC];
#pragma unroll
      for (int j = 0; j < VEC; ++j) {
        const float f = xv[it][j];
        float nw = (LN ? (f - mean) : f) * inv * ds::to_f32(wv[it][j]);
        if (LN && b != nullptr) nw += ds::to_f32(b[c + j]);
        out[j] = ds::from_f32<T>(nw);
      }
      *reinterpret_cast<VecT*>(y + at + c) =
          *reinterpret_cast<const VecT*>(out);
    }
  }
}

template <typename T, bool LN, int ITERS, bool RES>
__global__ void norm_fwd_cached_kernel(const T* __restrict__ x,
                                       const T* __restrict__ res,  // RES
                                       T* __restrict__ sum_out,    // RES
                                       const T* __restrict__ w,
                                       const T* __restrict__ b,  // LN bias or null
                                       T* __restrict__ y,
                                       float* __restrict__ invrms_out,
                                       float* __restrict__ mean_out,
                                       const int rows, const int H,
                                       const float eps) {
  __shared__ float red[BLOCK / WAVE_SIZE];
  for (int row = blockIdx.x; row < rows; row += gridDim.x) {
    const long long at = (long long)row * H;
    norm_row<T, LN, ITERS, RES>(
        [&](int c, T* v) {
          *reinterpret_cast<ds::bf16x8*>(v) =
              *reinterpret_cast<const ds::bf16x8*>(x + at + c);
        },
        at, res, sum_out, w, b, y, invrms_out, mean_out, row, H, eps, red);
    __syncthreads();
  }
}

// The same of res + x where x is still in parts, part[splits][rows][H], that
// tile_linear.hip's split contraction left: added up in their order and rounded
// as its merge would, by all 1024 threads (the loads of 8 splits in flight) into
// LDS, from where 256 go on as above. A launch and a pass less: 32 x 4096 5.5 us,
// the merge and the norm 4.2 and 4.0 under the profiler, which shows the launches
// longer than they are; four layers of 32 requests 895 -> 880 us with the append's.
constexpr int WIDE = 1024;

template <int ITERS>
__global__ __launch_bounds__(WIDE) void add_norm_parts_kernel(
    const float* __restrict__ part, const int splits,
    const ds::bf16* __restrict__ res, ds::bf16* __restrict__ sum_out,
    const ds::bf16* __restrict__ w, ds::bf16* __restrict__ y, const int rows,
    const int H, const float eps) {
  typedef float f4 __attribute__((ext_vector_type(4)));
  __shared__ float red[WIDE / WAVE_SIZE];
  __shared__ __attribute__((aligned(16))) ds::bf16 x[ITERS * BLOCK * VEC];
  const int row = blockIdx.x;
  const long long at = (long long)row * H, step = (long long)rows * H;
  for (int c = threadIdx.x * 4; c < H; c += WIDE * 4) {
    f4 t = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
    for (int s = 0; s < splits; ++s)
      t += *reinterpret_cast<const f4*>(part + s * step + at + c);
#pragma unroll
    for (int e = 0; e < 4; ++e) x[c + e] = ds::from_f32<ds::bf16>(t[e]);
  }
  __syncthreads();
  norm_row<ds::bf16, false, ITERS, true>(
      [&](int c, ds::bf16* v) {
        *reinterpret_cast<ds::bf16x8*>(v) =
            *reinterpret_cast<const ds::bf16x8*>(x + c);
      },
      at, res, sum_out, w, (const ds::bf16*)nullptr, y, (float*)nullptr,
      (float*)nullptr, row, H, eps, red);
}

// Generic fallback (any H, scalar loads, row re-read).
template <typename T, bool LN>
__global__ void norm_fwd_generic_kernel(const T* __restrict__ x,
                                        const T* __restrict__ w,
                                        const T* __restrict__ b,
                                        T* __restrict__ y,
                                        float* __restrict__ invrms_out,
                                        float* __restrict__ mean_out,
                                        const int rows, const int H,
                                        const float eps) {
  __shared__ float red[BLOCK / WAVE_SIZE];
  for (int row = blockIdx.x; row < rows; row += gridDim.x) {
    const T* xr = x + (long long)row * H;
    T* yr = y + (long long)row * H;
    float sum = 0.f, sumsq = 0.f;
    for (int c = threadIdx.x; c < H; c += BLOCK) {
      const float f = ds::to_f32(xr[c]);
      if (LN) sum += f;
      sumsq += f * f;
    }
    float mean = 0.f;
    if (LN) {
      mean = ds::block_reduce_sum<BLOCK>(sum, red) / H;
      __syncthreads();
    }
    float var = ds::block_reduce_sum<BLOCK>(sumsq, red) / H;
    if (LN) var -= mean * mean;
    const float inv = rsqrtf(var + eps);
    if (threadIdx.x == 0) {
      invrms_out[row] = inv;
      if (LN) mean_out[row] = mean;
    }
    __syncthreads();
    for (int c = threadIdx.x; c < H; c += BLOCK) {
      float f = ds::to_f32(xr[c]);
      float nw = (LN ? (f - mean) : f) * inv * ds::to_f32(w[c]);
      if (LN && b != nullptr) nw += ds::to_f32(b[c]);
      yr[c] = ds::from_f32<T>(nw);
    }
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// Backward.
//   xhat = (x - mean?) * invrms
//   dyw  = dy * w
//   RMS: dx = invrms * (dyw - xhat * mean_c(dyw*xhat))
//   LN : dx = invrms * (dyw - mean_c(dyw) - xhat * mean_c(dyw*xhat))
//   dw  = sum_rows dy * xhat ; db = sum_rows dy (LN)
// dweight partials accumulate in LDS fp32 across each block's rows, then one
// device-scope atomicAdd per column per block into the fp32 workspace.
// ---------------------------------------------------------------------------

template <typename T, bool LN>
__global__ void norm_bwd_kernel(const T* __restrict__ dy,
                                const T* __restrict__ x,
                                const T* __restrict__ w,
                                const float* __restrict__ invrms,
                                const float* __restrict__ mean,
                                T* __restrict__ dx,
                                float* __restrict__ dw,  // fp32 [H]
                                float* __restrict__ db,  // fp32 [H] (LN)
                                const int rows, const int H) {
  extern __shared__ float lds[];  // dw accum [H] (+ db accum [H] for LN)
  __shared__ float red[BLOCK / WAVE_SIZE];
  float* dw_lds = lds;
  float* db_lds = LN ? (lds + H) : nullptr;
  for (int c = threadIdx.x; c < H; c += BLOCK) {
    dw_lds[c] = 0.f;
    if (LN) db_lds[c] = 0.f;
  }
  __syncthreads();

  for (int row = blockIdx.x; row < rows; row += gridDim.x) {
    const T* dyr = dy + (long long)row * H;
    const T* xr = x + (long long)row * H;
    T* dxr = dx + (long long)row * H;
    const float inv = invrms[row];
    const float mu = LN ? mean[row] : 0.f;

    float dot = 0.f, dsum = 0.f;
    for (int c = threadIdx.x; c < H; c += BLOCK) {
      const float xhat = (ds::to_f32(xr[c]) - mu) * inv;
      const float dyv = ds::to_f32(dyr[c]);
      const float dyw = dyv * ds::to_f32(w[c]);
      dot += dyw * xhat;
      if (LN) dsum += dyw;
      dw_lds[c] += dyv * xhat;
      if (LN) db_lds[c] += dyv;
    }
    dot = ds::block_reduce_sum<BLOCK>(dot, red) / H;
    if (LN) {
      __syncthreads();
      dsum = ds::block_reduce_sum<BLOCK>(dsum, red) / H;
    }
    for (int c = threadIdx.x; c < H; c += BLOCK) {
      const float xhat = (ds::to_f32(xr[c]) - mu) * inv;
      const float dyw = ds::to_f32(dyr[c]) * ds::to_f32(w[c]);
      float v = dyw - xhat * dot;
      if (LN) v -= dsum;
      dxr[c] = ds::from_f32<T>(v * inv);
    }
    __syncthreads();
  }

  for (int c = threadIdx.x; c < H; c += BLOCK) {
    atomicAdd(dw + c, dw_lds[c]);
    if (LN) atomicAdd(db + c, db_lds[c]);
  }
}

// Rows in registers. Partial sums of dw (and db) over a block's rows go to
// row blockIdx.x of part [grid, (LN ? 2 : 1) * H]. The next row's loads are in
// flight during a row's reduction.
template <typename T, bool LN, int ITERS, bool RES>
__global__ __launch_bounds__(BLOCK) void norm_bwd_rows_kernel(
    const T* __restrict__ dy, const T* __restrict__ x,
    const T* __restrict__ w, const float* __restrict__ invrms,
    const float* __restrict__ mean,
    const T* __restrict__ dres,  // RES: added to dx
    T* __restrict__ dx, float* __restrict__ part, const int rows,
    const int H) {
  using VecT = ds::bf16x8;
  __shared__ float red[2][BLOCK / WAVE_SIZE][2];
  struct Row {
    VecT dy[ITERS], x[ITERS], r[ITERS];
    float inv, mu;
  };
  auto load = [&](Row& a, int row) {
    a.inv = invrms[row];
    a.mu = LN ? mean[row] : 0.f;
#pragma unroll
    for (int it = 0; it < ITERS; ++it) {
      const int c = (it * BLOCK + threadIdx.x) * VEC;
      if (c < H) {
        const long long at = (long long)row * H + c;
        a.dy[it] = *reinterpret_cast<const VecT*>(dy + at);
        a.x[it] = *reinterpret_cast<const VecT*>(x + at);
        if (RES) a.r[it] = *reinterpret_cast<const VecT*>(dres + at);
      }
    }
  };
  auto f32 = [](const VecT& v, int j) {
    return ds::to_f32(reinterpret_cast<const T*>(&v)[j]);
  };
  float wv[ITERS][VEC], dw[ITERS][VEC] = {}, db[LN ? ITERS : 1][VEC] = {};
#pragma unroll
  for (int it = 0; it < ITERS; ++it) {
    const int c = (it * BLOCK + threadIdx.x) * VEC;
#pragma unroll
    for (int j = 0; j < VEC; ++j)
      wv[it][j] = c < H ? ds::to_f32(w[c + j]) : 0.f;
  }
  Row next;
  int row = blockIdx.x, flip = 0;
  if (row < rows) load(next, row);
  for (; row < rows; row += gridDim.x, flip ^= 1) {
    const Row a = next;
    if (row + gridDim.x < rows) load(next, row + gridDim.x);
    float dot = 0.f, dsum = 0.f;
#pragma unroll
    for (int it = 0; it < ITERS; ++it) {
      if ((it * BLOCK + (int)threadIdx.x) * VEC < H) {
#pragma unroll
        for (int j = 0; j < VEC; ++j) {
          const float xhat = (f32(a.x[it], j) - a.mu) * a.inv;
          const float d = f32(a.dy[it], j);
          dot += d * wv[it][j] * xhat;
          dw[it][j] += d * xhat;
          if (LN) {
            dsum += d * wv[it][j];
            db[LN ? it : 0][j] += d;
          }
        }
      }
    }
    dot = ds::wave_reduce_sum(dot);
    if (LN) dsum = ds::wave_reduce_sum(dsum);
    if ((threadIdx.x & 63) == 0) {
      red[flip][threadIdx.x >> 6][0] = dot;
      red[flip][threadIdx.x >> 6][1] = dsum;
    }
    __syncthreads();     // two buffers: a wave can be one row ahead at most
    dot = dsum = 0.f;
#pragma unroll
    for (int i = 0; i < BLOCK / WAVE_SIZE; ++i) {
      dot += red[flip][i][0];
      if (LN) dsum += red[flip][i][1];
    }
    dot /= H;
    dsum /= H;
#pragma unroll
    for (int it = 0; it < ITERS; ++it) {
      const int c = (it * BLOCK + threadIdx.x) * VEC;
      if (c < H) {
        T out[VEC];
#pragma unroll
        for (int j = 0; j < VEC; ++j) {
          const float xhat = (f32(a.x[it], j) - a.mu) * a.inv;
          float v = f32(a.dy[it], j) * wv[it][j] - xhat * dot;
          if (LN) v -= dsum;
          v *= a.inv;
          if (RES) v += f32(a.r[it], j);
          out[j] = ds::from_f32<T>(v);
        }
        *reinterpret_cast<VecT*>(dx + (long long)row * H + c) =
            *reinterpret_cast<const VecT*>(out);
      }
    }
  }
  const long long width = (LN ? 2LL : 1LL) * H;
#pragma unroll
  for (int it = 0; it < ITERS; ++it) {
    const int c = (it * BLOCK + threadIdx.x) * VEC;
    if (c < H) {
      float* p = part + blockIdx.x * width + c;
#pragma unroll
      for (int j = 0; j < VEC; ++j) {
        p[j] = dw[it][j];
        if (LN) p[H + j] = db[LN ? it : 0][j];
      }
    }
  }
}

// out[c] = sum over n rows of part[., c]: 64 columns a workgroup, 16 waves
// each with every sixteenth row. In the weight's type where that is asked for: a
// conversion behind it was a launch a norm, ten a step of two layers with the
// additions to the flat buffer that went with it.
template <typename O>
__global__ __launch_bounds__(1024) void norm_parts_kernel(
    const float* __restrict__ part, O* __restrict__ out, const int n,
    const int width) {
  __shared__ float sums[16][64];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int c = blockIdx.x * 64 + lane;
  float s = 0.f;
  if (c < width) {
#pragma unroll 8
    for (int i = wid; i < n; i += 16) s += part[(long long)i * width + c];
  }
  sums[wid][lane] = s;
  __syncthreads();
  if (wid == 0 && c < width) {
#pragma unroll
    for (int i = 1; i < 16; ++i) s += sums[i][lane];
    out[c] = ds::from_f32<O>(s);
  }
}

template <typename T>
bool rows_cached(int H, std::initializer_list<const void*> p) {
  // register-cached vector path is for 16-bit dtypes (bf16x8 = 16 B/lane)
  bool ok = sizeof(T) == 2 && (H % VEC == 0) && (H <= BLOCK * VEC * 8);
  for (const void* q : p) ok = ok && reinterpret_cast<uintptr_t>(q) % 16 == 0;
  return ok;
}

template <typename T>
void launch_norm_fwd(const void* x, const void* w, const void* b, void* y,
                     float* invrms, float* mean, int rows, int H, float eps,
                     bool ln, hipStream_t s) {
  const int grid = rows < 8192 ? rows : 8192;
  const bool vec_ok = rows_cached<T>(H, {x, y});
  const T* xt = reinterpret_cast<const T*>(x);
  const T* wt = reinterpret_cast<const T*>(w);
  const T* bt = reinterpret_cast<const T*>(b);
  T* yt = reinterpret_cast<T*>(y);
#define LAUNCH_IT(LNV, ITERS)                                               \
  hipLaunchKernelGGL((norm_fwd_cached_kernel<T, LNV, ITERS, false>),       \
                     dim3(grid), dim3(BLOCK), 0, s, xt, (const T*)nullptr,  \
                     (T*)nullptr, wt, bt, yt, invrms, mean, rows, H, eps)
  if (vec_ok) {
    const int iters = (H + BLOCK * VEC - 1) / (BLOCK * VEC);
    if (ln) {
      if (iters <= 1) LAUNCH_IT(true, 1);
      else if (iters <= 2) LAUNCH_IT(true, 2);
      else if (iters <= 4) LAUNCH_IT(true, 4);
      else LAUNCH_IT(true, 8);
    } else {
      if (iters <= 1) LAUNCH_IT(false, 1);
      else if (iters <= 2) LAUNCH_IT(false, 2);
      else if (iters <= 4) LAUNCH_IT(false, 4);
      else LAUNCH_IT(false, 8);
    }
  } else if (ln) {
    hipLaunchKernelGGL((norm_fwd_generic_kernel<T, true>), dim3(grid),
                       dim3(BLOCK), 0, s, xt, wt, bt, yt, invrms, mean, rows, H,
                       eps);
  } else {
    hipLaunchKernelGGL((norm_fwd_generic_kernel<T, false>), dim3(grid),
                       dim3(BLOCK), 0, s, xt, wt, bt, yt, invrms, mean, rows, H,
                       eps);
  }
#undef LAUNCH_IT
}

// Blocks of the backward by rows (and rows of its partial sums): four a CU and
// at least four rows a block, so that writing and adding up the partial sums
// stays small beside the rows themselves.
int bwd_blocks(int rows) {
  const int b = rows / 4;
  return b < 1 ? 1 : b > 1024 ? 1024 : b;
}

template <typename T, bool LN, bool RES>
void launch_norm_bwd_rows(const T* dy, const T* x, const T* w,
                          const float* invrms, const float* mean,
                          const T* dres, T* dx, void* dwb, bool narrow,
                          float* part, int rows, int H, hipStream_t s) {
  const int grid = bwd_blocks(rows);
  const int iters = (H + BLOCK * VEC - 1) / (BLOCK * VEC);
#define ROWS(ITERS)                                                          \
  hipLaunchKernelGGL((norm_bwd_rows_kernel<T, LN, ITERS, RES>), dim3(grid),  \
                     dim3(BLOCK), 0, s, dy, x, w, invrms, mean, dres, dx,    \
                     part, rows, H)
  if (iters <= 1) ROWS(1);
  else if (iters <= 2) ROWS(2);
  else ROWS(4);
#undef ROWS
  const int width = (LN ? 2 : 1) * H;
  const dim3 columns((width + 63) / 64);
  if (narrow)
    hipLaunchKernelGGL(norm_parts_kernel<T>, columns, dim3(1024), 0, s, part,
                       (T*)dwb, grid, width);
  else
    hipLaunchKernelGGL(norm_parts_kernel<float>, columns, dim3(1024), 0, s,
                       part, (float*)dwb, grid, width);
}

// dwb: dw [H] and, LN, db [H] behind it; fp32, or with `narrow` (and part) T
template <typename T>
void launch_norm_bwd(const void* dy, const void* x, const void* w,
                     const float* invrms, const float* mean, const void* dres,
                     void* dx, void* dwb, bool narrow, float* part, int rows,
                     int H, bool ln, hipStream_t s) {
  const T* dyt = reinterpret_cast<const T*>(dy);
  const T* xt = reinterpret_cast<const T*>(x);
  const T* wt = reinterpret_cast<const T*>(w);
  const T* rt = reinterpret_cast<const T*>(dres);
  T* dxt = reinterpret_cast<T*>(dx);
  if (part != nullptr) {
    if constexpr (sizeof(T) == 2) {
      if (ln)
        launch_norm_bwd_rows<T, true, false>(dyt, xt, wt, invrms, mean, rt,
                                             dxt, dwb, narrow, part, rows, H, s);
      else if (dres != nullptr)
        launch_norm_bwd_rows<T, false, true>(dyt, xt, wt, invrms, mean, rt,
                                             dxt, dwb, narrow, part, rows, H, s);
      else
        launch_norm_bwd_rows<T, false, false>(dyt, xt, wt, invrms, mean, rt,
                                              dxt, dwb, narrow, part, rows, H, s);
    }
    return;
  }
  int grid = rows < 2048 ? rows : 2048;
  const size_t lds_bytes = (size_t)H * sizeof(float) * (ln ? 2 : 1);
  float* dw = (float*)dwb;
  float* db = dw + H;
  if (ln) {
    hipLaunchKernelGGL((norm_bwd_kernel<T, true>), dim3(grid), dim3(BLOCK),
                       lds_bytes, s, dyt, xt, wt, invrms, mean, dxt, dw, db,
                       rows, H);
  } else {
    hipLaunchKernelGGL((norm_bwd_kernel<T, false>), dim3(grid), dim3(BLOCK),
                       lds_bytes, s, dyt, xt, wt, invrms, mean, dxt, dw, db,
                       rows, H);
  }
}

}  // namespace

// dtype codes: 0=fp32, 1=bf16, 2=fp16
extern "C" void ds_norm_fwd(const void* x, const void* w, const void* b,
                            void* y, float* invrms, float* mean, int rows,
                            int H, float eps, int ln, int dtype, void* stream) {
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  if (dtype == 1)
    launch_norm_fwd<ds::bf16>(x, w, b, y, invrms, mean, rows, H, eps, ln, s);
  else if (dtype == 2)
    launch_norm_fwd<ds::f16>(x, w, b, y, invrms, mean, rows, H, eps, ln, s);
  else
    launch_norm_fwd<float>(x, w, b, y, invrms, mean, rows, H, eps, ln, s);
}

// RMS norm of x + res (16-bit, H a multiple of 8 up to 16384, 16-byte rows):
// the sum and its norm.
extern "C" void ds_add_norm_fwd(const void* x, const void* res, const void* w,
                                void* sum, void* y, float* invrms, int rows,
                                int H, float eps, int dtype, void* stream) {
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const int grid = rows < 8192 ? rows : 8192;
  const int iters = (H + BLOCK * VEC - 1) / (BLOCK * VEC);
#define GO(T, ITERS)                                                          \
  hipLaunchKernelGGL((norm_fwd_cached_kernel<T, false, ITERS, true>),         \
                     dim3(grid), dim3(BLOCK), 0, s, (const T*)x,              \
                     (const T*)res, (T*)sum, (const T*)w, (const T*)nullptr,  \
                     (T*)y, invrms, (float*)nullptr, rows, H, eps)
#define BY_H(T)                  \
  if (iters <= 1) GO(T, 1);      \
  else if (iters <= 2) GO(T, 2); \
  else if (iters <= 4) GO(T, 4); \
  else GO(T, 8)
  if (dtype == 1) { BY_H(ds::bf16); }
  else { BY_H(ds::f16); }
#undef BY_H
#undef GO
}

// The same, bf16, with x in parts [splits][rows][H] fp32; no 1/rms.
extern "C" void ds_add_norm_parts(const float* part, int splits,
                                  const void* res, const void* w, void* sum,
                                  void* y, int rows, int H, float eps,
                                  void* stream) {
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const int iters = (H + BLOCK * VEC - 1) / (BLOCK * VEC);
#define GO(ITERS)                                                           \
  hipLaunchKernelGGL((add_norm_parts_kernel<ITERS>), dim3(rows),            \
                     dim3(WIDE), 0, s, part, splits, (const ds::bf16*)res,  \
                     (ds::bf16*)sum, (const ds::bf16*)w, (ds::bf16*)y, rows,\
                     H, eps)
  if (iters <= 1) GO(1);
  else if (iters <= 2) GO(2);
  else if (iters <= 4) GO(4);
  else GO(8);
#undef GO
}

// Floats of workspace that ds_norm_bwd wants for its rows kernel; 0: it takes
// the general one, and dwb has to be zeroed.
extern "C" long long ds_norm_bwd_parts(const void* dy, const void* x,
                                       const void* dres, const void* dx,
                                       int rows, int H, int ln, int dtype) {
  // up to 8192: twice that needs more registers than a wave has
  const bool ok = dtype != 0 && H <= BLOCK * VEC * 4 &&
                  rows_cached<ds::bf16>(H, {dy, x, dres, dx});
  return ok ? (long long)bwd_blocks(rows) * H * (ln ? 2 : 1) : 0;
}

extern "C" void ds_norm_bwd(const void* dy, const void* x, const void* w,
                            const float* invrms, const float* mean,
                            const void* dres, void* dx, void* dwb, int narrow,
                            float* part, int rows, int H, int ln, int dtype,
                            void* stream) {
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  if (dtype == 1)
    launch_norm_bwd<ds::bf16>(dy, x, w, invrms, mean, dres, dx, dwb, narrow,
                              part, rows, H, ln, s);
  else if (dtype == 2)
    launch_norm_bwd<ds::f16>(dy, x, w, invrms, mean, dres, dx, dwb, narrow,
                             part, rows, H, ln, s);
  else
    launch_norm_bwd<float>(dy, x, w, invrms, mean, dres, dx, dwb, narrow, part,
                           rows, H, ln, s);
}
