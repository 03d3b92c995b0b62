// Python bindings for the deepspeed_amd CDNA4 kernels.
//
// Uses torch-ROCm's native HIP stream API (c10::hip) — no CUDA shims.

#include <torch/extension.h>
#include <pybind11/numpy.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>

#include <tuple>

std::tuple<at::Tensor, int64_t, int64_t, int64_t, bool, int64_t, int64_t>
step_plan(const pybind11::sequence& slots,
          pybind11::array_t<int64_t, pybind11::array::c_style |
                                         pybind11::array::forcecast> pos,
          const pybind11::object& tables, int64_t block_size, int64_t heads,
          int64_t kv_heads, const std::vector<int64_t>& lines, bool pinned);

extern "C" void ds_fused_adam_flat(float* p, const void* g, int grad_dtype,
                                   float* m, float* v, void* p16, long long n,
                                   float lr, float beta1, float beta2, float eps,
                                   float weight_decay, int step, float inv_scale,
                                   int adamw, void* stream);
extern "C" void ds_fused_lion(float* p, const void* g, int grad_dtype,
                              float* m, void* p16, long long n, float lr,
                              float beta1, float beta2, float weight_decay,
                              float inv_scale, void* stream);
extern "C" void ds_fused_lamb(float* p, const void* g, int grad_dtype,
                              float* m, float* v, float* u, float* norms2,
                              void* p16, long long n, float lr, float beta1,
                              float beta2, float eps, float weight_decay,
                              int step, float max_coeff, float min_coeff,
                              float inv_scale, void* stream);
extern "C" void ds_norm_fwd(const void* x, const void* w, const void* b,
                            void* y, float* invrms, float* mean, int rows,
                            int H, float eps, int ln, int dtype, void* stream);
extern "C" void ds_add_norm_fwd(const void* x, const void* res, const void* w,
                                void* sum, void* y, float* invrms, int rows,
                                int H, float eps, int dtype, void* stream);
extern "C" void ds_add_norm_parts(const float* part, int splits,
                                  const void* res, const void* w, void* sum,
                                  void* y, int rows, int H, float eps,
                                  void* stream);
extern "C" long long ds_norm_bwd_parts(const void* dy, const void* x,
                                       const void* dres, const void* dx,
                                       int rows, int H, int ln, int dtype);
extern "C" void ds_norm_bwd(const void* dy, const void* x, const void* w,
                            const float* invrms, const float* mean,
                            const void* dres, void* dx, void* dwb, int narrow,
                            float* part, int rows, int H, int ln, int dtype,
                            void* stream);
extern "C" void ds_rope(const void* x1, void* y1, int heads1, const void* x2,
                        void* y2, int heads2, const float* cos_table,
                        const float* sin_table, const int* positions,
                        long long batch, long long seq, long long dim, int bwd,
                        int dtype, void* stream);
extern "C" void ds_gated_act_fwd(const void* gate, const void* up, void* out,
                                 long long n, int act, int dtype, void* stream);
extern "C" void ds_gated_act_bwd(const void* dout, const void* gate,
                                 const void* up, void* dgate, void* dup,
                                 long long n, int act, int dtype, void* stream);
extern "C" void ds_nhwc_bias_add(const void* act, const void* bias,
                                 const void* other, const void* other_bias,
                                 void* out, long long n, int channels,
                                 int dtype, void* stream);
extern "C" void ds_token_move(const void* x, void* y, const int* idx, int B,
                              int S, int K, int D, int gather, int dtype,
                              void* stream);
extern "C" void ds_cpu_adam_flat(float* p, const void* g, int grad_dtype,
                                 float* m, float* v, void* p16, long long n,
                                 float lr, float beta1, float beta2, float eps,
                                 float weight_decay, int step, float inv_scale,
                                 int adamw);
extern "C" void ds_groupwise_quant(const void* x, int dtype, void* q,
                                   float* scales, long long n, int group_size,
                                   int bits, void* stream);
extern "C" void ds_groupwise_dequant(const void* q, const float* scales,
                                     void* out, int dtype, long long n,
                                     int group_size, int bits, void* stream);
extern "C" void ds_fp_quantize(const void* x, int dtype, void* out,
                               float* scales, long long n, int group_size,
                               int bits, int dequant, void* stream);
extern "C" int ds_sumsq_parts(const long long* n, int count);
extern "C" void ds_sumsq(const void* const* p, const long long* n, int count,
                         int dtype, float* part, float* out, void* stream);
extern "C" void ds_flash_fwd(const void* q, const void* k, const void* v,
                             void* o, float* lse, const long long* strides,
                             int B, int S, int H, int Hkv, int D, float scale,
                             int causal, void* stream);
extern "C" int ds_flash_bwd_splits(int B, int S, int H, int Hkv);
extern "C" void ds_flash_bwd(const void* q, const void* k, const void* v,
                             const void* o, const void* dout, const float* lse,
                             float* stat, float* part, int splits, void* dq,
                             void* dk, void* dv, const long long* strides,
                             int B, int S, int H, int Hkv, int D, float scale,
                             int causal, void* stream);
extern "C" void ds_paged_append(const void* q, const void* k, const void* v,
                                const float* part, int splits, void* qout,
                                void* kpool, void* vpool, const int* dst,
                                const float* cs, const float* sn,
                                const int* positions, int T, int S, int H,
                                int Hkv, int BS, void* stream);
extern "C" int ds_paged_rows(const void* q, const void* kpool,
                              const void* vpool, const int* table,
                              const int* runs, const int* items,
                              const int* merges, const int* lens, void* out,
                              float* part, float* part_ml, int n_items,
                              int n_merges, int any_merge, int nq, int H,
                              int Hkv, int BS, int max_blocks, int splits,
                              float scale, void* stream);
extern "C" int ds_rows_linear(const void* x, int layers, const void* const* w,
                              const float* const* scales,
                              const void* const* bias, void* const* out,
                              const int* n, int M, int K, int group, int mode,
                              void* stream);
extern "C" int ds_rows_append(const void* x, const void* const* w,
                              const float* const* scales,
                              const void* const* bias, void* q, const int* n,
                              int M, int K, int group, void* kpool,
                              void* vpool, const int* dst, const float* cs,
                              const float* sn, const int* positions, int S,
                              int BS, void* stream);
extern "C" int ds_tile_linear_plan(const int* n, int layers, int M, int K,
                                   int mode, int* splits);
extern "C" int ds_tile_linear_stages(int tile, int mode);
extern "C" int ds_tile_linear(const void* const* x, int layers,
                              const void* const* w, const void* const* bias,
                              void* const* out, const int* n, int M, int K,
                              int mode, int tile, int splits, float* part,
                              int merge, void* stream);
extern "C" void ds_transpose_bf16(const void* src, void* dst, int n_batch,
                                  int R, int C, long long row_stride,
                                  int inner, long long inner_stride,
                                  long long outer_stride, void* stream);
extern "C" void ds_transpose_2d(const void* src, void* dst, int R, int C,
                                int ld, void* stream);
extern "C" void ds_fused_softmax(const void* x, const void* mask, void* y,
                                 const float* alibi_slopes, long long rows,
                                 int n, int heads, int sq, int mask_stride,
                                 float scale, int causal, int dtype,
                                 void* stream);
extern "C" void ds_fused_dropout(const void* x, const void* bias,
                                 const void* residual, void* y,
                                 unsigned char* mask_out, long long n,
                                 int cols, float ratio,
                                 unsigned long long seed, int dtype,
                                 void* stream);
extern "C" void ds_dropout_bwd(const void* dy, const unsigned char* mask,
                               void* dx, long long n, float ratio, int dtype,
                               void* stream);
extern "C" void* ds_shm_open(const char* name, int rank, int world,
                             long long max_elems);
extern "C" int ds_shm_allreduce(void* handle, float* data, long long n);
extern "C" void ds_shm_close(void* handle);
extern "C" void* ds_aio_create(long long block_size, int n_threads);
extern "C" void ds_aio_destroy(void* h);
extern "C" int ds_aio_pwrite(void* h, const void* data, long long nbytes,
                             const char* path);
extern "C" int ds_aio_pread(void* h, void* data, long long nbytes,
                            const char* path);
extern "C" int ds_aio_wait(void* h);
extern "C" void ds_cpu_lion_flat(float* p, const void* g, int grad_dtype,
                                 float* m, void* p16, long long n, float lr,
                                 float beta1, float beta2, float weight_decay,
                                 float inv_scale);
extern "C" void ds_ce_fwd(const void* logits, const long long* labels,
                          float* loss, float* lse, int N, long long V,
                          long long ignore_index, void* stream);
extern "C" int ds_embedding_block();
extern "C" void ds_embedding_bwd(const long long* ids, const void* grad,
                                 int* order, int* key, unsigned* has,
                                 int* spans, void* out, int T, int V, int H,
                                 long long padding, void* stream);
extern "C" void ds_ce_total(const float* loss, const long long* labels,
                            float* sum, float* count, float* mean, int N,
                            long long ignore_index, void* stream);
extern "C" void ds_ce_bwd(const void* logits, const long long* labels,
                          const float* lse, const float* gscale, int stride,
                          const float* count, void* dlogits, int N,
                          long long V, long long ignore_index, void* stream);

namespace {

int dtype_code(const at::Tensor& t) {
  switch (t.scalar_type()) {
    case at::kFloat: return 0;
    case at::kBFloat16: return 1;
    case at::kHalf: return 2;
    default:
      TORCH_CHECK(false, "unsupported dtype ", t.scalar_type());
  }
}

void* cur_stream() {
  return reinterpret_cast<void*>(c10::hip::getCurrentHIPStream().stream());
}

// A call's tensors lie on one device, the first's, and its kernels run there,
// whichever device is the current one. Pointers of another device are no error
// to a kernel: it faults on them or reads what is not its own.
struct OneDevice {
  const char* what;
  const c10::Device device;
  const c10::DeviceGuard guard;
  template <typename... Ts>
  OneDevice(const char* what_, const at::Tensor& first, const Ts&... more)
      : what(what_), device(first.device()), guard(device) {
    (check(more), ...);
  }
  void check(const at::Tensor& t) const {
    TORCH_CHECK(t.device() == device, what, ": tensors on different devices, ",
                device, " and ", t.device());
  }
  void check(const c10::optional<at::Tensor>& t) const {
    if (t.has_value() && t->defined()) check(*t);
  }
};

void fused_adam_flat(at::Tensor p, at::Tensor g, at::Tensor m, at::Tensor v,
                     c10::optional<at::Tensor> p16, double lr, double beta1,
                     double beta2, double eps, double weight_decay,
                     int64_t step, double inv_scale, bool adamw) {
  TORCH_CHECK(p.is_contiguous() && g.is_contiguous() && m.is_contiguous() &&
              v.is_contiguous(), "fused_adam_flat: tensors must be contiguous");
  TORCH_CHECK(p.scalar_type() == at::kFloat && m.scalar_type() == at::kFloat &&
              v.scalar_type() == at::kFloat, "p/m/v must be fp32");
  TORCH_CHECK(p.numel() == g.numel() && p.numel() == m.numel() &&
              p.numel() == v.numel(), "numel mismatch");
  void* p16_ptr = nullptr;
  if (p16.has_value() && p16->defined()) {
    TORCH_CHECK(p16->scalar_type() == at::kBFloat16 && p16->is_contiguous() &&
                p16->numel() == p.numel(), "p16 must be contiguous bf16");
    p16_ptr = p16->data_ptr();
  }
  ds_fused_adam_flat(p.data_ptr<float>(), g.data_ptr(), dtype_code(g),
                     m.data_ptr<float>(), v.data_ptr<float>(), p16_ptr,
                     p.numel(), (float)lr, (float)beta1, (float)beta2,
                     (float)eps, (float)weight_decay, (int)step,
                     (float)inv_scale, adamw ? 1 : 0, cur_stream());
}

void fused_lion(at::Tensor p, at::Tensor g, at::Tensor m,
                c10::optional<at::Tensor> p16, double lr, double beta1,
                double beta2, double weight_decay, double inv_scale) {
  TORCH_CHECK(p.is_contiguous() && g.is_contiguous() && m.is_contiguous(),
              "fused_lion: tensors must be contiguous");
  TORCH_CHECK(p.scalar_type() == at::kFloat && m.scalar_type() == at::kFloat,
              "p/m must be fp32");
  void* p16_ptr = nullptr;
  if (p16.has_value() && p16->defined()) p16_ptr = p16->data_ptr();
  ds_fused_lion(p.data_ptr<float>(), g.data_ptr(), dtype_code(g),
                m.data_ptr<float>(), p16_ptr, p.numel(), (float)lr,
                (float)beta1, (float)beta2, (float)weight_decay,
                (float)inv_scale, cur_stream());
}

void fused_lamb(at::Tensor p, at::Tensor g, at::Tensor m, at::Tensor v,
                at::Tensor u, at::Tensor norms2,
                c10::optional<at::Tensor> p16, double lr, double beta1,
                double beta2, double eps, double weight_decay, int64_t step,
                double max_coeff, double min_coeff, double inv_scale) {
  TORCH_CHECK(p.is_contiguous() && g.is_contiguous() && m.is_contiguous() &&
              v.is_contiguous() && u.is_contiguous(),
              "fused_lamb: tensors must be contiguous");
  TORCH_CHECK(norms2.numel() == 2 && norms2.scalar_type() == at::kFloat,
              "norms2 must be fp32[2]");
  void* p16_ptr = nullptr;
  if (p16.has_value() && p16->defined()) p16_ptr = p16->data_ptr();
  ds_fused_lamb(p.data_ptr<float>(), g.data_ptr(), dtype_code(g),
                m.data_ptr<float>(), v.data_ptr<float>(), u.data_ptr<float>(),
                norms2.data_ptr<float>(), p16_ptr, p.numel(), (float)lr,
                (float)beta1, (float)beta2, (float)eps, (float)weight_decay,
                (int)step, (float)max_coeff, (float)min_coeff,
                (float)inv_scale, cur_stream());
}

std::vector<at::Tensor> fp_quantize(at::Tensor x, int64_t group_size,
                                    int64_t bits) {
  TORCH_CHECK(x.is_contiguous() && x.is_cuda(), "fp_quantize: cuda contiguous");
  TORCH_CHECK(bits == 4 || bits == 6 || bits == 8 || bits == 12,
              "bits must be 4/6/8/12");
  TORCH_CHECK(group_size % 8 == 0, "group_size % 8 == 0");
  const long long n = x.numel();
  const long long groups = (n + group_size - 1) / group_size;
  const int vper3 = 24 / (int)bits;
  const long long gu = (group_size + vper3 - 1) / vper3;  // units/group
  auto out = at::empty({groups * gu * 3}, x.options().dtype(at::kByte));
  auto scales = at::empty({groups}, x.options().dtype(at::kFloat));
  ds_fp_quantize(x.data_ptr(), dtype_code(x), out.data_ptr(),
                 scales.data_ptr<float>(), n, (int)group_size, (int)bits, 0,
                 cur_stream());
  return {out, scales};
}

at::Tensor fp_dequantize(at::Tensor q, at::Tensor scales, int64_t numel,
                         int64_t group_size, int64_t bits,
                         at::ScalarType out_dtype) {
  TORCH_CHECK(q.is_contiguous() && q.is_cuda(), "fp_dequantize: cuda");
  auto out = at::empty({numel}, q.options().dtype(out_dtype));
  ds_fp_quantize(q.data_ptr(), dtype_code(out), out.data_ptr(),
                 scales.data_ptr<float>(), numel, (int)group_size, (int)bits,
                 1, cur_stream());
  return out;
}

at::Tensor transpose_bf16(at::Tensor src, int64_t n_batch, int64_t R,
                          int64_t C, int64_t row_stride, int64_t inner,
                          int64_t inner_stride, int64_t outer_stride) {
  TORCH_CHECK(src.is_cuda() && src.scalar_type() == at::kBFloat16,
              "transpose_bf16: cuda bf16");
  auto dst = at::empty({n_batch, C, R}, src.options());
  ds_transpose_bf16(src.data_ptr(), dst.data_ptr(), (int)n_batch, (int)R,
                    (int)C, row_stride, (int)inner, inner_stride,
                    outer_stride, cur_stream());
  return dst;
}

// x [R, C] bf16 -> its transpose [C, R], whose rows start on 16 bytes (their
// stride is R rounded up to 8).
at::Tensor transpose_2d(at::Tensor x) {
  const OneDevice on("transpose_2d", x);
  TORCH_CHECK(x.is_cuda() && x.scalar_type() == at::kBFloat16 &&
              x.dim() == 2 && x.is_contiguous(), "transpose_2d: bf16 matrix");
  const int64_t R = x.size(0), C = x.size(1), ld = (R + 7) / 8 * 8;
  TORCH_CHECK(R < (1ll << 31) && C < (1ll << 31) && (C + 255) / 256 <= 65535,
              "transpose_2d: size");
  auto dst = at::empty({C, ld}, x.options());
  if (R && C)
    ds_transpose_2d(x.data_ptr(), dst.data_ptr(), (int)R, (int)C, (int)ld,
                    cur_stream());
  return dst.narrow(1, 0, R);
}

at::Tensor fused_softmax(at::Tensor x, c10::optional<at::Tensor> mask,
                         c10::optional<at::Tensor> alibi, int64_t heads,
                         int64_t sq, double scale, bool causal) {
  TORCH_CHECK(x.is_cuda() && x.is_contiguous(), "fused_softmax: cuda");
  const int n = x.size(-1);
  const long long rows = x.numel() / n;
  auto y = at::empty_like(x);
  const void* mp = nullptr;
  int mstride = 0;
  if (mask.has_value() && mask->defined()) {
    TORCH_CHECK(mask->scalar_type() == x.scalar_type(), "mask dtype");
    mp = mask->data_ptr();
    mstride = mask->numel() / mask->size(0);
  }
  const float* sl = nullptr;
  if (alibi.has_value() && alibi->defined())
    sl = alibi->data_ptr<float>();
  ds_fused_softmax(x.data_ptr(), mp, y.data_ptr(), sl, rows, n, (int)heads,
                   (int)sq, mstride, (float)scale, causal ? 1 : 0,
                   dtype_code(x), cur_stream());
  return y;
}

std::vector<at::Tensor> fused_dropout(at::Tensor x,
                                      c10::optional<at::Tensor> bias,
                                      c10::optional<at::Tensor> residual,
                                      double ratio, int64_t seed) {
  TORCH_CHECK(x.is_cuda() && x.is_contiguous(), "fused_dropout: cuda");
  auto y = at::empty_like(x);
  auto m = at::empty({x.numel()}, x.options().dtype(at::kByte));
  const void* bp = bias.has_value() && bias->defined() ? bias->data_ptr()
                                                       : nullptr;
  const void* rp = residual.has_value() && residual->defined()
                       ? residual->data_ptr() : nullptr;
  ds_fused_dropout(x.data_ptr(), bp, rp, y.data_ptr(),
                   m.data_ptr<unsigned char>(), x.numel(),
                   (int)x.size(-1), (float)ratio,
                   (unsigned long long)seed, dtype_code(x), cur_stream());
  return {y, m};
}

at::Tensor dropout_bwd(at::Tensor dy, at::Tensor mask, double ratio) {
  auto dx = at::empty_like(dy);
  ds_dropout_bwd(dy.contiguous().data_ptr(),
                 mask.data_ptr<unsigned char>(), dx.data_ptr(), dy.numel(),
                 (float)ratio, dtype_code(dy), cur_stream());
  return dx;
}

static void check_pool(const at::Tensor& q, const at::Tensor& kpool,
                       const at::Tensor& vpool, const char* what) {
  TORCH_CHECK(q.is_cuda() && q.scalar_type() == at::kBFloat16 &&
              q.is_contiguous() && q.dim() == 3 &&
              kpool.scalar_type() == at::kBFloat16 && kpool.is_cuda() &&
              kpool.is_contiguous() && kpool.dim() == 4 &&
              vpool.scalar_type() == at::kBFloat16 && vpool.is_cuda() &&
              vpool.is_contiguous() && kpool.sizes() == vpool.sizes(),
              what, ": bf16 cuda contiguous");
  TORCH_CHECK(q.size(2) == 128 && kpool.size(3) == 128, what,
              ": D must be 128");
  for (auto& t : {q, kpool, vpool})
    TORCH_CHECK(((uintptr_t)t.data_ptr() & 15) == 0, what,
                ": 16-byte accesses");
  TORCH_CHECK(kpool.size(1) > 0 && q.size(1) % kpool.size(1) == 0, what,
              ": H must be a multiple of Hkv");
}

at::Tensor paged_decode(at::Tensor q, at::Tensor kpool, at::Tensor vpool,
                        at::Tensor block_table, at::Tensor lens,
                        int64_t splits, double scale) {
  const OneDevice on("paged_decode", q, kpool, vpool, block_table, lens);
  check_pool(q, kpool, vpool, "paged_decode");
  const int n = q.size(0), H = q.size(1);
  const int Hkv = kpool.size(1), BS = kpool.size(2);
  TORCH_CHECK(H / Hkv <= 16, "paged_decode: at most 16 heads a key head");
  TORCH_CHECK(block_table.scalar_type() == at::kInt &&
              block_table.is_cuda() && block_table.is_contiguous() &&
              block_table.dim() == 2 && block_table.size(0) == n &&
              lens.scalar_type() == at::kInt && lens.is_cuda() &&
              lens.is_contiguous() && lens.numel() == n,
              "table/lens must be int32, one row each");
  TORCH_CHECK(splits >= 1, "paged_decode: at least one split");
  const long items = (long)n * splits;
  auto f32 = q.options().dtype(at::kFloat);
  auto part = at::empty({splits > 1 ? items * Hkv * 16 * 128 : 0}, f32);
  auto part_ml = at::empty({splits > 1 ? items * Hkv * 16 * 2 : 0}, f32);
  auto o = at::empty_like(q);
  if (n == 0) return o;
  const int e = ds_paged_rows(
      q.data_ptr(), kpool.data_ptr(), vpool.data_ptr(),
      block_table.data_ptr<int>(), nullptr, nullptr, nullptr,
      lens.data_ptr<int>(), o.data_ptr(), part.data_ptr<float>(),
      part_ml.data_ptr<float>(), (int)items, n, splits > 1, 1, H, Hkv, BS,
      (int)block_table.size(1), (int)splits, (float)scale, cur_stream());
  TORCH_CHECK(e == 0, "paged_decode: launch failed, hipError_t ", e);
  return o;
}

// meta: int32 [items 4 each | runs 4 each | merges 2 each | table ...], the
// plan of one serving step (built on the host from the cache's block lists).
at::Tensor paged_rows(at::Tensor q, at::Tensor kpool, at::Tensor vpool,
                      at::Tensor meta, int64_t n_items, int64_t n_runs,
                      int64_t n_merges, bool any_merge, int64_t nq,
                      double scale) {
  const OneDevice on("paged_rows", q, kpool, vpool, meta);
  check_pool(q, kpool, vpool, "paged_rows");
  TORCH_CHECK(meta.scalar_type() == at::kInt && meta.is_cuda() &&
              meta.is_contiguous() &&
              meta.numel() >= 4 * n_items + 4 * n_runs + 2 * n_merges &&
              (nq == 1 || nq == 2 || nq == 8), "paged_rows: plan");
  const int H = q.size(1), Hkv = kpool.size(1);
  const int* p = meta.data_ptr<int>();
  auto f32 = q.options().dtype(at::kFloat);
  const long cols = any_merge ? n_items * Hkv * 16 * nq : 0;
  auto part = at::empty({cols * 128}, f32);
  auto part_ml = at::empty({cols * 2}, f32);
  auto o = at::empty_like(q);
  if (n_items == 0) return o;
  const int e = ds_paged_rows(
      q.data_ptr(), kpool.data_ptr(), vpool.data_ptr(),
      p + 4 * (n_items + n_runs) + 2 * n_merges, p + 4 * n_items, p,
      p + 4 * (n_items + n_runs), nullptr, o.data_ptr(),
      part.data_ptr<float>(), part_ml.data_ptr<float>(), (int)n_items,
      (int)n_merges, any_merge, (int)nq, H, Hkv, (int)kpool.size(2), 0, 0,
      (float)scale, cur_stream());
  TORCH_CHECK(e == 0, "paged_rows: launch failed, hipError_t ", e);
  return o;
}

// Angles of a step's T rows, and that these have each a row of the pool.
struct Turn {
  const float *cs = nullptr, *sn = nullptr;
  const int* pos = nullptr;

  Turn(int64_t T, const at::Tensor& dst,
       const c10::optional<at::Tensor>& cos_table,
       const c10::optional<at::Tensor>& sin_table,
       const c10::optional<at::Tensor>& positions, int64_t S) {
    TORCH_CHECK(dst.scalar_type() == at::kInt && dst.is_cuda() &&
                dst.is_contiguous() && dst.numel() == T, "paged_append: dst");
    TORCH_CHECK(S >= 1 && T % S == 0, "paged_append: S");
    if (!cos_table.has_value()) return;
    for (auto& t : {*cos_table, *sin_table})
      TORCH_CHECK(t.scalar_type() == at::kFloat && t.is_cuda() &&
                  t.is_contiguous() && t.dim() == 2 && t.size(1) == 64,
                  "paged_append: tables must be fp32 [positions, 64]");
    cs = cos_table->data_ptr<float>();
    sn = sin_table->data_ptr<float>();
    if (positions.has_value()) {
      TORCH_CHECK(positions->scalar_type() == at::kInt &&
                  positions->is_cuda() && positions->is_contiguous() &&
                  positions->numel() == T, "paged_append: positions");
      pos = positions->data_ptr<int>();
    } else {
      TORCH_CHECK(cos_table->size(0) >= S, "table shorter than sequence");
    }
  }
};

// What both forms below share; q of T rows and H heads: its values, or what it
// is like.
at::Tensor append_rows(const at::Tensor& q, const void* k, const void* v,
                       const void* q_or_bias, const float* part, int splits,
                       at::Tensor kpool, at::Tensor vpool, at::Tensor dst,
                       c10::optional<at::Tensor> cos_table,
                       c10::optional<at::Tensor> sin_table,
                       c10::optional<at::Tensor> positions, int64_t S,
                       at::Tensor out) {
  const int T = q.size(0), H = q.size(1), Hkv = kpool.size(1);
  const Turn turn(T, dst, cos_table, sin_table, positions, S);
  if (T == 0) return out;
  ds_paged_append(q_or_bias, k, v, part, splits, out.data_ptr(),
                  kpool.data_ptr(), vpool.data_ptr(), dst.data_ptr<int>(),
                  turn.cs, turn.sn, turn.pos, T, (int)S, H, Hkv,
                  (int)kpool.size(2),
                  cur_stream());
  return out;
}

// New rows k, v [T, Hkv, 128] into the pool rows dst [T]; with tables also
// the rotary embedding of k on its way there and of q [T, H, 128], returned.
at::Tensor paged_append(at::Tensor q, at::Tensor k, at::Tensor v,
                        at::Tensor kpool, at::Tensor vpool, at::Tensor dst,
                        c10::optional<at::Tensor> cos_table,
                        c10::optional<at::Tensor> sin_table,
                        c10::optional<at::Tensor> positions, int64_t S) {
  const OneDevice on("paged_append", q, k, v, kpool, vpool, dst, cos_table,
                     sin_table, positions);
  check_pool(q, kpool, vpool, "paged_append");
  for (auto& x : {k, v})
    TORCH_CHECK(x.is_cuda() && x.scalar_type() == at::kBFloat16 &&
                x.is_contiguous() && x.dim() == 3 && x.size(0) == q.size(0) &&
                x.size(1) == kpool.size(1) && x.size(2) == 128 &&
                ((uintptr_t)x.data_ptr() & 15) == 0, "paged_append: k/v");
  return append_rows(q, k.data_ptr(), v.data_ptr(), q.data_ptr(), nullptr, 1,
                     kpool, vpool, dst, cos_table, sin_table, positions, S,
                     cos_table.has_value() ? at::empty_like(q) : q);
}

// Whether rows_linear.hip is ahead of tile_linear.hip for bf16 layers of `all`
// features: up to 16 rows, past which x is most of what it reads, and up to 32 for
// layers of two rounds of tiles of 16 features (us, either at 24 and 32 rows, K 4096
// unless said: 4096 9.1 / 11.5 and 9.8 / 11.8; q, k and v of that 12.2 / 14.7 and 12.9 /
// 15.1; 2048, K 2048 5.8 / 8.3 and 6.0 / 8.3; gate and up 2816, K 1024 5.2 / 7.4 and 5.4 /
// 7.5; but 9216, K 3072 15.8 / 15.5; gate and up 5632, K 2048 11.5 / 12.1 and 11.8 /
// 12.2, 14336 38.1 / 38.2 and 39.5 / 38.0). Over 3700 layers of the time of the latter
// 0.5 to 0.9 up to K 4096, 1.1 to 1.4 at 8192 and fewer than 192 tiles; gates 0.5 to 0.75
// at any K; three rounds 1.1.
bool few_rows(int64_t M, int64_t all, int64_t K, int64_t mode) {
  return M <= 16 || (M <= 32 && all <= 8192 && (mode == 1 || K <= 4096));
}

// bf16 weights on one input, pointers and features of each; outputs made anew:
// one each, or with mode 1 silu(layer 0) * layer 1.
struct Layers {
  const void *w[3], *b[3];
  const float* sc[3];
  void* o[3];
  int n[3];
  int count = 0;
  int64_t all = 0;
  std::vector<at::Tensor> out;

  void add(const char* what, const at::Tensor& x, const at::Tensor& weight,
           const c10::optional<at::Tensor>& bias, at::ScalarType type,
           int64_t mode, bool output = true) {
    const int64_t M = x.size(0), K = x.size(1);
    const int i = count++;
    TORCH_CHECK(weight.is_cuda() && weight.is_contiguous() &&
                weight.scalar_type() == type && weight.numel() % K == 0 &&
                (type == at::kChar ||
                 (weight.dim() == 2 && weight.size(1) == K)) &&
                weight.numel() > 0 && weight.numel() / K < (1 << 30) &&
                ((uintptr_t)weight.data_ptr() & 15) == 0, what, ": weight");
    n[i] = weight.numel() / K;
    all += n[i];
    w[i] = weight.data_ptr();
    b[i] = nullptr;
    if (bias.has_value()) {
      TORCH_CHECK(bias->is_cuda() && bias->is_contiguous() &&
                  bias->scalar_type() == at::kBFloat16 &&
                  bias->numel() == n[i], what, ": bias");
      b[i] = bias->data_ptr();
    }
    if (output && (mode == 0 || i == 0))
      out.push_back(at::empty({M, n[i]}, x.options()));
    o[i] = output ? out.back().data_ptr() : nullptr;
    TORCH_CHECK(mode == 0 || n[0] == n[i], what, ": gate and up");
  }
  // The last one's scales.
  void scaled(const char* what, const at::Tensor& weight,
              const at::Tensor& scales, int64_t group) {
    TORCH_CHECK(scales.is_cuda() && scales.is_contiguous() &&
                scales.scalar_type() == at::kFloat && group > 0 &&
                group % 256 == 0 &&
                scales.numel() == (weight.numel() + group - 1) / group,
                what, ": scales");
    sc[count - 1] = scales.data_ptr<float>();
  }
  // Whether tile_linear.hip takes them; does it if so. A tile and a number of
  // splits may be asked for. With `parts`, sums in parts [splits, M, all] are left
  // there, and the outputs are not written.
  bool tiled(const at::Tensor& x, int64_t mode, int tile = -1, int splits = 1,
             at::Tensor* parts = nullptr) {
    const int64_t M = x.size(0), K = x.size(1);
    if (K % 64 || K > (1 << 22) || M >= (1 << 30)) return false;
    for (int i = 0; i < count; ++i)
      if (n[i] % 4) return false;
    if (tile < 0)
      tile = ds_tile_linear_plan(n, count, (int)M, (int)K, (int)mode, &splits);
    const int stages = ds_tile_linear_stages(tile, (int)mode);
    if (stages < 1 || splits < 1 || K / 64 / splits < stages ||
        (mode && splits > 1))
      return false;
    at::Tensor part;
    if (splits > 1)
      part = at::empty({splits, M, all}, x.options().dtype(at::kFloat));
    const void* xs[1] = {x.data_ptr()};
    const int e = ds_tile_linear(
        xs, count, w, b, o, n, (int)M, (int)K, (int)mode, tile, splits,
        splits > 1 ? part.data_ptr<float>() : nullptr, parts == nullptr,
        cur_stream());
    TORCH_CHECK(e == 0, "tile_linear: launch failed with error ", e);
    if (parts) *parts = part;
    return true;
  }
};

// Linear layers on one input of a few rows, by rows_linear.hip or tile_linear.hip
// (few_rows). weights: bf16 [N, K], or int8 (any
// shape, N * K long) with their groupwise scales. mode 1 returns
// silu(layer 0) * layer 1.
std::vector<at::Tensor> rows_linear(
    at::Tensor x, std::vector<at::Tensor> weights,
    std::vector<at::Tensor> scales,
    std::vector<c10::optional<at::Tensor>> biases, int64_t group,
    int64_t mode) {
  const OneDevice on("rows_linear", x);
  for (auto& t : weights) on.check(t);
  for (auto& t : scales) on.check(t);
  for (auto& t : biases) on.check(t);
  const int L = weights.size();
  TORCH_CHECK(x.is_cuda() && x.scalar_type() == at::kBFloat16 &&
              x.is_contiguous() && x.dim() == 2, "rows_linear: x");
  const int64_t M = x.size(0), K = x.size(1);
  TORCH_CHECK(M >= 1 && M <= (scales.empty() ? 32 : 64) && K > 0 &&
              K % 256 == 0 && L >= 1 && L <= 3 && (mode == 0 || L == 2) &&
              (scales.empty() || (int)scales.size() == L) &&
              (int)biases.size() == L, "rows_linear: shape");
  TORCH_CHECK(((uintptr_t)x.data_ptr() & 15) == 0, "rows_linear: alignment");
  const bool i8 = !scales.empty();
  Layers y;
  for (int i = 0; i < L; ++i) {
    y.add("rows_linear", x, weights[i], biases[i],
          i8 ? at::kChar : at::kBFloat16, mode);
    if (i8) y.scaled("rows_linear", weights[i], scales[i], group);
  }
  if (!i8 && !few_rows(M, y.all, K, mode) && y.tiled(x, mode)) return y.out;
  const int e = ds_rows_linear(x.data_ptr(), L, y.w, i8 ? y.sc : nullptr, y.b,
                               y.o, y.n, (int)M, (int)K, (int)group, (int)mode,
                               cur_stream());
  TORCH_CHECK(e == 0, "rows_linear: launch failed with error ", e);
  return y.out;
}

// Linear layers on one input of any number of rows, bf16 (tile_linear.hip).
std::vector<at::Tensor> tile_linear(
    at::Tensor x, std::vector<at::Tensor> weights,
    std::vector<c10::optional<at::Tensor>> biases, int64_t mode, int64_t tile,
    int64_t splits) {
  const OneDevice on("tile_linear", x);
  for (auto& t : weights) on.check(t);
  for (auto& t : biases) on.check(t);
  const int L = weights.size();
  TORCH_CHECK(x.is_cuda() && x.scalar_type() == at::kBFloat16 &&
              x.is_contiguous() && x.dim() == 2 && x.numel() > 0 &&
              ((uintptr_t)x.data_ptr() & 15) == 0, "tile_linear: x");
  TORCH_CHECK(L >= 1 && L <= 3 && (mode == 0 || (mode == 1 && L == 2)) &&
              (int)biases.size() == L, "tile_linear: shape");
  Layers y;
  for (int i = 0; i < L; ++i)
    y.add("tile_linear", x, weights[i], biases[i], at::kBFloat16, mode);
  TORCH_CHECK(y.tiled(x, mode, (int)tile, (int)splits),
              "tile_linear: features in fours, inputs in 64s, 192 or more");
  return y.out;
}

// Gradients of linear layers y = x W^T on one input, bf16 (tile_linear.hip). mode
// 2: of the input, the sum over the layers of dy W; mode 3: of each weight, dy^T
// x, to `into` where that holds a tensor. others: the weights, or the input alone.
std::vector<at::Tensor> tile_linear_grad(
    const std::vector<at::Tensor>& dys, const std::vector<at::Tensor>& others,
    int mode, int tile, int splits,
    const std::vector<c10::optional<at::Tensor>>& into = {}) {
  const int L = dys.size();
  TORCH_CHECK(L >= 1 && L <= 3 && (int)others.size() == (mode == 2 ? L : 1),
              "tile_linear_grad: layers");
  const OneDevice on("tile_linear_grad", dys[0]);
  for (auto& t : dys) on.check(t);
  for (auto& t : others) on.check(t);
  for (auto& t : into) on.check(t);
  const int64_t M = dys[0].size(0), K = others[0].size(1);
  const void *x[3], *w[3], *b[3] = {};
  void* o[3];
  int n[3];
  int64_t all = 0;
  auto good = [](const at::Tensor& t) {
    return t.is_cuda() && t.scalar_type() == at::kBFloat16 && t.dim() == 2 &&
        t.is_contiguous() && t.numel() > 0 &&
        ((uintptr_t)t.data_ptr() & 15) == 0;
  };
  std::vector<at::Tensor> out;
  for (int i = 0; i < L; ++i) {
    const auto& other = others[mode == 2 ? i : 0];
    TORCH_CHECK(good(dys[i]) && good(other) && dys[i].size(0) == M &&
                other.size(1) == K &&
                other.size(0) == (mode == 2 ? dys[i].size(1) : M) &&
                dys[i].size(1) <= (1 << 23) && K % 8 == 0 &&
                dys[i].size(1) % (mode == 2 ? 64 : 8) == 0,
                "tile_linear_grad: operands");
    x[i] = dys[i].data_ptr();
    w[i] = other.data_ptr();
    n[i] = dys[i].size(1);
    all += n[i];
    const int64_t rows = mode == 2 ? M : n[i];
    if (i < (int)into.size() && into[i].has_value()) {
      TORCH_CHECK(good(*into[i]) && into[i]->size(0) == rows &&
                  into[i]->size(1) == K, "tile_linear_grad: into");
      out.push_back(*into[i]);
    } else if (mode == 3 || i == 0) {
      out.push_back(at::empty({rows, K}, dys[0].options()));
    }
    o[i] = out.back().data_ptr();
  }
  TORCH_CHECK(K <= (1 << 22) && M < (1 << 30) && all < (1ll << 31),
              "tile_linear_grad: size");
  if (tile < 0)
    tile = ds_tile_linear_plan(n, L, (int)M, (int)K, mode, &splits);
  const int stages = ds_tile_linear_stages(tile, mode);
  const int64_t steps = mode == 2 ? all / 64 : (M + 63) / 64;
  TORCH_CHECK(stages > 0 && splits > 0 && steps / splits >= stages,
              "tile_linear_grad: too little to add up");
  at::Tensor part;
  if (splits > 1)
    part = at::empty({splits * (mode == 2 ? M : all) * K},
                     dys[0].options().dtype(at::kFloat));
  const int e = ds_tile_linear(
      x, L, w, b, o, n, (int)M, (int)K, mode, tile, splits,
      splits > 1 ? part.data_ptr<float>() : nullptr, 1, cur_stream());
  TORCH_CHECK(e == 0, "tile_linear_grad: launch failed with error ", e);
  return out;
}

// (tile, splits) that tile_linear.hip takes for layers of ns features.
std::tuple<int64_t, int64_t> tile_linear_plan(const std::vector<int64_t>& ns,
                                              int64_t M, int64_t K,
                                              int64_t mode) {
  TORCH_CHECK(ns.size() >= 1 && ns.size() <= 3 && M > 0 && M < (1 << 30) &&
              K > 0 && K <= (1 << 22) && mode >= 0 && mode <= 3,
              "tile_linear_plan: layers");
  int n[3], splits = 1;
  for (size_t i = 0; i < ns.size(); ++i) {
    TORCH_CHECK(ns[i] > 0 && ns[i] <= (1 << 29), "tile_linear_plan: features");
    n[i] = (int)ns[i];
  }
  const int tile = ds_tile_linear_plan(n, (int)ns.size(), (int)M, (int)K,
                                       (int)mode, &splits);
  return {tile, splits};
}

at::Tensor tile_linear_dx(std::vector<at::Tensor> dys,
                          std::vector<at::Tensor> weights, int64_t tile,
                          int64_t splits) {
  return tile_linear_grad(dys, weights, 2, (int)tile, (int)splits)[0];
}

std::vector<at::Tensor> tile_linear_dw(at::Tensor x,
                                       std::vector<at::Tensor> dys,
                                       int64_t tile, int64_t splits,
                                       std::vector<c10::optional<at::Tensor>>
                                           into) {
  return tile_linear_grad(dys, {x}, 3, (int)tile, (int)splits, into);
}

at::Tensor sum_of_squares(std::vector<at::Tensor> ts) {
  TORCH_CHECK(!ts.empty(), "sum_of_squares: no tensors");
  const OneDevice on("sum_of_squares", ts[0]);
  std::vector<const void*> p;
  std::vector<long long> n;
  for (auto& t : ts) {
    TORCH_CHECK(t.is_cuda() && t.is_contiguous() &&
                t.scalar_type() == ts[0].scalar_type() &&
                t.device() == ts[0].device() &&
                (t.scalar_type() == at::kFloat ||
                 t.scalar_type() == at::kBFloat16) &&
                t.numel() < (1ll << 45), "sum_of_squares: bf16 or fp32 GPU");
    p.push_back(t.data_ptr());
    n.push_back(t.numel());
  }
  auto f32 = ts[0].options().dtype(at::kFloat);
  auto part = at::empty({ds_sumsq_parts(n.data(), (int)n.size())}, f32);
  auto out = at::empty({}, f32);
  ds_sumsq(p.data(), n.data(), (int)n.size(), dtype_code(ts[0]),
           part.data_ptr<float>(), out.data_ptr<float>(), cur_stream());
  return out;
}

class ShmComm {
 public:
  ShmComm(const std::string& name, int64_t rank, int64_t world,
          int64_t max_elems) {
    h_ = ds_shm_open(name.c_str(), (int)rank, (int)world, max_elems);
    TORCH_CHECK(h_ != nullptr, "shm_open failed for group ", name);
  }
  ~ShmComm() {
    if (h_) ds_shm_close(h_);
  }
  void all_reduce(at::Tensor t) {
    TORCH_CHECK(t.device().is_cpu() && t.scalar_type() == at::kFloat &&
                t.is_contiguous(), "shm all_reduce: contiguous fp32 CPU");
    TORCH_CHECK(ds_shm_allreduce(h_, t.data_ptr<float>(), t.numel()) == 0,
                "shm all_reduce failed (tensor larger than max_elems?)");
  }

 private:
  void* h_ = nullptr;
};

void cpu_adam_flat(at::Tensor p, at::Tensor g, at::Tensor m, at::Tensor v,
                   c10::optional<at::Tensor> p16, double lr, double beta1,
                   double beta2, double eps, double weight_decay, int64_t step,
                   double inv_scale, bool adamw) {
  TORCH_CHECK(!p.is_cuda() && !g.is_cuda(), "cpu_adam_flat: host tensors only");
  TORCH_CHECK(p.is_contiguous() && g.is_contiguous() && m.is_contiguous() &&
              v.is_contiguous(), "cpu_adam_flat: tensors must be contiguous");
  TORCH_CHECK(p.scalar_type() == at::kFloat && m.scalar_type() == at::kFloat &&
              v.scalar_type() == at::kFloat, "p/m/v must be fp32");
  TORCH_CHECK(p.numel() == g.numel() && p.numel() == m.numel() &&
              p.numel() == v.numel(), "numel mismatch");
  void* p16_ptr = nullptr;
  if (p16.has_value() && p16->defined()) {
    TORCH_CHECK(p16->scalar_type() == at::kBFloat16 && p16->is_contiguous() &&
                !p16->is_cuda() && p16->numel() == p.numel(),
                "p16 must be contiguous host bf16");
    p16_ptr = p16->data_ptr();
  }
  ds_cpu_adam_flat(p.data_ptr<float>(), g.data_ptr(), dtype_code(g),
                   m.data_ptr<float>(), v.data_ptr<float>(), p16_ptr,
                   p.numel(), (float)lr, (float)beta1, (float)beta2, (float)eps,
                   (float)weight_decay, (int)step, (float)inv_scale,
                   adamw ? 1 : 0);
}

std::tuple<at::Tensor, at::Tensor, at::Tensor> norm_fwd(
    at::Tensor x, at::Tensor w, c10::optional<at::Tensor> b, double eps,
    bool layernorm) {
  const OneDevice on("norm_fwd", x, w, b);
  TORCH_CHECK(x.is_contiguous() && w.is_contiguous(), "must be contiguous");
  const int64_t H = x.size(-1);
  const int64_t rows = x.numel() / H;
  TORCH_CHECK(w.numel() == H, "weight shape mismatch");
  // the kernel reads the weight in x's type
  TORCH_CHECK(w.scalar_type() == x.scalar_type(), "norm_fwd: types");
  auto y = at::empty_like(x);
  auto f32opts = x.options().dtype(at::kFloat);
  auto invrms = at::empty({rows}, f32opts);
  auto mean = layernorm ? at::empty({rows}, f32opts) : at::empty({0}, f32opts);
  const void* bptr = nullptr;
  if (b.has_value() && b->defined()) {
    TORCH_CHECK(b->is_contiguous() && b->numel() == H, "bias shape mismatch");
    TORCH_CHECK(b->scalar_type() == x.scalar_type(), "norm_fwd: types");
    bptr = b->data_ptr();
  }
  TORCH_CHECK(x.is_cuda(), "norm_fwd: GPU tensors");
  ds_norm_fwd(x.data_ptr(), w.data_ptr(), bptr, y.data_ptr(),
              invrms.data_ptr<float>(),
              layernorm ? mean.data_ptr<float>() : nullptr, (int)rows, (int)H,
              (float)eps, layernorm ? 1 : 0, dtype_code(x), cur_stream());
  return {y, invrms, mean};
}

// dres (RMS only): a further gradient of x, added to dx.
// (dx, dw, LN: db); dw and db in fp32, or dw in `into`, which has x's type.
std::tuple<at::Tensor, at::Tensor, at::Tensor> norm_bwd(
    at::Tensor dy, at::Tensor x, at::Tensor w, at::Tensor invrms,
    c10::optional<at::Tensor> mean, bool layernorm,
    c10::optional<at::Tensor> dres, c10::optional<at::Tensor> into) {
  const OneDevice on("norm_bwd", x, dy, w, invrms, mean, dres, into);
  TORCH_CHECK(dy.is_contiguous() && x.is_contiguous() && w.is_contiguous(),
              "must be contiguous");
  const int64_t H = x.size(-1);
  const int64_t rows = x.numel() / H;
  TORCH_CHECK(w.numel() == H && dy.numel() == x.numel() &&
              w.scalar_type() == x.scalar_type() &&
              dy.scalar_type() == x.scalar_type() &&
              invrms.scalar_type() == at::kFloat && invrms.numel() == rows &&
              invrms.is_contiguous() &&
              (!layernorm || (mean.has_value() && mean->numel() == rows &&
                              mean->scalar_type() == at::kFloat &&
                              mean->is_contiguous())),
              "norm_bwd: types or sizes");
  auto dx = at::empty_like(x);
  auto f32opts = x.options().dtype(at::kFloat);
  const void* rp = nullptr;
  if (dres.has_value()) {
    TORCH_CHECK(!layernorm && dres->is_contiguous() &&
                dres->scalar_type() == x.scalar_type() &&
                dres->numel() == x.numel(), "norm_bwd: dres");
    rp = dres->data_ptr();
  }
  const int code = dtype_code(x), ln = layernorm ? 1 : 0;
  const long long n = rows ? ds_norm_bwd_parts(
      dy.data_ptr(), x.data_ptr(), rp, dx.data_ptr(), (int)rows, (int)H, ln,
      code) : 0;
  auto part = at::empty({n}, f32opts);
  const int64_t width = layernorm ? 2 * H : H;
  TORCH_CHECK(!into || (!layernorm && into->is_contiguous() &&
                        into->numel() == H &&
                        into->scalar_type() == x.scalar_type()),
              "norm_bwd: into");
  const bool narrow = into.has_value() && n;
  auto dwb = narrow ? *into
      : n ? at::empty({width}, f32opts) : at::zeros({width}, f32opts);
  if (rows)
    ds_norm_bwd(dy.data_ptr(), x.data_ptr(), w.data_ptr(),
                invrms.data_ptr<float>(),
                layernorm ? mean->data_ptr<float>() : nullptr, n ? rp : nullptr,
                dx.data_ptr(), dwb.data_ptr(), narrow,
                n ? part.data_ptr<float>() : nullptr, (int)rows, (int)H, ln,
                code, cur_stream());
  if (rp != nullptr && !n) dx.add_(*dres);
  if (into) {
    if (!narrow) into->copy_(dwb.view(into->sizes()));
    return {dx, *into, at::empty({0}, f32opts)};
  }
  return {dx, dwb.narrow(0, 0, H),
          layernorm ? dwb.narrow(0, H, H) : at::empty({0}, f32opts)};
}

// RMS norm of x + res -> (norm, sum, 1/rms); add_rms_norm in ops/norms.py
// takes another way for what the kernel does not.
std::tuple<at::Tensor, at::Tensor, at::Tensor> add_norm_fwd(
    at::Tensor x, at::Tensor res, at::Tensor w, double eps) {
  const OneDevice on("add_norm_fwd", x, res, w);
  const int64_t H = x.size(-1);
  for (auto& t : {x, res})
    TORCH_CHECK(t.is_cuda() && t.is_contiguous() &&
                t.scalar_type() == w.scalar_type() &&
                t.sizes() == x.sizes() &&
                (t.scalar_type() == at::kBFloat16 ||
                 t.scalar_type() == at::kHalf) &&
                ((uintptr_t)t.data_ptr() & 15) == 0, "add_norm_fwd");
  TORCH_CHECK(H % 8 == 0 && H > 0 && H <= 16384 && w.numel() == H &&
              w.is_cuda() && w.is_contiguous(), "add_norm_fwd: size");
  const int64_t rows = x.numel() / H;
  auto y = at::empty_like(x), sum = at::empty_like(x);
  auto inv = at::empty({rows}, x.options().dtype(at::kFloat));
  if (rows)
    ds_add_norm_fwd(x.data_ptr(), res.data_ptr(), w.data_ptr(),
                    sum.data_ptr(), y.data_ptr(), inv.data_ptr<float>(),
                    (int)rows, (int)H, (float)eps, dtype_code(x),
                    cur_stream());
  return {y, sum, inv};
}

// own_forward of ops/linear.py, for what Layers::tiled takes.
bool own_forward(int64_t M, const std::vector<int64_t>& ns, int64_t K,
                 int64_t mode) {
  if (M < 2560 || mode == 1) return true;
  int64_t most = 0, all = 0, tiles = 0;
  for (const int64_t n : ns) {
    most = std::max(most, n);
    all += n;
    tiles += (M + 255) / 256 * ((n + 255) / 256);
  }
  if (ns.size() == 1 && K >= 16384)
    return all % 4096 != 0 || (all < 16384 && M % 256 != 0) ||
        (all < 8192 && tiles % 256 != 0);
  if (ns.size() == 1)
    return M % 256 != 0 || (all < 65536 && (K < 3072 || tiles % 256 != 0));
  return M % 256 != 0 || (most * K < (1 << 26) &&
                          (M < 16384 || 1.0 * M * all * K < 4e11));
}

// A decoder layer of a serving step over the paged pool, from the residual
// stream x [.., H] that still lacks the last layer's output delta, to the same:
// norm, q k v, rotation and append, attention, output, norm, gated MLP. What the
// modules of models/llama.py call one by one, without their host time between
// the launches (a layer of nine 180 us there, 40 here). norms: two weights.
// weights: q, k, v, o, gate, up, down; int8 with scales. meta.. nq: StepPlan.
// Products whose contraction is split leave their sums in parts to what reads
// them next: the append, the norms, and with `parts` the next layer's, whose
// delta is fp32 [splits, rows, H] then (and which is called with `behind`: another
// delta has x's type).
std::tuple<at::Tensor, at::Tensor> paged_decoder_layer(
    at::Tensor x, c10::optional<at::Tensor> delta,
    const std::vector<at::Tensor>& norms, double eps0, double eps1,
    const std::vector<at::Tensor>& weights,
    const std::vector<at::Tensor>& scales,
    const std::vector<c10::optional<at::Tensor>>& biases, int64_t group,
    at::Tensor cos_table, at::Tensor sin_table,
    c10::optional<at::Tensor> positions, int64_t S, at::Tensor kpool,
    at::Tensor vpool, at::Tensor dst, at::Tensor meta, int64_t n_items,
    int64_t n_runs, int64_t n_merges, bool any_merge, int64_t nq,
    double scale, bool behind, bool parts) {
  const OneDevice on("paged_decoder_layer", x, delta, cos_table, sin_table,
                     positions, kpool, vpool, dst, meta);
  TORCH_CHECK(norms.size() == 2 && weights.size() == 7 && biases.size() == 7 &&
              (scales.empty() || scales.size() == 7) && x.is_contiguous() &&
              x.numel() > 0 && x.scalar_type() == at::kBFloat16 &&
              kpool.dim() == 4, "paged_decoder_layer");
  TORCH_CHECK(!delta || behind || delta->scalar_type() == x.scalar_type(),
              "paged_decoder_layer: delta");
  const int64_t H = x.size(-1), M = x.numel() / H;
  auto own = [&](const at::Tensor& in, int first, int count, int64_t mode) {
    std::vector<int64_t> ns;
    for (int i = first; i < first + count; ++i)
      ns.push_back(weights[i].numel() / in.size(1));
    return own_forward(M, ns, in.size(1), mode);
  };
  auto linears = [&](const at::Tensor& in, int first, int count,
                     int64_t mode) {
    const std::vector<at::Tensor> w(weights.begin() + first,
                                    weights.begin() + first + count);
    const std::vector<c10::optional<at::Tensor>> b(
        biases.begin() + first, biases.begin() + first + count);
    if (!scales.empty() || M <= 32) {
      std::vector<at::Tensor> s;
      if (!scales.empty())
        s.assign(scales.begin() + first, scales.begin() + first + count);
      return rows_linear(in, w, s, b, group, mode);
    }
    if (!own(in, first, count, mode)) {
      std::vector<at::Tensor> y;
      for (int i = 0; i < count; ++i) y.push_back(at::linear(in, w[i], b[i]));
      return y;
    }
    return tile_linear(in, w, b, mode, -1, 1);
  };
  // outputs, or their sums in parts
  using Sums = std::pair<std::vector<at::Tensor>, at::Tensor>;
  auto sums = [&](const at::Tensor& in, int first, int count) -> Sums {
    int64_t all = 0;
    for (int i = first; i < first + count; ++i)
      all += weights[i].numel() / in.size(1);
    if (!scales.empty() || few_rows(M, all, in.size(1), 0) ||
        !own(in, first, count, 0))
      return {linears(in, first, count, 0), at::Tensor()};
    Layers y;
    at::Tensor part;
    for (int i = first; i < first + count; ++i)
      y.add("paged_decoder_layer", in, weights[i], biases[i], at::kBFloat16, 0);
    if (!y.tiled(in, 0, -1, 1, &part))
      return {linears(in, first, count, 0), at::Tensor()};
    return {y.out, part};
  };
  at::Tensor stream = x.view({M, H}), h;
  auto add_norm = [&](const at::Tensor& d, const at::Tensor& w, double eps) {
    if (d.scalar_type() != at::kFloat) {
      std::tie(h, stream, std::ignore) =
          add_norm_fwd(d.view({M, H}), stream, w, eps);
      return;
    }
    TORCH_CHECK(d.dim() == 3 && d.size(1) == M && d.size(2) == H &&
                d.is_contiguous() && w.is_contiguous() && w.numel() == H &&
                w.scalar_type() == at::kBFloat16 && H % 8 == 0 &&
                H <= 16384 && ((uintptr_t)stream.data_ptr() & 15) == 0,
                "paged_decoder_layer: norm");
    auto sum = at::empty_like(stream);
    h = at::empty_like(stream);
    ds_add_norm_parts(d.data_ptr<float>(), (int)d.size(0), stream.data_ptr(),
                      w.data_ptr(), sum.data_ptr(), h.data_ptr(), (int)M,
                      (int)H, (float)eps, cur_stream());
    stream = sum;
  };
  // here, not where each is used: sums() launches on what it is given
  for (auto& w : norms) on.check(w);
  for (auto& w : weights) on.check(w);
  for (auto& s : scales) on.check(s);
  for (auto& b : biases) on.check(b);
  if (delta.has_value())
    add_norm(*delta, norms[0], eps0);
  else
    h = std::get<0>(norm_fwd(stream, norms[0], c10::nullopt, eps0, false));
  // q turned, k and v in the pool, by the product of few rows itself
  auto few_append = [&]() -> at::Tensor {
    const bool i8 = !scales.empty();
    const int64_t all =
        (weights[0].numel() + weights[1].numel() + weights[2].numel()) / H;
    if (M > 32 || H % 256 || !(i8 || few_rows(M, all, H, 0)))
      return at::Tensor();
    Layers y;
    for (int i = 0; i < 3; ++i) {
      y.add("paged_decoder_layer", h, weights[i], biases[i],
            i8 ? at::kChar : at::kBFloat16, 0, i == 0);
      if (i8)
        y.scaled("paged_decoder_layer", weights[i], scales[i], group);
      if (y.n[i] % 128) return at::Tensor();
    }
    auto out = y.out[0].view({M, -1, 128});
    check_pool(out, kpool, vpool, "paged_decoder_layer");
    TORCH_CHECK(y.n[1] == kpool.size(1) * 128 && y.n[2] == y.n[1],
                "paged_decoder_layer: heads");
    const Turn turn(M, dst, cos_table, sin_table, positions, S);
    const int e = ds_rows_append(
        h.data_ptr(), y.w, i8 ? y.sc : nullptr, y.b, y.o[0], y.n, (int)M,
        (int)H, (int)group, kpool.data_ptr(), vpool.data_ptr(),
        dst.data_ptr<int>(), turn.cs, turn.sn, turn.pos, (int)S,
        (int)kpool.size(2), cur_stream());
    if (e < 0) return at::Tensor();
    TORCH_CHECK(e == 0, "paged_decoder_layer: launch failed with error ", e);
    return out;
  };
  auto q = few_append();
  std::vector<at::Tensor> qkv;
  at::Tensor qkv_part;
  if (!q.defined()) {
    std::tie(qkv, qkv_part) = sums(h, 0, 3);
    for (auto& t : qkv) t = t.view({M, -1, 128});
    check_pool(qkv[0], kpool, vpool, "paged_decoder_layer");
    TORCH_CHECK(qkv[1].size(1) == kpool.size(1) &&
                qkv[2].size(1) == kpool.size(1), "paged_decoder_layer: heads");
  }
  if (q.defined()) {
  } else if (qkv_part.defined()) {
    const void* b[3];
    for (int i = 0; i < 3; ++i)
      b[i] = biases[i].has_value() ? biases[i]->data_ptr() : nullptr;
    q = append_rows(qkv[0], b[1], b[2], b[0], qkv_part.data_ptr<float>(),
                    (int)qkv_part.size(0), kpool, vpool, dst, cos_table,
                    sin_table, positions, S, qkv[0]);
  } else {
    q = paged_append(qkv[0], qkv[1], qkv[2], kpool, vpool, dst, cos_table,
                     sin_table, positions, S);
  }
  auto o = paged_rows(q, kpool, vpool, meta, n_items, n_runs, n_merges,
                      any_merge, nq, scale);
  // the norm of sums in parts takes no bias
  auto output = [&](const at::Tensor& in, int i, bool in_parts) {
    if (!in_parts || biases[i].has_value()) return linears(in, i, 1, 0)[0];
    auto [y, part] = sums(in, i, 1);
    return part.defined() ? part : y[0];
  };
  add_norm(output(o.view({M, -1}), 3, true), norms[1], eps1);
  h = output(linears(h, 4, 2, 1)[0], 6, parts);
  return {stream.view(x.sizes()),
          h.scalar_type() == at::kFloat ? h : h.view(x.sizes())};
}

// What paged_decoder_layer asks of a layer's tensors, H wide, with kv features of
// keys; int8 weights have scales, and are as large as their modules say. Looked at
// one by one in Python, with their modules, they took 36 us of a layer's host time;
// the modules alone take 15.
bool paged_layer_fits(const std::vector<at::Tensor>& norms,
                      const std::vector<at::Tensor>& weights,
                      const std::vector<at::Tensor>& scales,
                      const std::vector<c10::optional<at::Tensor>>& biases,
                      int64_t H, int64_t kv) {
  auto plain = [](const at::Tensor& t) {
    return t.scalar_type() == at::kBFloat16 && t.is_contiguous();
  };
  if (weights.size() != 7 || biases.size() != 7 || H < 256 || H % 256)
    return false;
  for (auto& w : norms)
    if (!plain(w)) return false;
  const int64_t F = weights[4].numel() / H;
  const int64_t N[] = {H, kv, kv, H, F, F, H};
  for (int i = 0; i < 7; ++i) {
    const auto& w = weights[i];
    const int64_t K = i == 6 ? F : H;
    if (K % 256 || N[i] % 4 || !N[i] || w.numel() != N[i] * K ||
        !w.is_contiguous() || (uintptr_t)w.data_ptr() % 16 ||
        (scales.empty() && (!plain(w) || w.dim() != 2 || w.size(1) != K)) ||
        (biases[i].has_value() && !plain(*biases[i])))
      return false;
  }
  return true;
}

// Gradient [V, H] of an embedding's table for tokens ids [T] with the gradients
// grad [T, H] bf16; rows of `padding` (-1: none) get nothing. `into` is zero.
at::Tensor embedding_bwd(at::Tensor ids, at::Tensor grad, int64_t V,
                         int64_t padding, c10::optional<at::Tensor> into) {
  const OneDevice on("embedding_bwd", grad, ids, into);
  const int64_t T = ids.numel(), H = grad.size(-1);
  TORCH_CHECK(ids.scalar_type() == at::kLong && ids.is_contiguous() &&
              grad.is_cuda() && grad.is_contiguous() && grad.dim() == 2 &&
              grad.scalar_type() == at::kBFloat16 && grad.size(0) == T &&
              T > 0 && T <= 32768 && H > 0 && H % 8 == 0 && H <= (1 << 20) &&
              V > 0 && V < (1 << 30) &&
              ((uintptr_t)grad.data_ptr() & 15) == 0, "embedding_bwd");
  TORCH_CHECK(!into || (into->is_contiguous() && into->dim() == 2 &&
                        into->scalar_type() == at::kBFloat16 &&
                        into->size(0) == V && into->size(1) == H &&
                        ((uintptr_t)into->data_ptr() & 15) == 0),
              "embedding_bwd: into");
  auto out = into ? *into : at::zeros({V, H}, grad.options());
  const int64_t blk = ds_embedding_block(), blocks = (T + blk - 1) / blk;
  auto i32 = grad.options().dtype(at::kInt);
  auto places = at::empty({2 * T}, i32), spans = at::empty({V * blocks}, i32);
  auto has = at::zeros({V * ((blocks + 31) / 32)}, i32);
  ds_embedding_bwd((const long long*)ids.data_ptr<int64_t>(),
                   grad.data_ptr(), places.data_ptr<int>(),
                   places.data_ptr<int>() + T, (unsigned*)has.data_ptr<int>(),
                   spans.data_ptr<int>(), out.data_ptr(), (int)T, (int)V,
                   (int)H, padding, cur_stream());
  return out;
}

// Cross-entropy of bf16 logits [N, V] with labels [N]: (sum of the rows, labels
// other than ignore_index, mean over these, lse [N]).
std::tuple<at::Tensor, at::Tensor, at::Tensor, at::Tensor> ce_loss(
    at::Tensor logits, at::Tensor labels, int64_t ignore_index) {
  const OneDevice on("ce_loss", logits, labels);
  TORCH_CHECK(logits.is_cuda() && logits.is_contiguous() &&
              logits.dim() == 2 && logits.scalar_type() == at::kBFloat16 &&
              labels.scalar_type() == at::kLong && labels.is_contiguous() &&
              labels.numel() == logits.size(0) &&
              logits.size(0) < (1ll << 31), "ce_loss args");
  const int N = logits.size(0);
  auto f32 = logits.options().dtype(at::kFloat);
  auto loss = at::empty({N}, f32), lse = at::empty({N}, f32);
  // apart: the caller may change one in place
  auto sum = at::empty({}, f32), count = at::empty({}, f32),
       mean = at::empty({}, f32);
  const long long* y = (const long long*)labels.data_ptr<int64_t>();
  ds_ce_fwd(logits.data_ptr(), y, loss.data_ptr<float>(),
            lse.data_ptr<float>(), N, logits.size(1), ignore_index,
            cur_stream());
  ds_ce_total(loss.data_ptr<float>(), y, sum.data_ptr<float>(),
              count.data_ptr<float>(), mean.data_ptr<float>(), N,
              ignore_index, cur_stream());
  return {sum, count, mean, lse};
}

// gscale: [N], or one for all rows; of the mean over `count` labels, if given.
at::Tensor ce_bwd(at::Tensor logits, at::Tensor labels, at::Tensor lse,
                  at::Tensor gscale, int64_t ignore_index,
                  c10::optional<at::Tensor> count) {
  const OneDevice on("ce_bwd", logits, labels, lse, gscale, count);
  const int64_t N = logits.size(0);
  TORCH_CHECK(logits.is_cuda() && logits.is_contiguous() &&
              logits.dim() == 2 && logits.scalar_type() == at::kBFloat16 &&
              labels.scalar_type() == at::kLong && labels.is_contiguous() &&
              labels.numel() == N && lse.is_contiguous() &&
              lse.scalar_type() == at::kFloat && lse.numel() == N &&
              gscale.is_contiguous() && gscale.scalar_type() == at::kFloat &&
              (gscale.numel() == N || gscale.numel() == 1) &&
              (!count || (count->scalar_type() == at::kFloat &&
                          count->numel() == 1)), "ce_bwd args");
  auto d = at::empty_like(logits);
  ds_ce_bwd(logits.data_ptr(), (const long long*)labels.data_ptr<int64_t>(),
            lse.data_ptr<float>(), gscale.data_ptr<float>(),
            gscale.numel() == 1 ? 0 : 1,
            count ? count->data_ptr<float>() : nullptr, d.data_ptr(), (int)N,
            logits.size(1), ignore_index, cur_stream());
  return d;
}

at::Tensor token_gather(at::Tensor x, at::Tensor idx) {
  TORCH_CHECK(x.dim() == 3 && x.is_cuda() && x.is_contiguous(),
              "token_gather: contiguous [B,S,D] GPU tensor");
  TORCH_CHECK(idx.dim() == 2 && idx.scalar_type() == at::kInt &&
              idx.is_contiguous() && idx.size(0) == x.size(0),
              "token_gather: int32 [B,K] indices");
  const int64_t D = x.size(2);
  const int64_t vec = 16 / x.element_size();
  TORCH_CHECK(D % vec == 0, "token_gather: D % ", vec, " == 0");
  auto y = at::empty({x.size(0), idx.size(1), D}, x.options());
  ds_token_move(x.data_ptr(), y.data_ptr(), idx.data_ptr<int>(),
                (int)x.size(0), (int)x.size(1), (int)idx.size(1), (int)D,
                1, dtype_code(x), cur_stream());
  return y;
}

at::Tensor token_scatter(at::Tensor base, at::Tensor sub, at::Tensor idx) {
  TORCH_CHECK(base.dim() == 3 && sub.dim() == 3 && base.is_cuda() &&
              base.is_contiguous() && sub.is_contiguous() &&
              base.scalar_type() == sub.scalar_type(),
              "token_scatter: contiguous [B,S,D]/[B,K,D] GPU tensors");
  TORCH_CHECK(idx.dim() == 2 && idx.scalar_type() == at::kInt &&
              idx.is_contiguous() && idx.size(1) == sub.size(1),
              "token_scatter: int32 [B,K] indices");
  const int64_t D = base.size(2);
  const int64_t vec = 16 / base.element_size();
  TORCH_CHECK(D % vec == 0, "token_scatter: D % ", vec, " == 0");
  auto y = base.clone();
  ds_token_move(sub.data_ptr(), y.data_ptr(), idx.data_ptr<int>(),
                (int)base.size(0), (int)base.size(1), (int)sub.size(1),
                (int)D, 0, dtype_code(base), cur_stream());
  return y;
}

at::Tensor nhwc_bias_add(at::Tensor act, at::Tensor bias,
                         c10::optional<at::Tensor> other,
                         c10::optional<at::Tensor> other_bias) {
  TORCH_CHECK(act.is_cuda() && act.is_contiguous() && bias.is_contiguous(),
              "nhwc_bias_add: contiguous GPU tensors");
  TORCH_CHECK(act.scalar_type() == at::kBFloat16 ||
              act.scalar_type() == at::kHalf, "nhwc_bias_add: bf16/fp16");
  const int64_t C = bias.numel();
  TORCH_CHECK(C % 8 == 0 && act.numel() % C == 0,
              "nhwc_bias_add: channels % 8 == 0, act a multiple of channels");
  const void* other_p = nullptr;
  const void* ob_p = nullptr;
  if (other.has_value() && other->defined()) {
    TORCH_CHECK(other->is_contiguous() && other->numel() == act.numel() &&
                other->scalar_type() == act.scalar_type(),
                "nhwc_bias_add: other mismatched");
    other_p = other->data_ptr();
  }
  if (other_bias.has_value() && other_bias->defined()) {
    TORCH_CHECK(other_bias->is_contiguous() && other_bias->numel() == C &&
                other_bias->scalar_type() == act.scalar_type(),
                "nhwc_bias_add: other_bias mismatched");
    ob_p = other_bias->data_ptr();
  }
  auto out = at::empty_like(act);
  ds_nhwc_bias_add(act.data_ptr(), bias.data_ptr(), other_p, ob_p,
                   out.data_ptr(), act.numel(), (int)C, dtype_code(act),
                   cur_stream());
  return out;
}

// Rotates x [B, S, H, D] (and x2, of other heads) into new tensors, or in
// place.
std::vector<at::Tensor> rope(at::Tensor x, c10::optional<at::Tensor> x2,
                             at::Tensor cos_table, at::Tensor sin_table,
                             c10::optional<at::Tensor> positions,
                             bool backward, bool inplace) {
  const OneDevice on("rope", x, x2, cos_table, sin_table, positions);
  TORCH_CHECK(x.dim() == 4 && x.is_contiguous() && x.is_cuda(),
              "rope expects [B,S,H,D]");
  for (auto& t : {cos_table, sin_table})
    TORCH_CHECK(t.scalar_type() == at::kFloat && t.is_contiguous() &&
                t.is_cuda(), "tables must be fp32");
  const int64_t B = x.size(0), S = x.size(1), D = x.size(3);
  TORCH_CHECK(cos_table.size(-1) == D / 2, "table dim mismatch");
  TORCH_CHECK(cos_table.size(0) >= S || positions.has_value(),
              "cos table shorter than sequence");
  const int* pos_ptr = nullptr;
  if (positions.has_value() && positions->defined()) {
    TORCH_CHECK(positions->scalar_type() == at::kInt &&
                positions->is_contiguous() && positions->numel() == B * S,
                "positions must be int32 [B,S]");
    pos_ptr = positions->data_ptr<int>();
  }
  std::vector<at::Tensor> in = {x}, out;
  if (x2.has_value()) {
    TORCH_CHECK(x2->dim() == 4 && x2->is_contiguous() && x2->is_cuda() &&
                x2->size(0) == B && x2->size(1) == S && x2->size(3) == D &&
                x2->scalar_type() == x.scalar_type(), "rope: second tensor");
    in.push_back(*x2);
  }
  for (auto& t : in) out.push_back(inplace ? t : at::empty_like(t));
  const bool two = in.size() == 2;
  ds_rope(in[0].data_ptr(), out[0].data_ptr(), (int)x.size(2),
          two ? in[1].data_ptr() : nullptr, two ? out[1].data_ptr() : nullptr,
          two ? (int)in[1].size(2) : 0, cos_table.data_ptr<float>(),
          sin_table.data_ptr<float>(), pos_ptr, B, S, D, backward ? 1 : 0,
          dtype_code(x), cur_stream());
  return out;
}

at::Tensor gated_act_fwd(at::Tensor gate, at::Tensor up, int64_t act) {
  const OneDevice on("gated_act_fwd", gate, up);
  TORCH_CHECK(gate.is_contiguous() && up.is_contiguous() &&
              gate.sizes() == up.sizes(), "shape mismatch");
  TORCH_CHECK(gate.scalar_type() == up.scalar_type(), "gated_act_fwd: types");
  auto out = at::empty_like(gate);
  ds_gated_act_fwd(gate.data_ptr(), up.data_ptr(), out.data_ptr(),
                   gate.numel(), (int)act, dtype_code(gate), cur_stream());
  return out;
}

std::tuple<at::Tensor, at::Tensor> gated_act_bwd(at::Tensor dout,
                                                 at::Tensor gate,
                                                 at::Tensor up, int64_t act) {
  const OneDevice on("gated_act_bwd", gate, dout, up);
  TORCH_CHECK(dout.is_contiguous() && gate.is_contiguous() &&
              up.is_contiguous(), "must be contiguous");
  TORCH_CHECK(gate.scalar_type() == up.scalar_type() &&
              gate.scalar_type() == dout.scalar_type() &&
              gate.numel() == up.numel() && gate.numel() == dout.numel(),
              "gated_act_bwd: types or sizes");
  auto dgate = at::empty_like(gate);
  auto dup = at::empty_like(up);
  ds_gated_act_bwd(dout.data_ptr(), gate.data_ptr(), up.data_ptr(),
                   dgate.data_ptr(), dup.data_ptr(), dout.numel(), (int)act,
                   dtype_code(gate), cur_stream());
  return {dgate, dup};
}

std::tuple<at::Tensor, at::Tensor> groupwise_quant(at::Tensor x,
                                                   int64_t group_size,
                                                   int64_t bits) {
  TORCH_CHECK(x.is_contiguous() && x.is_cuda(), "x must be contiguous GPU");
  TORCH_CHECK(bits == 8 || bits == 4, "bits must be 4 or 8");
  TORCH_CHECK(group_size % 2 == 0, "group_size must be even");
  const long long n = x.numel();
  const long long groups = (n + group_size - 1) / group_size;
  const long long qbytes = bits == 8 ? n : (n + 1) / 2;
  auto q = at::empty({qbytes}, x.options().dtype(at::kChar));
  auto scales = at::empty({groups}, x.options().dtype(at::kFloat));
  ds_groupwise_quant(x.data_ptr(), dtype_code(x), q.data_ptr(),
                     scales.data_ptr<float>(), n, (int)group_size, (int)bits,
                     cur_stream());
  return {q, scales};
}

at::Tensor groupwise_dequant(at::Tensor q, at::Tensor scales, int64_t numel,
                             int64_t group_size, int64_t bits,
                             at::ScalarType dtype) {
  TORCH_CHECK(q.is_contiguous() && q.is_cuda() && scales.is_contiguous(),
              "q/scales must be contiguous GPU");
  auto out = at::empty({numel}, q.options().dtype(dtype));
  ds_groupwise_dequant(q.data_ptr(), scales.data_ptr<float>(), out.data_ptr(),
                       dtype_code(out), numel, (int)group_size, (int)bits,
                       cur_stream());
  return out;
}

// q, o, do [B, S, H, D], k, v [B, S, Hkv, D] with any strides between tokens
// and heads that keep 16-byte rows: (batch, token, head) strides, in order.
struct FlashArgs {
  int B, S, H, Hkv, D;
  std::vector<long long> strides;
  FlashArgs(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v,
            double scale) {
    TORCH_CHECK(q.dim() == 4 && k.dim() == 4 && k.sizes() == v.sizes() &&
                q.size(0) == k.size(0) && q.size(1) == k.size(1) &&
                q.size(3) == k.size(3), "flash: q [B,S,H,D], k/v [B,S,Hkv,D]");
    B = q.size(0); S = q.size(1); H = q.size(2); D = q.size(3);
    Hkv = k.size(2);
    TORCH_CHECK(D == 64 || D == 96 || D == 128, "flash: D of 64, 96 or 128");
    TORCH_CHECK(Hkv > 0 && H % Hkv == 0, "flash: H a multiple of Hkv");
    TORCH_CHECK(scale > 0, "flash: scale must be positive");
    TORCH_CHECK(q.size(1) < (1 << 30) && q.size(0) * (int64_t)H *
                ((S + 127) / 128) < (1ll << 31), "flash: size");
  }
  void add(const at::Tensor& t, const at::Tensor& like) {
    TORCH_CHECK(t.is_cuda() && t.scalar_type() == at::kBFloat16 &&
                t.sizes() == like.sizes() && t.stride(3) == 1 &&
                ((uintptr_t)t.data_ptr() & 15) == 0 &&
                t.stride(0) % 8 == 0 && t.stride(1) % 8 == 0 &&
                t.stride(2) % 8 == 0 && t.stride(1) >= 0 &&
                t.stride(1) < (1 << 24), "flash: bf16 GPU, 16-byte rows");
    for (int d = 0; d < 3; ++d) strides.push_back(t.stride(d));
  }
};

std::tuple<at::Tensor, at::Tensor> flash_attn_fwd(
    at::Tensor q, at::Tensor k, at::Tensor v, double scale, bool causal,
    bool with_lse) {
  const OneDevice on("flash_attn_fwd", q, k, v);
  FlashArgs a(q, k, v, scale);
  auto o = at::empty({a.B, a.S, a.H, a.D}, q.options());
  auto lse = at::empty({with_lse ? a.B : 0, a.H, a.S},
                       q.options().dtype(at::kFloat));
  a.add(q, q); a.add(k, k); a.add(v, k); a.add(o, q);
  if (q.numel())
    ds_flash_fwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(),
                 with_lse ? lse.data_ptr<float>() : nullptr, a.strides.data(),
                 a.B, a.S, a.H, a.Hkv, a.D, (float)scale, causal ? 1 : 0,
                 cur_stream());
  return {o, lse};
}

std::tuple<at::Tensor, at::Tensor, at::Tensor> flash_attn_bwd(
    at::Tensor q, at::Tensor k, at::Tensor v, at::Tensor o, at::Tensor dout,
    at::Tensor lse, double scale, bool causal, int64_t splits) {
  const OneDevice on("flash_attn_bwd", q, k, v, o, dout, lse);
  FlashArgs a(q, k, v, scale);
  if (splits == 0) splits = ds_flash_bwd_splits(a.B, a.S, a.H, a.Hkv);
  TORCH_CHECK(splits >= 1 && splits <= a.H / a.Hkv, "flash_bwd: splits");
  TORCH_CHECK(lse.is_cuda() && lse.scalar_type() == at::kFloat &&
              lse.is_contiguous() &&
              lse.numel() == (int64_t)a.B * a.H * a.S, "flash_bwd: lse");
  auto dq = at::empty({a.B, a.S, a.H, a.D}, q.options());
  auto dk = at::empty({a.B, a.S, a.Hkv, a.D}, q.options());
  auto dv = at::empty({a.B, a.S, a.Hkv, a.D}, q.options());
  auto stat = at::empty({2, lse.numel()}, lse.options());
  auto part = at::empty({splits > 1 ? 2 * splits * dk.numel() : 0},
                        lse.options());
  a.add(q, q); a.add(k, k); a.add(v, k); a.add(o, q); a.add(dout, q);
  a.add(dq, q); a.add(dk, k); a.add(dv, k);
  if (q.numel())
    ds_flash_bwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(),
                 dout.data_ptr(), lse.data_ptr<float>(),
                 stat.data_ptr<float>(), part.data_ptr<float>(), (int)splits,
                 dq.data_ptr(), dk.data_ptr(), dv.data_ptr(),
                 a.strides.data(), a.B, a.S, a.H, a.Hkv, a.D, (float)scale,
                 causal ? 1 : 0, cur_stream());
  return {dq, dk, dv};
}

class AioHandle {
 public:
  AioHandle(int64_t block_size, int n_threads)
      : h_(ds_aio_create(block_size, n_threads)) {}
  ~AioHandle() { ds_aio_destroy(h_); }
  void async_pwrite(at::Tensor t, const std::string& path) {
    TORCH_CHECK(!t.is_cuda() && t.is_contiguous(),
                "aio: host contiguous tensors only");
    keep_.push_back(t);  // hold storage until wait()
    TORCH_CHECK(ds_aio_pwrite(h_, t.data_ptr(),
                              t.numel() * t.element_size(),
                              path.c_str()) == 0, "aio pwrite setup failed");
  }
  void async_pread(at::Tensor t, const std::string& path) {
    TORCH_CHECK(!t.is_cuda() && t.is_contiguous(),
                "aio: host contiguous tensors only");
    keep_.push_back(t);
    TORCH_CHECK(ds_aio_pread(h_, t.data_ptr(),
                             t.numel() * t.element_size(),
                             path.c_str()) == 0, "aio pread setup failed");
  }
  int wait() {
    int e;
    {
      pybind11::gil_scoped_release nogil;
      e = ds_aio_wait(h_);
    }
    keep_.clear();
    return e;
  }

 private:
  void* h_;
  std::vector<at::Tensor> keep_;
};

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  pybind11::class_<ShmComm>(m, "ShmComm")
      .def(pybind11::init<const std::string&, int64_t, int64_t, int64_t>())
      .def("all_reduce", &ShmComm::all_reduce);
  m.def("paged_decode", &paged_decode,
        "split-KV decode attention over a paged KV block table");
  m.def("rows_linear", &rows_linear,
        "linear layers of a few rows, bf16 or groupwise int8 weights");
  m.def("tile_linear", &tile_linear, "linear layers of many rows, bf16",
        py::arg("x"), py::arg("weights"), py::arg("biases"), py::arg("mode"),
        py::arg("tile") = -1, py::arg("splits") = 1);
  m.def("tile_linear_plan", &tile_linear_plan,
        "tile and splits of layers of ns features", pybind11::arg("ns"),
        pybind11::arg("rows"), pybind11::arg("inputs"), pybind11::arg("mode"));
  m.def("tile_linear_dx", &tile_linear_dx,
        "input's gradient, summed over linear layers", py::arg("dys"),
        py::arg("weights"), py::arg("tile") = -1, py::arg("splits") = 1);
  m.def("tile_linear_dw", &tile_linear_dw, "weights' gradients",
        py::arg("x"), py::arg("dys"), py::arg("tile") = -1,
        py::arg("splits") = 1,
        py::arg("into") = std::vector<c10::optional<at::Tensor>>());
  m.def("sum_of_squares", &sum_of_squares,
        "sum of squares over a list of tensors");
  m.def("paged_rows", &paged_rows,
        "attention of a serving step's runs of tokens over the paged pool");
  m.def("paged_append", &paged_append,
        "rotary embedding and cache write of a serving step's new rows");
  m.def("fused_softmax", &fused_softmax,
        "fused masked/alibi/causal softmax");
  m.def("fused_dropout", &fused_dropout, "fused bias+dropout(+residual)");
  m.def("dropout_bwd", &dropout_bwd, "dropout backward from saved mask");
  m.def("transpose_2d", &transpose_2d, "bf16 matrix transpose");
  m.def("transpose_bf16", &transpose_bf16, "tiled bf16 batched transpose");
  m.def("fp_quantize", &fp_quantize, "groupwise FP4/6/8/12 quantize");
  m.def("fp_dequantize", &fp_dequantize, "groupwise FP dequantize");
  m.def("fused_lion", &fused_lion, "fused Lion step (GPU)");
  m.def("fused_lamb", &fused_lamb, "fused LAMB step (GPU, 2-phase)");
  m.def("fused_adam_flat", &fused_adam_flat,
        "Fused Adam/AdamW on flat fp32 master + 16-bit grad shard");
  m.def("cpu_adam_flat", &cpu_adam_flat,
        "Host Adam/AdamW on flat pinned fp32 master (ZeRO-Offload)");
  m.def("cpu_lion_flat",
        [](at::Tensor p, at::Tensor g, at::Tensor m,
           c10::optional<at::Tensor> p16, double lr, double beta1,
           double beta2, double weight_decay, double inv_scale) {
          TORCH_CHECK(!p.is_cuda() && p.is_contiguous() && g.is_contiguous()
                      && m.is_contiguous(), "cpu_lion: host contiguous");
          TORCH_CHECK(p.scalar_type() == at::kFloat &&
                      m.scalar_type() == at::kFloat, "p/m must be fp32");
          void* p16_ptr = nullptr;
          if (p16.has_value() && p16->defined()) p16_ptr = p16->data_ptr();
          ds_cpu_lion_flat(p.data_ptr<float>(), g.data_ptr(), dtype_code(g),
                           m.data_ptr<float>(), p16_ptr, p.numel(), (float)lr,
                           (float)beta1, (float)beta2, (float)weight_decay,
                           (float)inv_scale);
        },
        "Host Lion on flat fp32 master");
  m.def("norm_fwd", &norm_fwd, "RMSNorm/LayerNorm forward");
  m.def("norm_bwd", &norm_bwd, "RMSNorm/LayerNorm backward",
        pybind11::arg("dy"), pybind11::arg("x"), pybind11::arg("w"),
        pybind11::arg("invrms"), pybind11::arg("mean"),
        pybind11::arg("layernorm"), pybind11::arg("dres") = c10::nullopt,
        pybind11::arg("into") = c10::nullopt);
  m.def("paged_decoder_layer", &paged_decoder_layer,
        "a decoder layer of a serving step over the paged pool");
  m.def("own_forward", &own_forward, "which products paged_decoder_layer makes",
        pybind11::arg("rows"), pybind11::arg("ns"), pybind11::arg("inputs"),
        pybind11::arg("mode"));
  m.def("paged_layer_fits", &paged_layer_fits,
        "whether paged_decoder_layer takes a layer's tensors");
  m.def("step_plan", &step_plan, "plan of a serving step over the paged pool");
  m.def("add_norm_fwd", &add_norm_fwd, "RMS norm of a sum, and the sum");
  m.def("rope", &rope, "Rotary position embedding of one or two tensors",
        pybind11::arg("x"), pybind11::arg("x2"), pybind11::arg("cos"),
        pybind11::arg("sin"), pybind11::arg("positions"),
        pybind11::arg("backward"), pybind11::arg("inplace") = false);
  m.def("token_gather", &token_gather,
        "row-coalesced token gather [B,S,D] x [B,K] -> [B,K,D]");
  m.def("token_scatter", &token_scatter,
        "row-coalesced token scatter-back into a cloned base");
  m.def("nhwc_bias_add", &nhwc_bias_add,
        "fused channels-last bias (+residual +residual-bias) add",
        pybind11::arg("act"), pybind11::arg("bias"),
        pybind11::arg("other") = c10::nullopt,
        pybind11::arg("other_bias") = c10::nullopt);
  m.def("gated_act_fwd", &gated_act_fwd, "SwiGLU/GeGLU forward");
  m.def("gated_act_bwd", &gated_act_bwd, "SwiGLU/GeGLU backward");
  m.def("groupwise_quant", &groupwise_quant,
        "Groupwise symmetric int8/int4 quantization");
  m.def("groupwise_dequant", &groupwise_dequant,
        "Groupwise symmetric int8/int4 dequantization");
  m.def("ce_fwd",
        [](at::Tensor logits, at::Tensor labels, int64_t ignore_index) {
          TORCH_CHECK(logits.is_cuda() && logits.is_contiguous() &&
                      logits.scalar_type() == at::kBFloat16 &&
                      labels.scalar_type() == at::kLong, "ce_fwd args");
          const int N = logits.size(0);
          const long long V = logits.size(1);
          auto loss = at::empty({N}, logits.options().dtype(at::kFloat));
          auto lse = at::empty({N}, logits.options().dtype(at::kFloat));
          ds_ce_fwd(logits.data_ptr(), (const long long*)labels.data_ptr<int64_t>(),
                    loss.data_ptr<float>(), lse.data_ptr<float>(), N, V,
                    ignore_index, cur_stream());
          return std::make_tuple(loss, lse);
        },
        "fused CE forward: bf16 logits -> per-token loss + lse");
  m.def("embedding_bwd", &embedding_bwd, "gradient of an embedding's table",
        py::arg("ids"), py::arg("grad"), py::arg("rows"), py::arg("padding"),
        py::arg("into") = c10::nullopt);
  m.def("ce_loss", &ce_loss,
        "fused CE forward: bf16 logits -> sum, labels, mean, lse");
  m.def("ce_bwd", &ce_bwd, "fused CE backward: dlogits in bf16",
        py::arg("logits"), py::arg("labels"), py::arg("lse"),
        py::arg("gscale"), py::arg("ignore_index"),
        py::arg("count") = c10::nullopt);
  m.def("flash_attn_fwd", &flash_attn_fwd,
        "flash attention forward (bf16, MFMA): (o, logsumexp)");
  m.def("flash_attn_bwd", &flash_attn_bwd,
        "flash attention backward (bf16, MFMA): (dq, dk, dv)",
        pybind11::arg("q"), pybind11::arg("k"), pybind11::arg("v"),
        pybind11::arg("o"), pybind11::arg("dout"), pybind11::arg("lse"),
        pybind11::arg("scale"), pybind11::arg("causal"),
        pybind11::arg("splits") = 0);
  pybind11::class_<AioHandle>(m, "AioHandle")
      .def(pybind11::init<int64_t, int>(),
           pybind11::arg("block_size") = 1 << 20,
           pybind11::arg("n_threads") = 8)
      .def("async_pwrite", &AioHandle::async_pwrite)
      .def("async_pread", &AioHandle::async_pread)
      .def("wait", &AioHandle::wait);
}
