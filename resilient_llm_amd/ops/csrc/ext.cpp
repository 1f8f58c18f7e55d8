// Torch bindings for the gfx950 kernels (TORCH_LIBRARY, not pybind — the
// ops dispatch through torch.ops.rlli.* and stay graph-capturable).
// This is the only translation unit that includes torch headers; the
// kernels live in pure-HIP .hip files behind kernels.h.

#include <torch/library.h>
#include <ATen/ATen.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <ATen/hip/impl/HIPGuardImplMasqueradingAsCUDA.h>
#include <c10/hip/HIPGraphsC10Utils.h>

#include "kernels.h"

#include <algorithm>
#include <cstdlib>
#include <vector>

namespace {

using at::Tensor;

hipStream_t current_stream(const Tensor& t) {
  return at::hip::getCurrentHIPStreamMasqueradingAsCUDA(
      t.device().index()).stream();
}

// after-launch error check (skipped inside hipGraph capture, where the
// runtime reports capture-sequencing pseudo-errors)
void check_launch(const char* op) {
  if (c10::hip::currentStreamCaptureStatusMayInitCtx() !=
      c10::hip::CaptureStatus::None)
    return;
  hipError_t e = hipGetLastError();
  TORCH_CHECK(e == hipSuccess, op, " launch failed: ", hipGetErrorString(e));
}

uint16_t* bf16_ptr(const Tensor& t) {
  return reinterpret_cast<uint16_t*>(t.data_ptr());
}

void check_bf16_contig(const Tensor& t, const char* name) {
  TORCH_CHECK(t.scalar_type() == at::kBFloat16, name, " must be bf16");
  TORCH_CHECK(t.is_contiguous(), name, " must be contiguous");
  TORCH_CHECK(t.is_cuda(), name, " must be on the GPU");
}


// ``t`` from a multiple of 16 bytes on, copied if it is elsewhere: what direct
// global -> LDS loads of 16 bytes are made for
Tensor aligned(const Tensor& t) {
  return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 ? t.clone() : t;
}

// cache tensors: bf16 or fp8-e4m3 (common.h codecs); returns the fp8
// flag after validating dtype/contiguity/device
bool check_cache(const Tensor& k_cache, const Tensor& v_cache) {
  TORCH_CHECK(k_cache.scalar_type() == v_cache.scalar_type(),
              "k/v cache dtype mismatch");
  const bool fp8 = k_cache.scalar_type() == at::kFloat8_e4m3fn;
  TORCH_CHECK(fp8 || k_cache.scalar_type() == at::kBFloat16,
              "kv cache must be bf16 or float8_e4m3fn");
  TORCH_CHECK(k_cache.is_contiguous() && v_cache.is_contiguous() &&
              k_cache.is_cuda() && v_cache.is_cuda());
  return fp8;
}

// ------------------------------------------------------------- rmsnorm
Tensor rmsnorm(const Tensor& x, const Tensor& w, double eps) {
  check_bf16_contig(x, "x");
  check_bf16_contig(w, "w");
  const int dim = int(x.size(-1));
  TORCH_CHECK(dim % 8 == 0, "dim must be a multiple of 8");
  TORCH_CHECK(w.numel() == dim, "weight/dim mismatch");
  const int rows = int(x.numel() / dim);
  Tensor y = at::empty_like(x);
  c10::hip::HIPGuardMasqueradingAsCUDA guard(x.device());
  rlli::launch_rmsnorm(bf16_ptr(x), nullptr, bf16_ptr(w), bf16_ptr(y), rows,
                       dim, float(eps), current_stream(x));
  check_launch("rmsnorm");
  return y;
}

Tensor rmsnorm_residual_(const Tensor& x, Tensor residual, const Tensor& w,
                         double eps) {
  check_bf16_contig(x, "x");
  check_bf16_contig(residual, "residual");
  check_bf16_contig(w, "w");
  TORCH_CHECK(x.sizes() == residual.sizes(), "x/residual shape mismatch");
  const int dim = int(x.size(-1));
  TORCH_CHECK(dim % 8 == 0 && w.numel() == dim, "bad dim/weight");
  const int rows = int(x.numel() / dim);
  Tensor y = at::empty_like(x);
  c10::hip::HIPGuardMasqueradingAsCUDA guard(x.device());
  rlli::launch_rmsnorm(bf16_ptr(x), bf16_ptr(residual), bf16_ptr(w),
                       bf16_ptr(y), rows, dim, float(eps), current_stream(x));
  check_launch("rmsnorm_residual_");
  return y;
}

// ---- fp8-activation emitters (quantized-weight GEMM path) ----
std::tuple<Tensor, Tensor> rmsnorm_fp8(const Tensor& x, const Tensor& w,
                                       double eps) {
  check_bf16_contig(x, "x");
  check_bf16_contig(w, "w");
  const int dim = int(x.size(-1));
  TORCH_CHECK(dim % 8 == 0 && dim <= 8192 && w.numel() == dim,
              "bad dim/weight for fp8 rmsnorm");
  const int rows = int(x.numel() / dim);
  Tensor y8 = at::empty(x.sizes(), x.options().dtype(at::kFloat8_e4m3fn));
  Tensor scales = at::empty({rows}, x.options().dtype(at::kFloat));
  c10::hip::HIPGuardMasqueradingAsCUDA guard(x.device());
  rlli::launch_rmsnorm_fp8(bf16_ptr(x), nullptr, bf16_ptr(w),
                           reinterpret_cast<uint8_t*>(y8.data_ptr()),
                           scales.data_ptr<float>(), rows, dim, float(eps),
                           current_stream(x));
  check_launch("rmsnorm_fp8");
  return {y8, scales};
}

// rmsnorm_residual_ with x = the sum of f32 parts [n, rows, dim]
Tensor rmsnorm_residual_parts_(const Tensor& parts, Tensor residual,
                               const Tensor& w, double eps) {
  check_bf16_contig(residual, "residual");
  check_bf16_contig(w, "w");
  const int64_t dim = residual.size(-1);
  TORCH_CHECK(parts.scalar_type() == at::kFloat && parts.is_cuda() &&
                  parts.is_contiguous() && parts.dim() == 3 &&
                  parts.size(0) >= 1 && parts.size(2) == dim &&
                  parts.size(1) * dim == residual.numel() &&
                  w.numel() == dim,
              "parts must be contiguous f32 [n, rows, dim]");
  TORCH_CHECK(dim % 8 == 0 && dim <= 8192, "dim must be a multiple of 8, at "
              "most 8192, got ", dim);
  Tensor y = at::empty_like(residual);
  c10::hip::HIPGuardMasqueradingAsCUDA guard(residual.device());
  rlli::launch_rmsnorm_parts(parts.data_ptr<float>(), int(parts.size(0)),
                             bf16_ptr(residual), bf16_ptr(w), bf16_ptr(y),
                             int(parts.size(1)), int(dim), float(eps),
                             current_stream(residual));
  check_launch("rmsnorm_residual_parts_");
  return y;
}

std::tuple<Tensor, Tensor> rmsnorm_residual_fp8(const Tensor& x,
                                                Tensor residual,
                                                const Tensor& w, double eps) {
  check_bf16_contig(x, "x");
  check_bf16_contig(residual, "residual");
  check_bf16_contig(w, "w");
  TORCH_CHECK(x.sizes() == residual.sizes(), "x/residual shape mismatch");
  const int dim = int(x.size(-1));
  TORCH_CHECK(dim % 8 == 0 && dim <= 8192 && w.numel() == dim,
              "bad dim/weight for fp8 rmsnorm");
  const int rows = int(x.numel() / dim);
  Tensor y8 = at::empty(x.sizes(), x.options().dtype(at::kFloat8_e4m3fn));
  Tensor scales = at::empty({rows}, x.options().dtype(at::kFloat));
  c10::hip::HIPGuardMasqueradingAsCUDA guard(x.device());
  rlli::launch_rmsnorm_fp8(bf16_ptr(x), bf16_ptr(residual), bf16_ptr(w),
                           reinterpret_cast<uint8_t*>(y8.data_ptr()),
                           scales.data_ptr<float>(), rows, dim, float(eps),
                           current_stream(x));
  check_launch("rmsnorm_residual_fp8");
  return {y8, scales};
}

std::tuple<Tensor, Tensor> silu_mul_fp8(const Tensor& gate_up) {
  check_bf16_contig(gate_up, "gate_up");
  const int64_t inter = gate_up.size(-1) / 2;
  TORCH_CHECK(inter % 8 == 0, "inter must be a multiple of 8");
  const int rows = int(gate_up.numel() / (2 * inter));
  auto sizes = gate_up.sizes().vec();
  sizes.back() = inter;
  Tensor y8 = at::empty(sizes, gate_up.options().dtype(at::kFloat8_e4m3fn));
  Tensor scales = at::empty({rows}, gate_up.options().dtype(at::kFloat));
  c10::hip::HIPGuardMasqueradingAsCUDA guard(gate_up.device());
  rlli::launch_silu_mul_fp8(bf16_ptr(gate_up),
                            reinterpret_cast<uint8_t*>(y8.data_ptr()),
                            scales.data_ptr<float>(), rows, int(inter),
                            current_stream(gate_up));
  check_launch("silu_mul_fp8");
  return {y8, scales};
}

// ------------------------------------------------------------ silu_mul
Tensor silu_mul(const Tensor& gate_up) {
  check_bf16_contig(gate_up, "gate_up");
  const int twoi = int(gate_up.size(-1));
  TORCH_CHECK(twoi % 16 == 0, "2*intermediate must be a multiple of 16");
  const int inter = twoi / 2;
  const int rows = int(gate_up.numel() / twoi);
  auto sizes = gate_up.sizes().vec();
  sizes.back() = inter;
  Tensor y = at::empty(sizes, gate_up.options());
  c10::hip::HIPGuardMasqueradingAsCUDA guard(gate_up.device());
  rlli::launch_silu_mul(bf16_ptr(gate_up), bf16_ptr(y), rows, inter,
                        current_stream(gate_up));
  check_launch("silu_mul");
  return y;
}

// ------------------------------------------------------- rope_kv_append
void rope_kv_append_(Tensor q, Tensor k, const Tensor& v,
                     const Tensor& positions, const Tensor& cos_sin,
                     Tensor k_cache, Tensor v_cache,
                     const Tensor& slot_mapping) {
  check_bf16_contig(q, "q");
  check_bf16_contig(k, "k");
  check_bf16_contig(v, "v");
  const bool cache_fp8 = check_cache(k_cache, v_cache);
  TORCH_CHECK(positions.scalar_type() == at::kInt && positions.is_contiguous());
  TORCH_CHECK(slot_mapping.scalar_type() == at::kInt && slot_mapping.is_contiguous());
  TORCH_CHECK(cos_sin.scalar_type() == at::kFloat && cos_sin.is_contiguous());
  const int tokens = int(q.size(0));
  const int n_q = int(q.size(1));
  const int n_kv = int(k.size(1));
  const int D = int(q.size(2));
  TORCH_CHECK(k.size(2) == D && v.size(1) == n_kv && v.size(2) == D);
  TORCH_CHECK(D % 16 == 0, "head_dim must be a multiple of 16");
  TORCH_CHECK(cos_sin.size(1) == D, "cos_sin must be [max_pos, head_dim]");
  TORCH_CHECK(k_cache.size(1) == n_kv && k_cache.size(3) == D);
  const int block_size = int(k_cache.size(2));
  TORCH_CHECK(positions.numel() == tokens && slot_mapping.numel() == tokens);
  c10::hip::HIPGuardMasqueradingAsCUDA guard(q.device());
  rlli::launch_rope_kv_append(
      bf16_ptr(q), bf16_ptr(k), bf16_ptr(v),
      positions.data_ptr<int32_t>(), cos_sin.data_ptr<float>(),
      k_cache.data_ptr(), v_cache.data_ptr(),
      slot_mapping.data_ptr<int32_t>(),
      tokens, n_q, n_kv, D, block_size, n_q * D, n_kv * D, cache_fp8,
      current_stream(q));
  check_launch("rope_kv_append_");
}

// Fused-QKV form: qkv is the raw [T, (n_q + 2*n_kv) * D] GEMM output;
// rope + cache append run on strided views, zero copies.
void rope_kv_append_qkv_(Tensor qkv, const Tensor& positions,
                         const Tensor& cos_sin, Tensor k_cache,
                         Tensor v_cache, const Tensor& slot_mapping,
                         int64_t n_q) {
  check_bf16_contig(qkv, "qkv");
  const bool cache_fp8 = check_cache(k_cache, v_cache);
  const int n_kv = int(k_cache.size(1));
  const int D = int(k_cache.size(3));
  const int block_size = int(k_cache.size(2));
  const int stride = int(qkv.size(1));
  TORCH_CHECK(stride == (n_q + 2 * n_kv) * D, "qkv width mismatch");
  const int tokens = int(qkv.size(0));
  TORCH_CHECK(positions.numel() == tokens && slot_mapping.numel() == tokens);
  TORCH_CHECK(cos_sin.size(1) == D && D % 16 == 0);
  uint16_t* base = bf16_ptr(qkv);
  c10::hip::HIPGuardMasqueradingAsCUDA guard(qkv.device());
  rlli::launch_rope_kv_append(
      base, base + n_q * D, base + (n_q + n_kv) * D,
      positions.data_ptr<int32_t>(), cos_sin.data_ptr<float>(),
      k_cache.data_ptr(), v_cache.data_ptr(),
      slot_mapping.data_ptr<int32_t>(),
      tokens, int(n_q), n_kv, D, block_size, stride, stride, cache_fp8,
      current_stream(qkv));
  check_launch("rope_kv_append_qkv_");
}

// The same without the queries, which stay as they are.
void kv_append_qkv_(Tensor qkv, const Tensor& positions,
                    const Tensor& cos_sin, Tensor k_cache, Tensor v_cache,
                    const Tensor& slot_mapping, int64_t n_q) {
  check_bf16_contig(qkv, "qkv");
  const bool cache_fp8 = check_cache(k_cache, v_cache);
  const int n_kv = int(k_cache.size(1));
  const int D = int(k_cache.size(3));
  const int stride = int(qkv.size(1));
  const int tokens = int(qkv.size(0));
  TORCH_CHECK(stride == (n_q + 2 * n_kv) * D, "qkv width mismatch");
  TORCH_CHECK(positions.numel() == tokens && slot_mapping.numel() == tokens);
  TORCH_CHECK(cos_sin.size(1) == D && D % 16 == 0);
  uint16_t* base = bf16_ptr(qkv);
  c10::hip::HIPGuardMasqueradingAsCUDA guard(qkv.device());
  rlli::launch_rope_kv_append(
      base, base + n_q * D, base + (n_q + n_kv) * D,
      positions.data_ptr<int32_t>(), cos_sin.data_ptr<float>(),
      k_cache.data_ptr(), v_cache.data_ptr(),
      slot_mapping.data_ptr<int32_t>(), tokens, 0, n_kv, D,
      int(k_cache.size(2)), stride, stride, cache_fp8, current_stream(qkv));
  check_launch("kv_append_qkv_");
}

// ---------------------------------------------------------- decode_attn
Tensor rows_linear_parts(const Tensor& x, const Tensor& w);

// whether rows_linear takes x w^T
static bool rows_take(const Tensor& x, const Tensor& w) {
  return w.scalar_type() == at::kBFloat16 && w.is_contiguous() &&
         x.is_contiguous() && w.device() == x.device() &&
         x.size(1) % 64 == 0 && w.size(0) % 16 == 0 &&
         (reinterpret_cast<uintptr_t>(x.data_ptr()) |
          reinterpret_cast<uintptr_t>(w.data_ptr())) % 16 == 0;
}

// One launch for all forms.  q: bf16 rows that start with the query heads
// ([batch, .., stride]), or f32 parts [n, batch, stride] whose sum they are.
// With ``positions`` queries are rotated here; with ``slot_mapping`` as well
// the rows are q | k | v, and key and value are appended.
static Tensor decode_attn_any(const Tensor& q, int64_t n_q,
                              const Tensor& k_cache, const Tensor& v_cache,
                              const Tensor& block_table,
                              const Tensor& seq_lens, double scale,
                              const Tensor* positions, const Tensor* cos_sin,
                              const Tensor* slot_mapping,
                              const Tensor* into = nullptr,
                              const Tensor* w_next = nullptr) {
  const bool parts = q.scalar_type() == at::kFloat;
  if (parts) {
    TORCH_CHECK(q.is_cuda() && q.is_contiguous() && q.dim() == 3 &&
                    q.size(0) >= 1,
                "parts must be contiguous f32 [n, batch, width]");
  } else {
    check_bf16_contig(q, "q");
  }
  const bool cache_fp8 = check_cache(k_cache, v_cache);
  for (const Tensor* t : {&block_table, &seq_lens})
    TORCH_CHECK(t->scalar_type() == at::kInt && t->is_contiguous(),
                "tables and lengths must be contiguous int32");
  const int batch = int(q.size(parts ? 1 : 0));
  const int stride = batch ? int(q.numel() / batch / (parts ? q.size(0) : 1))
                           : 0;
  const int n_kv = int(k_cache.size(1));
  const int block_size = int(k_cache.size(2));
  const int D = int(k_cache.size(3));
  const int max_blocks = int(block_table.size(1));
  const int group = int(n_q) / n_kv;
  TORCH_CHECK(n_q % n_kv == 0 && (group == 1 || group == 2 || group == 4 ||
                                  group == 8),
              "GQA group must be 1/2/4/8, got ", group);
  TORCH_CHECK(D == 64 || D == 128, "head_dim must be 64 or 128, got ", D);
  TORCH_CHECK(block_size > 0 &&
              v_cache.sizes().slice(1) == k_cache.sizes().slice(1));
  // (longer ones, as a batch's buffers are, end in what nobody reads)
  TORCH_CHECK(block_table.size(0) >= batch && seq_lens.numel() >= batch,
              "tables and lengths of ", batch, " sequences are needed");
  if (into) {
    check_bf16_contig(*into, "out");
    TORCH_CHECK(into->dim() == 2 && into->size(0) >= batch &&
                    into->size(1) == n_q * D &&
                    into->device() == q.device() &&
                    reinterpret_cast<uintptr_t>(into->data_ptr()) % 16 == 0,
                "out: rows of the queries' width");
  }
  Tensor out = into ? *into
                    : at::empty({batch, n_q * D},
                                q.options().dtype(at::kBFloat16));
  if (batch == 0) return out;
  c10::hip::HIPGuardMasqueradingAsCUDA guard(q.device());
  // scratch of sequences that several workgroups share; allocated here, so
  // that a captured step keeps its own
  const int shares =
      rlli::decode_attn_shares(batch, n_kv, max_blocks * block_size);
  Tensor part, ml;
  if (shares > 0) {
    const int64_t slots = int64_t(n_kv) * (shares + batch) * group;
    auto opt = q.options().dtype(at::kFloat);
    part = at::empty({slots, D}, opt);
    ml = at::empty({slots, 2}, opt);
  }
  // of one row, the product behind it puts the shares together
  const int K = int(n_q) * D, N = w_next ? int(w_next->size(0)) : 0;
  const bool apart = w_next && shares > 0 && batch == 1 &&
                     rows_take(out, *w_next) && w_next->size(1) == K &&
                     rlli::rows_combine_ok(N, K, max_blocks * block_size);
  rlli::launch_decode_attn(
      parts ? nullptr : bf16_ptr(q), parts ? q.data_ptr<float>() : nullptr,
      parts ? int(q.size(0)) : 0, k_cache.data_ptr(), v_cache.data_ptr(),
      block_table.data_ptr<int32_t>(), seq_lens.data_ptr<int32_t>(),
      positions ? positions->data_ptr<int32_t>() : nullptr,
      cos_sin ? cos_sin->data_ptr<float>() : nullptr,
      slot_mapping ? slot_mapping->data_ptr<int32_t>() : nullptr,
      bf16_ptr(out), batch, int(n_q), n_kv, D, block_size, max_blocks,
      float(scale), stride, shares,
      shares > 0 ? part.data_ptr<float>() : nullptr,
      shares > 0 ? ml.data_ptr<float>() : nullptr, cache_fp8, apart,
      current_stream(q));
  check_launch("decode_attn");
  if (!w_next) return out;
  if (!apart)
    return rows_take(out, *w_next) ? rows_linear_parts(out, *w_next)
                                   : at::linear(out, *w_next);
  const int splits = rlli::rows_gemm_splits(N, K);
  Tensor y = at::empty({splits, 1, N}, out.options().dtype(at::kFloat));
  rlli::launch_rows_combine(
      rlli::RowsCombine{part.data_ptr<float>(), ml.data_ptr<float>(),
                        bf16_ptr(out), seq_lens.data_ptr<int32_t>(), shares,
                        group, D},
      bf16_ptr(*w_next), y.data_ptr<float>(), N, K, splits, current_stream(q));
  check_launch("rows_combine");
  return y;
}

Tensor decode_attn(const Tensor& q, const Tensor& k_cache,
                   const Tensor& v_cache, const Tensor& block_table,
                   const Tensor& seq_lens, double scale) {
  check_bf16_contig(q, "q");
  TORCH_CHECK(q.dim() == 3 && q.size(2) == k_cache.size(3) &&
              v_cache.sizes() == k_cache.sizes());
  TORCH_CHECK(block_table.size(0) == q.size(0) &&
              seq_lens.numel() == q.size(0));
  const int gpw = 64 / (int(q.size(2)) / 8);
  TORCH_CHECK(k_cache.size(2) % gpw == 0, "block_size must be a multiple of ",
              gpw);
  return decode_attn_any(q, q.size(1), k_cache, v_cache, block_table,
                         seq_lens, scale, nullptr, nullptr, nullptr)
      .view(q.sizes());
}

static void check_qkv_width(const Tensor& qkv, const Tensor& k_cache,
                            int64_t n_q) {
  TORCH_CHECK(qkv.dim() == (qkv.scalar_type() == at::kFloat ? 3 : 2) &&
                  qkv.size(-1) ==
                      (n_q + 2 * k_cache.size(1)) * k_cache.size(3),
              "qkv width mismatch");
}

// Fused-QKV decode attention: q read strided from the qkv GEMM output.
Tensor decode_attn_qkv(const Tensor& qkv, const Tensor& k_cache,
                       const Tensor& v_cache, const Tensor& block_table,
                       const Tensor& seq_lens, double scale, int64_t n_q) {
  check_bf16_contig(qkv, "qkv");
  check_qkv_width(qkv, k_cache, n_q);
  return decode_attn_any(qkv, n_q, k_cache, v_cache, block_table, seq_lens,
                         scale, nullptr, nullptr, nullptr);
}

// The same to the first rows of ``out``.
void decode_attn_qkv_out(const Tensor& qkv, const Tensor& k_cache,
                         const Tensor& v_cache, const Tensor& block_table,
                         const Tensor& seq_lens, double scale, int64_t n_q,
                         Tensor out) {
  check_bf16_contig(qkv, "qkv");
  check_qkv_width(qkv, k_cache, n_q);
  decode_attn_any(qkv, n_q, k_cache, v_cache, block_table, seq_lens, scale,
                  nullptr, nullptr, nullptr, &out);
}

static void check_rope_qkv(const Tensor& qkv, const Tensor& positions,
                           const Tensor& cos_sin, const Tensor& k_cache,
                           const Tensor& slot_mapping, int64_t n_q) {
  TORCH_CHECK(positions.scalar_type() == at::kInt && positions.is_contiguous());
  TORCH_CHECK(slot_mapping.scalar_type() == at::kInt && slot_mapping.is_contiguous());
  TORCH_CHECK(cos_sin.scalar_type() == at::kFloat && cos_sin.is_contiguous());
  TORCH_CHECK(cos_sin.size(1) == k_cache.size(3));
  check_qkv_width(qkv, k_cache, n_q);
  const int64_t batch = qkv.size(qkv.dim() == 3 ? 1 : 0);
  TORCH_CHECK(positions.numel() >= batch && slot_mapping.numel() >= batch,
              "positions and slots of ", batch, " sequences are needed");
}

// Fused decode: rope + append + attention in one kernel.  qkv: bf16 rows, or
// the f32 parts of rows_linear_parts.
Tensor decode_attn_rope_qkv(const Tensor& qkv, const Tensor& positions,
                            const Tensor& cos_sin, Tensor k_cache,
                            Tensor v_cache, const Tensor& slot_mapping,
                            const Tensor& block_table, const Tensor& seq_lens,
                            double scale, int64_t n_q) {
  check_rope_qkv(qkv, positions, cos_sin, k_cache, slot_mapping, n_q);
  return decode_attn_any(qkv, n_q, k_cache, v_cache, block_table, seq_lens,
                         scale, &positions, &cos_sin, &slot_mapping);
}

// The product with w of decode_attn_rope_qkv's result, as rows_linear_parts has
// it.
Tensor decode_attn_rope_linear(const Tensor& qkv, const Tensor& positions,
                               const Tensor& cos_sin, Tensor k_cache,
                               Tensor v_cache, const Tensor& slot_mapping,
                               const Tensor& block_table,
                               const Tensor& seq_lens, double scale,
                               int64_t n_q, const Tensor& w) {
  check_rope_qkv(qkv, positions, cos_sin, k_cache, slot_mapping, n_q);
  return decode_attn_any(qkv, n_q, k_cache, v_cache, block_table, seq_lens,
                         scale, &positions, &cos_sin, &slot_mapping, nullptr,
                         &w);
}

// Queries rotated here, everything they see already in the cache.
Tensor decode_attn_q_rope(const Tensor& qkv, const Tensor& positions,
                          const Tensor& cos_sin, const Tensor& k_cache,
                          const Tensor& v_cache, const Tensor& block_table,
                          const Tensor& seq_lens, double scale, int64_t n_q) {
  check_bf16_contig(qkv, "qkv");
  TORCH_CHECK(positions.scalar_type() == at::kInt && positions.is_contiguous());
  TORCH_CHECK(cos_sin.scalar_type() == at::kFloat && cos_sin.is_contiguous());
  TORCH_CHECK(cos_sin.size(1) == k_cache.size(3) &&
              positions.numel() == qkv.size(0));
  check_qkv_width(qkv, k_cache, n_q);
  return decode_attn_any(qkv, n_q, k_cache, v_cache, block_table, seq_lens,
                         scale, &positions, &cos_sin, nullptr);
}

// Block table [rows, width] and length [rows] of every row of a mixed step;
// tables and lengths of the decoding sequences may be absent if there are none.
std::tuple<Tensor, Tensor> mixed_row_tables(
    int64_t rows, int64_t n_decode, const c10::optional<Tensor>& tables_dec,
    const c10::optional<Tensor>& lens_dec, const Tensor& row0,
    const Tensor& pos0, const Tensor& nrows, const Tensor& btrow,
    const Tensor& tables_pre) {
  auto check = [&](const Tensor& t) {
    TORCH_CHECK(t.scalar_type() == at::kInt && t.is_contiguous() &&
                t.device() == tables_pre.device(),
                "tables, lengths and tiles must be contiguous int32 on one "
                "GPU");
  };
  rlli::RowTables a{};
  for (const Tensor* t : {&row0, &pos0, &nrows, &btrow, &tables_pre})
    check(*t);
  a.n_tiles = int(row0.numel());
  TORCH_CHECK(tables_pre.dim() == 2 && pos0.numel() == a.n_tiles &&
              nrows.numel() == a.n_tiles && btrow.numel() == a.n_tiles);
  TORCH_CHECK(n_decode >= 0 && n_decode <= rows);
  a.n_decode = int(n_decode);
  a.pre_width = int(tables_pre.size(1));
  if (n_decode > 0) {
    TORCH_CHECK(tables_dec && lens_dec);
    check(*tables_dec);
    check(*lens_dec);
    TORCH_CHECK(tables_dec->dim() == 2 && tables_dec->size(0) >= n_decode &&
                lens_dec->numel() >= n_decode);
    a.tables_dec = tables_dec->data_ptr<int32_t>();
    a.lens_dec = lens_dec->data_ptr<int32_t>();
    a.dec_width = int(tables_dec->size(1));
  }
  a.row0 = row0.data_ptr<int32_t>();
  a.pos0 = pos0.data_ptr<int32_t>();
  a.nrows = nrows.data_ptr<int32_t>();
  a.btrow = btrow.data_ptr<int32_t>();
  a.tables_pre = tables_pre.data_ptr<int32_t>();
  const int wide = std::max(a.pre_width, a.dec_width);
  c10::hip::HIPGuardMasqueradingAsCUDA guard(tables_pre.device());
  Tensor tables = at::empty({rows, wide}, tables_pre.options());
  Tensor lens = at::empty({rows}, tables_pre.options());
  rlli::launch_row_tables(a, tables.data_ptr<int32_t>(),
                          lens.data_ptr<int32_t>(), int(rows), wide,
                          current_stream(tables_pre));
  check_launch("mixed_row_tables");
  return {tables, lens};
}

// --------------------------------------------------------- prefill_attn
Tensor prefill_attn(const Tensor& q, const Tensor& k, const Tensor& v,
                    const Tensor& cu_seqlens, double scale) {
  check_bf16_contig(q, "q");
  check_bf16_contig(k, "k");
  check_bf16_contig(v, "v");
  TORCH_CHECK(cu_seqlens.scalar_type() == at::kInt && cu_seqlens.is_contiguous());
  const int T = int(q.size(0));
  const int n_q = int(q.size(1));
  const int D = int(q.size(2));
  const int n_kv = int(k.size(1));
  const int group = n_q / n_kv;
  TORCH_CHECK(n_q % n_kv == 0 && (group == 1 || group == 2 || group == 4 || group == 8),
              "GQA group must be 1/2/4/8, got ", group);
  TORCH_CHECK(D == 64 || D == 128, "head_dim must be 64 or 128, got ", D);
  TORCH_CHECK(k.size(0) == T && v.size(0) == T && k.size(2) == D);
  const int n_seqs = int(cu_seqlens.numel()) - 1;
  Tensor out = at::empty_like(q);
  c10::hip::HIPGuardMasqueradingAsCUDA guard(q.device());
  rlli::launch_prefill_attn(
      bf16_ptr(q), bf16_ptr(k), bf16_ptr(v), cu_seqlens.data_ptr<int32_t>(),
      bf16_ptr(out), n_seqs, T, n_q, n_kv, D, float(scale),
      n_q * D, n_kv * D, current_stream(q));
  check_launch("prefill_attn");
  return out;
}

// Fused-QKV prefill attention: q/k/v all read strided from qkv (k was
// rope-rotated in place by rope_kv_append_qkv_).
Tensor prefill_attn_qkv(const Tensor& qkv, const Tensor& cu_seqlens,
                        double scale, int64_t n_q, int64_t n_kv,
                        int64_t head_dim) {
  check_bf16_contig(qkv, "qkv");
  TORCH_CHECK(cu_seqlens.scalar_type() == at::kInt &&
              cu_seqlens.is_contiguous());
  const int T = int(qkv.size(0));
  const int D = int(head_dim);
  const int stride = int(qkv.size(1));
  TORCH_CHECK(stride == (n_q + 2 * n_kv) * D, "qkv width mismatch");
  const int group = int(n_q) / int(n_kv);
  TORCH_CHECK(group == 1 || group == 2 || group == 4 || group == 8);
  TORCH_CHECK(D == 64 || D == 128);
  const int n_seqs = int(cu_seqlens.numel()) - 1;
  TORCH_CHECK(T == 0 || n_seqs >= 1, "rows without a sequence: cu_seqlens has ",
              cu_seqlens.numel(), " entries");
  Tensor out = at::empty({T, n_q * D}, qkv.options());
  c10::hip::HIPGuardMasqueradingAsCUDA guard(qkv.device());
  // on the host it may be too
  const Tensor cu = cu_seqlens.to(qkv.device());
  const Tensor rows = aligned(qkv);
  rlli::launch_prefill_rows(
      bf16_ptr(rows), cu.data_ptr<int32_t>(), bf16_ptr(out), n_seqs, T,
      int(n_kv), group, D, stride, float(scale), current_stream(qkv));
  check_launch("prefill_attn_qkv");
  return out;
}

// rope_kv_append_qkv_ and prefill_attn_qkv: of up to 64 rows in one launch, which
// leaves qkv as it is.
static Tensor prompt_rows_attn(Tensor qkv, const Tensor& positions,
                               const Tensor& cos_sin, Tensor k_cache,
                               Tensor v_cache, const Tensor& slot_mapping,
                               const Tensor& cu_seqlens, double scale,
                               int64_t n_q) {
  const int64_t T = qkv.size(0), n_kv = k_cache.size(1), D = k_cache.size(3);
  if (T > 64 || (D != 64 && D != 128) || n_q % n_kv != 0) {
    rope_kv_append_qkv_(qkv, positions, cos_sin, k_cache, v_cache,
                        slot_mapping, n_q);
    return prefill_attn_qkv(qkv, cu_seqlens, scale, n_q, n_kv, D);
  }
  check_bf16_contig(qkv, "qkv");
  const bool cache_fp8 = check_cache(k_cache, v_cache);
  TORCH_CHECK(qkv.size(1) == (n_q + 2 * n_kv) * D, "qkv width mismatch");
  TORCH_CHECK(positions.numel() == T && slot_mapping.numel() == T);
  TORCH_CHECK(cos_sin.size(1) == D);
  TORCH_CHECK(cu_seqlens.scalar_type() == at::kInt &&
              cu_seqlens.is_contiguous());
  const int group = int(n_q / n_kv), n_seqs = int(cu_seqlens.numel()) - 1;
  TORCH_CHECK(group == 1 || group == 2 || group == 4 || group == 8);
  TORCH_CHECK(T == 0 || n_seqs >= 1, "rows without a sequence: cu_seqlens has ",
              cu_seqlens.numel(), " entries");
  Tensor out = at::empty({T, n_q * D}, qkv.options());
  c10::hip::HIPGuardMasqueradingAsCUDA guard(qkv.device());
  const Tensor cu = cu_seqlens.to(qkv.device());
  const Tensor rows = aligned(qkv);
  rlli::launch_prompt_rows_attn(
      bf16_ptr(rows), cu.data_ptr<int32_t>(), positions.data_ptr<int32_t>(),
      cos_sin.data_ptr<float>(), k_cache.data_ptr(), v_cache.data_ptr(),
      slot_mapping.data_ptr<int32_t>(), bf16_ptr(out), n_seqs, int(T),
      int(n_kv), group, int(D), int(k_cache.size(2)), int(qkv.size(1)),
      float(scale), cache_fp8, current_stream(qkv));
  check_launch("prompt_rows_attn");
  return out;
}

// ------------------------------------------------------ prefill (paged)
Tensor prefill_paged_attn(const Tensor& qkv, const Tensor& k_cache,
                          const Tensor& v_cache, const Tensor& chunk_row0,
                          const Tensor& chunk_pos0, const Tensor& chunk_nrows,
                          const Tensor& chunk_btrow,
                          const Tensor& block_tables, double scale,
                          int64_t n_q) {
  check_bf16_contig(qkv, "qkv");
  const bool cache_fp8 = check_cache(k_cache, v_cache);
  for (const Tensor* t : {&chunk_row0, &chunk_pos0, &chunk_nrows,
                          &chunk_btrow, &block_tables}) {
    TORCH_CHECK(t->scalar_type() == at::kInt && t->is_contiguous() &&
                t->is_cuda(), "chunk/table tensors must be contiguous "
                "int32 on the GPU");
  }
  const int T = int(qkv.size(0));
  const int n_kv = int(k_cache.size(1));
  const int block_size = int(k_cache.size(2));
  const int D = int(k_cache.size(3));
  const int stride = int(qkv.size(1));
  TORCH_CHECK(stride >= n_q * D, "qkv too narrow");
  const int group = int(n_q) / n_kv;
  TORCH_CHECK(group == 1 || group == 2 || group == 4 || group == 8);
  TORCH_CHECK(D == 64 || D == 128);
  const int n_chunks = int(chunk_row0.numel());
  const int max_blocks = int(block_tables.size(1));
  Tensor out = at::empty({T, n_q * D}, qkv.options());
  c10::hip::HIPGuardMasqueradingAsCUDA guard(qkv.device());
  const Tensor k = aligned(k_cache), v = aligned(v_cache);
  rlli::PrefillParts parts{nullptr, nullptr,
                           rlli::prefill_splits(n_chunks, n_kv, group,
                                                max_blocks * block_size),
                           T};
  Tensor part, ml;
  if (parts.splits > 1) {
    const auto f32 = qkv.options().dtype(at::kFloat);
    part = at::empty({parts.splits, T, n_q * D}, f32);
    ml = at::empty({parts.splits, T, n_q, 2}, f32);
    parts.o = part.data_ptr<float>();
    parts.ml = ml.data_ptr<float>();
  }
  rlli::launch_prefill_paged(
      bf16_ptr(qkv), k.data_ptr(), v.data_ptr(),
      chunk_row0.data_ptr<int32_t>(), chunk_pos0.data_ptr<int32_t>(),
      chunk_nrows.data_ptr<int32_t>(), chunk_btrow.data_ptr<int32_t>(),
      block_tables.data_ptr<int32_t>(), bf16_ptr(out), n_chunks, n_kv,
      group, D, stride, max_blocks, block_size, float(scale), cache_fp8, parts,
      current_stream(qkv));
  check_launch("prefill_paged_attn");
  return out;
}

// Attention of a mixed step: rows [0, n_decode) are decoding sequences', the
// others the tiles'.  In one launch where mixed_attn_plan takes the sizes (with
// the parts and shares of ``given`` if there are any), one after the other
// elsewhere.
Tensor mixed_attn_qkv(const Tensor& qkv, const Tensor& k_cache,
                      const Tensor& v_cache, const Tensor& chunk_row0,
                      const Tensor& chunk_pos0, const Tensor& chunk_nrows,
                      const Tensor& chunk_btrow, const Tensor& tables_pre,
                      const Tensor& tables_dec, const Tensor& lens_dec,
                      int64_t n_decode, double scale, int64_t n_q,
                      at::IntArrayRef given) {
  check_bf16_contig(qkv, "qkv");
  check_qkv_width(qkv, k_cache, n_q);
  const bool cache_fp8 = check_cache(k_cache, v_cache);
  TORCH_CHECK(n_decode >= 0 && n_decode <= qkv.size(0), "decoding rows: ",
              n_decode, " of ", qkv.size(0));
  const int T = int(qkv.size(0)), batch = int(n_decode);
  const int n_kv = int(k_cache.size(1)), block_size = int(k_cache.size(2));
  const int D = int(k_cache.size(3)), group = int(n_q) / n_kv;
  const int n_tiles = int(chunk_row0.numel());
  auto table = [&](const Tensor& t) {
    return t.scalar_type() == at::kInt && t.is_contiguous() &&
           t.device() == qkv.device();
  };
  rlli::MixedPlan plan{0, 0, false};
  if (n_tiles > 0 && batch > 0 && n_q % n_kv == 0 && (D == 64 || D == 128) &&
      table(chunk_row0) && table(chunk_pos0) && table(chunk_nrows) &&
      table(chunk_btrow) && table(tables_pre) && table(tables_dec) &&
      table(lens_dec) && tables_pre.dim() == 2 && tables_dec.dim() == 2 &&
      chunk_pos0.numel() == n_tiles && chunk_nrows.numel() == n_tiles &&
      chunk_btrow.numel() == n_tiles && tables_dec.size(0) >= batch &&
      lens_dec.numel() >= batch && v_cache.sizes() == k_cache.sizes() &&
      k_cache.device() == qkv.device() && v_cache.device() == qkv.device() &&
      (reinterpret_cast<uintptr_t>(qkv.data_ptr()) |
       reinterpret_cast<uintptr_t>(k_cache.data_ptr()) |
       reinterpret_cast<uintptr_t>(v_cache.data_ptr())) % 16 == 0)
    plan = rlli::mixed_attn_plan(
        n_tiles, batch, n_kv, group, D, int(tables_pre.size(1)) * block_size,
        int(tables_dec.size(1)) * block_size, int(k_cache.element_size()),
        block_size);
  if (!given.empty()) {
    TORCH_CHECK(plan.splits > 0 && given.size() == 2 && given[0] >= 1 &&
                    given[0] <= 16 && given[1] >= 0 && given[1] <= 512,
                "no such division for these sizes");
    plan = {int(given[0]), int(given[1]), true};
  }
  if (!plan.faster) {
    Tensor out = prefill_paged_attn(qkv, k_cache, v_cache, chunk_row0,
                                    chunk_pos0, chunk_nrows, chunk_btrow,
                                    tables_pre, scale, n_q);
    if (batch > 0)
      decode_attn_qkv_out(qkv.narrow(0, 0, batch), k_cache, v_cache,
                          tables_dec, lens_dec, scale, n_q, out);
    return out;
  }
  Tensor out = at::empty({T, n_q * D}, qkv.options());
  c10::hip::HIPGuardMasqueradingAsCUDA guard(qkv.device());
  const auto f32 = qkv.options().dtype(at::kFloat);
  rlli::PrefillParts parts{nullptr, nullptr, plan.splits, T};
  Tensor tile_part, tile_ml, part, ml;
  if (plan.splits > 1) {
    tile_part = at::empty({plan.splits, T, n_q * D}, f32);
    tile_ml = at::empty({plan.splits, T, n_q, 2}, f32);
    parts.o = tile_part.data_ptr<float>();
    parts.ml = tile_ml.data_ptr<float>();
  }
  if (plan.shares > 0) {
    const int64_t slots = int64_t(n_kv) * (plan.shares + batch) * group;
    part = at::empty({slots, D}, f32);
    ml = at::empty({slots, 2}, f32);
  }
  rlli::launch_mixed_attn(
      bf16_ptr(qkv), k_cache.data_ptr(), v_cache.data_ptr(),
      chunk_row0.data_ptr<int32_t>(), chunk_pos0.data_ptr<int32_t>(),
      chunk_nrows.data_ptr<int32_t>(), chunk_btrow.data_ptr<int32_t>(),
      tables_pre.data_ptr<int32_t>(), int(tables_pre.size(1)),
      tables_dec.data_ptr<int32_t>(), lens_dec.data_ptr<int32_t>(),
      int(tables_dec.size(1)), bf16_ptr(out), n_tiles, batch, n_kv, group, D,
      int(qkv.size(1)), float(scale), cache_fp8, parts, plan.shares,
      plan.shares > 0 ? part.data_ptr<float>() : nullptr,
      plan.shares > 0 ? ml.data_ptr<float>() : nullptr, current_stream(qkv));
  check_launch("mixed_attn_qkv");
  return out;
}

// ------------------------------------------------------------ rows_gemm
static void check_rows(const Tensor& x, const Tensor& w) {
  check_bf16_contig(x, "x");
  check_bf16_contig(w, "w");
  TORCH_CHECK(x.device() == w.device(), "x and W on one GPU");
  TORCH_CHECK(x.dim() == 2 && w.dim() == 2 && w.size(1) == x.size(1),
              "x/W K mismatch");
  TORCH_CHECK(x.size(0) >= 1 && x.size(0) <= 128, "1 to 128 rows, got ",
              x.size(0));
  TORCH_CHECK(x.size(1) % 64 == 0 && x.size(1) > 0 && w.size(0) % 4 == 0 &&
                  w.size(0) > 0,
              "K % 64 == 0 and N % 4 == 0, got K=", x.size(1), " N=",
              w.size(0));
  TORCH_CHECK(reinterpret_cast<uintptr_t>(x.data_ptr()) % 16 == 0 &&
                  reinterpret_cast<uintptr_t>(w.data_ptr()) % 16 == 0,
              "x and W start at multiples of 16 bytes");
}

// y = x w^T in f32 parts [splits, M, N] to be summed, or whole in bf16
// [M, N] where K is not divided.
Tensor rows_linear_parts(const Tensor& x, const Tensor& w) {
  check_rows(x, w);
  const int M = int(x.size(0)), N = int(w.size(0)), K = int(x.size(1));
  c10::hip::HIPGuardMasqueradingAsCUDA guard(x.device());
  const int splits = rlli::rows_gemm_splits(N, K);
  Tensor out = splits > 1
                   ? at::empty({splits, M, N}, x.options().dtype(at::kFloat))
                   : at::empty({M, N}, x.options());
  rlli::launch_rows_gemm(
      bf16_ptr(x), bf16_ptr(w), splits > 1 ? out.data_ptr<float>() : nullptr,
      splits > 1 ? nullptr : bf16_ptr(out), M, N, K, splits,
      current_stream(x));
  check_launch("rows_linear");
  return out;
}

// whole products of at most 64 rows by workgroups that divide K themselves,
// with or without the squared positive part; undefined where those are not
// the faster ones
Tensor rows_short(const Tensor& x, const Tensor& w, bool relu2) {
  check_rows(x, w);
  const int M = int(x.size(0)), N = int(w.size(0)), K = int(x.size(1));
  if (M > 64 || !rlli::rows_short_ok(N, K)) return Tensor();
  c10::hip::HIPGuardMasqueradingAsCUDA guard(x.device());
  Tensor out = at::empty({M, N}, x.options());
  rlli::launch_rows_short(bf16_ptr(x), bf16_ptr(w), bf16_ptr(out), M, N, K,
                          relu2, current_stream(x));
  check_launch("rows_short");
  return out;
}

Tensor rows_linear(const Tensor& x, const Tensor& w) {
  Tensor whole = rows_short(x, w, false);
  if (whole.defined()) return whole;
  Tensor parts = rows_linear_parts(x, w);
  if (parts.dim() == 2) return parts;
  c10::hip::HIPGuardMasqueradingAsCUDA guard(x.device());
  Tensor out = at::empty({x.size(0), w.size(0)}, x.options());
  rlli::launch_sum_parts(parts.data_ptr<float>(), bf16_ptr(out),
                         int(parts.size(0)), out.numel(), current_stream(x));
  check_launch("sum_parts");
  return out;
}

// the squared positive part of x w^T, of the f32 sums
Tensor rows_linear_relu2(const Tensor& x, const Tensor& w) {
  Tensor whole = rows_short(x, w, true);
  TORCH_CHECK(whole.defined(), "rows_whole_ok says which products these are");
  return whole;
}

bool rows_whole_ok(int64_t M, int64_t N, int64_t K) {
  return M <= 64 && N <= 8192 && K <= 8192 &&
         rlli::rows_short_ok(int(N), int(K));
}

Tensor rows_linear_silu(const Tensor& x, const Tensor& w) {
  check_rows(x, w);
  const int inter = int(w.size(0)) / 2;
  TORCH_CHECK(w.size(0) % 16 == 0, "gate and up rows are multiples of 8");
  if (!rlli::rows_gemm_silu_ok(inter)) return silu_mul(rows_linear(x, w));
  c10::hip::HIPGuardMasqueradingAsCUDA guard(x.device());
  Tensor out = at::empty({x.size(0), inter}, x.options());
  rlli::launch_rows_gemm_silu(bf16_ptr(x), bf16_ptr(w), bf16_ptr(out),
                              int(x.size(0)), inter, int(x.size(1)),
                              current_stream(x));
  check_launch("rows_linear_silu");
  return out;
}

bool rows_norm_ok(int64_t N, int64_t K, bool silu) {
  return N <= 1 << 20 && K <= 8192 &&
         rlli::rows_norm_ok(int(N), int(K), silu);
}

// Of one row: rows_linear_parts or (silu) rows_linear_silu of the rmsnorm of
// residual + the sum of parts [n, 1, K], in one launch; and the new residual.
std::tuple<Tensor, Tensor> rows_norm_linear(const Tensor& parts,
                                            const Tensor& residual,
                                            const Tensor& gain, double eps,
                                            const Tensor& w, bool silu) {
  check_rows(residual, w);
  check_bf16_contig(gain, "gain");
  const int K = int(residual.size(1)), N = int(w.size(0));
  TORCH_CHECK(residual.size(0) == 1 && rows_norm_ok(N, K, silu) &&
                  (!silu || N % 16 == 0),
              "one row; rows_norm_ok says which products these are");
  TORCH_CHECK(parts.scalar_type() == at::kFloat && parts.is_contiguous() &&
                  parts.device() == residual.device() && parts.dim() == 3 &&
                  parts.size(0) >= 1 && parts.size(1) == 1 &&
                  parts.size(2) == K,
              "parts: f32 [n, 1, K]");
  TORCH_CHECK(gain.numel() == K && gain.device() == residual.device(),
              "a gain of K");
  TORCH_CHECK(reinterpret_cast<uintptr_t>(parts.data_ptr()) % 16 == 0,
              "parts start at multiples of 16 bytes");
  c10::hip::HIPGuardMasqueradingAsCUDA guard(residual.device());
  const hipStream_t st = current_stream(residual);
  const Tensor whole_gain = aligned(gain);
  Tensor after = at::empty_like(residual);
  const rlli::RowsNorm norm{parts.data_ptr<float>(), bf16_ptr(residual),
                            bf16_ptr(after), bf16_ptr(whole_gain),
                            int(parts.size(0)), float(eps)};
  Tensor out;
  if (silu) {
    out = at::empty({1, N / 2}, residual.options());
    rlli::launch_rows_norm_silu(norm, bf16_ptr(w), bf16_ptr(out), N / 2, K,
                                st);
  } else {
    const int splits = rlli::rows_gemm_splits(N, K);
    out = at::empty({splits, 1, N}, parts.options());
    rlli::launch_rows_norm(norm, bf16_ptr(w), out.data_ptr<float>(), N, K,
                           splits, st);
  }
  check_launch("rows_norm_linear");
  return {out, after};
}

// Of up to 32 rows, the first of two products that share a norm: x w^T into the
// streams, what is normed of them times the gains, and sums of squares
// [N / 16, 16 or 32].
std::tuple<Tensor, Tensor> rows_linear_streams_(
    const Tensor& x, const Tensor& w, Tensor streams, const Tensor& mix,
    const Tensor& out_w, const Tensor& in_w, const Tensor& gain) {
  check_rows(x, w);
  auto f32 = [&](const Tensor& t, int64_t n, const char* name) {
    TORCH_CHECK(t.scalar_type() == at::kFloat && t.is_contiguous() &&
                    t.numel() == n && t.device() == x.device(),
                name, " must be ", n, " contiguous f32 beside x");
  };
  const int M = int(x.size(0)), N = int(w.size(0)), K = int(x.size(1));
  TORCH_CHECK(streams.dim() == 3 && streams.size(0) == M &&
                  streams.size(2) == N, "streams of the product's rows");
  const int S = int(streams.size(1));
  TORCH_CHECK(rlli::rows_adds_ok(M, N, K, S), "not for these sizes: ", M,
              " rows, ", N, " x ", K, ", ", S, " streams");
  f32(streams, streams.numel(), "streams");
  f32(mix, S * S, "mix");
  f32(out_w, S, "out_w");
  f32(in_w, S, "in_w");
  f32(gain, N, "gain");
  Tensor h = at::empty({M, N}, x.options());
  Tensor ss = at::empty({N / 16, M <= 16 ? 16 : 32},
                        x.options().dtype(at::kFloat));
  c10::hip::HIPGuardMasqueradingAsCUDA guard(x.device());
  rlli::launch_rows_adds(
      bf16_ptr(x), bf16_ptr(w), bf16_ptr(h), M, N, K, S,
      rlli::RowsAdds{streams.data_ptr<float>(), mix.data_ptr<float>(),
                     out_w.data_ptr<float>(), in_w.data_ptr<float>(),
                     gain.data_ptr<float>(), ss.data_ptr<float>()},
      current_stream(x));
  check_launch("rows_linear_streams_");
  return {h, ss};
}

// Whether the two take m rows, weights [n, k] and then [next, n].
bool rows_streams_ok(int64_t m, int64_t n, int64_t k, int64_t streams,
                     int64_t next) {
  return rlli::rows_adds_ok(int(m), int(n), int(k), int(streams)) &&
         rlli::rows_scaled_ok(int(m), int(next), int(n));
}

// The second of them, the squared positive part of its result.
Tensor rows_linear_scaled_relu2(const Tensor& h, const Tensor& ss, double eps,
                                const Tensor& w) {
  check_rows(h, w);
  const int M = int(h.size(0)), N = int(w.size(0)), K = int(h.size(1));
  TORCH_CHECK(rlli::rows_scaled_ok(M, N, K), "not for these sizes: ", M,
              " rows, ", N, " x ", K);
  TORCH_CHECK(ss.scalar_type() == at::kFloat && ss.is_contiguous() &&
                  ss.dim() == 2 && ss.size(0) * 16 == K && ss.size(0) <= 256 &&
                  ss.size(1) == (M <= 16 ? 16 : 32) &&
                  ss.device() == h.device() &&
                  reinterpret_cast<uintptr_t>(ss.data_ptr()) % 16 == 0,
              "sums of squares of the rows by sixteen columns");
  Tensor out = at::empty({M, N}, h.options());
  c10::hip::HIPGuardMasqueradingAsCUDA guard(h.device());
  rlli::launch_rows_scaled_relu2(
      bf16_ptr(h), bf16_ptr(w), bf16_ptr(out), M, N, K,
      rlli::RowsScale{ss.data_ptr<float>(), int(ss.size(0)), K, float(eps)},
      current_stream(h));
  check_launch("rows_linear_scaled_relu2");
  return out;
}

static void check_tiles(const Tensor& x, const Tensor& w, int multiple) {
  check_bf16_contig(x, "x");
  check_bf16_contig(w, "w");
  TORCH_CHECK(x.device() == w.device(), "x and W on one GPU");
  TORCH_CHECK(x.dim() == 2 && w.dim() == 2 && w.size(1) == x.size(1),
              "x/W K mismatch");
  TORCH_CHECK(x.size(0) >= 1 && x.size(1) % 64 == 0 && x.size(1) > 0 &&
                  w.size(0) % multiple == 0 && w.size(0) > 0,
              "K % 64 == 0 and N % ", multiple, " == 0, got K=", x.size(1),
              " N=", w.size(0));
  TORCH_CHECK(x.numel() < int64_t(1) << 31 && w.numel() < int64_t(1) << 31,
              "x and W below 4 GiB");
  TORCH_CHECK(reinterpret_cast<uintptr_t>(x.data_ptr()) % 16 == 0 &&
                  reinterpret_cast<uintptr_t>(w.data_ptr()) % 16 == 0,
              "x and W start at multiples of 16 bytes");
}

// Rows of x and w that a workgroup of rows_tall has; 0: it does not take M rows
// by N columns.
int64_t rows_tall_work(int64_t M, int64_t N) {
  if (M < 1 || N < 1 || M > 1 << 20 || N > 1 << 20) return 0;
  const rlli::TallPlan plan = rlli::rows_tall_plan(int(M), int(N));
  return plan.rows + 8 * plan.eights;
}

// x w^T of some hundred rows, or the squared positive part of it in 16 bits, by
// workgroups that divide K themselves
Tensor rows_tall(const Tensor& x, const Tensor& w, bool relu2) {
  check_tiles(x, w, 4);
  TORCH_CHECK(rows_tall_work(x.size(0), w.size(0)) > 0,
              "too many rows and columns to run at once");
  const int M = int(x.size(0)), N = int(w.size(0)), K = int(x.size(1));
  c10::hip::HIPGuardMasqueradingAsCUDA guard(x.device());
  Tensor out = at::empty({M, N}, x.options());
  rlli::launch_rows_tall(bf16_ptr(x), bf16_ptr(w), bf16_ptr(out), M, N, K,
                         relu2, rlli::rows_tall_plan(M, N),
                         current_stream(x));
  check_launch("rows_tall");
  return out;
}

// The tile and the division of K that should take least, or those of ``plan``:
// a tile's 64 rows and 128 columns, and parts.
static rlli::TilePlan tile_plan(int M, int N, int K, bool whole,
                                at::IntArrayRef plan) {
  if (plan.empty()) return rlli::tile_gemm_plan(M, N, K, whole);
  TORCH_CHECK(plan.size() == 3 && std::all_of(plan.begin(), plan.end(),
                                              [](int64_t v) {
                                                return v > 0 && v < 16;
                                              }),
              "a plan: 64 rows and 128 columns of a tile, parts");
  const rlli::TilePlan p{int(plan[0]), int(plan[1]), int(plan[2])};
  TORCH_CHECK(rlli::tile_gemm_ok(p, K, whole), "there is no such plan");
  return p;
}

// x w^T in f32 parts [splits, M, N], or in bf16 [M, N] where K is not divided
Tensor tile_linear_parts(const Tensor& x, const Tensor& w,
                         at::IntArrayRef by) {
  check_tiles(x, w, 8);
  const int M = int(x.size(0)), N = int(w.size(0)), K = int(x.size(1));
  c10::hip::HIPGuardMasqueradingAsCUDA guard(x.device());
  const rlli::TilePlan plan = tile_plan(M, N, K, false, by);
  const bool parts = plan.splits > 1;
  Tensor out = parts ? at::empty({plan.splits, M, N},
                                 x.options().dtype(at::kFloat))
                     : at::empty({M, N}, x.options());
  rlli::launch_tile_gemm(bf16_ptr(x), bf16_ptr(w),
                         parts ? out.data_ptr<float>() : nullptr,
                         parts ? nullptr : bf16_ptr(out), M, N, K,
                         rlli::TileAct::none, plan, current_stream(x));
  check_launch("tile_linear_parts");
  return out;
}

// the whole product in bf16
Tensor tile_linear(const Tensor& x, const Tensor& w, at::IntArrayRef by) {
  const Tensor parts = tile_linear_parts(x, w, by);
  if (parts.dim() == 2) return parts;
  c10::hip::HIPGuardMasqueradingAsCUDA guard(x.device());
  Tensor out = at::empty({x.size(0), w.size(0)}, x.options());
  rlli::launch_sum_parts(parts.data_ptr<float>(), bf16_ptr(out),
                         int(parts.size(0)), out.numel(), current_stream(x));
  check_launch("sum_parts");
  return out;
}

static Tensor tile_linear_act(const Tensor& x, const Tensor& w,
                              rlli::TileAct act, at::IntArrayRef by) {
  const bool silu = act == rlli::TileAct::silu;
  check_tiles(x, w, silu ? 16 : 8);
  const int M = int(x.size(0)), N = int(w.size(0)), K = int(x.size(1));
  c10::hip::HIPGuardMasqueradingAsCUDA guard(x.device());
  Tensor out = at::empty({M, silu ? N / 2 : N}, x.options());
  rlli::launch_tile_gemm(bf16_ptr(x), bf16_ptr(w), nullptr, bf16_ptr(out), M,
                         N, K, act, tile_plan(M, N, K, true, by),
                         current_stream(x));
  check_launch("tile_linear");
  return out;
}

// silu(x w[:I]^T) * (x w[I:]^T) for w [2 I, K]
Tensor tile_linear_silu(const Tensor& x, const Tensor& w,
                       at::IntArrayRef by) {
  return tile_linear_act(x, w, rlli::TileAct::silu, by);
}

// the squared positive part of the 16-bit x w^T
Tensor tile_linear_relu2(const Tensor& x, const Tensor& w,
                        at::IntArrayRef by) {
  return tile_linear_act(x, w, rlli::TileAct::relu2, by);
}

// The same under the names and limits of earlier kernels; ``splitk`` has no
// effect any more.
static void check_skinny(const char* op, const Tensor& x, const Tensor& w,
                         int64_t K) {
  check_bf16_contig(x, "x");
  check_bf16_contig(w, "w");
  const int64_t M = x.size(0), N = w.size(0);
  TORCH_CHECK(w.size(1) == K, "x/W K mismatch");
  TORCH_CHECK(M >= 1 && M <= 64, op, " needs 1 <= M <= 64, got ", M);
  TORCH_CHECK(K % 256 == 0 && N % 64 == 0, op,
              " needs K%256==0 and N%64==0, got K=", K, " N=", N);
}

Tensor skinny_linear(const Tensor& x, const Tensor& w) {
  check_skinny("skinny_linear", x, w, x.size(1));
  return rows_linear(aligned(x), aligned(w));
}

Tensor skinny2_linear(const Tensor& x, const Tensor& w, int64_t /*splitk*/) {
  check_skinny("skinny2_linear", x, w, x.size(1));
  return rows_linear(aligned(x), aligned(w));
}

// down-proj behind SwiGLU: (silu(gu[:, :K]) * gu[:, K:]) @ w^T, gu [M, 2K]
Tensor skinny2_silu_linear(const Tensor& gu, const Tensor& w,
                           int64_t /*splitk*/) {
  TORCH_CHECK(gu.size(1) % 2 == 0, "gu must be [M, 2K]");
  check_skinny("skinny2_silu", gu, w, gu.size(1) / 2);
  return rows_linear(silu_mul(gu), aligned(w));
}

Tensor stream_probe(const Tensor& w, int64_t splitk) {
  check_bf16_contig(w, "w");
  Tensor sink = at::zeros({256}, w.options().dtype(at::kFloat));
  c10::hip::HIPGuardMasqueradingAsCUDA guard(w.device());
  rlli::launch_stream_probe(bf16_ptr(w), sink.data_ptr<float>(),
                            int(w.size(0)), int(w.size(1)), int(splitk),
                            current_stream(w));
  check_launch("stream_probe");
  return sink;
}

// --------------------------------------------------------------- sample
Tensor sample(const Tensor& logits, const Tensor& temperatures,
              const Tensor& seeds, int64_t step) {
  const bool f32 = logits.scalar_type() == at::kFloat;
  TORCH_CHECK(f32 || logits.scalar_type() == at::kBFloat16,
              "logits must be bf16 or f32");
  TORCH_CHECK(logits.is_contiguous() && logits.is_cuda() &&
              logits.dim() == 2, "logits must be [batch, vocab] on the GPU");
  TORCH_CHECK(temperatures.scalar_type() == at::kFloat &&
              temperatures.is_contiguous() && temperatures.is_cuda());
  TORCH_CHECK(seeds.scalar_type() == at::kLong && seeds.is_contiguous() &&
              seeds.is_cuda());
  const int batch = int(logits.size(0));
  const int vocab = int(logits.size(1));
  TORCH_CHECK(temperatures.numel() == batch && seeds.numel() == batch);
  Tensor out = at::empty({batch}, logits.options().dtype(at::kInt));
  c10::hip::HIPGuardMasqueradingAsCUDA guard(logits.device());
  const int n_split = rlli::sample_n_split(batch);
  uint64_t* pptr = nullptr;
  Tensor partials;
  if (n_split > 1) {
    // caching-allocator tensor: participates in hipGraph capture pools
    partials = at::empty({int64_t(batch) * n_split},
                         logits.options().dtype(at::kLong));
    pptr = reinterpret_cast<uint64_t*>(partials.data_ptr<int64_t>());
  }
  rlli::launch_sample(logits.data_ptr(), f32, temperatures.data_ptr<float>(),
                      reinterpret_cast<const uint64_t*>(seeds.data_ptr<int64_t>()),
                      uint64_t(step), out.data_ptr<int32_t>(), batch, vocab,
                      pptr, n_split, current_stream(logits));
  check_launch("sample");
  return out;
}

// ------------------------------------------------- a captured step's state
static void check_rows_of(const Tensor& t, at::ScalarType type, int64_t rows,
                          int64_t width, const Tensor& like, const char* name) {
  TORCH_CHECK(t.is_cuda() && t.device() == like.device() &&
                  t.scalar_type() == type && t.is_contiguous() &&
                  t.dim() == (width < 0 ? 1 : 2) && t.size(0) == rows &&
                  (width < 0 || t.size(1) == width),
              name, ": ", rows, " rows of the step's type on its GPU");
}

// The first ``bucket`` rows of a step's buffers from a batch; those that it
// does not fill have nothing but the scratch block and slot.
void decode_load(Tensor ids_to, Tensor positions_to, Tensor tables_to,
                 Tensor temps_to, Tensor seeds_to, Tensor slots_to,
                 const Tensor& ids, const Tensor& positions,
                 const Tensor& tables, const Tensor& temps,
                 const Tensor& seeds, const std::optional<Tensor>& slots,
                 int64_t bucket, int64_t scratch_block, int64_t scratch_slot) {
  TORCH_CHECK(ids_to.dim() == 1 && tables_to.dim() == 2 && ids.dim() == 1 &&
                  tables.dim() == 2,
              "rows of ids and of tables");
  const int64_t rows = ids_to.size(0), width = tables_to.size(1);
  const int64_t batch = ids.size(0), wide = tables.size(1);
  TORCH_CHECK(batch <= bucket && bucket >= 1 && bucket <= rows &&
                  wide <= width,
              "a batch of ", batch, " by ", wide, " in ", bucket, " of ", rows,
              " rows by ", width);
  const Tensor& at = ids_to;
  check_rows_of(ids_to, at::kInt, rows, -1, at, "ids_to");
  check_rows_of(positions_to, at::kInt, rows, -1, at, "positions_to");
  check_rows_of(tables_to, at::kInt, rows, width, at, "tables_to");
  check_rows_of(temps_to, at::kFloat, rows, -1, at, "temps_to");
  check_rows_of(seeds_to, at::kLong, rows, -1, at, "seeds_to");
  check_rows_of(slots_to, at::kInt, rows, -1, at, "slots_to");
  check_rows_of(ids, at::kInt, batch, -1, at, "ids");
  check_rows_of(positions, at::kInt, batch, -1, at, "positions");
  check_rows_of(tables, at::kInt, batch, wide, at, "tables");
  check_rows_of(temps, at::kFloat, batch, -1, at, "temps");
  check_rows_of(seeds, at::kLong, batch, -1, at, "seeds");
  if (slots) check_rows_of(*slots, at::kInt, batch, -1, at, "slots");
  c10::hip::HIPGuardMasqueradingAsCUDA guard(at.device());
  auto state = [](const Tensor& i, const Tensor& p, const Tensor& t,
                  const Tensor& f, const Tensor& s, const Tensor* slot) {
    return rlli::DecodeState{
        i.data_ptr<int32_t>(), p.data_ptr<int32_t>(), t.data_ptr<int32_t>(),
        f.data_ptr<float>(),   s.data_ptr<int64_t>(),
        slot ? slot->data_ptr<int32_t>() : nullptr, int(t.size(1))};
  };
  rlli::launch_decode_load(
      state(ids_to, positions_to, tables_to, temps_to, seeds_to, &slots_to),
      state(ids, positions, tables, temps, seeds, slots ? &*slots : nullptr),
      int(bucket), int(batch), int(wide), int(scratch_block),
      int(scratch_slot), current_stream(at));
  check_launch("decode_load");
}

// Rows of decoding sequences at ``positions``: where their keys and values go,
// and how many tokens they see.
std::tuple<Tensor, Tensor> decode_begin(const Tensor& positions,
                                        const Tensor& tables,
                                        int64_t block_size) {
  TORCH_CHECK(positions.dim() == 1 && tables.dim() == 2 &&
                  tables.size(1) >= 1 && block_size >= 1,
              "positions, their tables and a block's size");
  const int64_t batch = positions.size(0);
  check_rows_of(positions, at::kInt, batch, -1, positions, "positions");
  check_rows_of(tables, at::kInt, batch, tables.size(1), positions, "tables");
  Tensor slots = at::empty_like(positions), lens = at::empty_like(positions);
  if (batch == 0) return {slots, lens};
  c10::hip::HIPGuardMasqueradingAsCUDA guard(positions.device());
  rlli::launch_decode_begin(positions.data_ptr<int32_t>(),
                            tables.data_ptr<int32_t>(),
                            slots.data_ptr<int32_t>(),
                            lens.data_ptr<int32_t>(), int(batch),
                            int(tables.size(1)), int(block_size),
                            current_stream(positions));
  check_launch("decode_begin");
  return {slots, lens};
}

// One token on: the sampled tokens are the next ids.
void decode_advance_(Tensor ids, Tensor positions, Tensor seeds,
                     const Tensor& tokens, int64_t seed_step) {
  TORCH_CHECK(ids.dim() == 1, "rows of ids");
  const int64_t batch = ids.size(0);
  check_rows_of(ids, at::kInt, batch, -1, ids, "ids");
  check_rows_of(positions, at::kInt, batch, -1, ids, "positions");
  check_rows_of(seeds, at::kLong, batch, -1, ids, "seeds");
  check_rows_of(tokens, at::kInt, batch, -1, ids, "tokens");
  if (batch == 0) return;
  c10::hip::HIPGuardMasqueradingAsCUDA guard(ids.device());
  rlli::launch_decode_advance(ids.data_ptr<int32_t>(),
                              positions.data_ptr<int32_t>(),
                              seeds.data_ptr<int64_t>(),
                              tokens.data_ptr<int32_t>(), int(batch),
                              seed_step, current_stream(ids));
  check_launch("decode_advance_");
}

// ------------------------------------------------------- a prompt's layer
static Tensor norm_any(const Tensor& x, const Tensor& residual,
                       const Tensor& gain, double eps) {
  return x.dim() == 3 && x.scalar_type() == at::kFloat
             ? rmsnorm_residual_parts_(x, residual, gain, eps)
             : rmsnorm_residual_(x, residual, gain, eps);
}

// All of a Llama layer but the first for the rows of a few short prompts, whose
// step waits for the host: the ops in their order, rotation, append and attention
// as one, launched from here; the last product and the new residual, which is
// ``residual`` itself unless the one row's norm is made inside gate and up.
// (A prompt of 45 tokens through 16 layers of 2048: 8 us a launch from Python, 5
// from here; 1150 -> 1040 us.)
std::tuple<Tensor, Tensor> prompt_rows_layer(
    const Tensor& x, Tensor residual, const Tensor& ln1, const Tensor& w_qkv,
    const Tensor& w_o, const Tensor& ln2, const Tensor& w_gate_up,
    const Tensor& w_down, const Tensor& positions, const Tensor& cos_sin,
    Tensor k_cache, Tensor v_cache, const Tensor& slot_mapping,
    const Tensor& cu_seqlens, double eps, double scale, int64_t n_q) {
  const Tensor h = norm_any(x, residual, ln1, eps);
  Tensor qkv = rows_take(h, w_qkv) ? rows_linear(h, w_qkv)
                                   : at::linear(h, w_qkv);
  const Tensor seen =
      prompt_rows_attn(qkv, positions, cos_sin, k_cache, v_cache, slot_mapping,
                       cu_seqlens, scale, n_q);
  const Tensor mixed = rows_take(seen, w_o) ? rows_linear_parts(seen, w_o)
                                            : at::linear(seen, w_o);
  Tensor act, after = residual;
  if (mixed.dim() == 3 && mixed.size(1) == 1 &&
      rows_take(residual, w_gate_up) &&
      rows_norm_ok(w_gate_up.size(0), w_gate_up.size(1), true)) {
    std::tie(act, after) =
        rows_norm_linear(mixed, residual, ln2, eps, w_gate_up, true);
  } else {
    const Tensor h2 = norm_any(mixed, residual, ln2, eps);
    act = rows_take(h2, w_gate_up) ? rows_linear_silu(h2, w_gate_up)
                                   : silu_mul(at::linear(h2, w_gate_up));
  }
  return {rows_take(act, w_down) ? rows_linear_parts(act, w_down)
                                 : at::linear(act, w_down),
          after};
}

}  // namespace

TORCH_LIBRARY(rlli, m) {
  m.def("rmsnorm(Tensor x, Tensor w, float eps) -> Tensor");
  m.def("rmsnorm_residual_(Tensor x, Tensor(a!) residual, Tensor w, float eps) -> Tensor");
  m.def("rmsnorm_residual_parts_(Tensor parts, Tensor(a!) residual, Tensor w, float eps) -> Tensor");
  m.def("silu_mul(Tensor gate_up) -> Tensor");
  m.def("rmsnorm_fp8(Tensor x, Tensor w, float eps) -> (Tensor, Tensor)");
  m.def("rmsnorm_residual_fp8(Tensor x, Tensor(a!) residual, Tensor w, float eps) -> (Tensor, Tensor)");
  m.def("silu_mul_fp8(Tensor gate_up) -> (Tensor, Tensor)");
  m.def("rope_kv_append_(Tensor(a!) q, Tensor(b!) k, Tensor v, Tensor positions, "
        "Tensor cos_sin, Tensor(c!) k_cache, Tensor(d!) v_cache, "
        "Tensor slot_mapping) -> ()");
  m.def("decode_attn(Tensor q, Tensor k_cache, Tensor v_cache, "
        "Tensor block_table, Tensor seq_lens, float scale) -> Tensor");
  m.def("rope_kv_append_qkv_(Tensor(a!) qkv, Tensor positions, Tensor cos_sin, "
        "Tensor(b!) k_cache, Tensor(c!) v_cache, Tensor slot_mapping, "
        "int n_q) -> ()");
  m.def("decode_attn_qkv(Tensor qkv, Tensor k_cache, Tensor v_cache, "
        "Tensor block_table, Tensor seq_lens, float scale, int n_q) -> Tensor");
  m.def("decode_attn_qkv_out(Tensor qkv, Tensor k_cache, Tensor v_cache, "
        "Tensor block_table, Tensor seq_lens, float scale, int n_q, "
        "Tensor(a!) out) -> ()");
  m.def("decode_attn_rope_qkv(Tensor qkv, Tensor positions, Tensor cos_sin, "
        "Tensor(a!) k_cache, Tensor(b!) v_cache, Tensor slot_mapping, "
        "Tensor block_table, Tensor seq_lens, float scale, int n_q) -> Tensor");
  m.def("decode_attn_rope_linear(Tensor qkv, Tensor positions, "
        "Tensor cos_sin, Tensor(a!) k_cache, Tensor(b!) v_cache, "
        "Tensor slot_mapping, Tensor block_table, Tensor seq_lens, "
        "float scale, int n_q, Tensor w) -> Tensor");
  m.def("kv_append_qkv_(Tensor(a!) qkv, Tensor positions, Tensor cos_sin, "
        "Tensor(b!) k_cache, Tensor(c!) v_cache, Tensor slot_mapping, "
        "int n_q) -> ()");
  m.def("decode_attn_q_rope(Tensor qkv, Tensor positions, Tensor cos_sin, "
        "Tensor k_cache, Tensor v_cache, Tensor block_table, "
        "Tensor seq_lens, float scale, int n_q) -> Tensor");
  m.def("mixed_row_tables(int rows, int n_decode, Tensor? tables_dec, "
        "Tensor? lens_dec, Tensor row0, Tensor pos0, Tensor nrows, "
        "Tensor btrow, Tensor tables_pre) -> (Tensor, Tensor)");
  m.def("prefill_attn_qkv(Tensor qkv, Tensor cu_seqlens, float scale, "
        "int n_q, int n_kv, int head_dim) -> Tensor");
  m.def("prompt_rows_layer(Tensor x, Tensor(a!) residual, Tensor ln1, "
        "Tensor w_qkv, Tensor w_o, Tensor ln2, Tensor w_gate_up, "
        "Tensor w_down, Tensor positions, Tensor cos_sin, "
        "Tensor(b!) k_cache, Tensor(c!) v_cache, Tensor slot_mapping, "
        "Tensor cu_seqlens, float eps, float scale, int n_q) -> "
        "(Tensor, Tensor(a!))");
  m.def("prefill_attn(Tensor q, Tensor k, Tensor v, Tensor cu_seqlens, "
        "float scale) -> Tensor");
  m.def("decode_load(Tensor(a!) ids_to, Tensor(b!) positions_to, "
        "Tensor(c!) tables_to, Tensor(d!) temps_to, Tensor(e!) seeds_to, "
        "Tensor(f!) slots_to, Tensor ids, Tensor positions, Tensor tables, "
        "Tensor temps, Tensor seeds, Tensor? slots, int bucket, "
        "int scratch_block, int scratch_slot) -> ()");
  m.def("decode_begin(Tensor positions, Tensor tables, int block_size) -> "
        "(Tensor, Tensor)");
  m.def("decode_advance_(Tensor(a!) ids, Tensor(b!) positions, "
        "Tensor(c!) seeds, Tensor tokens, int seed_step) -> ()");
  m.def("sample(Tensor logits, Tensor temperatures, Tensor seeds, int step) -> Tensor");
  m.def("rows_linear_parts(Tensor x, Tensor w) -> Tensor");
  m.def("rows_linear(Tensor x, Tensor w) -> Tensor");
  m.def("rows_linear_silu(Tensor x, Tensor w) -> Tensor");
  m.def("rows_linear_relu2(Tensor x, Tensor w) -> Tensor");
  m.def("rows_tall(Tensor x, Tensor w, bool relu2) -> Tensor");
  m.def("rows_tall_work(int m, int n) -> int", &rows_tall_work);
  m.def("rows_whole_ok(int m, int n, int k) -> bool", &rows_whole_ok);
  m.def("rows_norm_ok(int n, int k, bool silu) -> bool",
        &rows_norm_ok);
  m.def("rows_norm_linear(Tensor parts, Tensor residual, Tensor gain, "
        "float eps, Tensor w, bool silu) -> (Tensor, Tensor)");
  m.def("rows_streams_ok(int m, int n, int k, int streams, int next) -> bool",
        &rows_streams_ok);
  m.def("rows_linear_streams_(Tensor x, Tensor w, Tensor(a!) streams, "
        "Tensor mix, Tensor out_w, Tensor in_w, Tensor gain) -> "
        "(Tensor, Tensor)");
  m.def("rows_linear_scaled_relu2(Tensor h, Tensor ss, float eps, Tensor w) "
        "-> Tensor");
  m.def("tile_linear_parts(Tensor x, Tensor w, int[] plan=[]) -> Tensor");
  m.def("tile_linear(Tensor x, Tensor w, int[] plan=[]) -> Tensor");
  m.def("tile_linear_silu(Tensor x, Tensor w, int[] plan=[]) -> Tensor");
  m.def("tile_linear_relu2(Tensor x, Tensor w, int[] plan=[]) -> Tensor");
  m.def("skinny_linear(Tensor x, Tensor w) -> Tensor");
  m.def("skinny2_linear(Tensor x, Tensor w, int splitk) -> Tensor");
  m.def("skinny2_silu_linear(Tensor gu, Tensor w, int splitk) -> Tensor");
  m.def("stream_probe(Tensor w, int splitk) -> Tensor");
  m.def("prefill_paged_attn(Tensor qkv, Tensor k_cache, Tensor v_cache, "
        "Tensor chunk_row0, Tensor chunk_pos0, Tensor chunk_nrows, "
        "Tensor chunk_btrow, Tensor block_tables, float scale, int n_q) "
        "-> Tensor");
  m.def("mixed_attn_qkv(Tensor qkv, Tensor k_cache, Tensor v_cache, "
        "Tensor chunk_row0, Tensor chunk_pos0, Tensor chunk_nrows, "
        "Tensor chunk_btrow, Tensor tables_pre, Tensor tables_dec, "
        "Tensor lens_dec, int n_decode, float scale, int n_q, int[] plan=[]) "
        "-> Tensor");
}

TORCH_LIBRARY_IMPL(rlli, CUDA, m) {
  m.impl("rmsnorm", &rmsnorm);
  m.impl("rmsnorm_residual_", &rmsnorm_residual_);
  m.impl("rmsnorm_residual_parts_", &rmsnorm_residual_parts_);
  m.impl("silu_mul", &silu_mul);
  m.impl("rmsnorm_fp8", &rmsnorm_fp8);
  m.impl("rmsnorm_residual_fp8", &rmsnorm_residual_fp8);
  m.impl("silu_mul_fp8", &silu_mul_fp8);
  m.impl("rope_kv_append_", &rope_kv_append_);
  m.impl("decode_attn", &decode_attn);
  m.impl("rope_kv_append_qkv_", &rope_kv_append_qkv_);
  m.impl("decode_attn_qkv", &decode_attn_qkv);
  m.impl("decode_attn_qkv_out", &decode_attn_qkv_out);
  m.impl("decode_attn_rope_qkv", &decode_attn_rope_qkv);
  m.impl("decode_attn_rope_linear", &decode_attn_rope_linear);
  m.impl("kv_append_qkv_", &kv_append_qkv_);
  m.impl("decode_attn_q_rope", &decode_attn_q_rope);
  m.impl("mixed_row_tables", &mixed_row_tables);
  m.impl("prefill_attn_qkv", &prefill_attn_qkv);
  m.impl("prompt_rows_layer", &prompt_rows_layer);
  m.impl("prefill_attn", &prefill_attn);
  m.impl("decode_load", &decode_load);
  m.impl("decode_begin", &decode_begin);
  m.impl("decode_advance_", &decode_advance_);
  m.impl("sample", &sample);
  m.impl("rows_linear_parts", &rows_linear_parts);
  m.impl("rows_linear", &rows_linear);
  m.impl("rows_linear_silu", &rows_linear_silu);
  m.impl("rows_linear_relu2", &rows_linear_relu2);
  m.impl("rows_tall", &rows_tall);
  m.impl("rows_norm_linear", &rows_norm_linear);
  m.impl("rows_linear_streams_", &rows_linear_streams_);
  m.impl("rows_linear_scaled_relu2", &rows_linear_scaled_relu2);
  m.impl("tile_linear_parts", &tile_linear_parts);
  m.impl("tile_linear", &tile_linear);
  m.impl("tile_linear_silu", &tile_linear_silu);
  m.impl("tile_linear_relu2", &tile_linear_relu2);
  m.impl("skinny_linear", &skinny_linear);
  m.impl("skinny2_linear", &skinny2_linear);
  m.impl("skinny2_silu_linear", &skinny2_silu_linear);
  m.impl("stream_probe", &stream_probe);
  m.impl("prefill_paged_attn", &prefill_paged_attn);
  m.impl("mixed_attn_qkv", &mixed_attn_qkv);
}
