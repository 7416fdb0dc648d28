// Python binding of the per-layer calls: tensors in, the checks and the C ABI
// call in native code. A decode layer is two kernels of 2-7 us at a small batch,
// and the wrappers' shape checks, stride reads and 25-argument foreign calls cost
// more than that on the host in Python (33 us a layer).
//
// `stream` is the raw handle of torch's current stream on the tensors' device.
// Errors are RuntimeError with the same messages wherever the call came from.
#include <torch/extension.h>

#include <optional>
#include <tuple>

#include "infrared_amd.h"

namespace {

using at::Tensor;
using OptTensor = std::optional<Tensor>;

template <typename... Msg>
void require(bool cond, const Msg&... msg) {
  if (!cond) throw std::runtime_error(c10::str(msg...));
}

void check(int rc, const char* what) {
  if (rc != 0) throw std::runtime_error(c10::str(what, " failed (code ", rc, "): ", ir_last_error()));
}

void require_device(std::initializer_list<const Tensor*> ts) {
  const Tensor* first = nullptr;
  for (const Tensor* t : ts) {
    if (!t->is_cuda())
      throw std::runtime_error(
          c10::str("infrared_amd runs on ROCm device tensors only; got a tensor on ", t->device()));
    if (!first)
      first = t;
    else if (t->device() != first->device())
      throw std::runtime_error(c10::str("tensors on different devices: ", first->device(), " and ", t->device()));
  }
}

int dtype_code(const Tensor& t) {
  switch (t.scalar_type()) {
    case at::kFloat: return IR_DTYPE_F32;
    case at::kHalf: return IR_DTYPE_F16;
    case at::kBFloat16: return IR_DTYPE_BF16;
    default:
      throw std::runtime_error(c10::str("dtype ", t.scalar_type(), " is not supported (float32, float16, bfloat16)"));
  }
}

void unit_last(const char* name, const Tensor& t) {
  require(t.dim() > 0 && t.stride(-1) == 1, name, ": the last (head_dim) dimension must be contiguous");
}

void cache_layer(const char* name, const Tensor& c) {
  require(c.dim() == 3, name, ": expected one pool layer [num_slots, num_kv_heads, head_dim]");
  unit_last(name, c);
}

void check_tables(const char* name, const Tensor& bt, const Tensor& ctx) {
  require(bt.scalar_type() == at::kInt && bt.dim() == 2 && bt.stride(1) == 1, name,
          ": block_tables must be int32 [B, max_blocks] with contiguous rows");
  require(ctx.scalar_type() == at::kInt && ctx.dim() == 1 && ctx.size(0) == bt.size(0), name,
          ": context_lens must be int32 [B]");
  require(ctx.is_contiguous(), name, ": context_lens must be contiguous");
}

// A block size the C ABI's int holds (truncated it could divide by zero here).
void check_block_size(const char* name, int64_t block_size) {
  require(block_size > 0 && block_size <= INT32_MAX, name, "block_size must be positive and fit 32 bits, got ",
          block_size);
}

void* ptr(const OptTensor& t) { return t ? t->data_ptr() : nullptr; }
ir_stream_t stream_of(int64_t s) { return (ir_stream_t)(intptr_t)s; }

Tensor scratch(const OptTensor& given, int64_t need, const Tensor& like) {
  if (given && given->numel() >= need) return *given;
  return at::empty({need}, like.options().dtype(at::kByte));
}

Tensor counters_for(const OptTensor& given, int64_t n, const Tensor& like) {
  if (!given) return at::zeros({std::max<int64_t>(n, 1)}, like.options().dtype(at::kInt));
  require(given->scalar_type() == at::kInt && given->is_contiguous() && given->numel() >= n,
          "decode counters must be a contiguous int32 tensor of >= ", n, " zeros");
  return *given;
}

void kv_scatter(const Tensor& kc, const Tensor& vc, const Tensor& k, const Tensor& v, const Tensor& slots,
                const OptTensor& err, int64_t stream) {
  require_device({&kc, &vc, &k, &v, &slots});
  cache_layer("kv_scatter", kc);
  require(vc.sizes() == kc.sizes() && vc.strides() == kc.strides(),
          "kv_scatter: k_cache and v_cache must have the same shape and strides");
  require(k.dim() == 3 && v.sizes() == k.sizes() && k.size(1) == kc.size(1) && k.size(2) == kc.size(2),
          "kv_scatter: k ", k.sizes(), " / v ", v.sizes(), " do not match pool rows ", kc.sizes().slice(1));
  require(k.scalar_type() == kc.scalar_type() && v.scalar_type() == kc.scalar_type(), "kv_scatter: dtype mismatch (",
          k.scalar_type(), ", ", v.scalar_type(), " vs pool ", kc.scalar_type(), ")");
  const int64_t n = k.size(0);
  require(slots.scalar_type() == at::kLong && slots.dim() == 1 && slots.size(0) == n,
          "kv_scatter: slots must be int64 [", n, "], got ", slots.scalar_type(), " ", slots.sizes());
  unit_last("kv_scatter k", k);
  unit_last("kv_scatter v", v);
  const Tensor s = slots.contiguous();
  check(ir_kv_scatter(k.data_ptr(), k.stride(0), k.stride(1), v.data_ptr(), v.stride(0), v.stride(1), kc.data_ptr(),
                      vc.data_ptr(), kc.stride(0), kc.stride(1), kc.size(0), (const int64_t*)s.data_ptr(), n,
                      (int)k.size(1), (int)k.size(2), dtype_code(kc), (int32_t*)ptr(err), stream_of(stream)),
        "ir_kv_scatter");
}

Tensor paged_decode(const Tensor& q, const Tensor& kc, const Tensor& vc, const Tensor& bt, const Tensor& ctx,
                    int64_t block_size, double scale, const OptTensor& out_, int64_t partition,
                    const OptTensor& workspace, const OptTensor& err, const OptTensor& counters, int64_t stream) {
  require_device({&q, &kc, &vc, &bt, &ctx});
  cache_layer("paged_decode", kc);
  check_tables("paged_decode", bt, ctx);
  require(q.dim() == 3, "paged_decode: q must be [B, H_q, D], got ", q.sizes());
  check_block_size("paged_decode: ", block_size);
  const int b = (int)q.size(0), hq = (int)q.size(1), d = (int)q.size(2), h_kv = (int)kc.size(1);
  require(d == kc.size(2) && q.scalar_type() == kc.scalar_type() && vc.sizes() == kc.sizes(),
          "paged_decode: q / pool shape or dtype mismatch");
  require(bt.size(0) == b, "paged_decode: block_tables rows != batch");
  unit_last("paged_decode q", q);
  const Tensor out = out_ ? *out_ : at::empty({b, hq, d}, q.options());
  const int max_blocks = (int)bt.size(1), bs = (int)block_size;
  const int part = partition > 0 ? (int)partition : ir_paged_decode_default_partition(b, h_kv, max_blocks, bs);
  const int64_t need = ir_paged_decode_workspace_size(b, hq, h_kv, d, max_blocks, bs, part);
  Tensor ws, ctr;
  int64_t n_ctr = 0;
  if (need > 0) {
    ws = scratch(workspace, need, q);
    n_ctr = ir_paged_decode_num_counters(b, hq, h_kv);
    ctr = counters_for(counters, n_ctr, q);
  }
  check(ir_paged_decode(q.data_ptr(), q.stride(0), q.stride(1), kc.data_ptr(), vc.data_ptr(), kc.stride(0),
                        kc.stride(1), kc.size(0) / bs, bs, (const int32_t*)bt.data_ptr(), bt.stride(0), max_blocks,
                        (const int32_t*)ctx.data_ptr(), out.data_ptr(), out.stride(0), out.stride(1), b, hq, h_kv, d,
                        (float)scale, dtype_code(q), part, need > 0 ? (int32_t*)ctr.data_ptr() : nullptr, n_ctr,
                        need > 0 ? ws.data_ptr() : nullptr, need, (int32_t*)ptr(err), stream_of(stream)),
        "ir_paged_decode");
  return out;
}

// `plan`: the fields of a decode plan in the order of its dataclass, buffer and
// dtype apart (num_seqs, num_q_heads, num_kv_heads, max_blocks, block_size,
// num_blocks, slot_stride, head_stride).
Tensor paged_decode_planned(const Tensor& q, const Tensor& kc, const Tensor& vc, const Tensor& plan_buf,
                            const std::tuple<int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t>& p,
                            at::ScalarType plan_dtype, int64_t flags, double scale, const OptTensor& out_,
                            const OptTensor& workspace, const OptTensor& err, const OptTensor& counters,
                            int64_t stream) {
  require_device({&q, &kc, &vc, &plan_buf});
  cache_layer("paged_decode_planned", kc);
  require(q.dim() == 3, "paged_decode_planned: q must be [B, H_q, D], got ", q.sizes());
  const auto& [seqs, p_hq, p_hkv, max_blocks, bs, num_blocks, slot_stride, head_stride] = p;
  check_block_size("paged_decode_planned: the plan's ", bs);
  const int b = (int)q.size(0), hq = (int)q.size(1), d = (int)q.size(2);
  require(b == seqs && hq == p_hq && kc.size(1) == p_hkv, "paged_decode_planned: q / pool heads differ from the plan's");
  require(kc.size(0) / bs == num_blocks && kc.stride(0) == slot_stride && kc.stride(1) == head_stride &&
              kc.scalar_type() == plan_dtype,
          "paged_decode_planned: pool layout differs from the plan's");
  require(vc.sizes() == kc.sizes() && vc.strides() == kc.strides(),
          "paged_decode_planned: v_cache must match k_cache's shape and strides");
  require(d == kc.size(2) && q.scalar_type() == kc.scalar_type(),
          "paged_decode_planned: q / pool shape or dtype mismatch");
  unit_last("paged_decode_planned q", q);
  const Tensor out = out_ ? *out_ : at::empty({b, hq, d}, q.options());
  const Tensor ws = scratch(workspace, ir_paged_decode_planned_workspace_bytes(b, hq, (int)p_hkv, d), q);
  const int64_t n_ctr = ir_paged_decode_num_counters(b, hq, (int)p_hkv);
  const Tensor ctr = counters_for(counters, n_ctr, q);
  check(ir_paged_decode_planned(q.data_ptr(), q.stride(0), q.stride(1), kc.data_ptr(), vc.data_ptr(), kc.stride(0),
                                out.data_ptr(), out.stride(0), out.stride(1), b, hq, (int)p_hkv, d, (int)max_blocks,
                                (int)bs, (float)scale, dtype_code(q), (int)flags, plan_buf.data_ptr(),
                                (int32_t*)ctr.data_ptr(), n_ctr, ws.data_ptr(), ws.numel(), (int32_t*)ptr(err),
                                stream_of(stream)),
        "ir_paged_decode_planned");
  return out;
}

Tensor paged_attention_masked(const Tensor& q, const Tensor& kc, const Tensor& vc, const Tensor& gs,
                              const Tensor& mask, double scale, const OptTensor& out_, const OptTensor& err,
                              const OptTensor& run_if, int64_t stream) {
  require_device({&q, &kc, &vc, &gs, &mask});
  cache_layer("paged_attention_masked", kc);
  require(q.dim() == 4, "paged_attention_masked: q must be [B, Sq, H_q, D], got ", q.sizes());
  const int b = (int)q.size(0), sq = (int)q.size(1), hq = (int)q.size(2), d = (int)q.size(3), h_kv = (int)kc.size(1);
  require(d == kc.size(2) && q.scalar_type() == kc.scalar_type(),
          "paged_attention_masked: q / pool shape or dtype mismatch");
  require(gs.scalar_type() == at::kLong && gs.dim() == 2 && gs.size(0) == b,
          "paged_attention_masked: gather_slots must be int64 [B, T]");
  const int t = (int)gs.size(1);
  require(mask.dim() == 4 && mask.size(1) == 1, "paged_attention_masked: mask must be [B, 1, Sq, T], got ",
          mask.sizes());
  const Tensor m = mask.expand({b, 1, sq, t});
  unit_last("paged_attention_masked q", q);
  const Tensor out = out_ ? *out_ : at::empty({b, sq, hq, d}, q.options());
  if (run_if) {
    require_device({&q, &*run_if});
    require(run_if->scalar_type() == at::kInt && run_if->numel() >= 1,
            "paged_attention_masked: run_if must be an int32 device tensor");
  }
  // a gated call of few columns takes its parts in one launch, without a workspace
  Tensor ws;
  if (h_kv > 0 && (!run_if || (int64_t)sq * (hq / h_kv) > IR_MASKED_FEW_COLUMNS)) {
    const int64_t need = ir_paged_attention_masked_workspace_size(b, sq, t, hq, h_kv, d, dtype_code(q), dtype_code(m),
                                                                  m.stride(3));
    if (need > 0) {
      try {
        ws = at::empty({need}, q.options().dtype(at::kByte));
      } catch (const c10::OutOfMemoryError&) {
        // a pool that leaves no room for it: one part, every tile, no workspace
      }
    }
  }
  check(ir_paged_attention_masked_ws(
            q.data_ptr(), q.stride(0), q.stride(1), q.stride(2), kc.data_ptr(), vc.data_ptr(), kc.stride(0),
            kc.stride(1), kc.size(0), (const int64_t*)gs.data_ptr(), gs.stride(0), gs.stride(1), m.data_ptr(),
            m.stride(0), m.stride(2), m.stride(3), dtype_code(m), out.data_ptr(), out.stride(0), out.stride(1),
            out.stride(2), b, sq, t, hq, h_kv, d, (float)scale, dtype_code(q), (int32_t*)ptr(err),
            (const int32_t*)ptr(run_if), ws.defined() ? ws.data_ptr() : nullptr, ws.defined() ? ws.numel() : 0,
            stream_of(stream)),
        "ir_paged_attention_masked");
  return out;
}

Tensor rope_kv_scatter(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& cos, const Tensor& sin,
                       const Tensor& kc, const Tensor& vc, const Tensor& slots, const OptTensor& q_out_,
                       const OptTensor& err, int64_t stream) {
  require_device({&q, &k, &v, &cos, &sin, &kc, &vc, &slots});
  cache_layer("rope_kv_scatter", kc);
  require(q.dim() == 3 && k.dim() == 3 && v.sizes() == k.sizes(),
          "rope_kv_scatter: q [N, H_q, D], k and v [N, H_kv, D] expected");
  const int64_t n = q.size(0), d = q.size(2);
  require(k.size(0) == n && k.size(2) == d && k.size(1) == kc.size(1) && d == kc.size(2),
          "rope_kv_scatter: k/v rows do not match q or the pool");
  require(q.scalar_type() == k.scalar_type() && k.scalar_type() == kc.scalar_type() &&
              v.scalar_type() == k.scalar_type(),
          "rope_kv_scatter: dtype mismatch");
  require(vc.strides() == kc.strides(), "rope_kv_scatter: k_cache and v_cache must share strides");
  for (const auto& [name, t] : {std::pair<const char*, const Tensor*>{"cos", &cos}, {"sin", &sin}})
    require(t->scalar_type() == at::kFloat && t->dim() == 2 && t->size(0) == n && t->size(1) == d && t->stride(1) == 1,
            "rope_kv_scatter: ", name, " must be fp32 [N, D] with unit column stride");
  require(cos.stride(0) == sin.stride(0), "rope_kv_scatter: cos and sin must share strides");
  require(slots.scalar_type() == at::kLong && slots.dim() == 1 && slots.size(0) == n,
          "rope_kv_scatter: slots must be int64 [N]");
  unit_last("rope_kv_scatter q", q);
  unit_last("rope_kv_scatter k", k);
  unit_last("rope_kv_scatter v", v);
  const Tensor qo = q_out_ ? *q_out_ : at::empty_like(q);
  const Tensor s = slots.contiguous();
  check(ir_rope_kv_scatter(q.data_ptr(), q.stride(0), q.stride(1), qo.data_ptr(), qo.stride(0), qo.stride(1),
                           k.data_ptr(), k.stride(0), k.stride(1), v.data_ptr(), v.stride(0), v.stride(1),
                           (const float*)cos.data_ptr(), (const float*)sin.data_ptr(), cos.stride(0), kc.data_ptr(),
                           vc.data_ptr(), kc.stride(0), kc.stride(1), kc.size(0), (const int64_t*)s.data_ptr(), n,
                           (int)q.size(1), (int)k.size(1), (int)d, dtype_code(q), (int32_t*)ptr(err),
                           stream_of(stream)),
        "ir_rope_kv_scatter");
  return qo;
}

Tensor paged_prefill(const Tensor& q, const Tensor& kc, const Tensor& vc, const Tensor& bt, const Tensor& cu,
                     const Tensor& q_start, int64_t max_q_len, int64_t block_size, double scale, const OptTensor& out_,
                     const OptTensor& err, const OptTensor& plan_buf, const OptTensor& kn, const OptTensor& vn,
                     const OptTensor& slots_, int64_t src_row0, int64_t stream) {
  require_device({&q, &kc, &vc, &bt, &cu, &q_start});
  cache_layer("paged_prefill", kc);
  require(q.dim() == 3, "paged_prefill: q must be [total_q, H_q, D], got ", q.sizes());
  check_block_size("paged_prefill: ", block_size);
  const int hq = (int)q.size(1), d = (int)q.size(2), h_kv = (int)kc.size(1);
  require(d == kc.size(2) && q.scalar_type() == kc.scalar_type() && vc.sizes() == kc.sizes(),
          "paged_prefill: q / pool shape or dtype mismatch");
  require(vc.strides() == kc.strides(), "paged_prefill: k_cache and v_cache must share strides");
  require(bt.scalar_type() == at::kInt && bt.dim() == 2 && bt.stride(1) == 1,
          "paged_prefill: block_tables must be int32 [B, max_blocks] with unit column stride");
  const int64_t b = bt.size(0);
  for (const auto& [name, t, n] : {std::tuple<const char*, const Tensor*, int64_t>{"cu_seqlens_q", &cu, b + 1},
                                   {"q_start", &q_start, b}})
    require(t->scalar_type() == at::kInt && t->dim() == 1 && t->size(0) == n && t->is_contiguous(),
            "paged_prefill: ", name, " must be contiguous int32 [", n, "]");
  unit_last("paged_prefill q", q);
  if (plan_buf) require_device({&q, &*plan_buf});
  const Tensor out = out_ ? *out_ : at::empty(q.sizes(), q.options());
  int64_t n_write = 0;
  Tensor slots;
  require(kn.has_value() == vn.has_value() && kn.has_value() == slots_.has_value(),
          "paged_prefill: new_kv must be (k, v, slots), each of them a tensor");
  if (kn) {
    require_device({&q, &*kn, &*vn, &*slots_});
    n_write = kn->size(0);
    require(kn->dim() == 3 && kn->size(1) == h_kv && kn->size(2) == d && vn->sizes() == kn->sizes() &&
                kn->scalar_type() == q.scalar_type() && vn->scalar_type() == q.scalar_type() &&
                slots_->scalar_type() == at::kLong && slots_->dim() == 1 && slots_->size(0) == n_write,
            "paged_prefill: new_kv must be (k, v [N, H_kv, D] of q's dtype, slots int64 [N])");
    unit_last("paged_prefill new k", *kn);
    unit_last("paged_prefill new v", *vn);
    slots = slots_->contiguous();
  }
  check(ir_paged_prefill(q.data_ptr(), q.stride(0), q.stride(1), kc.data_ptr(), vc.data_ptr(), kc.stride(0),
                         kc.stride(1), kc.size(0) / block_size, (int)block_size, (const int32_t*)bt.data_ptr(),
                         bt.stride(0), (int)bt.size(1), (const int32_t*)cu.data_ptr(),
                         (const int32_t*)q_start.data_ptr(), (int)b, (int)q.size(0), (int)max_q_len, out.data_ptr(),
                         out.stride(0), out.stride(1), hq, h_kv, d, (float)scale, dtype_code(q), ptr(plan_buf),
                         plan_buf ? plan_buf->numel() : 0, ptr(kn), kn ? kn->stride(0) : 0, kn ? kn->stride(1) : 0,
                         ptr(vn), vn ? vn->stride(0) : 0, vn ? vn->stride(1) : 0,
                         slots.defined() ? (const int64_t*)slots.data_ptr() : nullptr, n_write, src_row0,
                         (int32_t*)ptr(err), stream_of(stream)),
        "ir_paged_prefill");
  return out;
}

// The seam's forms of the calls above: k, v [B, Sq, H_kv, D], q and the result
// [B, 1, H_q, D].
void write_step(const Tensor& kc, const Tensor& vc, const Tensor& k, const Tensor& v, const Tensor& slots,
                const OptTensor& err, int64_t stream) {
  const int64_t h = k.size(-2), d = k.size(-1);
  kv_scatter(kc, vc, k.reshape({-1, h, d}), v.reshape({-1, h, d}), slots, err, stream);
}

Tensor decode_step(const Tensor& q, const Tensor& kc, const Tensor& vc, const Tensor& bt, const Tensor& ctx,
                   int64_t block_size, double scale, const OptTensor& out, const OptTensor& workspace,
                   const OptTensor& err, const OptTensor& counters, int64_t stream) {
  return paged_decode(q.select(1, 0), kc, vc, bt, ctx, block_size, scale, out, 0, workspace, err, counters, stream)
      .unsqueeze(1);
}

Tensor decode_step_planned(const Tensor& q, const Tensor& kc, const Tensor& vc, const Tensor& plan_buf,
                           const std::tuple<int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t>& p,
                           at::ScalarType plan_dtype, int64_t flags, double scale, const OptTensor& out,
                           const OptTensor& workspace, const OptTensor& err, const OptTensor& counters,
                           int64_t stream) {
  return paged_decode_planned(q.select(1, 0), kc, vc, plan_buf, p, plan_dtype, flags, scale, out, workspace, err,
                              counters, stream)
      .unsqueeze(1);
}

}  // namespace

PYBIND11_MODULE(_seam, m) {
  // (the calls release the interpreter lock, as foreign calls do: a launch can
  // wait for room in its queue)
  using nogil = pybind11::call_guard<pybind11::gil_scoped_release>;
  m.def("kv_scatter", &kv_scatter, nogil());
  m.def("paged_decode", &paged_decode, nogil());
  m.def("paged_decode_planned", &paged_decode_planned, nogil());
  m.def("paged_attention_masked", &paged_attention_masked, nogil());
  m.def("rope_kv_scatter", &rope_kv_scatter, nogil());
  m.def("paged_prefill", &paged_prefill, nogil());
  m.def("write_step", &write_step, nogil());
  m.def("decode_step", &decode_step, nogil());
  m.def("decode_step_planned", &decode_step_planned, nogil());
  m.def("decode_plan_bytes", &ir_paged_decode_plan_bytes);
  m.def("decode_workspace_size", &ir_paged_decode_workspace_size);
  m.def("decode_num_counters", &ir_paged_decode_num_counters);
  m.def("planned_workspace_bytes", &ir_paged_decode_planned_workspace_bytes);
}
