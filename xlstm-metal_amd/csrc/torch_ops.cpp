// The xlstm_hip::* torch operators in native code: shape and dtype checks, output allocation (torch's
// caching allocator) and the call through the C ABI, on the tensor's device and its current stream.
//
// Schemas and fake kernels are declared in xlstm_hip/ops.py, which loads this library.  Reason for being
// native: a call is 2-30 us of GPU work at one decoded token or a short prompt, and checks, allocations,
// ctypes and the Python operator wrapper took 25-40 us of host time per call (B1 NH8 DQK256 DV512 bf16
// decode step through the backend module: 38 us a call for a 5.5 us kernel, 17 us so; forward and backward
// at B2 NH8 S1024 DQK128 DV256 275 -> 106 us).
// Errors: bad arguments raise ValueError, unsupported ones NotImplementedError, launch and device errors
// RuntimeError, with the library's message.
#include <ATen/ATen.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <c10/core/DeviceGuard.h>
#include <torch/csrc/autograd/autograd_not_implemented_fallback.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/functions/basic_ops.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/library.h>

#include <optional>
#include <tuple>
#include <vector>

#include "xlstm_hip.h"

// Constants that xlstm_hip/ops.py reads: the backward's padding tokens; the most rows of lm_head_softcap and the
// LDS bytes its staged form has for rows * (D + 8) 16-bit values.
extern "C" {
extern const double xl_pad_i, xl_pad_f;
extern const int64_t xl_lm_head_max_rows, xl_lm_head_max_lds;
const double xl_pad_i = -3.0e4, xl_pad_f = 30.0;
const int64_t xl_lm_head_max_rows = 16, xl_lm_head_max_lds = 160 * 1024;
}

namespace {

using at::Tensor;
using OptTensor = std::optional<Tensor>;

#define XL_CHECK(cond, what, ...) TORCH_CHECK_VALUE(cond, what, ": ", __VA_ARGS__)

// Every given tensor on one GPU; the guard makes it current and st is its current stream.
struct Gpu {
  c10::OptionalDeviceGuard guard;
  void* st = nullptr;
  Gpu(const char* what, std::initializer_list<const Tensor*> tensors) {
    const Tensor* first = nullptr;
    for (const Tensor* t : tensors) {
      if (!t || !t->defined()) continue;
      TORCH_CHECK(t->is_cuda(), what, ": tensors must be on the GPU (got ", t->device(), "); there is no CPU path");
      if (!first) first = t;
      TORCH_CHECK(t->device() == first->device(), what, ": tensors on different devices (", first->device(), " vs ",
                  t->device(), ")");
    }
    guard.reset_device(first->device());
    st = (void*)c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(first->device().index()).stream();
  }
};

const Tensor* opt(const OptTensor& t) { return t.has_value() ? &*t : nullptr; }

// contiguous and 16-byte aligned
Tensor prep(const Tensor& t) {
  Tensor c = t.contiguous();
  return (uintptr_t)c.const_data_ptr() & 15u ? c.clone() : c;
}
Tensor prep(const OptTensor& t) { return t.has_value() && t->defined() ? prep(*t) : Tensor(); }
Tensor f32(const Tensor& t) { return prep(t.scalar_type() == at::kFloat ? t : t.to(at::kFloat)); }
Tensor f32(const OptTensor& t) { return t.has_value() && t->defined() ? f32(*t) : Tensor(); }

template <typename T = void>
T* ptr(const Tensor& t) {
  return t.defined() ? (T*)t.data_ptr() : nullptr;
}

int dtype_code(const Tensor& t, const char* what) {
  switch (t.scalar_type()) {
    case at::kFloat: return XL_DTYPE_F32;
    case at::kBFloat16: return XL_DTYPE_BF16;
    case at::kHalf: return XL_DTYPE_F16;
    default: break;
  }
  TORCH_CHECK_VALUE(false, what, ": unsupported dtype ", t.scalar_type(), " (float32, bfloat16, float16)");
}

void check_rc(int rc, const char* what) {
  if (rc == XL_OK) return;
  const char* msg = xl_last_error();
  TORCH_CHECK_VALUE(rc != XL_ERR_INVALID_ARG, what, ": ", msg, " (invalid argument)");
  TORCH_CHECK_NOT_IMPLEMENTED(rc != XL_ERR_UNSUPPORTED, what, ": ", msg, " (unsupported)");
  TORCH_CHECK(rc != XL_ERR_WORKSPACE, what, ": ", msg, " (workspace)");
  TORCH_CHECK(rc != XL_ERR_LAUNCH, what, ": ", msg, " (launch)");
  TORCH_CHECK(false, what, ": ", msg, " (code ", rc, ")");
}

at::TensorOptions f32_on(const Tensor& t) { return t.options().dtype(at::kFloat); }
Tensor like(const Tensor& t) { return at::empty(t.sizes(), t.options()); }
int i32(int64_t v, const char* what) {
  XL_CHECK(v >= INT32_MIN && v <= INT32_MAX, what, "size ", v, " out of range");
  return (int)v;
}

// ------------------------------------------------------------------ soft_cap
Tensor soft_cap(const Tensor& x_, double cap) {
  const char* what = "soft_cap";
  Gpu gpu(what, {&x_});
  const Tensor x = prep(x_), y = like(x);
  check_rc(xl_soft_cap_fwd(ptr(x), ptr(y), x.numel(), (float)cap, dtype_code(x, what), gpu.st), what);
  return y;
}

// ---------------------------------------------------------------- mLSTM step
struct StepShape {
  int64_t B, NH, DQK, DV;
};
StepShape step_shapes(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& i, const Tensor& f, const Tensor& c,
                      const Tensor& n, const Tensor& m, const char* what) {
  XL_CHECK(q.dim() == 3, what, "q must be (B, NH, DHQK), got ", q.sizes());
  const int64_t B = q.size(0), NH = q.size(1), DQK = q.size(2);
  XL_CHECK(k.sizes() == q.sizes(), what, "q and k must have the same shape");
  XL_CHECK(v.dim() == 3 && v.size(0) == B && v.size(1) == NH, what, "v must be (B, NH, DHV), got ", v.sizes());
  const int64_t DV = v.size(2);
  XL_CHECK(q.scalar_type() == k.scalar_type() && k.scalar_type() == v.scalar_type(), what, "q, k, v must share a dtype");
  XL_CHECK(c.sizes() == at::IntArrayRef({B, NH, DQK, DV}), what, "matC_old has wrong shape, got ", c.sizes());
  XL_CHECK(n.sizes() == at::IntArrayRef({B, NH, DQK}), what, "vecN_old has wrong shape, got ", n.sizes());
  XL_CHECK(m.numel() == B * NH, what, "scaM_old has wrong shape, got ", m.sizes());
  XL_CHECK(i.numel() == B * NH, what, "scaI has wrong shape, got ", i.sizes());
  XL_CHECK(f.numel() == B * NH, what, "scaF has wrong shape, got ", f.sizes());
  XL_CHECK(i.scalar_type() == f.scalar_type(), what, "i and f must share a dtype");
  return {B, NH, DQK, DV};
}

// c_new: where C' goes (c itself for the in-place step)
std::tuple<Tensor, Tensor, Tensor> launch_step(const Tensor& q_, const Tensor& k_, const Tensor& v_, const Tensor& i_,
                                               const Tensor& f_, const Tensor& c, const Tensor& n_, const Tensor& m_,
                                               const Tensor& c_new, const StepShape& s, double eps, double qk_scale,
                                               const Gpu& gpu, const char* what) {
  const Tensor q = prep(q_), k = prep(k_), v = prep(v_), i = prep(i_), f = prep(f_), n = f32(n_), m = f32(m_);
  const Tensor h = at::empty({s.B, s.NH, s.DV}, q.options());
  const Tensor n_new = at::empty({s.B, s.NH, s.DQK}, f32_on(q)), m_new = at::empty({s.B, s.NH, 1}, f32_on(q));
  check_rc(xl_mlstm_step_fwd(ptr(q), ptr(k), ptr(v), ptr(i), ptr(f), ptr<float>(c), ptr<float>(n), ptr<float>(m), ptr(h),
                             ptr<float>(c_new), ptr<float>(n_new), ptr<float>(m_new), i32(s.B, what), i32(s.NH, what),
                             i32(s.DQK, what), i32(s.DV, what), (float)qk_scale, (float)eps, dtype_code(q, what),
                             dtype_code(i, what), gpu.st),
           what);
  return {h, n_new, m_new};
}

std::tuple<Tensor, Tensor, Tensor, Tensor> mlstm_step(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& i,
                                                      const Tensor& f, const Tensor& c_, const Tensor& n, const Tensor& m,
                                                      double eps, double qk_scale) {
  const char* what = "mlstm_step";
  Gpu gpu(what, {&q, &k, &v, &i, &f, &c_, &n, &m});
  const StepShape s = step_shapes(q, k, v, i, f, c_, n, m, what);
  const Tensor c = f32(c_), c_new = at::empty({s.B, s.NH, s.DQK, s.DV}, f32_on(q));
  auto [h, n_new, m_new] = launch_step(q, k, v, i, f, c, n, m, c_new, s, eps, qk_scale, gpu, what);
  return {h, c_new, n_new, m_new};
}

std::tuple<Tensor, Tensor, Tensor> mlstm_step_(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& i,
                                               const Tensor& f, const Tensor& c, const Tensor& n, const Tensor& m,
                                               double eps, double qk_scale) {
  const char* what = "mlstm_step_";
  Gpu gpu(what, {&q, &k, &v, &i, &f, &c, &n, &m});
  const StepShape s = step_shapes(q, k, v, i, f, c, n, m, what);
  XL_CHECK(c.scalar_type() == at::kFloat && c.is_contiguous() && ((uintptr_t)c.const_data_ptr() & 15u) == 0, what,
           "in-place C must be a contiguous, 16-byte aligned float32 tensor");
  return launch_step(q, k, v, i, f, c, n, m, c, s, eps, qk_scale, gpu, what);
}

// -------------------------------------------------------- chunkwise / sequence
struct SeqShape {
  int64_t B, NH, S, DQK, DV;
};
SeqShape seq_shapes(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& i, const Tensor& f,
                    const OptTensor& c0, const OptTensor& n0, const OptTensor& m0, const char* what) {
  XL_CHECK(q.dim() == 4, what, "q must be (B, NH, S, DHQK), got ", q.sizes());
  const int64_t B = q.size(0), NH = q.size(1), S = q.size(2), DQK = q.size(3);
  XL_CHECK(k.sizes() == q.sizes(), what, "q and k must have the same shape");
  XL_CHECK(v.dim() == 4 && v.size(0) == B && v.size(1) == NH && v.size(2) == S, what, "v must be (B, NH, S, DHV), got ",
           v.sizes());
  const int64_t DV = v.size(3);
  XL_CHECK(q.scalar_type() == k.scalar_type() && k.scalar_type() == v.scalar_type(), what, "q, k, v must share a dtype");
  const at::IntArrayRef g = q.sizes().slice(0, 3);
  XL_CHECK(i.sizes() == g && f.sizes() == g, what, "i and f must be (B, NH, S)");
  XL_CHECK(i.scalar_type() == f.scalar_type(), what, "i and f must share a dtype");
  const bool c = opt(c0), n = opt(n0), m = opt(m0);
  XL_CHECK(c == n && n == m, what, "Initial states must be provided together.");
  if (c) {
    XL_CHECK(c0->sizes() == at::IntArrayRef({B, NH, DQK, DV}), what, "c_initial has wrong shape, got ", c0->sizes());
    XL_CHECK(n0->sizes() == at::IntArrayRef({B, NH, DQK}), what, "n_initial has wrong shape, got ", n0->sizes());
    XL_CHECK(m0->numel() == B * NH, what, "m_initial has wrong shape, got ", m0->sizes());
  }
  return {B, NH, S, DQK, DV};
}

// the last states, or three distinct empties (operator outputs may not alias each other)
std::tuple<Tensor, Tensor, Tensor> state_outs(bool ret, const SeqShape& s, const Tensor& q) {
  const auto o = f32_on(q);
  if (!ret) return {at::empty({0}, o), at::empty({0}, o), at::empty({0}, o)};
  return {at::empty({s.B, s.NH, s.DQK, s.DV}, o), at::empty({s.B, s.NH, s.DQK}, o), at::empty({s.B, s.NH, 1}, o)};
}

// {batch, head, row} strides of each [B, NH, S, D] tensor for the pipelined kernel; false where one of them
// has to be copied: columns contiguous, 16-byte rows and base, rows apart
bool row_strides(std::initializer_list<const Tensor*> tensors, int64_t (&out)[9]) {
  int at = 0;
  for (const Tensor* t : tensors) {
    const int64_t b = t->size(0) > 1 ? t->stride(0) : 0, h = t->size(1) > 1 ? t->stride(1) : 0, r = t->stride(2);
    if (t->stride(3) != 1 || ((b | h | r) & 7) || r < t->size(3) || r > (1 << 22) ||
        ((uintptr_t)t->const_data_ptr() & 15u))
      return false;
    out[at++] = b;
    out[at++] = h;
    out[at++] = r;
  }
  return true;
}

using FourTensors = std::tuple<Tensor, Tensor, Tensor, Tensor>;

FourTensors mlstm_chunkwise(const Tensor& q_, const Tensor& k_, const Tensor& v_, const Tensor& i_, const Tensor& f_,
                            const OptTensor& c0_, const OptTensor& n0_, const OptTensor& m0_, double qk_scale,
                            int64_t chunk_size, double eps, bool return_last_states, int64_t algo) {
  const char* what = "mlstm_chunkwise";
  Gpu gpu(what, {&q_, &k_, &v_, &i_, &f_, opt(c0_), opt(n0_), opt(m0_)});
  const SeqShape s = seq_shapes(q_, k_, v_, i_, f_, c0_, n0_, m0_, what);
  XL_CHECK(chunk_size > 0 && (s.S % chunk_size == 0 || algo == XL_CHUNKWISE_FUSED || algo == XL_CHUNKWISE_PIPELINED), what,
           "Sequence length ", s.S, " is not divisible by chunk size ", chunk_size, ".");
  const int dq = dtype_code(q_, what);
  const int B = i32(s.B, what), NH = i32(s.NH, what), S = i32(s.S, what), DQK = i32(s.DQK, what), DV = i32(s.DV, what),
            L = i32(chunk_size, what), al = i32(algo, what);
  // q, k, v as a projection's permuted views: the pipelined kernel reads them in place
  int64_t strides[9];
  const bool strided = dq != XL_DTYPE_F32 && !(q_.is_contiguous() && k_.is_contiguous() && v_.is_contiguous()) &&
                       row_strides({&q_, &k_, &v_}, strides) &&
                       xl_mlstm_chunkwise_algo(B, NH, S, DQK, DV, L, dq, al) == XL_CHUNKWISE_PIPELINED;
  const Tensor q = strided ? q_ : prep(q_), k = strided ? k_ : prep(k_), v = strided ? v_ : prep(v_);
  const Tensor i = prep(i_), f = prep(f_), c0 = f32(c0_), n0 = f32(n0_), m0 = f32(m0_);
  const Tensor h = at::empty({s.B, s.NH, s.S, s.DV}, q.options());
  auto [cl, nl, ml] = state_outs(return_last_states, s, q);
  const size_t ws_bytes = xl_mlstm_chunkwise_workspace_size(B, NH, S, DQK, DV, L, dq, al);
  const Tensor ws = ws_bytes ? at::empty({(int64_t)ws_bytes}, q.options().dtype(at::kByte)) : Tensor();
  float* last[3] = {return_last_states ? ptr<float>(cl) : nullptr, return_last_states ? ptr<float>(nl) : nullptr,
                    return_last_states ? ptr<float>(ml) : nullptr};
  const int dg = dtype_code(i, what);
  const int rc =
      strided ? xl_mlstm_chunkwise_fwd_strided(ptr(q), ptr(k), ptr(v), strides, ptr(i), ptr(f), ptr<float>(c0),
                                               ptr<float>(n0), ptr<float>(m0), ptr(h), last[0], last[1], last[2], B, NH, S,
                                               DQK, DV, L, (float)qk_scale, (float)eps, dq, dg, al, ptr(ws), ws_bytes, gpu.st)
              : xl_mlstm_chunkwise_fwd(ptr(q), ptr(k), ptr(v), ptr(i), ptr(f), ptr<float>(c0), ptr<float>(n0),
                                       ptr<float>(m0), ptr(h), last[0], last[1], last[2], B, NH, S, DQK, DV, L,
                                       (float)qk_scale, (float)eps, dq, dg, al, ptr(ws), ws_bytes, gpu.st);
  check_rc(rc, what);
  return {h, cl, nl, ml};
}

std::tuple<Tensor, Tensor, Tensor, Tensor, Tensor, Tensor> mlstm_chunkwise_bwd(
    const Tensor& q_, const Tensor& k_, const Tensor& v_, const Tensor& i_, const Tensor& f_, const OptTensor& c0_,
    const OptTensor& n0_, const OptTensor& m0_, const Tensor& dh_, const OptTensor& dc_last, double qk_scale,
    int64_t chunk_size, double eps) {
  const char* what = "mlstm_chunkwise_bwd";
  Gpu gpu(what, {&q_, &k_, &v_, &i_, &f_, opt(c0_), opt(n0_), opt(m0_), &dh_, opt(dc_last)});
  const SeqShape s = seq_shapes(q_, k_, v_, i_, f_, c0_, n0_, m0_, what);
  XL_CHECK(dh_.sizes() == at::IntArrayRef({s.B, s.NH, s.S, s.DV}), what, "dh must be (B, NH, S, DHV), got ", dh_.sizes());
  XL_CHECK(!opt(dc_last) || dc_last->sizes() == at::IntArrayRef({s.B, s.NH, s.DQK, s.DV}), what,
           "dC_last must be (B, NH, DHQK, DHV)");
  XL_CHECK(chunk_size > 0 && s.S % chunk_size == 0, what, "Sequence length ", s.S, " is not divisible by chunk size ",
           chunk_size, ".");
  const Tensor q = prep(q_), k = prep(k_), v = prep(v_), i = prep(i_), f = prep(f_);
  const Tensor dh = prep(dh_.scalar_type() == q.scalar_type() ? dh_ : dh_.to(q.scalar_type()));
  const Tensor c0 = f32(c0_), n0 = f32(n0_), m0 = f32(m0_), dcl = f32(dc_last);
  const Tensor dq = like(q), dk = like(k), dv = like(v), di = like(i), df = like(f);
  const Tensor dc0 = c0.defined() ? like(c0) : at::empty({0}, f32_on(q));
  const int B = i32(s.B, what), NH = i32(s.NH, what), S = i32(s.S, what), DQK = i32(s.DQK, what), DV = i32(s.DV, what),
            L = i32(chunk_size, what);
  const size_t ws_bytes = xl_mlstm_chunkwise_bwd_workspace_size(B, NH, S, DQK, DV, L);
  XL_CHECK(ws_bytes > 0, what, "unsupported shape or chunk_size ", chunk_size, " (16, 32 or 64)");
  const Tensor ws = at::empty({(int64_t)ws_bytes}, q.options().dtype(at::kByte));
  check_rc(xl_mlstm_chunkwise_bwd(ptr(q), ptr(k), ptr(v), ptr(i), ptr(f), ptr<float>(c0), ptr<float>(n0), ptr<float>(m0),
                                  ptr(dh), ptr<float>(dcl), ptr(dq), ptr(dk), ptr(dv), ptr(di), ptr(df),
                                  c0.defined() ? ptr<float>(dc0) : nullptr, B, NH, S, DQK, DV, L, (float)qk_scale,
                                  (float)eps, dtype_code(q, what), dtype_code(i, what), ptr(ws), ws_bytes, gpu.st),
           what);
  return {dq, dk, dv, di, df, dc0};
}

// Gradients of (h, C_last) through the reference's custom backward; those of n_last and m_last are dropped
// and the initial n and m get zeros, as there (bw.py:340-342).
//
// The backward kernels take chunk sizes 16, 32 and 64 and whole chunks.  The custom backward's gradients
// do not depend on the chunk size (tests/test_oracle_chunkwise_bw.py::test_chunk_size_invariant), so any other
// size runs at 64, and so does a sequence that the single-pass forward took with a ragged last chunk,
// padded to whole 64-token chunks with state-preserving tokens whose gradients are dropped: an input gate
// of xl_pad_i makes exp(i - m) = 0 and leaves every stabiliser alone, logsigmoid(xl_pad_f) = -9.4e-14 makes the
// forget factor 1 to float32 precision, so (C, n, m) and the last state's gradient pass through them
// unchanged (read by ops._PAD_I, ops._PAD_F; test_state_preserving_padding).

// Sizes stay symbolic from here to the backward's results: a traced training step then serves every
// sequence length (the kernels above get plain integers from the dispatcher).
FourTensors call_chunkwise(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& i, const Tensor& f,
                           const OptTensor& c0, const OptTensor& n0, const OptTensor& m0, double qk_scale,
                           c10::SymInt chunk, double eps, bool ret, c10::SymInt algo) {
  static const auto op = c10::Dispatcher::singleton().findSchemaOrThrow("xlstm_hip::mlstm_chunkwise", "")
                             .typed<decltype(call_chunkwise)>();
  at::AutoDispatchBelowADInplaceOrView below;
  return op.call(q, k, v, i, f, c0, n0, m0, qk_scale, chunk, eps, ret, algo);
}

using SixTensors = std::tuple<Tensor, Tensor, Tensor, Tensor, Tensor, Tensor>;
using ChunkwiseBwd = SixTensors(const Tensor&, const Tensor&, const Tensor&, const Tensor&, const Tensor&, const OptTensor&,
                                const OptTensor&, const OptTensor&, const Tensor&, const OptTensor&, double, c10::SymInt,
                                double);

struct ChunkwiseFn : public torch::autograd::Function<ChunkwiseFn> {
  static torch::autograd::variable_list forward(torch::autograd::AutogradContext* ctx, const Tensor& q, const Tensor& k,
                                                const Tensor& v, const Tensor& i, const Tensor& f, const OptTensor& c0,
                                                const OptTensor& n0, const OptTensor& m0, double qk_scale,
                                                c10::SymInt chunk, double eps, bool ret, c10::SymInt algo) {
    ctx->save_for_backward({q, k, v, i, f, c0.value_or(Tensor()), n0.value_or(Tensor()), m0.value_or(Tensor())});
    ctx->saved_data["qk_scale"] = qk_scale;
    ctx->saved_data["chunk"] = chunk;
    ctx->saved_data["eps"] = eps;
    ctx->saved_data["ret"] = ret;
    ctx->set_materialize_grads(false);
    auto [h, C, n, m] = call_chunkwise(q, k, v, i, f, c0, n0, m0, qk_scale, chunk, eps, ret, algo);
    return {h, C, n, m};
  }

  static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx,
                                                 torch::autograd::variable_list grads) {
    static const auto bwd = c10::Dispatcher::singleton().findSchemaOrThrow("xlstm_hip::mlstm_chunkwise_bwd", "")
                                .typed<ChunkwiseBwd>();
    auto saved = ctx->get_saved_variables();
    Tensor q = saved[0], k = saved[1], v = saved[2], i = saved[3], f = saved[4];
    const Tensor c0 = saved[5], n0 = saved[6], m0 = saved[7];
    auto given = [](const Tensor& t) { return t.defined() ? OptTensor(t) : OptTensor(); };
    const c10::SymInt S = q.sym_size(2);
    Tensor dh = grads[0];
    if (!dh.defined()) dh = at::zeros_symint({q.sym_size(0), q.sym_size(1), S, v.sym_size(3)}, q.options());
    const OptTensor dcl = ctx->saved_data["ret"].toBool() ? given(grads[1]) : OptTensor();
    int64_t L = ctx->saved_data["chunk"].toSymInt().guard_int(__FILE__, __LINE__);
    if ((L != 16 && L != 32 && L != 64) || S % L != 0) L = 64;
    const bool ragged = S % L != 0;
    if (ragged) {
      const c10::SymInt pad = L - S % L;
      for (Tensor* t : {&q, &k, &v, &dh}) *t = at::constant_pad_nd_symint(*t, {0, 0, 0, pad});
      i = at::constant_pad_nd_symint(i, {0, pad}, xl_pad_i);
      f = at::constant_pad_nd_symint(f, {0, pad}, xl_pad_f);
    }
    auto [dq, dk, dv, di, df, dc0] = bwd.call(q, k, v, i, f, given(c0), given(n0), given(m0), dh, dcl,
                                              ctx->saved_data["qk_scale"].toDouble(), L, ctx->saved_data["eps"].toDouble());
    if (ragged)
      for (Tensor* t : {&dq, &dk, &dv, &di, &df}) *t = t->slice_symint(2, 0, S).contiguous();
    const Tensor none;
    return {dq,
            dk,
            dv,
            di,
            df,
            c0.defined() ? dc0.to(c0.scalar_type()) : none,
            n0.defined() ? at::zeros_like(n0) : none,
            m0.defined() ? at::zeros_like(m0) : none,
            none,
            none,
            none,
            none,
            none};
  }
};

FourTensors mlstm_chunkwise_autograd(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& i, const Tensor& f,
                                     const OptTensor& c0, const OptTensor& n0, const OptTensor& m0, double qk_scale,
                                     c10::SymInt chunk, double eps, bool ret, c10::SymInt algo) {
  auto wants = [](const Tensor* t) { return t && t->defined() && (t->requires_grad() || t->_fw_grad(0).defined()); };
  bool any = false;
  for (const Tensor* t : {&q, &k, &v, &i, &f, opt(c0), opt(n0), opt(m0)}) any = any || wants(t);
  if (!any) return call_chunkwise(q, k, v, i, f, c0, n0, m0, qk_scale, chunk, eps, ret, algo);
  const auto r = ChunkwiseFn::apply(q, k, v, i, f, c0, n0, m0, qk_scale, chunk, eps, ret, algo);
  return {r[0], r[1], r[2], r[3]};
}

FourTensors mlstm_sequence(const Tensor& q_, const Tensor& k_, const Tensor& v_, const Tensor& i_, const Tensor& f_,
                           const OptTensor& c0_, const OptTensor& n0_, const OptTensor& m0_, double qk_scale, double eps,
                           bool return_last_states) {
  const char* what = "mlstm_sequence";
  Gpu gpu(what, {&q_, &k_, &v_, &i_, &f_, opt(c0_), opt(n0_), opt(m0_)});
  const SeqShape s = seq_shapes(q_, k_, v_, i_, f_, c0_, n0_, m0_, what);
  const Tensor q = prep(q_), k = prep(k_), v = prep(v_), i = prep(i_), f = prep(f_);
  const Tensor c0 = f32(c0_), n0 = f32(n0_), m0 = f32(m0_);
  const Tensor h = at::empty({s.B, s.NH, s.S, s.DV}, q.options());
  auto [cl, nl, ml] = state_outs(return_last_states, s, q);
  check_rc(xl_mlstm_sequence_fwd(ptr(q), ptr(k), ptr(v), ptr(i), ptr(f), ptr<float>(c0), ptr<float>(n0), ptr<float>(m0),
                                 ptr(h), return_last_states ? ptr<float>(cl) : nullptr,
                                 return_last_states ? ptr<float>(nl) : nullptr, return_last_states ? ptr<float>(ml) : nullptr,
                                 i32(s.B, what), i32(s.NH, what), i32(s.S, what), i32(s.DQK, what), i32(s.DV, what),
                                 (float)qk_scale, (float)eps, dtype_code(q, what), dtype_code(i, what), gpu.st),
           what);
  return {h, cl, nl, ml};
}

// ------------------------------------------------------------------- sLSTM
at::ScalarType slstm_dtype(const Tensor& z, const Tensor& i, const Tensor* c) {
  const auto t = at::promote_types(z.scalar_type(), i.scalar_type());
  return c ? at::promote_types(t, c->scalar_type()) : t;
}

std::tuple<Tensor, Tensor> slstm_step(const Tensor& z_, const Tensor& i_, const Tensor& f_, const Tensor& o_,
                                      const Tensor& c_, const Tensor& n_, const Tensor& m_, double eps) {
  const char* what = "slstm_step";
  Gpu gpu(what, {&z_, &i_, &f_, &o_, &c_, &n_, &m_});
  XL_CHECK(z_.dim() == 3, what, "z must be (B, NH, H), got ", z_.sizes());
  const int64_t B = z_.size(0), NH = z_.size(1), H = z_.size(2), per = B * NH * H;
  const at::IntArrayRef bn = z_.sizes().slice(0, 2);
  XL_CHECK(i_.sizes() == bn, what, "i_preact must be (B, NH), got ", i_.sizes());
  XL_CHECK(f_.sizes() == bn, what, "f_preact must be (B, NH), got ", f_.sizes());
  XL_CHECK(o_.sizes() == bn, what, "o_preact must be (B, NH), got ", o_.sizes());
  XL_CHECK(m_.sizes() == bn, what, "m_state must be (B, NH), got ", m_.sizes());
  XL_CHECK(c_.sizes() == z_.sizes() && n_.sizes() == z_.sizes(), what, "c_state and n_state must be (B, NH, H)");
  XL_CHECK(i_.scalar_type() == f_.scalar_type() && f_.scalar_type() == o_.scalar_type(), what, "gates must share a dtype");
  const auto out = slstm_dtype(z_, i_, &c_);
  const Tensor z = prep(z_), i = prep(i_), f = prep(f_), o = prep(o_), c = f32(c_), n = f32(n_), m = f32(m_);
  const Tensor h = at::empty({B, NH, H}, z.options().dtype(out)), st = at::empty({2 * per + B * NH}, f32_on(z));
  float* s = ptr<float>(st);
  check_rc(xl_slstm_step_fwd(ptr(z), ptr(i), ptr(f), ptr(o), ptr<float>(c), ptr<float>(n), ptr<float>(m), ptr(h), s, s + per,
                             s + 2 * per, i32(B, what), i32(NH, what), i32(H, what), (float)eps, dtype_code(z, what),
                             dtype_code(i, what), dtype_code(h, what), gpu.st),
           what);
  return {h, out == at::kFloat ? st : st.to(out)};
}

std::tuple<Tensor, Tensor> slstm_sequence(const Tensor& z_, const Tensor& i_, const Tensor& f_, const Tensor& o_,
                                          const OptTensor& c0_, const OptTensor& n0_, const OptTensor& m0_, double eps) {
  const char* what = "slstm_sequence";
  Gpu gpu(what, {&z_, &i_, &f_, &o_, opt(c0_), opt(n0_), opt(m0_)});
  XL_CHECK(z_.dim() == 4, what, "z must be (B, S, NH, H), got ", z_.sizes());
  const int64_t B = z_.size(0), S = z_.size(1), NH = z_.size(2), H = z_.size(3), per = B * NH * H;
  const at::IntArrayRef g = z_.sizes().slice(0, 3);
  XL_CHECK(i_.sizes() == g, what, "i_preact must be (B, S, NH), got ", i_.sizes());
  XL_CHECK(f_.sizes() == g, what, "f_preact must be (B, S, NH), got ", f_.sizes());
  XL_CHECK(o_.sizes() == g, what, "o_preact must be (B, S, NH), got ", o_.sizes());
  XL_CHECK(i_.scalar_type() == f_.scalar_type() && f_.scalar_type() == o_.scalar_type(), what, "gates must share a dtype");
  const bool hc = opt(c0_), hn = opt(n0_), hm = opt(m0_);
  XL_CHECK(hc == hn && hn == hm, what, "initial states must be provided together");
  if (hc)
    XL_CHECK(c0_->sizes() == at::IntArrayRef({B, NH, H}) && n0_->sizes() == at::IntArrayRef({B, NH, H}) &&
                 m0_->sizes() == at::IntArrayRef({B, NH}),
             what, "state must be c, n (B, NH, H) and m (B, NH)");
  const auto out = slstm_dtype(z_, i_, opt(c0_));
  const Tensor z = prep(z_), i = prep(i_), f = prep(f_), o = prep(o_), c0 = f32(c0_), n0 = f32(n0_), m0 = f32(m0_);
  const Tensor h = at::empty({B, S, NH, H}, z.options().dtype(out)), st = at::empty({2 * per + B * NH}, f32_on(z));
  float* s = ptr<float>(st);
  check_rc(xl_slstm_seq_fwd(ptr(z), ptr(i), ptr(f), ptr(o), ptr<float>(c0), ptr<float>(n0), ptr<float>(m0), ptr(h), s, s + per,
                            s + 2 * per, i32(B, what), i32(S, what), i32(NH, what), i32(H, what), (float)eps,
                            dtype_code(z, what), dtype_code(i, what), dtype_code(h, what), gpu.st),
           what);
  return {h, out == at::kFloat ? st : st.to(out)};
}

// ------------------------------------------- sLSTM layer: causal conv1d + SiLU, GroupNorm
Tensor causal_conv1d(const Tensor& x_, const Tensor& w_, const OptTensor& b_, int64_t act) {
  const char* what = "causal_conv1d";
  Gpu gpu(what, {&x_, &w_, opt(b_)});
  XL_CHECK(x_.dim() == 3, what, "x must be (B, S, D) channels last, got ", x_.sizes());
  const int64_t B = x_.size(0), S = x_.size(1), D = x_.size(2);
  XL_CHECK((w_.dim() == 2 || w_.dim() == 3) && w_.size(0) == D && (w_.dim() == 2 || w_.size(1) == 1), what,
           "weight must be (D, K) or (D, 1, K) with D = ", D, ", got ", w_.sizes());
  XL_CHECK(!opt(b_) || b_->sizes() == at::IntArrayRef({D}), what, "bias must be (", D, ",)");
  XL_CHECK(w_.scalar_type() == x_.scalar_type() && (!opt(b_) || b_->scalar_type() == x_.scalar_type()), what,
           "x, weight and bias must share a dtype (as nn.Conv1d requires)");
  XL_CHECK(act == 0 || act == 1, what, "act must be 0 (none) or 1 (SiLU), got ", act);
  const Tensor x = prep(x_), w = prep(w_), b = prep(b_), y = like(x);
  check_rc(xl_causal_conv1d_fwd(ptr(x), ptr(w), ptr(b), ptr(y), i32(B, what), i32(S, what), i32(D, what),
                                i32(w.size(-1), what), (int)act, dtype_code(x, what), gpu.st),
           what);
  return y;
}

Tensor group_norm(const Tensor& x_, int64_t groups, const OptTensor& w_, const OptTensor& b_, double eps) {
  const char* what = "group_norm";
  Gpu gpu(what, {&x_, opt(w_), opt(b_)});
  XL_CHECK(x_.dim() == 2, what, "x must be (N, C), got ", x_.sizes());
  const int64_t N = x_.size(0), C = x_.size(1);
  XL_CHECK(groups >= 1 && C % groups == 0, what, "C = ", C, " is not a multiple of num_groups = ", groups);
  for (const OptTensor* t : {&w_, &b_}) {
    if (!opt(*t)) continue;
    const char* name = t == &w_ ? "weight" : "bias";
    XL_CHECK((*t)->sizes() == at::IntArrayRef({C}), what, name, " must be (", C, ",)");
    XL_CHECK((*t)->scalar_type() == x_.scalar_type(), what, name, " must have x's dtype ", x_.scalar_type());
  }
  const Tensor x = prep(x_), w = prep(w_), b = prep(b_), y = like(x);
  check_rc(xl_group_norm_fwd(ptr(x), ptr(w), ptr(b), ptr(y), N, i32(groups, what), i32(C / groups, what), (float)eps,
                             dtype_code(x, what), gpu.st),
           what);
  return y;
}

// ------------------------------------------- mLSTM output cell: multi-head RMSNorm x sigmoid(o)
Tensor mh_rmsnorm_gate(const Tensor& h_, const OptTensor& w_, const OptTensor& o_, bool heads_first, double eps) {
  const char* what = "mh_rmsnorm_gate";
  Gpu gpu(what, {&h_, opt(w_), opt(o_)});
  XL_CHECK(h_.dim() == 4, what, "h must be 4-D, got ", h_.sizes());
  const int64_t B = h_.size(0), NH = h_.size(heads_first ? 1 : 2), S = h_.size(heads_first ? 2 : 1), DH = h_.size(3);
  XL_CHECK(!opt(w_) || w_->sizes() == at::IntArrayRef({NH * DH}), what, "weight must be (", NH * DH, ",)");
  XL_CHECK(!opt(o_) || o_->sizes() == at::IntArrayRef({B, S, NH * DH}) || o_->sizes() == at::IntArrayRef({B, S, NH, DH}),
           what, "o_preact must be (B, S, NH*DH) = (", B, ", ", S, ", ", NH * DH, ")");
  for (const OptTensor* t : {&w_, &o_})
    XL_CHECK(!opt(*t) || (*t)->scalar_type() == h_.scalar_type(), what, t == &w_ ? "weight" : "o_preact",
             " must have h's dtype ", h_.scalar_type());
  const Tensor h = prep(h_), w = prep(w_), o = prep(o_), y = at::empty({B, S, NH * DH}, h.options());
  check_rc(xl_mh_rmsnorm_gate_fwd(ptr(h), ptr(w), ptr(o), ptr(y), i32(B, what), i32(NH, what), i32(S, what), i32(DH, what),
                                  heads_first ? 1 : 0, (float)eps, dtype_code(h, what), gpu.st),
           what);
  return y;
}

// ------------------------------------------- projections with a soft-cap epilogue
// rows of x [..., D] and the output's shape [..., G]
int64_t rows_of(const Tensor& x, int64_t G, std::vector<int64_t>& shape) {
  shape = x.sizes().vec();
  shape.back() = G;
  int64_t M = 1;
  for (size_t d = 0; d + 1 < shape.size(); ++d) M *= shape[d];
  return M;
}

Tensor gate_proj_softcap(const Tensor& x_, const Tensor& w_, const OptTensor& b_, double cap, int64_t cap_rounding) {
  const char* what = "gate_proj_softcap";
  Gpu gpu(what, {&x_, &w_, opt(b_)});
  XL_CHECK(x_.dim() >= 1 && w_.dim() == 2 && w_.size(1) == x_.size(-1), what,
           "weight must be (G, D) with D = x.shape[-1], got ", w_.sizes(), " for x ", x_.sizes());
  const int64_t G = w_.size(0), D = w_.size(1);
  XL_CHECK(!opt(b_) || b_->sizes() == at::IntArrayRef({G}), what, "bias must be (", G, ",)");
  XL_CHECK(w_.scalar_type() == x_.scalar_type() && (!opt(b_) || b_->scalar_type() == x_.scalar_type()), what,
           "x, weight and bias must share a dtype");
  std::vector<int64_t> shape;
  const int64_t M = rows_of(x_, G, shape);
  const Tensor x = prep(x_), w = prep(w_), b = prep(b_), y = at::empty(shape, x.options());
  check_rc(xl_gate_proj_softcap_fwd(ptr(x), ptr(w), ptr(b), ptr(y), i32(M, what), i32(D, what), i32(G, what), (float)cap,
                                    i32(cap_rounding, what), dtype_code(x, what), gpu.st),
           what);
  return y;
}

std::tuple<Tensor, Tensor> gate_proj2_softcap(const Tensor& x_, const Tensor& w1_, const OptTensor& b1_, const Tensor& w2_,
                                              const OptTensor& b2_, double cap, int64_t cap_rounding, bool heads_first) {
  const char* what = "gate_proj_softcap";
  Gpu gpu(what, {&x_, &w1_, opt(b1_), &w2_, opt(b2_)});
  XL_CHECK(x_.dim() == 3, what, "x must be (B, S, D), got ", x_.sizes());
  const int64_t B = x_.size(0), S = x_.size(1), D = x_.size(2);
  auto check = [&](const Tensor& w, const OptTensor& b) {
    XL_CHECK(w.dim() == 2 && w.size(1) == D, what, "weight must be (G, D) with D = x.shape[-1], got ", w.sizes(), " for x ",
             x_.sizes());
    XL_CHECK(!opt(b) || b->sizes() == at::IntArrayRef({w.size(0)}), what, "bias must be (", w.size(0), ",)");
    XL_CHECK(w.scalar_type() == x_.scalar_type() && (!opt(b) || b->scalar_type() == x_.scalar_type()), what,
             "x, weight and bias must share a dtype");
  };
  check(w1_, b1_);
  check(w2_, b2_);
  const int64_t G1 = w1_.size(0), G2 = w2_.size(0);
  const Tensor x = prep(x_), w1 = prep(w1_), b1 = prep(b1_), w2 = prep(w2_), b2 = prep(b2_);
  auto out = [&](int64_t G) { return heads_first ? at::empty({B, G, S}, x.options()) : at::empty({B, S, G}, x.options()); };
  const Tensor y1 = out(G1), y2 = out(G2);
  check_rc(xl_gate_proj2_softcap_fwd(ptr(x), ptr(w1), ptr(b1), i32(G1, what), ptr(w2), ptr(b2), i32(G2, what), ptr(y1),
                                     ptr(y2), i32(B * S, what), i32(D, what), heads_first ? i32(S, what) : 0, (float)cap,
                                     i32(cap_rounding, what), dtype_code(x, what), gpu.st),
           what);
  return {y1, y2};
}

Tensor lm_head_softcap(const Tensor& x_, const Tensor& w_, double cap) {
  const char* what = "lm_head_softcap";
  Gpu gpu(what, {&x_, &w_});
  XL_CHECK(x_.dim() >= 1 && w_.dim() == 2 && w_.size(1) == x_.size(-1), what,
           "weight must be (V, D) with D = x.shape[-1], got ", w_.sizes(), " for x ", x_.sizes());
  XL_CHECK(w_.scalar_type() == x_.scalar_type(), what, "x and weight must share a dtype");
  const int64_t V = w_.size(0), D = w_.size(1);
  std::vector<int64_t> shape;
  const int64_t M = rows_of(x_, V, shape);
  XL_CHECK(M <= xl_lm_head_max_rows, what, M, " rows (at most ", xl_lm_head_max_rows,
           "; logits of every position are a GEMM: use the Linear and soft_cap)");
  XL_CHECK(M * (D + 8) * 2 <= xl_lm_head_max_lds, what, M, " rows of D=", D, " exceed the kernel's LDS staging");
  const Tensor x = prep(x_), w = prep(w_), y = at::empty(shape, x.options());
  check_rc(xl_lm_head_softcap_fwd(ptr(x), ptr(w), ptr(y), i32(M, what), i32(D, what), i32(V, what), (float)cap,
                                  dtype_code(x, what), gpu.st),
           what);
  return y;
}

// ------------------------------------------- a block's norm (with the residual before it), SwiGLU product
std::tuple<Tensor, Tensor> norm_impl(const char* what, const Tensor& x_, const Tensor* r_, const Tensor& w_, double eps,
                                     at::TensorList src, at::TensorList dst) {
  Gpu gpu(what, {&x_, r_, &w_});
  XL_CHECK(x_.dim() >= 1, what, "x must have a last axis");
  const int64_t D = x_.size(-1);
  XL_CHECK(w_.sizes() == at::IntArrayRef({D}) && w_.scalar_type() == x_.scalar_type(), what, "weight must be (", D,
           ",) of ", x_.scalar_type());
  XL_CHECK(!r_ || (r_->sizes() == x_.sizes() && r_->scalar_type() == x_.scalar_type()), what,
           "x and the residual must share shape and dtype");
  XL_CHECK(src.size() == dst.size() && src.size() <= 2, what, "at most two state copies");
  float* cp[2][2] = {};
  int n[2] = {};
  for (size_t c = 0; c < src.size(); ++c) {
    const Tensor &a = src[c], &b = dst[c];
    XL_CHECK(a.device() == x_.device() && b.device() == x_.device() && a.scalar_type() == at::kFloat &&
                 b.scalar_type() == at::kFloat && a.numel() == b.numel() && a.is_contiguous() && b.is_contiguous(),
             what, "state copies are between contiguous float32 tensors of one size");
    cp[c][0] = ptr<float>(a);
    cp[c][1] = ptr<float>(b);
    n[c] = i32(a.numel(), what);
  }
  const Tensor x = prep(x_), w = prep(w_), r = r_ ? prep(*r_) : Tensor(), y = like(x), s = r_ ? like(x) : Tensor();
  check_rc(xl_add_rmsnorm_fwd(ptr(x), ptr(r), ptr(w), ptr(s), ptr(y), i32(D ? x.numel() / D : 0, what), i32(D, what),
                              (float)eps, cp[0][0], cp[0][1], n[0], cp[1][0], cp[1][1], n[1], dtype_code(x, what), gpu.st),
           what);
  return {s, y};
}

Tensor rms_norm(const Tensor& x, const Tensor& w, double eps) {
  return std::get<1>(norm_impl("rms_norm", x, nullptr, w, eps, {}, {}));
}

std::tuple<Tensor, Tensor> add_rmsnorm(const Tensor& x, const Tensor& r, const Tensor& w, double eps, at::TensorList src,
                                       at::TensorList dst) {
  return norm_impl("add_rmsnorm", x, &r, w, eps, src, dst);
}

Tensor silu_mul(const Tensor& g_, const Tensor& u_) {
  const char* what = "silu_mul";
  Gpu gpu(what, {&g_, &u_});
  XL_CHECK(g_.sizes() == u_.sizes() && g_.scalar_type() == u_.scalar_type(), what, "gate and up must share shape and dtype");
  const Tensor g = prep(g_), u = prep(u_), y = like(g);
  check_rc(xl_silu_mul_fwd(ptr(g), ptr(u), ptr(y), y.numel(), dtype_code(y, what), gpu.st), what);
  return y;
}

// The operators that write an argument, under autograd's bookkeeping, on fake tensors as on real ones.  What they
// write is updated outside autograd, whatever it requires (a leaf too; its own history stays), a backward through
// the outputs raises, and the written tensors' version counters move (inference tensors have none).
template <typename Op, typename... Args>
auto without_backward(const char* name, const Op& op, c10::DispatchKeySet ks, at::TensorList given, const Args&... args) {
  bool grad = false;
  for (const Tensor& t : given) {
    TORCH_CHECK_NOT_IMPLEMENTED(!t._fw_grad(0).defined(), name, ": no forward-mode derivative");
    grad = grad || t.requires_grad();
  }
  grad = grad && c10::GradMode::is_enabled();
  auto out = [&] {
    at::AutoDispatchBelowAutograd below;
    return op.redispatch(ks & c10::after_autograd_keyset, args...);
  }();
  if (grad) {
    const auto none = std::make_shared<torch::autograd::NotImplemented>(name);
    none->set_next_edges(torch::autograd::collect_next_edges(given));
    std::apply([&](const auto&... t) { (torch::autograd::set_history(t, none), ...); }, out);
  }
  return out;
}

template <typename Op, typename... Args>
auto and_count(const Op& op, c10::DispatchKeySet ks, at::TensorList written, const Args&... args) {
  at::AutoDispatchBelowADInplaceOrView below;
  auto out = op.redispatch(ks & c10::after_ADInplaceOrView_keyset, args...);
  for (const Tensor& t : written)
    if (!t.is_inference()) t.unsafeGetTensorImpl()->bump_version();
  return out;
}

const auto& step_inplace_op() {
  static const auto op =
      c10::Dispatcher::singleton().findSchemaOrThrow("xlstm_hip::mlstm_step_", "").typed<decltype(mlstm_step_)>();
  return op;
}

std::tuple<Tensor, Tensor, Tensor> mlstm_step__autograd(c10::DispatchKeySet ks, const Tensor& q, const Tensor& k,
                                                        const Tensor& v, const Tensor& i, const Tensor& f, const Tensor& c,
                                                        const Tensor& n, const Tensor& m, double eps, double qk_scale) {
  return without_backward("xlstm_hip::mlstm_step_", step_inplace_op(), ks, {q, k, v, i, f, c, n, m}, q, k, v, i, f, c, n,
                          m, eps, qk_scale);
}

std::tuple<Tensor, Tensor, Tensor> mlstm_step__inplace(c10::DispatchKeySet ks, const Tensor& q, const Tensor& k,
                                                       const Tensor& v, const Tensor& i, const Tensor& f, const Tensor& c,
                                                       const Tensor& n, const Tensor& m, double eps, double qk_scale) {
  return and_count(step_inplace_op(), ks, {c}, q, k, v, i, f, c, n, m, eps, qk_scale);
}

const auto& add_rmsnorm_op() {
  static const auto op =
      c10::Dispatcher::singleton().findSchemaOrThrow("xlstm_hip::add_rmsnorm", "").typed<decltype(add_rmsnorm)>();
  return op;
}

std::tuple<Tensor, Tensor> add_rmsnorm_autograd(c10::DispatchKeySet ks, const Tensor& x, const Tensor& r, const Tensor& w,
                                                double eps, at::TensorList src, at::TensorList dst) {
  std::vector<Tensor> given = {x, r, w};
  given.insert(given.end(), src.begin(), src.end());
  given.insert(given.end(), dst.begin(), dst.end());
  return without_backward("xlstm_hip::add_rmsnorm", add_rmsnorm_op(), ks, given, x, r, w, eps, src, dst);
}

std::tuple<Tensor, Tensor> add_rmsnorm_inplace(c10::DispatchKeySet ks, const Tensor& x, const Tensor& r, const Tensor& w,
                                               double eps, at::TensorList src, at::TensorList dst) {
  return and_count(add_rmsnorm_op(), ks, dst, x, r, w, eps, src, dst);
}

// The kernels below call the library with this build's argument lists: none is registered over one of another ABI
// (xlstm_hip/_lib.py then says so in their place).
bool abi_matches() { return xl_abi_version() == XL_ABI_VERSION; }

}  // namespace

TORCH_LIBRARY_IMPL(xlstm_hip, CUDA, m) {
  if (!abi_matches()) return;
  m.impl("soft_cap", soft_cap);
  m.impl("mlstm_step", mlstm_step);
  m.impl("mlstm_step_", mlstm_step_);
  m.impl("mlstm_chunkwise", mlstm_chunkwise);
  m.impl("mlstm_chunkwise_bwd", mlstm_chunkwise_bwd);
  m.impl("mlstm_sequence", mlstm_sequence);
  m.impl("slstm_step", slstm_step);
  m.impl("slstm_sequence", slstm_sequence);
  m.impl("causal_conv1d", causal_conv1d);
  m.impl("group_norm", group_norm);
  m.impl("mh_rmsnorm_gate", mh_rmsnorm_gate);
  m.impl("gate_proj_softcap", gate_proj_softcap);
  m.impl("gate_proj2_softcap", gate_proj2_softcap);
  m.impl("lm_head_softcap", lm_head_softcap);
  m.impl("rms_norm", rms_norm);
  m.impl("add_rmsnorm", add_rmsnorm);
  m.impl("silu_mul", silu_mul);
}

// The chunkwise forward differentiates through its own backward; every other operator is forward-only and
// a backward through it raises.
#define XL_FORWARD_ONLY(m, kernel)                                                                                     \
  for (const char* op : {"soft_cap", "mlstm_step", "mlstm_chunkwise_bwd", "mlstm_sequence", "slstm_step",              \
                         "slstm_sequence", "causal_conv1d", "group_norm", "mh_rmsnorm_gate", "gate_proj_softcap",      \
                         "gate_proj2_softcap", "lm_head_softcap", "rms_norm", "silu_mul"})                             \
    m.impl(op, kernel());
TORCH_LIBRARY_IMPL(xlstm_hip, Autograd, m) {
  if (!abi_matches()) return;
  m.impl("mlstm_chunkwise", mlstm_chunkwise_autograd);
  m.impl("mlstm_step_", mlstm_step__autograd);
  m.impl("add_rmsnorm", add_rmsnorm_autograd);
  XL_FORWARD_ONLY(m, torch::autograd::autogradNotImplementedFallback)
}
TORCH_LIBRARY_IMPL(xlstm_hip, ADInplaceOrView, m) {
  if (!abi_matches()) return;
  m.impl("mlstm_step_", mlstm_step__inplace);
  m.impl("add_rmsnorm", add_rmsnorm_inplace);
}
