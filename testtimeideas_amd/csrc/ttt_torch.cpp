// ttt_torch.cpp — torch binding of the forward, backward and double backward
// of the C ABI (include/ttt_attn.h): ttt_attn_fwd, then ttt_attn_bwd and
// ttt_attn_gg, or, with a split of each kernel family's own (tiles per
// workgroup; 0 lets the library choose), ttt_attn_bwd_dq + ttt_attn_bwd_dkdv
// and ttt_attn_gg_row + ttt_attn_gg_col.
//
// The ctypes binding (testtimeideas_amd/_lib.py) spends tens of microseconds
// of Python per call building views, problems and outputs; the autograd path
// of one grad-grad step makes three such calls.  This module does the same
// work in C++: it takes tensors whose head dim is a multiple of 8 up to 128
// (the Python layer pads others), copies any whose strides the C ABI does not take (ready),
// allocates outputs, statistics and the workspace with torch's caching
// allocator on the tensors' device, and calls the C entry points on torch's
// current HIP stream.  A nonzero status raises
// RuntimeError with the library's message.  No kernel runs here and nothing
// falls back: the C ABI is the only compute path.
#include <torch/extension.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/functions/basic_ops.h>
#include <c10/hip/HIPStream.h>

#include <algorithm>
#include <atomic>
#include <string>
#include <cstring>
#include <vector>

#include "../../include/ttt_attn.h"

namespace {

int32_t dtype_code(const at::Tensor& t) {
  switch (t.scalar_type()) {
    case at::kHalf: return TTT_F16;
    case at::kBFloat16: return TTT_BF16;
    case at::kFloat: return TTT_F32;
    default: TORCH_CHECK(false, "unsupported dtype ", t.scalar_type(), "; expected float16, bfloat16 or float32");
  }
  return -1;
}

ttt_view view_of(const at::Tensor& t) {
  ttt_view v;
  v.data = t.data_ptr();
  v.stride_b = t.stride(0);
  v.stride_h = t.stride(1);
  v.stride_t = t.stride(2);
  return v;
}

// `t` itself when the C ABI takes it as it is (unit last stride, a positive
// T stride, 16-byte aligned base and B/H/T strides), else a contiguous copy
// (fresh strides, so a size-1 dimension's stride is positive too).
at::Tensor ready(const at::Tensor& t) {
  const int64_t eb = t.element_size();
  const bool ok = (t.stride(3) == 1 || t.size(3) <= 1) && t.stride(2) > 0 &&
                  reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0 && (t.stride(0) * eb) % 16 == 0 &&
                  (t.stride(1) * eb) % 16 == 0 && (t.stride(2) * eb) % 16 == 0;
  return ok ? t : at::empty(t.sizes(), t.options()).copy_(t);
}

c10::optional<at::Tensor> ready(const c10::optional<at::Tensor>& t) {
  if (!t || !t->defined()) return t;
  return ready(*t);
}

ttt_view none_view() {
  ttt_view v;
  v.data = nullptr;
  v.stride_b = v.stride_h = v.stride_t = 0;
  return v;
}

// The problem of [B,H,T,D] tensor x with the mask fields.
ttt_problem problem_of(const at::Tensor& x, bool causal, double scale, int64_t split_chunk, int64_t window,
                       int64_t window_kind, const c10::optional<at::Tensor>& bias, int64_t block_rows = 0) {
  ttt_problem pr;
  std::memset(&pr, 0, sizeof(pr));
  pr.dtype = dtype_code(x);
  pr.causal = causal ? 1 : 0;
  pr.batch = x.size(0);
  pr.heads = x.size(1);
  pr.seqlen = x.size(2);
  pr.head_dim = x.size(3);
  pr.scale = static_cast<float>(scale);
  pr.split_chunk = static_cast<int32_t>(split_chunk);
  pr.window = static_cast<int32_t>(window);
  pr.window_kind = static_cast<int32_t>(window_kind);
  pr.bias = (bias && bias->defined()) ? view_of(*bias) : none_view();
  pr.block_rows = static_cast<int32_t>(block_rows);
  return pr;
}

void check(int rc, const char* what) {
  TORCH_CHECK(rc == 0, what, " failed (status ", rc, "): ", ttt_last_error());
}

// The shape of q [B,H,Tq,d] against k [B,H,Tk,d]; its problem's head_dim is d
// rounded up to 64 or 128.
ttt_shape shape_of(const at::Tensor& q, const at::Tensor& k, ttt_problem* pr) {
  const int64_t d = q.size(3);
  pr->head_dim = d <= 64 ? 64 : d <= 128 ? 128 : d;
  ttt_shape sh;
  std::memset(&sh, 0, sizeof(sh));
  sh.keys = k.size(2);
  sh.cols = d;
  return sh;
}

at::Tensor stats_of(const at::Tensor& x) {
  return at::empty({x.size(0), x.size(1), x.size(2)}, x.options().dtype(at::kFloat));
}

// [B,H,Tq,Tk] P with rows padded to 8 elements (the kernels read rows in runs of 8).
at::Tensor alloc_p(const at::Tensor& x, int64_t t) {
  const int64_t tp = (t + 7) / 8 * 8;
  at::Tensor buf = at::empty({x.size(0), x.size(1), x.size(2), tp}, x.options());
  return tp == t ? buf : buf.narrow(3, 0, t);
}

// P as the forward wrote it, or, where it came back from a saved-tensor hook
// without the forward's row storage, a copy that has it.
c10::optional<at::Tensor> ready_p(const c10::optional<at::Tensor>& p) {
  if (!p || !p->defined()) return c10::nullopt;
  const int64_t eb = p->element_size();
  int64_t end = p->storage_offset() + (p->size(3) + 7) / 8 * 8;  // past the last element read
  bool ok = p->stride(3) == 1 && reinterpret_cast<uintptr_t>(p->data_ptr()) % 16 == 0;
  for (int i = 0; i < 3; ++i) {
    ok = ok && (p->stride(i) * eb) % 16 == 0;
    end += (p->size(i) - 1) * p->stride(i);
  }
  if (ok && end * eb <= static_cast<int64_t>(p->storage().nbytes())) return p;
  return alloc_p(*p, p->size(3)).copy_(*p);
}

int64_t workspace_size(const ttt_problem& pr, int32_t entry, bool gdo, const ttt_shape* shape) {
  const int64_t n = ttt_attn_workspace_size_shape(&pr, shape, entry, gdo ? 1 : 0);
  TORCH_CHECK(n >= 0, "ttt_attn_workspace_size failed: ", ttt_last_error());
  return n;
}

at::Tensor workspace(const ttt_problem& pr, const ttt_shape& shape, int32_t entry, bool gdo, const at::Tensor& like,
                     int64_t* bytes) {
  const int64_t n = workspace_size(pr, entry, gdo, &shape);
  *bytes = n;
  return n > 0 ? at::empty({n}, like.options().dtype(at::kByte)) : at::Tensor();
}

// One workspace for two launches in stream order (the second starts after
// the first, its combine included, has finished with it).
at::Tensor workspace2(const ttt_problem& pr0, int32_t e0, const ttt_problem& pr1, int32_t e1,
                      const ttt_shape& shape, bool gdo, const at::Tensor& like, int64_t* bytes) {
  const int64_t n = std::max(workspace_size(pr0, e0, gdo, &shape), workspace_size(pr1, e1, gdo, &shape));
  *bytes = n;
  return n > 0 ? at::empty({n}, like.options().dtype(at::kByte)) : at::Tensor();
}

void* ptr_or_null(const at::Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }

void* stream_of(const at::Tensor& x) {
  return static_cast<void*>(c10::hip::getCurrentHIPStream(x.device().index()).stream());
}

// Forward: (O, LSE, P or None).  Replaces TritonAttentionFn.forward's launches.
std::vector<at::Tensor> fwd(const at::Tensor& q_, const at::Tensor& k_, const at::Tensor& v_, bool causal,
                            double scale, bool want_p, int64_t split_chunk, int64_t window, int64_t window_kind,
                            const c10::optional<at::Tensor>& bias, int64_t block_rows) {
  const at::Tensor q = ready(q_), k = ready(k_), v = ready(v_);
  ttt_problem pr = problem_of(q, causal, scale, split_chunk, window, window_kind, bias, block_rows);
  const ttt_shape sh = shape_of(q, k, &pr);
  at::Tensor o = at::empty(q.sizes(), q.options());
  at::Tensor lse = stats_of(q);
  at::Tensor p = want_p ? alloc_p(q, k.size(2)) : at::Tensor();
  int64_t wsb = 0;
  at::Tensor ws = workspace(pr, sh, want_p ? TTT_ENTRY_FWD_P : TTT_ENTRY_FWD, false, q, &wsb);
  const ttt_view vq = view_of(q), vk = view_of(k), vv = view_of(v), vo = view_of(o);
  const ttt_view vp = want_p ? view_of(p) : none_view();
  check(ttt_attn_fwd_shape(&pr, &sh, &vq, &vk, &vv, &vo, lse.data_ptr<float>(), want_p ? &vp : nullptr, ptr_or_null(ws), wsb,
                     stream_of(q)),
        "ttt_attn_fwd");
  return {o, lse, p};
}

// First backward: (dQ, dK, dV, D).  split_dq, split_dkdv: each family's split.
std::vector<at::Tensor> bwd(const at::Tensor& q_, const at::Tensor& k_, const at::Tensor& v_, const at::Tensor& o_,
                            const at::Tensor& dout_, const at::Tensor& lse, const c10::optional<at::Tensor>& p_,
                            bool causal, double scale, int64_t split_dq, int64_t split_dkdv, int64_t window,
                            int64_t window_kind, const c10::optional<at::Tensor>& bias) {
  const at::Tensor q = ready(q_), k = ready(k_), v = ready(v_), o = ready(o_), dout = ready(dout_);
  ttt_problem pq = problem_of(q, causal, scale, split_dq, window, window_kind, bias);
  const ttt_shape sh = shape_of(q, k, &pq);
  ttt_problem pk = pq;
  pk.split_chunk = static_cast<int32_t>(split_dkdv);
  at::Tensor dq = at::empty(q.sizes(), q.options());
  at::Tensor dk = at::empty(k.sizes(), k.options());
  at::Tensor dv = at::empty(v.sizes(), v.options());
  at::Tensor rowsum = stats_of(q);
  int64_t wsb = 0;
  at::Tensor ws = workspace2(pq, TTT_ENTRY_BWD_DQ, pk, TTT_ENTRY_BWD_DKDV, sh, false, q, &wsb);
  const c10::optional<at::Tensor> p = ready_p(p_);
  const bool lp = p.has_value();
  const ttt_view vq = view_of(q), vk = view_of(k), vv = view_of(v), vo = view_of(o), vdo = view_of(dout);
  const ttt_view vp = lp ? view_of(*p) : none_view();
  const ttt_view vdq = view_of(dq), vdk = view_of(dk), vdv = view_of(dv);
  void* st = stream_of(q);
  float* rs = rowsum.data_ptr<float>();
  check(ttt_attn_bwd_dq_shape(&pq, &sh, &vq, &vk, &vv, &vo, &vdo, lse.data_ptr<float>(), lp ? &vp : nullptr, nullptr,
                              rs, &vdq, ptr_or_null(ws), wsb, st),
        "ttt_attn_bwd_dq");
  check(ttt_attn_bwd_dkdv_shape(&pk, &sh, &vq, &vk, &vv, &vdo, lse.data_ptr<float>(), lp ? &vp : nullptr, rs, &vdk,
                                &vdv, ptr_or_null(ws), wsb, st),
        "ttt_attn_bwd_dkdv");
  return {dq, dk, dv, rowsum};
}

// The same through ttt_attn_bwd, both families with one split (0: the
// library's): the dK/dV launch also finishes dQ's split blocks.
std::vector<at::Tensor> bwd_fused(const at::Tensor& q_, const at::Tensor& k_, const at::Tensor& v_,
                                  const at::Tensor& o_, const at::Tensor& dout_, const at::Tensor& lse,
                                  const c10::optional<at::Tensor>& p_, bool causal, double scale, int64_t window,
                                  int64_t window_kind, const c10::optional<at::Tensor>& bias, int64_t split) {
  const at::Tensor q = ready(q_), k = ready(k_), v = ready(v_), o = ready(o_), dout = ready(dout_);
  ttt_problem pr = problem_of(q, causal, scale, split, window, window_kind, bias);
  const ttt_shape sh = shape_of(q, k, &pr);
  at::Tensor dq = at::empty(q.sizes(), q.options());
  at::Tensor dk = at::empty(k.sizes(), k.options());
  at::Tensor dv = at::empty(v.sizes(), v.options());
  at::Tensor rowsum = stats_of(q);
  int64_t wsb = 0;
  at::Tensor ws = workspace(pr, sh, TTT_ENTRY_BWD, false, q, &wsb);
  const c10::optional<at::Tensor> p = ready_p(p_);
  const bool lp = p.has_value();
  const ttt_view vq = view_of(q), vk = view_of(k), vv = view_of(v), vo = view_of(o), vdo = view_of(dout);
  const ttt_view vp = lp ? view_of(*p) : none_view();
  const ttt_view vdq = view_of(dq), vdk = view_of(dk), vdv = view_of(dv);
  check(ttt_attn_bwd_shape(&pr, &sh, &vq, &vk, &vv, &vo, &vdo, lse.data_ptr<float>(), lp ? &vp : nullptr,
                     rowsum.data_ptr<float>(), &vdq, &vdk, &vdv, ptr_or_null(ws), wsb, stream_of(q)),
        "ttt_attn_bwd");
  return {dq, dk, dv, rowsum};
}

// Double backward: (GQ, GK, GV, GdO or None).  dq: the first backward's dQ,
// or None (ttt_attn_gg_row).
std::vector<at::Tensor> gg(const at::Tensor& q_, const at::Tensor& k_, const at::Tensor& v_, const at::Tensor& dout_,
                           const at::Tensor& lse, const c10::optional<at::Tensor>& p_, const at::Tensor& rowsum,
                           const c10::optional<at::Tensor>& dq_, const at::Tensor& gq_, const at::Tensor& gk_,
                           const at::Tensor& gv_, bool causal, double scale, bool want_gdo, int64_t split_row,
                           int64_t split_col, int64_t window, int64_t window_kind,
                           const c10::optional<at::Tensor>& bias) {
  const at::Tensor q = ready(q_), k = ready(k_), v = ready(v_), dout = ready(dout_);
  const at::Tensor gq = ready(gq_), gk = ready(gk_), gv = ready(gv_);
  const c10::optional<at::Tensor> dq = ready(dq_);
  ttt_problem pr = problem_of(q, causal, scale, split_row, window, window_kind, bias);
  const ttt_shape sh = shape_of(q, k, &pr);
  ttt_problem pc = pr;
  pc.split_chunk = static_cast<int32_t>(split_col);
  at::Tensor gq_out = at::empty(q.sizes(), q.options());
  at::Tensor gk_out = at::empty(k.sizes(), k.options());
  at::Tensor gv_out = at::empty(v.sizes(), v.options());
  at::Tensor gdo = want_gdo ? at::empty(dout.sizes(), dout.options()) : at::Tensor();
  at::Tensor e = stats_of(q), f = stats_of(q);
  int64_t wsb = 0;
  at::Tensor ws = workspace2(pr, TTT_ENTRY_GG_ROW, pc, TTT_ENTRY_GG_COL, sh, want_gdo, q, &wsb);
  const c10::optional<at::Tensor> p = ready_p(p_);
  const bool lp = p.has_value();
  const ttt_view vq = view_of(q), vk = view_of(k), vv = view_of(v), vdo = view_of(dout);
  const ttt_view vp = lp ? view_of(*p) : none_view();
  const ttt_view vgq = view_of(gq), vgk = view_of(gk), vgv = view_of(gv);
  const ttt_view ogq = view_of(gq_out), ogk = view_of(gk_out), ogv = view_of(gv_out);
  const ttt_view ogdo = want_gdo ? view_of(gdo) : none_view();
  const bool ldq = dq && dq->defined();
  const ttt_view vdq = ldq ? view_of(*dq) : none_view();
  void* st = stream_of(q);
  const float* rs = rowsum.data_ptr<float>();
  check(ttt_attn_gg_row_shape(&pr, &sh, &vq, &vk, &vv, &vdo, lse.data_ptr<float>(), lp ? &vp : nullptr, rs,
                              ldq ? &vdq : nullptr, &vgq, &vgk, &vgv, &ogq, want_gdo ? &ogdo : nullptr,
                              e.data_ptr<float>(), f.data_ptr<float>(), ptr_or_null(ws), wsb, st),
        "ttt_attn_gg_row");
  check(ttt_attn_gg_col_shape(&pc, &sh, &vq, &vk, &vv, &vdo, lse.data_ptr<float>(), lp ? &vp : nullptr, rs,
                              e.data_ptr<float>(), f.data_ptr<float>(), &vgq, &vgk, &vgv, &ogk, &ogv, ptr_or_null(ws),
                              wsb, st),
        "ttt_attn_gg_col");
  return {gq_out, gk_out, gv_out, gdo};
}

// The same through ttt_attn_gg, both passes with one split (0: the library's):
// the column launch also finishes the row pass's split blocks.
std::vector<at::Tensor> gg_fused(const at::Tensor& q_, const at::Tensor& k_, const at::Tensor& v_,
                                 const at::Tensor& dout_, const at::Tensor& lse, const c10::optional<at::Tensor>& p_,
                                 const at::Tensor& rowsum, const c10::optional<at::Tensor>& dq_,
                                 const at::Tensor& gq_, const at::Tensor& gk_, const at::Tensor& gv_, bool causal,
                                 double scale, bool want_gdo, int64_t window, int64_t window_kind,
                                 const c10::optional<at::Tensor>& bias, int64_t split) {
  const at::Tensor q = ready(q_), k = ready(k_), v = ready(v_), dout = ready(dout_);
  const at::Tensor gq = ready(gq_), gk = ready(gk_), gv = ready(gv_);
  const c10::optional<at::Tensor> dq = ready(dq_);
  ttt_problem pr = problem_of(q, causal, scale, split, window, window_kind, bias);
  const ttt_shape sh = shape_of(q, k, &pr);
  at::Tensor gq_out = at::empty(q.sizes(), q.options());
  at::Tensor gk_out = at::empty(k.sizes(), k.options());
  at::Tensor gv_out = at::empty(v.sizes(), v.options());
  at::Tensor gdo = want_gdo ? at::empty(dout.sizes(), dout.options()) : at::Tensor();
  at::Tensor e = stats_of(q), f = stats_of(q);
  int64_t wsb = 0;
  at::Tensor ws = workspace(pr, sh, TTT_ENTRY_GG, want_gdo, q, &wsb);
  const c10::optional<at::Tensor> p = ready_p(p_);
  const bool lp = p.has_value();
  const ttt_view vq = view_of(q), vk = view_of(k), vv = view_of(v), vdo = view_of(dout);
  const ttt_view vp = lp ? view_of(*p) : none_view();
  const ttt_view vgq = view_of(gq), vgk = view_of(gk), vgv = view_of(gv);
  const ttt_view ogq = view_of(gq_out), ogk = view_of(gk_out), ogv = view_of(gv_out);
  const ttt_view ogdo = want_gdo ? view_of(gdo) : none_view();
  const bool ldq = dq && dq->defined();
  const ttt_view vdq = ldq ? view_of(*dq) : none_view();
  check(ttt_attn_gg_shape(&pr, &sh, &vq, &vk, &vv, &vdo, lse.data_ptr<float>(), lp ? &vp : nullptr, rowsum.data_ptr<float>(),
                    ldq ? &vdq : nullptr, &vgq, &vgk, &vgv, &ogq, &ogk, &ogv, want_gdo ? &ogdo : nullptr,
                    e.data_ptr<float>(), f.data_ptr<float>(), ptr_or_null(ws), wsb, stream_of(q)),
        "ttt_attn_gg");
  return {gq_out, gk_out, gv_out, gdo};
}

// What library_choice() of testtimeideas_amd/_lib.py would say (_lib.py sets it
// whenever a split is forced, kernels are timed or tuning is switched), and its
// gg (set once, when the module is loaded, and never released: graphs may
// outlive the interpreter's modules).
std::atomic<bool> g_library_choice{true};
PyObject* g_python_gg = nullptr;

void set_library_choice(bool on) { g_library_choice.store(on); }

void set_python_gg(const py::function& gg) { g_python_gg = py::function(gg).release().ptr(); }

// The first backward as a differentiable function of (q, k, v, dO), for
// create_graph=True on operands that go to the kernels as they are; its
// backward is the double backward.  The Python Function of the same role
// (_AttnBwdFn in testtimeideas_amd/ttt_kernels/triton_attention.py) takes every
// other call and says what is saved and why.  In C++ neither pass enters the
// interpreter: a step at b1 h1 T64, where the host is all there is, takes 79
// instead of 93 us of host time (73 instead of 89 with P recomputed), the
// splits kept per thread (ttt_capi.hip) included.  Only where a split is forced
// or kernels are timed or tuned when the double backward runs does it go
// through _lib.py's gg, whatever held at the first backward (asking _lib.py each
// time took the step at T512 from 76 to 83 us).
struct SavedForward {
  at::Tensor o, lse;
  c10::optional<at::Tensor> p, bias;
  bool causal;
  double scale;
  int64_t window, window_kind;
};

struct AttnBwd : public torch::autograd::Function<AttnBwd> {
  static torch::autograd::variable_list forward(torch::autograd::AutogradContext* ctx, const at::Tensor& q,
                                                const at::Tensor& k, const at::Tensor& v, const at::Tensor& dout,
                                                const SavedForward& f) {
    std::vector<at::Tensor> r =
        bwd_fused(q, k, v, f.o, dout, f.lse, f.p, f.causal, f.scale, f.window, f.window_kind, f.bias, 0);
    const at::Tensor none;
    ctx->save_for_backward({q, k, v, dout, f.lse, f.p ? *f.p : none, r[3], r[0]});
    // the mask is a constant of the call
    ctx->saved_data["bias"] = f.bias;
    ctx->saved_data["causal"] = f.causal;
    ctx->saved_data["scale"] = f.scale;
    ctx->saved_data["window"] = f.window;
    ctx->saved_data["window_kind"] = f.window_kind;
    return {r[0], r[1], r[2]};
  }

  // The double backward through _lib.py's gg, unless every launch is to take the
  // library's choice.
  static bool forced(std::vector<at::Tensor>* r, const torch::autograd::variable_list& s,
                     const torch::autograd::variable_list& g, const c10::optional<at::Tensor>& p, bool causal,
                     double scale, bool want_gdo, int64_t window, int64_t window_kind,
                     const c10::optional<at::Tensor>& bias) {
    if (g_library_choice.load()) return false;
    py::gil_scoped_acquire gil;
    const py::tuple out = py::handle(g_python_gg)(s[0], s[1], s[2], s[3], s[4], p, s[6], s[7], g[0], g[1], g[2],
                                                  causal, scale, want_gdo, window, window_kind, bias);
    for (const py::handle t : out) r->push_back(t.is_none() ? at::Tensor() : t.cast<at::Tensor>());
    return true;
  }

  static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx,
                                                 torch::autograd::variable_list g) {
    const bool twice = at::GradMode::is_enabled() &&
                       std::any_of(g.begin(), g.end(), [](const at::Tensor& t) { return t.requires_grad(); });
    torch::autograd::variable_list out;
    {
      at::NoGradGuard no_grad;
      const torch::autograd::variable_list s = ctx->get_saved_variables();
      for (at::Tensor& t : g)
        if (t.scalar_type() != s[0].scalar_type()) t = t.to(s[0].scalar_type());
      const bool want_gdo = ctx->needs_input_grad(3);
      const c10::optional<at::Tensor> p = s[5].defined() ? c10::make_optional(s[5]) : c10::nullopt;
      const bool causal = ctx->saved_data["causal"].toBool();
      const double scale = ctx->saved_data["scale"].toDouble();
      const int64_t window = ctx->saved_data["window"].toInt(), window_kind = ctx->saved_data["window_kind"].toInt();
      const c10::optional<at::Tensor> bias = ctx->saved_data["bias"].toOptional<at::Tensor>();
      std::vector<at::Tensor> r;
      if (!forced(&r, s, g, p, causal, scale, want_gdo, window, window_kind, bias))
        r = gg_fused(s[0], s[1], s[2], s[3], s[4], p, s[6], s[7], g[0], g[1], g[2], causal, scale, want_gdo, window,
                     window_kind, bias, 0);
      for (int i = 0; i < 4; ++i)
        out.push_back(ctx->needs_input_grad(i) ? r[i] : at::Tensor());
      out.emplace_back();  // the saved forward
    }
    if (!twice) return out;
    // A third derivative fails when it is asked for, as once_differentiable's does.
    torch::autograd::variable_list vars;
    for (at::Tensor& t : out)
      if (t.defined()) vars.push_back(t.detach().set_requires_grad(true));
    const auto err = std::make_shared<torch::autograd::DelayedError>(
        "trying to differentiate twice a function that was marked with @once_differentiable", vars.size());
    vars = (*err)(std::move(vars));
    size_t n = 0;
    for (at::Tensor& t : out)
      if (t.defined()) t = vars[n++];
    return out;
  }
};

// (dQ, dK, dV) with the double backward behind them.
std::vector<at::Tensor> bwd_graph(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v,
                                  const at::Tensor& dout, const at::Tensor& o, const at::Tensor& lse,
                                  const c10::optional<at::Tensor>& p, bool causal, double scale, int64_t window,
                                  int64_t window_kind, const c10::optional<at::Tensor>& bias) {
  // O is detached: the saved node holds no edge into the forward's graph
  return AttnBwd::apply(q, k, v, dout,
                        SavedForward{o.detach(), lse, p, bias, causal, scale, window, window_kind});
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.doc() = "torch binding of the forward, backward and double backward of libttt_attn.so";
  m.def("fwd", &fwd, "forward: (O, LSE, P or None)");
  m.def("bwd", &bwd, "first backward: (dQ, dK, dV, D)");
  m.def("bwd_fused", &bwd_fused, "first backward in one entry call: (dQ, dK, dV, D)");
  m.def("bwd_graph", &bwd_graph, "differentiable first backward: (dQ, dK, dV)");
  m.def("set_library_choice", &set_library_choice, "whether bwd_graph's double backward takes the library's choice");
  m.def("set_python_gg", &set_python_gg, "the Python layer's double backward, for every other case");
  m.def("gg", &gg, "double backward: (GQ, GK, GV, GdO or None)");
  m.def("gg_fused", &gg_fused, "double backward in one entry call: (GQ, GK, GV, GdO or None)");
}
