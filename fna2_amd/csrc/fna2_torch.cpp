// fna2_torch.cpp — the launch path of the Python entry points in native code.
//
// Fills the argument structs of include/fna2.h from torch tensors, allocates
// outputs and workspace and calls the C ABI on torch's current HIP stream:
// what the Python launchers (flash_naylis_attn.py, decode.py, rope.py) do
// through ctypes.  What it saves is host time: a training pass of one small
// layer spends most of its time in these launchers, the backward's share of
// it on autograd's own thread, where every Python object the launcher
// touches is first fetched from the other core's cache (B1 H8 L512 d64,
// forward + backward: 240 us a pass, 85 of them GPU work).
//
// Each function takes the ordinary call only: tensors of the expected
// shapes and dtypes, on one device, laid out as the kernels read them.  For
// anything else, and for a call the C ABI refuses (nothing is launched
// then), it returns None, and the caller's Python launcher makes the copies
// or raises the error, as without this file.  A launch that fails raises
// here: other kernels of the call may be queued by then, so it is not
// repeated.
//
// The library's functions come as addresses (bind), so that the binding
// always calls the library that _capi.py loaded.
#include <c10/hip/HIPStream.h>
#include <torch/extension.h>

#include <cstring>
#include <map>
#include <optional>
#include <string>
#include <tuple>

#include "fna2.h"

namespace {

using at::Tensor;
using OptTensor = std::optional<Tensor>;

struct Lib {
  decltype(&fna2_fwd) fwd;
  decltype(&fna2_bwd) bwd;
  decltype(&fna2_fwd_workspace_bytes) fwd_workspace_bytes;
  decltype(&fna2_bwd_workspace_bytes) bwd_workspace_bytes;
  decltype(&fna2_bwd_split_bytes) bwd_split_bytes;
  decltype(&fna2_decode) decode;
  decltype(&fna2_decode_workspace_bytes) decode_workspace_bytes;
  decltype(&fna2_check_decode) check_decode;
  decltype(&fna2_decode_rows) decode_rows;
  decltype(&fna2_rope_varlen) rope_varlen;
  decltype(&fna2_rope_bwd) rope_bwd;
  decltype(&fna2_rope_bwd_workspace_bytes) rope_bwd_workspace_bytes;
};
Lib L{};

PyObject* launch_error = nullptr;  // the exception class (never freed)

// Whether a call was launched; false where the C ABI refused it.
bool launched(int status, const char* what) {
  if (status == FNA2_E_LAUNCH) {
    const py::gil_scoped_acquire gil;
    PyErr_Format(launch_error, "%s: FNA2_E_LAUNCH: kernel launch failed", what);
    throw py::error_already_set();
  }
  return status == FNA2_OK;
}

void bind(const std::map<std::string, uintptr_t>& f, py::object error) {
  launch_error = error.release().ptr();
#define FNA2_BIND(n) L.n = reinterpret_cast<decltype(L.n)>(f.at("fna2_" #n))
  FNA2_BIND(fwd);
  FNA2_BIND(bwd);
  FNA2_BIND(fwd_workspace_bytes);
  FNA2_BIND(bwd_workspace_bytes);
  FNA2_BIND(bwd_split_bytes);
  FNA2_BIND(decode);
  FNA2_BIND(decode_workspace_bytes);
  FNA2_BIND(check_decode);
  FNA2_BIND(decode_rows);
  FNA2_BIND(rope_varlen);
  FNA2_BIND(rope_bwd);
  FNA2_BIND(rope_bwd_workspace_bytes);
#undef FNA2_BIND
}

// A plain strided GPU tensor with data, on `dev`.
bool plain(const Tensor& t, const c10::Device& dev) {
  return t.defined() && t.is_cuda() && t.device() == dev && t.layout() == c10::kStrided &&
         !t.unsafeGetTensorImpl()->is_python_dispatch() && t.numel() > 0;
}

// Unit feature stride, 16-byte aligned rows.
bool rows16(const Tensor& t) {
  const int64_t d = t.dim(), unit = 16 / (int64_t)t.element_size();
  if (d < 1 || t.stride(d - 1) != 1 || (uintptr_t)t.data_ptr() % 16) return false;
  for (int64_t i = 0; i + 1 < d; ++i)
    if (t.stride(i) % unit) return false;
  return true;
}

bool int32_on(const Tensor& t, const c10::Device& dev) {
  return plain(t, dev) && t.scalar_type() == at::kInt && t.is_contiguous();
}

bool float_on(const Tensor& t, const c10::Device& dev, int64_t n) {
  return plain(t, dev) && t.scalar_type() == at::kFloat && t.is_contiguous() && t.numel() == n;
}

// Dense [B, h, S(, F)] or packed [T, h(, F)].
fna2_tensor view(const Tensor& t, bool packed) {
  fna2_tensor v{};
  if (!t.defined() || t.numel() == 0) return v;
  v.ptr = t.data_ptr();
  v.stride_b = packed ? 0 : t.stride(0);
  v.stride_s = packed ? t.stride(0) : t.stride(2);
  v.stride_h = t.stride(1);
  return v;
}

void* stream_of(const c10::Device& d) {
  return (void*)c10::hip::getCurrentHIPStream(d.index()).stream();
}

Tensor bytes_on(size_t n, const Tensor& like) {
  return at::empty({(int64_t)std::max<size_t>(n, 1)}, like.options().dtype(at::kByte));
}

// The backward's workspace, with room for dK/dV items in chunks where the
// library would use them (up to 512 MiB) and the memory is there: without
// the room it runs the items whole.
Tensor bwd_workspace(const fna2_problem& p, const Tensor& like) {
  const size_t need = L.bwd_workspace_bytes(&p), chunks = L.bwd_split_bytes(&p);
  if (chunks > 0) {
    try {
      return bytes_on(need + chunks, like);
    } catch (const c10::OutOfMemoryError&) {
    }
  }
  return bytes_on(need, like);
}

// The problem of an attention call, or false for the Python launcher.
struct Call {
  fna2_problem p{};
  bool packed = false;
  int64_t HG = 0;
};

bool problem(Call& c, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& rq,
             const Tensor& rk, const Tensor& gs, double scale, bool causal, const Tensor& cu_q,
             const Tensor& cu_k, int64_t max_q, int64_t max_k) {
  if (!L.fwd || !q.defined() || !q.is_cuda()) return false;
  const c10::Device dev = q.device();
  c.packed = cu_q.defined();
  const int64_t nd = c.packed ? 3 : 4, f = nd - 1, s = c.packed ? 0 : 2;
  const auto dt = q.scalar_type();
  if (dt != at::kBFloat16 && dt != at::kHalf) return false;
  for (const Tensor* t : {&q, &k, &v})
    if (!plain(*t, dev) || t->dim() != nd || t->scalar_type() != dt || !rows16(*t)) return false;
  const int64_t H = q.size(1), HKV = k.size(1), D = q.size(f);
  if ((D != 64 && D != 128) || k.size(f) != D || H % HKV || v.sizes() != k.sizes()) return false;
  if (!c.packed && k.size(0) != q.size(0)) return false;
  int64_t R = 0;
  c.HG = 0;
  if (rq.defined()) {
    if (!rk.defined() || !gs.defined()) return false;
    for (const Tensor* t : {&rq, &rk})
      if (!plain(*t, dev) || t->dim() != nd || t->scalar_type() != at::kBFloat16 || !rows16(*t))
        return false;
    c.HG = rq.size(1);
    R = rq.size(f);
    if (c.HG > H || rk.size(1) != c.HG || rk.size(f) != R || R % 8 || R > 64) return false;
    if (rq.size(s) != q.size(s) || rk.size(s) != k.size(s)) return false;
    if (!c.packed && (rq.size(0) != q.size(0) || rk.size(0) != q.size(0))) return false;
    if (!float_on(gs, dev, c.HG)) return false;
  } else if (rk.defined()) {
    return false;
  }
  fna2_problem& p = c.p;
  p.dtype = dt == at::kHalf ? FNA2_F16 : FNA2_BF16;
  p.varlen = c.packed;
  if (c.packed) {
    if (!int32_on(cu_q, dev) || !int32_on(cu_k, dev) || cu_q.dim() != 1 || cu_k.dim() != 1 ||
        cu_q.numel() < 2 || cu_k.numel() != cu_q.numel())
      return false;
    if (q.size(0) > INT32_MAX || k.size(0) > INT32_MAX) return false;
    p.batch = (int32_t)(cu_q.numel() - 1);
    p.seqlen_q = (int32_t)std::min<int64_t>(std::max<int64_t>(max_q, 0), INT32_MAX);
    p.seqlen_k = (int32_t)std::min<int64_t>(std::max<int64_t>(max_k, 0), INT32_MAX);
    p.total_q = (int32_t)q.size(0);
    p.total_k = (int32_t)k.size(0);
    p.cu_seqlens_q = cu_q.data_ptr<int32_t>();
    p.cu_seqlens_k = cu_k.data_ptr<int32_t>();
  } else {
    if (q.size(0) > INT32_MAX || q.size(2) > INT32_MAX || k.size(2) > INT32_MAX) return false;
    p.batch = (int32_t)q.size(0);
    p.seqlen_q = (int32_t)q.size(2);
    p.seqlen_k = (int32_t)k.size(2);
  }
  p.heads = (int32_t)H;
  p.heads_kv = (int32_t)HKV;
  p.heads_graph = (int32_t)c.HG;
  p.head_dim = (int32_t)D;
  p.rank = (int32_t)R;
  p.causal = causal;
  p.softmax_scale = (float)scale;
  return true;
}

const Tensor kNone;
const Tensor& opt(const OptTensor& t) { return t.has_value() ? *t : kNone; }

// _fna2_forward / _fna2_forward_varlen: (out, lse).
std::optional<std::tuple<Tensor, Tensor>> attn_fwd(
    const Tensor& q, const Tensor& k, const Tensor& v, const OptTensor& rq_, const OptTensor& rk_,
    const OptTensor& gs_, double scale, bool causal, const OptTensor& cu_q, const OptTensor& cu_k,
    int64_t max_q, int64_t max_k, const OptTensor& plan_, bool plan_filled, bool head_major) {
  const Tensor &rq = opt(rq_), &rk = opt(rk_), &gs = opt(gs_), &plan = opt(plan_);
  Call c;
  if (!problem(c, q, k, v, rq, rk, gs, scale, causal, opt(cu_q), opt(cu_k), max_q, max_k))
    return std::nullopt;
  const c10::DeviceGuard guard(q.device());
  const Tensor out = at::empty_like(q);
  const auto f32 = q.options().dtype(at::kFloat);
  const int64_t H = q.size(1);
  const Tensor lse = !c.packed    ? at::empty({q.size(0), H, q.size(2)}, f32)
                     : head_major ? at::empty({H, q.size(0)}, f32).t()
                                  : at::empty({q.size(0), H}, f32);
  const Tensor ws = bytes_on(L.fwd_workspace_bytes(&c.p), q);
  fna2_fwd_args a{};
  a.p = c.p;
  a.q = view(q, c.packed);
  a.k = view(k, c.packed);
  a.v = view(v, c.packed);
  if (c.HG) {
    a.r_q = view(rq, c.packed);
    a.r_k = view(rk, c.packed);
    a.graph_scale = gs.data_ptr<float>();
  }
  a.out = view(out, c.packed);
  a.lse = view(lse, c.packed);
  a.workspace = ws.data_ptr();
  a.workspace_bytes = (size_t)ws.numel();
  if (plan.defined()) {
    a.plan = plan.data_ptr();
    a.plan_bytes = (size_t)plan.numel();
    a.plan_filled = plan_filled;
  }
  if (!launched(L.fwd(&a, stream_of(q.device())), "fna2_fwd")) return std::nullopt;
  return std::make_tuple(out, lse);
}

using Grads = std::tuple<Tensor, Tensor, Tensor, OptTensor, OptTensor, OptTensor>;

// _fna2_backward / _fna2_backward_varlen: (dq, dk, dv, dr_q, dr_k, d_gs).
// dv_, drq_, drk_: where to write them (rows of any stride).
std::optional<Grads> attn_bwd(const Tensor& dout, const Tensor& q, const Tensor& k,
                              const Tensor& v, const OptTensor& rq_, const OptTensor& rk_,
                              const OptTensor& gs_, const Tensor& out, const Tensor& lse,
                              double scale, bool causal, const OptTensor& cu_q,
                              const OptTensor& cu_k, int64_t max_q, int64_t max_k,
                              const OptTensor& plan_, const OptTensor& dv_, const OptTensor& drq_,
                              const OptTensor& drk_) {
  const Tensor &rq = opt(rq_), &rk = opt(rk_), &gs = opt(gs_), &plan = opt(plan_);
  Call c;
  if (!problem(c, q, k, v, rq, rk, gs, scale, causal, opt(cu_q), opt(cu_k), max_q, max_k))
    return std::nullopt;
  const c10::Device dev = q.device();
  for (const Tensor* t : {&dout, &out})
    if (!plain(*t, dev) || t->scalar_type() != q.scalar_type() || t->sizes() != q.sizes() ||
        !rows16(*t))
      return std::nullopt;
  if (!plain(lse, dev) || lse.scalar_type() != at::kFloat ||
      lse.sizes() != q.sizes().slice(0, q.dim() - 1) || (!c.packed && !lse.is_contiguous()))
    return std::nullopt;
  auto given = [&](const OptTensor& g, const Tensor& like) {
    return !g.has_value() || (plain(*g, dev) && g->scalar_type() == like.scalar_type() &&
                              g->sizes() == like.sizes());
  };
  if (!given(dv_, v) || (c.HG && (!given(drq_, rq) || !given(drk_, rk)))) return std::nullopt;
  const c10::DeviceGuard guard(dev);
  const auto f32 = q.options().dtype(at::kFloat);
  const int64_t H = q.size(1);
  const Tensor delta = c.packed ? at::empty({H, q.size(0)}, f32).t()
                                : at::empty({q.size(0), H, q.size(2)}, f32);
  const Tensor dq = at::empty_like(q), dk = at::empty_like(k);
  const Tensor dv = dv_.has_value() ? *dv_ : at::empty_like(v);
  Tensor drq, drk, dgs;
  fna2_bwd_args a{};
  if (c.HG) {
    drq = drq_.has_value() ? *drq_ : at::empty_like(rq);
    drk = drk_.has_value() ? *drk_ : at::empty_like(rk);
    dgs = at::empty({c.HG}, f32);
    a.r_q = view(rq, c.packed);
    a.r_k = view(rk, c.packed);
    a.graph_scale = gs.data_ptr<float>();
    a.dr_q = view(drq, c.packed);
    a.dr_k = view(drk, c.packed);
    a.d_graph_scale = dgs.data_ptr<float>();
  }
  const Tensor ws = bwd_workspace(c.p, q);
  a.p = c.p;
  a.q = view(q, c.packed);
  a.k = view(k, c.packed);
  a.v = view(v, c.packed);
  a.out = view(out, c.packed);
  a.lse = view(lse, c.packed);
  a.dout = view(dout, c.packed);
  a.delta = view(delta, c.packed);
  a.dq = view(dq, c.packed);
  a.dk = view(dk, c.packed);
  a.dv = view(dv, c.packed);
  a.workspace = ws.data_ptr();
  a.workspace_bytes = (size_t)ws.numel();
  if (plan.defined()) {
    a.plan = plan.data_ptr();
    a.plan_bytes = (size_t)plan.numel();
  }
  if (!launched(L.bwd(&a, stream_of(dev)), "fna2_bwd")) return std::nullopt;
  auto some = [](const Tensor& t) { return t.defined() ? OptTensor(t) : std::nullopt; };
  return Grads(dq, dk, dv, some(drq), some(drk), some(dgs));
}

// flash_naylis_decode: (out, lse).
std::optional<std::tuple<Tensor, Tensor>> decode(const Tensor& q_, const Tensor& kc,
                                                 const Tensor& vc, const OptTensor& rq_,
                                                 const OptTensor& rkc_, const OptTensor& gs_,
                                                 double scale, const OptTensor& seq_,
                                                 int64_t num_splits) {
  const Tensor &rkc = opt(rkc_), &seq = opt(seq_);
  Tensor gs = opt(gs_);
  if (!L.decode || !q_.defined() || !q_.is_cuda()) return std::nullopt;
  const c10::Device dev = q_.device();
  // [B, H, F], or [B, H, 1, F] with the row dimension dropped
  auto row = [&](const Tensor& t, Tensor& out) {
    if (!plain(t, dev) || t.scalar_type() != at::kBFloat16) return false;
    if (t.dim() == 4 && t.size(2) == 1)
      out = t.select(2, 0);
    else if (t.dim() == 3)
      out = t;
    else
      return false;
    return rows16(out);
  };
  auto cache = [&](const Tensor& t, int64_t B, int64_t F) {
    return plain(t, dev) && t.scalar_type() == at::kBFloat16 && t.dim() == 4 && t.size(0) == B &&
           t.size(3) == F && rows16(t);
  };
  Tensor q, rq;
  if (!row(q_, q)) return std::nullopt;
  const int64_t B = q.size(0), H = q.size(1), D = q.size(2);
  if (!cache(kc, B, D) || !cache(vc, B, D) || kc.sizes() != vc.sizes()) return std::nullopt;
  if (num_splits < 0 || num_splits > 64 || kc.size(2) > INT32_MAX) return std::nullopt;
  fna2_decode_args a{};
  a.batch = (int32_t)B;
  a.heads = (int32_t)H;
  a.heads_kv = (int32_t)kc.size(1);
  a.head_dim = (int32_t)D;
  a.max_seqlen_k = (int32_t)kc.size(2);
  a.num_splits = (int32_t)num_splits;
  a.softmax_scale = (float)scale;
  auto row_view = [](const Tensor& t) {
    fna2_tensor v{};
    v.ptr = t.data_ptr();
    v.stride_b = t.stride(0);
    v.stride_h = t.stride(1);
    return v;
  };
  if (rq_.has_value()) {
    if (!row(*rq_, rq) || rq.size(0) != B || !rkc.defined() || !plain(gs, dev) ||
        !gs.is_floating_point())
      return std::nullopt;
    gs = gs.detach().to(at::kFloat).contiguous();  // (a module's parameter is bf16)
    if (!cache(rkc, B, rq.size(2)) || rkc.size(1) != rq.size(1) || rkc.size(2) != kc.size(2) ||
        !float_on(gs, dev, rq.size(1)))
      return std::nullopt;
    a.heads_graph = (int32_t)rq.size(1);
    a.rank = (int32_t)rq.size(2);
    a.r_q = row_view(rq);
    a.rk_cache = view(rkc, false);
    a.graph_scale = gs.data_ptr<float>();
  }
  if (seq.defined()) {
    if (!int32_on(seq, dev) || seq.numel() != B) return std::nullopt;
    a.seqlens_k = seq.data_ptr<int32_t>();
  }
  const c10::DeviceGuard guard(dev);
  const Tensor out = at::empty({B, H, D}, q.options());
  const Tensor lse = at::empty({B, H}, q.options().dtype(at::kFloat));
  a.q = row_view(q);
  a.k_cache = view(kc, false);
  a.v_cache = view(vc, false);
  a.out = row_view(out);
  a.lse = row_view(lse);
  if (L.check_decode(&a) != FNA2_OK) return std::nullopt;
  const size_t need = L.decode_workspace_bytes(&a);
  Tensor ws;
  if (need > 0) {
    ws = bytes_on(need, q);
    a.workspace = ws.data_ptr();
    a.workspace_bytes = need;
  }
  if (!launched(L.decode(&a, stream_of(dev)), "fna2_decode")) return std::nullopt;
  return std::make_tuple(out, lse);
}

// The rows of a decode step: normalised and rotated q as [B, H, D]; k, v and
// r_k into k_out, v_out and rk_out.  All [B, heads, 1, F]; norm weights and
// the cos / sin rows [D], bf16.  None, with nothing written: not this call.
OptTensor decode_rows(const Tensor& q, const Tensor& k, const Tensor& v, const OptTensor& rk_,
                      const Tensor& k_out, const Tensor& v_out, const OptTensor& rko_,
                      const OptTensor& nq, double eps_q, const OptTensor& nk, double eps_k,
                      const OptTensor& cos, const OptTensor& sin) {
  if (!L.decode_rows || !q.defined() || !q.is_cuda()) return std::nullopt;
  const c10::Device dev = q.device();
  auto rows = [&](const Tensor& t) {
    return plain(t, dev) && t.scalar_type() == at::kBFloat16 && t.dim() == 4 && t.size(2) == 1 &&
           t.size(0) == q.size(0) && rows16(t);
  };
  if (!rows(q)) return std::nullopt;
  const int64_t D = q.size(3);
  for (const Tensor* t : {&k, &v, &k_out, &v_out})
    if (!rows(*t) || t->sizes() != k.sizes()) return std::nullopt;
  if (k.size(3) != D || rk_.has_value() != rko_.has_value()) return std::nullopt;
  fna2_decode_rows_args a{};
  auto vec = [&](const OptTensor& t, const void*& p) {
    if (!t.has_value()) return true;
    if (!plain(*t, dev) || t->scalar_type() != at::kBFloat16 || !t->is_contiguous() ||
        t->numel() != D || (uintptr_t)t->data_ptr() % 16)
      return false;
    p = t->data_ptr();
    return true;
  };
  if (!vec(nq, a.norm_q) || !vec(nk, a.norm_k) || !vec(cos, a.cos) || !vec(sin, a.sin))
    return std::nullopt;
  auto row_view = [](const Tensor& t) {
    fna2_tensor v{};
    v.ptr = t.data_ptr();
    v.stride_b = t.stride(0);
    v.stride_h = t.stride(1);
    return v;
  };
  a.batch = (int32_t)q.size(0);
  a.heads = (int32_t)q.size(1);
  a.heads_kv = (int32_t)k.size(1);
  a.head_dim = (int32_t)D;
  if (rk_.has_value()) {
    if (!rows(*rk_) || !rows(*rko_) || rk_->sizes() != rko_->sizes()) return std::nullopt;
    a.heads_graph = (int32_t)rk_->size(1);
    a.rank = (int32_t)rk_->size(3);
    a.r_k = row_view(*rk_);
    a.rk_out = row_view(*rko_);
  }
  // The cache rows are written in place, as torch's copy_ would: an inference
  // tensor only in inference mode, any other with its version counted up.
  const Tensor* written[3] = {&k_out, &v_out, rko_.has_value() ? &*rko_ : nullptr};
  for (const Tensor* t : written)
    if (t && t->is_inference() && !c10::InferenceMode::is_enabled()) return std::nullopt;
  const c10::DeviceGuard guard(dev);
  const Tensor out = at::empty({q.size(0), q.size(1), D}, q.options());
  a.q = row_view(q);
  a.k = row_view(k);
  a.v = row_view(v);
  a.q_out = row_view(out);
  a.k_out = row_view(k_out);
  a.v_out = row_view(v_out);
  a.eps_q = (float)eps_q;
  a.eps_k = (float)eps_k;
  if (!launched(L.decode_rows(&a, stream_of(dev)), "fna2_decode_rows")) return std::nullopt;
  for (const Tensor* t : written)
    if (t && !t->is_inference()) t->unsafeGetTensorImpl()->bump_version();
  return out;
}

// The arguments rope_varlen's forward and backward share.  w: the norm
// weights and inv_freq in fp32 (kept by the caller).
bool rope_args(fna2_rope_args& a, const Tensor& q, const Tensor& k, const Tensor& cu,
               const Tensor& inv, int64_t sign, const OptTensor& nq, const OptTensor& nk,
               double eps, Tensor (&w)[3]) {
  if (!L.rope_varlen || !q.defined() || !q.is_cuda()) return false;
  const c10::Device dev = q.device();
  const auto dt = q.scalar_type();
  if (dt != at::kBFloat16 && dt != at::kHalf && dt != at::kFloat) return false;
  for (const Tensor* t : {&q, &k})
    if (!plain(*t, dev) || t->dim() != 3 || t->scalar_type() != dt || !rows16(*t)) return false;
  const int64_t D = q.size(2);
  if (k.size(0) != q.size(0) || k.size(2) != D || q.size(0) > INT32_MAX) return false;
  if (!int32_on(cu, dev) || !plain(inv, dev) || inv.numel() != D / 2 || !inv.is_floating_point())
    return false;
  w[2] = inv.to(at::kFloat).contiguous();
  const OptTensor* norms[2] = {&nq, &nk};
  for (int i = 0; i < 2; ++i) {
    if (!norms[i]->has_value()) continue;
    const Tensor& n = **norms[i];
    if (!plain(n, dev) || n.numel() != D || !n.is_floating_point()) return false;
    w[i] = n.detach().to(at::kFloat).contiguous();
  }
  a.dtype = dt == at::kHalf ? FNA2_F16 : dt == at::kFloat ? FNA2_F32 : FNA2_BF16;
  a.total_tokens = (int32_t)q.size(0);
  a.heads_q = (int32_t)q.size(1);
  a.heads_k = (int32_t)k.size(1);
  a.head_dim = (int32_t)D;
  a.nseq = (int32_t)(cu.numel() - 1);
  a.sign = (int32_t)sign;
  a.cu_seqlens = cu.data_ptr<int32_t>();
  a.inv_freq = w[2].data_ptr<float>();
  a.q = view(q, true);
  a.k = view(k, true);
  a.norm_q = w[0].defined() ? w[0].data_ptr<float>() : nullptr;
  a.norm_k = w[1].defined() ? w[1].data_ptr<float>() : nullptr;
  a.norm_eps = (float)eps;
  return true;
}

std::optional<std::tuple<Tensor, Tensor>> rope_fwd(const Tensor& q, const Tensor& k,
                                                   const Tensor& cu, const Tensor& inv,
                                                   int64_t sign, const OptTensor& nq,
                                                   const OptTensor& nk, double eps) {
  fna2_rope_args a{};
  Tensor w[3];
  const c10::OptionalDeviceGuard guard(at::device_of(q));
  if (!rope_args(a, q, k, cu, inv, sign, nq, nk, eps, w)) return std::nullopt;
  const Tensor qo = at::empty_like(q, at::MemoryFormat::Contiguous);
  const Tensor ko = at::empty_like(k, at::MemoryFormat::Contiguous);
  a.q_out = view(qo, true);
  a.k_out = view(ko, true);
  if (!launched(L.rope_varlen(&a, stream_of(q.device())), "fna2_rope_varlen")) return std::nullopt;
  return std::make_tuple(qo, ko);
}

// rope_varlen_bwd: (dq, dk, dnorm_q, dnorm_k).
std::optional<std::tuple<Tensor, Tensor, OptTensor, OptTensor>> rope_bwd(
    const Tensor& dqo, const Tensor& dko, const Tensor& q, const Tensor& k, const Tensor& cu,
    const Tensor& inv, int64_t sign, const OptTensor& nq, const OptTensor& nk, double eps,
    const OptTensor& dq_, const OptTensor& dk_) {
  fna2_rope_bwd_args b{};
  Tensor w[3];
  const c10::OptionalDeviceGuard guard(at::device_of(q));
  if (!rope_args(b.fwd, q, k, cu, inv, sign, nq, nk, eps, w)) return std::nullopt;
  const c10::Device dev = q.device();
  auto like = [&](const Tensor& t, const Tensor& x) {
    return plain(t, dev) && t.scalar_type() == x.scalar_type() && t.sizes() == x.sizes();
  };
  if (!like(dqo, q) || !like(dko, k) || !rows16(dqo) || !rows16(dko)) return std::nullopt;
  if ((dq_.has_value() && !like(*dq_, q)) || (dk_.has_value() && !like(*dk_, k)))
    return std::nullopt;
  const Tensor dq = dq_.has_value() ? *dq_ : at::empty_like(q, at::MemoryFormat::Contiguous);
  const Tensor dk = dk_.has_value() ? *dk_ : at::empty_like(k, at::MemoryFormat::Contiguous);
  b.dq_out = view(dqo, true);
  b.dk_out = view(dko, true);
  b.dq = view(dq, true);
  b.dk = view(dk, true);
  OptTensor dn[2];
  for (int i = 0; i < 2; ++i)
    if (w[i].defined()) dn[i] = at::empty_like(w[i]);
  b.dnorm_q = dn[0] ? dn[0]->data_ptr<float>() : nullptr;
  b.dnorm_k = dn[1] ? dn[1]->data_ptr<float>() : nullptr;
  const size_t need = L.rope_bwd_workspace_bytes(&b.fwd);
  Tensor ws;
  if (need > 0) {
    ws = bytes_on(need, q);
    b.workspace = ws.data_ptr();
    b.workspace_bytes = need;
  }
  if (!launched(L.rope_bwd(&b, stream_of(dev)), "fna2_rope_bwd")) return std::nullopt;
  return std::make_tuple(dq, dk, dn[0], dn[1]);
}

}  // namespace

PYBIND11_MODULE(_torch_binding, m) {
  // (no Python object is touched inside: other threads run meanwhile)
  using Free = py::call_guard<py::gil_scoped_release>;
  m.def("bind", &bind);
  m.def("attn_fwd", &attn_fwd, Free());
  m.def("attn_bwd", &attn_bwd, Free());
  m.def("decode", &decode, Free());
  m.def("decode_rows", &decode_rows, Free());
  m.def("rope_fwd", &rope_fwd, Free());
  m.def("rope_bwd", &rope_bwd, Free());
}
