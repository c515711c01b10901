// Host side of the Python package in native code: fills the C ABI's argument structs from torch tensors, allocates
// results and workspaces from torch's caching allocator and issues the launch sequences of the flash-entropy and
// VMonarch attention, forward and backward.
//
// Why native: a VMonarch forward of two iterations is five or six launches (R- and L-steps, the exact recompute beside
// R-step 0, the merge of its key ranges where it has several), in some orders with a second stream's fork and join.
// Issued from Python through ctypes each launch cost ~20 us of host time (struct fields, views, allocations, stream
// queries) against 4-20 us of GPU time at small sizes, so small calls ran at the host's pace.  Back to back on one box,
// the same launches from Python -> from here, in us: VMonarch forward of a 4 x 64 grid 135 -> 61, of 16 x 256 (batch 2,
// 4 heads) 139 -> 70 (with the recompute in R-step 0's launch, without the fork: 21 and 58); flash-entropy forward
// (1, 2, 1024, 64) 30 -> 17 (key-group kernel: 9.6), its training step at (2, 4, 1000, 64) 224 -> 115.
//
// Every call only issues work on the current stream (and the given side stream, joined before returning); nothing
// is kept between calls, and no check is cached.  Types and devices are checked here, sizes, strides and alignment by
// the C ABI (include/vmonarch_amd.h), all before a launch.
#include <Python.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/extension.h>

#include <algorithm>
#include <array>
#include <initializer_list>
#include <optional>
#include <stdexcept>
#include <string>
#include <tuple>
#include <utility>
#include <vector>

#include "../../include/vmonarch_amd.h"

namespace py = pybind11;
using at::Tensor;
using OptT = std::optional<Tensor>;

namespace {

// Everything below runs without the interpreter lock, so that other Python threads go on through launches, allocations
// and whatever waits they lead to in the driver: no Python object is touched, and errors are C++ exceptions that the
// binding turns into Python's once it holds the lock again.  (std::runtime_error: RuntimeError.)
struct assertion_error : py::builtin_exception {
  using builtin_exception::builtin_exception;
  void set_error() const override { PyErr_SetString(PyExc_AssertionError, what()); }
};
struct zero_division_error : py::builtin_exception {
  using builtin_exception::builtin_exception;
  void set_error() const override { PyErr_SetString(PyExc_ZeroDivisionError, what()); }
};

void require(bool ok, const char* msg) {
  if (!ok) throw assertion_error(msg);
}

void whole_frames(int64_t nq, int64_t nk, int64_t frames) {
  if (frames == 0) throw zero_division_error("no frames");
  require(nq % frames == 0 && nk % frames == 0, "whole frames");
}

int dtype_code(const Tensor& t) {
  if (t.scalar_type() == at::kBFloat16) return VMO_DTYPE_BF16;
  if (t.scalar_type() == at::kHalf) return VMO_DTYPE_F16;
  throw py::key_error(std::string("torch.") + c10::toString(t.scalar_type()));
}

// The kernels take every tensor's type and place from q, so a tensor of another type would be read as what it is not, and
// one elsewhere through an address the GPU does not have.
// OnGpuOf(q): q's GPU is the current one while this lives, as a null stream and an event's creation take that.
struct OnGpuOf {
  c10::OptionalDeviceGuard guard;
  explicit OnGpuOf(const Tensor& q) {
    if (!q.is_cuda()) throw py::value_error("vmonarch_amd: needs GPU tensors, got " + q.device().str());
    if (c10::hip::current_device() != q.device().index()) guard.reset_device(q.device());
  }
};
void same_device(const Tensor& q, const Tensor& t) { require(t.device() == q.device(), "all tensors on one GPU: q's device"); }
void like(const Tensor& q, const Tensor& t) {
  require(t.scalar_type() == q.scalar_type(), "all of one dtype: q's");
  same_device(q, t);
}
void like(const Tensor& q, std::initializer_list<const Tensor*> ts) {
  for (const Tensor* t : ts)
    if (t) like(q, *t);
}
void same_device(const Tensor& q, std::initializer_list<const Tensor*> ts) {
  for (const Tensor* t : ts)
    if (t) same_device(q, *t);
}

// (B, H, N, F) tensor -> view (element strides, feature dim contiguous)
vmo_view view(const Tensor& t) {
  require(t.dim() == 4 && t.stride(3) == 1, "feature dimension must be contiguous");
  return vmo_view{t.data_ptr(), t.stride(0), t.stride(1), t.stride(2)};
}

// t itself when its rows are 16-byte aligned with a contiguous feature dim, else a contiguous copy
Tensor row_aligned(const Tensor& t) {
  bool ok = t.stride(-1) == 1 && reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
  for (int64_t d = 0; ok && d < t.dim() - 1; ++d) ok = t.stride(d) % 8 == 0;
  return ok ? t : t.contiguous();
}

using Order = std::array<int, 3>;
// order of t's (B, H, N) dims in memory, outermost first (by stride)
Order layout_order(const Tensor& t) {
  Order o{0, 1, 2};
  std::stable_sort(o.begin(), o.end(), [&](int a, int b) { return t.stride(a) > t.stride(b); });
  return o;
}
// an uninitialised (B, H, N, feat) tensor whose (B, H, N) dims lie in memory in `order`, feature dim innermost
Tensor empty_in_order(const Order& order, const int64_t (&dims)[3], int64_t feat, const at::TensorOptions& opt) {
  int64_t st[3], s = feat;
  for (int i = 2; i >= 0; --i) {
    st[order[i]] = s;
    s *= std::max<int64_t>(dims[order[i]], 1);   // (torch's strides of an empty dim)
  }
  return at::empty_strided({dims[0], dims[1], dims[2], feat}, {st[0], st[1], st[2], 1}, opt);
}
Tensor empty_in_layout(const Tensor& ref, int64_t feat) {
  const int64_t dims[3] = {ref.size(0), ref.size(1), ref.size(2)};
  return empty_in_order(layout_order(ref), dims, feat, ref.options());
}
at::TensorOptions f32(const Tensor& t) { return t.options().dtype(at::kFloat); }

void* stream_of(const Tensor& t) { return (void*)c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

void check(int rc, const char* what) {
  if (rc != 0)
    throw std::runtime_error(std::string(what) + " failed (code " + std::to_string(rc) + "): " + vmo_last_error());
}

// ---- single launches -------------------------------------------------------------------------------------------

// q: F*nq rows; k, w0, w1: F*nk rows; o, lse, ent optional outputs.  rows >= 0: only the first `rows` queries.
struct FwdCall {
  const Tensor &q, &k, &w0;
  const Tensor* w1;
  double sm_scale;
  int64_t frames;
  const Tensor &o;
  const Tensor* lse;
  const Tensor* ent;
  int64_t splits;
  bool fp8;
  int64_t rows;
};
vmo_fea_fwd_args fwd_args(const FwdCall& c) {
  like(c.q, {&c.k, &c.w0, c.w1, &c.o});
  same_device(c.q, {c.lse, c.ent});
  vmo_fea_fwd_args a{};
  a.dtype = dtype_code(c.q);
  a.batch = c.q.size(0); a.heads = c.q.size(1); a.frames = c.frames;
  const int64_t nq = c.rows >= 0 ? c.rows : c.q.size(2), nk = c.k.size(2);
  whole_frames(nq, nk, c.frames);
  a.nq = nq / c.frames; a.nk = nk / c.frames;
  a.d = c.q.size(3); a.dw0 = c.w0.size(3); a.dw1 = c.w1 ? c.w1->size(3) : 0;
  a.q = view(c.q); a.k = view(c.k); a.w0 = view(c.w0); a.o = view(c.o);
  if (c.w1) a.w1 = view(*c.w1);
  if (c.lse) a.lse = c.lse->data_ptr<float>();
  if (c.ent) a.ent = c.ent->data_ptr<float>();
  if (c.lse && c.ent)
    require(c.lse->stride(0) == c.ent->stride(0) && c.lse->stride(1) == c.ent->stride(1), "lse and ent strides");
  if (const Tensor* st = c.lse ? c.lse : c.ent) {
    require(st->stride(2) == 1, "lse / ent token stride");
    a.stat_stride_b = st->stride(0); a.stat_stride_h = st->stride(1);
  }
  a.sm_scale = (float)c.sm_scale;
  a.num_splits = (int32_t)c.splits;
  a.qk_fp8 = c.fp8;
  return a;
}
Tensor workspace(size_t bytes, const Tensor& like) { return at::empty({(int64_t)bytes}, like.options().dtype(at::kByte)); }
// launched on `stream`; returns the workspace (undefined when none is needed), which must outlive the work: on the
// current stream the caching allocator sees to that, on another the caller keeps it until it has joined that stream
Tensor run_fwd(const FwdCall& c, void* stream) {
  vmo_fea_fwd_args a = fwd_args(c);
  Tensor ws;
  if (const size_t bytes = vmo_fea_fwd_workspace_size(&a)) {
    ws = workspace(bytes, c.q);
    a.workspace = ws.data_ptr();
    a.workspace_bytes = bytes;
  }
  check(vmo_fea_fwd(&a, stream), "vmo_fea_fwd");
  return ws;
}
// a and b together (vmo_fea_fwd_pair) on the current stream
void run_pair(const FwdCall& ca, const FwdCall& cb, void* stream) {
  vmo_fea_fwd_args a = fwd_args(ca), b = fwd_args(cb);
  Tensor wa, wb;
  auto reserve = [&](vmo_fea_fwd_args& x, Tensor& ws) {
    if (const size_t bytes = vmo_fea_fwd_workspace_size(&x)) {
      ws = workspace(bytes, ca.q);
      x.workspace = ws.data_ptr();
      x.workspace_bytes = bytes;
    }
  };
  reserve(a, wa);
  reserve(b, wb);
  check(vmo_fea_fwd_pair(&a, &b, stream), "vmo_fea_fwd_pair");
}
const Tensor* ptr(const OptT& t) { return t ? &*t : nullptr; }

std::tuple<Tensor, OptT, OptT> fea_fwd(const Tensor& q, const Tensor& k, const Tensor& w0, const OptT& w1, double sm_scale,
                                       int64_t frames, OptT o, OptT lse, OptT ent, bool want_ent, bool want_lse,
                                       int64_t num_splits, bool qk_fp8) {
  const int64_t B = q.size(0), H = q.size(1), NQ = q.size(2);
  if (!o) o = at::empty({B, H, NQ, w0.size(3) + (w1 ? w1->size(3) : 0)}, q.options());
  if (!lse && want_lse) lse = at::empty({B, H, NQ}, f32(q));
  if (!ent && want_ent) ent = at::empty({B, H, NQ}, f32(q));
  run_fwd({q, k, w0, ptr(w1), sm_scale, frames, *o, ptr(lse), ptr(ent), num_splits, qk_fp8, -1}, stream_of(q));
  return {*o, lse, ent};
}

struct BwdCall {
  const Tensor &q, &k, &v, &o, &lse, &ent, &dO, &dE;
  double sm_scale;
  const Tensor *dq, *dk, *dv, *v1;
  int64_t frames;
  int32_t flags;
  const Tensor *dq_base, *dk_base, *dv_base, *delta;
  int64_t rows;   // >= 0: only the first `rows` queries
};
void run_bwd(const BwdCall& c) {
  like(c.q, {&c.k, &c.v, c.v1, &c.o, &c.dO});
  same_device(c.q, {&c.lse, &c.ent, &c.dE, c.dq, c.dk, c.dv, c.dq_base, c.dk_base, c.dv_base, c.delta});
  vmo_fea_bwd_args a{};
  a.flags = c.flags;
  a.dtype = dtype_code(c.q);
  const int64_t nq = c.rows >= 0 ? c.rows : c.q.size(2), nk = c.k.size(2);
  whole_frames(nq, nk, c.frames);
  a.batch = c.q.size(0); a.heads = c.q.size(1); a.nq = nq / c.frames; a.nk = nk / c.frames;
  a.d = c.q.size(3); a.dv = c.v.size(3) * (c.v1 ? 2 : 1); a.frames = c.frames;
  a.q = view(c.q); a.k = view(c.k); a.v = view(c.v); a.o = view(c.o); a.grad_o = view(c.dO);
  a.grad_q = view(*c.dq); a.grad_k = view(*c.dk);
  if (c.dv) a.grad_v = view(*c.dv);
  auto base = [](const Tensor* b, const Tensor* g, vmo_view& out) {
    if (!b) return;
    require(g && b->sizes() == g->sizes(), "a base is shaped like its gradient");
    out = view(*b);
  };
  base(c.dq_base, c.dq, a.grad_q_base); base(c.dk_base, c.dk, a.grad_k_base); base(c.dv_base, c.dv, a.grad_v_base);
  require(c.lse.strides() == c.ent.strides() && c.lse.stride(2) == 1 && c.dE.stride(2) == 1, "lse / ent / de strides");
  a.lse = c.lse.data_ptr<float>(); a.ent = c.ent.data_ptr<float>(); a.grad_ent = c.dE.data_ptr<float>();
  a.stat_stride_b = c.lse.stride(0); a.stat_stride_h = c.lse.stride(1);
  a.grad_ent_stride_b = c.dE.stride(0); a.grad_ent_stride_h = c.dE.stride(1);
  a.sm_scale = (float)c.sm_scale;
  if (c.v1) {
    require(c.v1->sizes() == c.v.sizes() && c.v1->strides() == c.v.strides() && c.v1->dtype() == c.v.dtype(),
            "v1 has the shape, strides and dtype of v");
    a.v1 = view(*c.v1); a.dv1 = c.v1->size(3);
  }
  if (c.delta) {
    require(c.delta->scalar_type() == at::kFloat && c.delta->stride(2) == 1, "delta: float32, unit token stride");
    a.delta = c.delta->data_ptr<float>();
    a.delta_stride_b = c.delta->stride(0); a.delta_stride_h = c.delta->stride(1);
  }
  const size_t bytes = vmo_fea_bwd_workspace_size(&a);
  const Tensor ws = workspace(bytes, c.q);
  a.workspace = ws.data_ptr(); a.workspace_bytes = bytes;
  check(vmo_fea_bwd(&a, stream_of(c.q)), "vmo_fea_bwd");
}

std::tuple<Tensor, Tensor, OptT> fea_bwd(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& o, const Tensor& lse,
                                         const Tensor& ent, const Tensor& dO, const Tensor& dE, double sm_scale, OptT dq,
                                         OptT dk, OptT dv, const std::string& overwrite, const OptT& v1, bool fold_k,
                                         const OptT& dk_base, const OptT& dv_base, int64_t frames, int64_t route_flags,
                                         const OptT& dq_base, const OptT& delta) {
  int32_t flags = (fold_k ? VMO_BWD_FOLD_K : 0) | (int32_t)route_flags;
  struct G { const OptT& t; char name; int accum, f32_bit, sum; const OptT& base; };
  for (const G& g : {G{dq, 'q', VMO_BWD_ACCUM_Q, VMO_BWD_F32_Q, VMO_BWD_SUM_Q, dq_base},
                     G{dk, 'k', VMO_BWD_ACCUM_K, VMO_BWD_F32_K, VMO_BWD_SUM_K, dk_base},
                     G{dv, 'v', VMO_BWD_ACCUM_V, VMO_BWD_F32_V, VMO_BWD_SUM_V, dv_base}}) {
    if (g.base) {
      require(g.base->scalar_type() == at::kFloat && (!g.t || g.t->scalar_type() == q.scalar_type()),
              "base fp32, result q.dtype");
      flags |= g.sum;
    } else if (g.t && g.t->scalar_type() != q.scalar_type()) {
      require(g.t->scalar_type() == at::kFloat, "a gradient passed in must be float32 or q's dtype");
      flags |= overwrite.find(g.name) != std::string::npos ? g.f32_bit : g.accum;
    }
  }
  const int64_t B = q.size(0), H = q.size(1), NQ = q.size(2), NK = k.size(2), D = q.size(3);
  if (!dq) dq = at::empty({B, H, NQ, D}, q.options());
  if (!dk) dk = at::empty({B, H, NK, D}, q.options());
  if (!dv && !(fold_k && !v1))
    dv = at::empty({B, H, NK, fold_k ? v1->size(3) : v.size(3) * (v1 ? 2 : 1)}, q.options());
  run_bwd({q, k, v, o, lse, ent, dO, dE, sm_scale, ptr(dq), ptr(dk), ptr(dv), ptr(v1), frames, flags, ptr(dq_base),
           ptr(dk_base), ptr(dv_base), ptr(delta), -1});
  return {*dq, *dk, dv};
}

void lstep_fwd(const Tensor& q, const Tensor& out, const Tensor& ent, const Tensor& res, int64_t m, int64_t b, double scale,
               bool last, int64_t skip, double min_col_mass) {
  like(q, {&out, &res});
  same_device(q, ent);
  vmo_lstep_args a{};
  a.dtype = dtype_code(q);
  a.batch = q.size(0); a.heads = q.size(1); a.num_blocks = m; a.block_size = b;
  a.d = q.size(3); a.dv = last ? out.size(3) - q.size(3) : 0;
  a.last = last; a.skip_tokens = (int32_t)skip;
  a.q = view(q); a.out = view(out); a.res = view(res);
  a.ent = ent.data_ptr<float>();
  a.ent_stride_b = ent.stride(0); a.ent_stride_h = ent.stride(1);
  a.scale = (float)scale; a.min_col_mass = (float)min_col_mass;
  check(vmo_lstep_fwd(&a, stream_of(q)), "vmo_lstep_fwd");
}

void lstep_bwd(const Tensor& q, const Tensor& out, const Tensor& ent, const Tensor& grad_res, const Tensor& grad_q,
               const Tensor& grad_out, int64_t m, int64_t b, double scale, bool last, int64_t skip, double min_col_mass,
               bool overwrite_q, const OptT& delta) {
  like(q, {&out, &grad_res, &grad_out});
  require(grad_q.scalar_type() == at::kFloat, "grad_q: float32");
  same_device(q, {&ent, &grad_q, ptr(delta)});
  vmo_lstep_bwd_args a{};
  a.dtype = dtype_code(q);
  a.batch = q.size(0); a.heads = q.size(1); a.num_blocks = m; a.block_size = b;
  a.d = q.size(3); a.dv = last ? out.size(3) - q.size(3) : 0;
  a.last = last; a.skip_tokens = (int32_t)skip;
  a.q = view(q); a.out = view(out); a.grad_res = view(grad_res); a.grad_q = view(grad_q); a.grad_out = view(grad_out);
  a.ent = ent.data_ptr<float>();
  a.ent_stride_b = ent.stride(0); a.ent_stride_h = ent.stride(1);
  a.scale = (float)scale; a.min_col_mass = (float)min_col_mass;
  a.flags = overwrite_q ? VMO_LSTEP_BWD_OVERWRITE_Q : 0;
  if (delta) {
    require(delta->scalar_type() == at::kFloat && delta->stride(2) == 1, "delta: float32, unit token stride");
    a.delta = delta->data_ptr<float>();
    a.delta_stride_b = delta->stride(0); a.delta_stride_h = delta->stride(1);
  }
  check(delta ? vmo_lstep_bwd_delta(&a, stream_of(q)) : vmo_lstep_bwd(&a, stream_of(q)), "vmo_lstep_bwd");
}

// ---- flash-entropy attention (all N rows valid, head dims the kernels take as they are) --------------------------

std::tuple<Tensor, Tensor, Tensor> fea_attention(const Tensor& q0, const Tensor& k0, const Tensor& v0, double sm_scale) {
  like(q0, {&k0, &v0});
  const OnGpuOf device(q0);
  const Tensor q = row_aligned(q0), k = row_aligned(k0), v = row_aligned(v0);
  const int64_t B = q.size(0), H = q.size(1), N = q.size(2);
  Tensor o = empty_in_layout(q0, v.size(3));
  Tensor lse = at::empty({B, H, N}, f32(q)), ent = at::empty({B, H, N}, f32(q));
  if (N > 0) run_fwd({q, k, v, nullptr, sm_scale, 1, o, &lse, &ent, 1, false, -1}, stream_of(q));
  return {o, ent, lse};
}

std::tuple<Tensor, Tensor, Tensor> fea_attention_bwd(const Tensor& q0, const Tensor& k0, const Tensor& v0, const Tensor& o0,
                                                     const Tensor& lse, const Tensor& ent, const Tensor& do0,
                                                     const Tensor& dE, double sm_scale) {
  like(q0, {&k0, &v0, &o0, &do0});
  const OnGpuOf device(q0);
  // the gradients in the memory order of the caller's q, k, v
  Tensor dq = empty_in_layout(q0, q0.size(3)), dk = empty_in_layout(k0, k0.size(3)), dv = empty_in_layout(v0, v0.size(3));
  const Tensor q = row_aligned(q0), k = row_aligned(k0), v = row_aligned(v0), o = row_aligned(o0), dO = row_aligned(do0);
  run_bwd({q, k, v, o, lse, ent, dO, dE, sm_scale, &dq, &dk, &dv, nullptr, 1, 0, nullptr, nullptr, nullptr, nullptr, -1});
  return {dq, dk, dv};
}

// ---- VMonarch attention ------------------------------------------------------------------------------------------

// A side stream's work between fork (it waits for the current stream) and join (the current stream waits for it).
struct SideStream {
  hipStream_t main, side;
  bool open = false;
  SideStream(void* m, int64_t s) : main((hipStream_t)m), side((hipStream_t)s) {}
  SideStream(const SideStream&) = delete;
  ~SideStream() {   // an error between fork and join: joined all the same, before the workspaces are given back
    if (!open) return;
    try { join(); } catch (const std::runtime_error&) {}
  }
  static void order(hipStream_t after, hipStream_t then) {   // work issued to `then` from here on follows `after`'s
    hipEvent_t e;
    if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) throw std::runtime_error("vmonarch: no event");
    hipError_t rc = hipEventRecord(e, after);
    if (rc == hipSuccess) rc = hipStreamWaitEvent(then, e, 0);
    (void)hipEventDestroy(e);   // (released once the recorded work is done)
    if (rc != hipSuccess) throw std::runtime_error(std::string("vmonarch: stream order: ") + hipGetErrorString(rc));
  }
  void fork() {
    order(main, side);
    open = true;
  }
  void join() {
    open = false;
    order(side, main);
  }
};

// Where the recompute runs: on the caller's stream after the chain; on the side stream, forked at the start, after
// R-step 0 or after the last R-step; or in one launch with R-step 0 (with more than one iteration: its values are k).
enum Overlap { kOff = 0, kStart = 1, kAfterR0 = 2, kAfterR1 = 3, kWithR0 = 4 };

// the caller's stage hook (None: none), with the torch stream objects it is told of; called with the interpreter lock
struct Stages {
  py::object hook, main, side;
  void operator()(const char* name, int it, const char* phase, bool on_side = false) const {
    if (hook.is_none()) return;
    const py::gil_scoped_acquire lock;
    hook(it < 0 ? std::string(name) : name + std::to_string(it), phase, on_side ? side : main);
  }
};

Tensor vmonarch_fwd(const Tensor& q0, const Tensor& k0, const Tensor& v0, int64_t m, int64_t b, int64_t iters,
                    int64_t recompute_tokens, double min_col_mass, double scale, bool qk_fp8, int64_t splits, int overlap,
                    int64_t side_handle, const Stages& stage) {
  like(q0, {&k0, &v0});
  const OnGpuOf device(q0);
  const Tensor q = row_aligned(q0), k = row_aligned(k0), v = row_aligned(v0);
  const int64_t B = q.size(0), H = q.size(1), N = q.size(2), D = q.size(3), Dv = v.size(3);
  const int64_t rt = std::min<int64_t>(recompute_tokens, N);
  void* const main = stream_of(q);
  Tensor ent = at::empty({B, H, N}, f32(q));
  Tensor z = empty_in_layout(q, Dv);   // in the caller's layout
  Tensor ws;                           // the recompute's workspace: held until its stream is joined
  SideStream ss(main, side_handle);
  // exact attention of the first rt queries, into rows of z that the L-steps do not write
  const FwdCall exact_rows{q, k, v, nullptr, scale, 1, z, nullptr, nullptr, splits, false, rt};
  const bool with_r0 = rt > 0 && iters > 1 && overlap == kWithR0;
  auto recompute = [&](void* stream, bool on_side) {
    stage("recompute", -1, "begin", on_side);
    ws = run_fwd(exact_rows, stream);
    stage("recompute", -1, "end", on_side);
  };
  bool forked = false;
  auto fork = [&] {
    forked = true;
    ss.fork();   // q, k, v and z are ready on the caller's stream
    recompute((void*)ss.side, true);
  };
  if (rt > 0 && overlap == kStart) fork();
  Tensor u, out;
  for (int64_t it = 0; it < iters; ++it) {
    const bool last = it == iters - 1;
    out = at::empty({B, H, N, D + (last ? Dv : 0)}, q.options());
    stage("rstep", it, "begin");   // iteration 0 folds u = q * scale into the softmax scale
    const FwdCall rstep{it == 0 ? q : u, k, k, last ? &v : nullptr, it == 0 ? scale : 1.0, m, out, nullptr, &ent, 1, qk_fp8, -1};
    if (with_r0 && it == 0) {   // one launch, both stages'
      stage("recompute", -1, "begin");
      run_pair(exact_rows, rstep, main);
      stage("recompute", -1, "end");
    } else {
      run_fwd(rstep, main);
    }
    stage("rstep", it, "end");
    if (rt > 0 && !forked && ((overlap == kAfterR0 && it == 0) || (overlap == kAfterR1 && last))) fork();
    stage("lstep", it, "begin");
    if (last) {
      lstep_fwd(q, out, ent, z, m, b, scale, true, rt, min_col_mass);
    } else {
      if (!u.defined()) u = at::empty({B, H, N, D}, q.options());
      lstep_fwd(q, out, ent, u, m, b, scale, false, 0, min_col_mass);
    }
    stage("lstep", it, "end");
  }
  if (rt > 0 && !with_r0) {
    if (forked) ss.join();   // z is complete on the caller's stream
    else recompute(main, false);
  }
  return z;
}

// The forward that keeps what the backward needs: (orders, q, k, v, z, lse_rt, [x, out, lse, ent] per iteration).
std::tuple<std::vector<int>, std::vector<Tensor>> vmonarch_fwd_train(const Tensor& q0, const Tensor& k0, const Tensor& v0,
                                                                     int64_t m, int64_t b, int64_t iters, int64_t rt,
                                                                     double min_col_mass, double scale, int64_t splits,
                                                                     int overlap, int64_t side_handle) {
  like(q0, {&k0, &v0});
  const OnGpuOf device(q0);
  std::vector<int> orders;
  for (const Tensor* t : {&q0, &k0, &v0})
    for (int d : layout_order(*t)) orders.push_back(d);
  Tensor z = empty_in_layout(q0, v0.size(3));
  // read in place in any memory order: the kernels take each head's m frames as m problems
  Tensor q = row_aligned(q0), k = row_aligned(k0), v = row_aligned(v0);
  if (k.strides() != v.strides()) {   // the backward reads the values [k | v] as two parts with one set of strides
    k = k.contiguous();
    v = v.contiguous();
  }
  const int64_t B = q.size(0), H = q.size(1), N = q.size(2), D = q.size(3), Dv = v.size(3);
  void* const main = stream_of(q);
  Tensor lse_rt, ws;
  SideStream ss(main, side_handle);
  if (rt > 0) lse_rt = at::empty({B, H, rt}, f32(q));
  const FwdCall exact_rows{q, k, v, nullptr, scale, 1, z, &lse_rt, nullptr, splits, false, rt};
  const bool with_r0 = rt > 0 && iters > 1 && overlap == kWithR0, forked = rt > 0 && overlap != kOff && overlap != kWithR0;
  if (forked) {
    ss.fork();
    ws = run_fwd(exact_rows, (void*)ss.side);
  }
  std::vector<Tensor> saved;
  Tensor u;
  for (int64_t it = 0; it < iters; ++it) {
    const bool last = it == iters - 1;
    Tensor out = at::empty({B, H, N, D + (last ? Dv : 0)}, q.options());
    Tensor lse = at::empty({B, H, N}, f32(q)), ent = at::empty({B, H, N}, f32(q));
    const Tensor x = it == 0 ? q : u;
    const FwdCall rstep{x, k, k, last ? &v : nullptr, it == 0 ? scale : 1.0, m, out, &lse, &ent, 1, false, -1};
    if (with_r0 && it == 0) run_pair(exact_rows, rstep, main);
    else run_fwd(rstep, main);
    if (last) {
      lstep_fwd(q, out, ent, z, m, b, scale, true, rt, min_col_mass);
    } else {
      u = at::empty({B, H, N, D}, q.options());
      lstep_fwd(q, out, ent, u, m, b, scale, false, 0, min_col_mass);
    }
    for (const Tensor& t : {x, out, lse, ent}) saved.push_back(t);
  }
  if (forked) ss.join();   // z and lse_rt are complete on the caller's stream
  else if (rt > 0 && !with_r0) run_fwd(exact_rows, main);
  std::vector<Tensor> all{q, k, v, z, rt > 0 ? lse_rt : at::empty({0}, q.options())};
  all.insert(all.end(), saved.begin(), saved.end());
  return {orders, all};
}

// Which L-steps' backward kernels form delta: one-tile grids every one, multi-block grids the last.
enum Delta { kNoDelta = 0, kEveryStep = 1, kLastStep = 2 };

// Call order: the L- and R-step backwards from the last iteration down, R-step 0's last of all and the recompute's
// (rows [0, rt), vmonarch.py:66-68) just before it.  Every gradient is written once, in the caller's dtype and
// memory order, by the last call that contributes to it: the fp32 sum of the earlier contributions plus its own
// (VMO_BWD_SUM_*), so no conversion pass follows.  dq: the L-steps (the first overwrites, the rest add), the
// recompute, then R-step 0 (x = q).  dk: every R-step (values start with k: the kernels fold k's value-role
// gradient into dk, as autograd's sum over k's uses at vmonarch.py:50 does), the recompute, R-step 0 last.  dv: the
// last R-step (values [k | v]) and the recompute.
std::tuple<Tensor, Tensor, Tensor> vmonarch_bwd(const std::vector<int>& orders, const std::vector<Tensor>& all, const Tensor& dz0,
                                                int64_t m, int64_t b, int64_t iters, int64_t rt, double min_col_mass,
                                                double scale, int want_delta) {
  const Tensor &q = all[0], &k = all[1], &v = all[2], &z = all[3], &lse_rt = all[4];
  const OnGpuOf device(q);
  same_device(q, dz0);
  const Tensor dz = row_aligned(dz0.to(q.scalar_type()));
  const int64_t B = q.size(0), H = q.size(1), N = q.size(2), D = q.size(3), Dv = v.size(3);
  const int64_t dims[3] = {B, H, N};
  auto grad = [&](int i, int64_t feat) {
    return empty_in_order(Order{orders[3 * i], orders[3 * i + 1], orders[3 * i + 2]}, dims, feat, q.options());
  };
  Tensor gq = grad(0, D), gk = grad(1, D), gv = grad(2, Dv);
  Tensor dq = at::empty({B, H, N, D}, f32(q));
  struct Sum {   // one gradient's fp32 partial sum and final tensor
    Tensor partial, result;
    bool started;
  } sk{at::empty({B, H, N, D}, f32(q)), gk, false}, sv{at::empty({B, H, N, Dv}, f32(q)), gv, false};
  const Tensor de = at::zeros({B, H, N}, f32(q));
  // rowsum(out * d out), formed by the L-step backward that writes d out and read by the R-step backward in place of
  // another pass over both
  OptT delta;
  if (want_delta != kNoDelta) delta = at::empty({B, H, N}, f32(q));
  // where one call puts its part of a gradient: into the fp32 partial sum (the first call overwrites it), or from
  // its last contribution into the result
  struct Put { const Tensor* g; const Tensor* base; int32_t flags; };
  auto put = [](Sum& s, bool last_writer, int accum, int f32_bit, int sum) {
    if (last_writer) return Put{&s.result, s.started ? &s.partial : nullptr, s.started ? sum : 0};
    const bool first = !s.started;
    s.started = true;
    return Put{&s.partial, nullptr, first ? f32_bit : accum};
  };
  auto put_k = [&](bool lw) { return put(sk, lw, VMO_BWD_ACCUM_K, VMO_BWD_F32_K, VMO_BWD_SUM_K); };
  auto put_v = [&](bool lw) { return put(sv, lw, VMO_BWD_ACCUM_V, VMO_BWD_F32_V, VMO_BWD_SUM_V); };
  Tensor g = dz;
  for (int64_t it = iters - 1; it >= 0; --it) {
    const bool last = it == iters - 1;
    const Tensor &x = all[5 + 4 * it], &out = all[6 + 4 * it], &lse = all[7 + 4 * it], &ent = all[8 + 4 * it];
    Tensor dout = at::empty_like(out);
    if (!last && want_delta != kEveryStep) delta.reset();
    lstep_bwd(q, out, ent, g, dq, dout, m, b, scale, last, last ? rt : 0, min_col_mass, last, delta);
    if (it == 0 && rt > 0) {   // the exact attention of the first rt queries; it reads every key and value
      const Tensor zeros = de.narrow(2, 0, rt);
      const Tensor ent0 = lse_rt;   // (multiplied by a zero entropy gradient)
      const Put pk = put_k(false), pv = put_v(iters > 1);
      run_bwd({q, k, v, z, lse_rt, ent0, dz, zeros, scale, &dq, pk.g, pv.g, nullptr, 1, VMO_BWD_ACCUM_Q | pk.flags | pv.flags,
               nullptr, pk.base, pv.base, nullptr, rt});
    }
    // values k, or [k | v] read from the two tensors in place (vmonarch.py:50); m frames per head
    const Put pk = put_k(it == 0);
    Put pv{nullptr, nullptr, 0};
    if (last) pv = put_v(iters == 1 || rt == 0);
    Tensor gx;
    if (it > 0) gx = at::empty({B, H, N, D}, q.options());
    run_bwd({x, k, k, out, lse, ent, dout, de, it == 0 ? scale : 1.0, it == 0 ? &gq : &gx, pk.g, pv.g, last ? &v : nullptr, m,
             VMO_BWD_FOLD_K | pk.flags | pv.flags | (it == 0 ? VMO_BWD_SUM_Q : 0), it == 0 ? &dq : nullptr, pk.base, pv.base,
             ptr(delta), -1});
    if (it > 0) g = gx;   // dL/du of the previous L-step's output
  }
  return {gq, gk, gv};
}

// A single launch as an entry of its own: on its first tensor's GPU.
template <class R, class... A>
auto on_its_gpu(R (*launch)(const Tensor&, A...)) {
  return [launch](const Tensor& q, A... rest) -> R {
    const OnGpuOf device(q);
    return launch(q, std::forward<A>(rest)...);
  };
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, mod) {
  using NoGil = py::call_guard<py::gil_scoped_release>;
  mod.def("fea_fwd", on_its_gpu(&fea_fwd), NoGil());
  mod.def("fea_bwd", on_its_gpu(&fea_bwd), NoGil());
  mod.def("lstep_fwd", on_its_gpu(&lstep_fwd), NoGil());
  mod.def("lstep_bwd", on_its_gpu(&lstep_bwd), NoGil());
  mod.def("fea_attention", &fea_attention, NoGil());
  mod.def("fea_attention_bwd", &fea_attention_bwd, NoGil());
  mod.def("vmonarch_fwd", [](const Tensor& q, const Tensor& k, const Tensor& v, int64_t m, int64_t b, int64_t iters,
                             int64_t recompute_tokens, double min_col_mass, double scale, bool qk_fp8, int64_t splits, int overlap,
                             int64_t side_handle, py::object hook, py::object main, py::object side) {
    const Stages stage{std::move(hook), std::move(main), std::move(side)};   // (outlives the release of the lock)
    const py::gil_scoped_release unlocked;
    return vmonarch_fwd(q, k, v, m, b, iters, recompute_tokens, min_col_mass, scale, qk_fp8, splits, overlap, side_handle, stage);
  });
  mod.def("vmonarch_fwd_train", &vmonarch_fwd_train, NoGil());
  mod.def("vmonarch_bwd", &vmonarch_bwd, NoGil());
}
