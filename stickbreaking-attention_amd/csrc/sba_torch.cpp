// Eager host path of the operators: argument checks, allocations, the autograd node and the C ABI calls in one native
// function, so that a call costs a few microseconds of host time instead of the ~35 (forward) and ~150 (forward and
// backward) it took in Python, which is more than the kernels of a short sequence need.  The backward runs in the autograd
// thread without the interpreter.  No kernels here; libsba.so has no torch types.
//
// Measured per pass, Python before -> now: 12 heads x 64 tokens, forward 32 -> 8.1 us; 24 heads x 64, 4 x 256 tokens, forward and
// backward 195 -> 75 us, or 43 in one process of four (its kernels take 40, and 51 replayed from a graph: the host is what
// such a pass waits for).
#include <torch/extension.h>

#include <ATen/ops/empty.h>
#include <ATen/ops/empty_like.h>
#include <ATen/ops/zeros_like.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/jit/frontend/tracer.h>

#include <atomic>
#include <cmath>
#include <optional>

#include "../../include/sba.h"
#include "sba_internal.hpp"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// Upper limit in bytes for the backward's workspace (negative: whatever the whole call needs); see
// set_backward_workspace_limit in _native.py.
std::atomic<int64_t> g_bwd_limit{-1};

// Debugging aids, as in _native.py: the caller passes the flags in force at the forward and they hold for its backward.
enum : int64_t { kPoison = 1, kDebugCheck = 2, kBackwardKernelsShift = 2 };

int32_t dtype_code(const Tensor& t) {
  switch (t.scalar_type()) {
    case at::kBFloat16: return SBA_BF16;
    case at::kHalf: return SBA_F16;
    case at::kFloat: return SBA_F32;
    default: TORCH_CHECK_TYPE(false, "unsupported dtype ", t.dtype());
  }
}

void check(int status, const char* what) {
  TORCH_CHECK(status == SBA_OK, what, " failed: ", sba_strerror(status), " (status ", status, ")");
}

void require_gpu(const Tensor& t) {
  TORCH_CHECK(t.is_cuda(), "stick-breaking attention runs on the GPU only (got a CPU tensor); there is no CPU path");
}

// The kernels need unit stride along head_dim.
Tensor rows_contiguous(const Tensor& t) { return t.stride(-1) == 1 ? t : t.contiguous(); }

void same_dtype(const Tensor& q, const Tensor& t, const char* name) {
  TORCH_CHECK_TYPE(t.scalar_type() == q.scalar_type(), name, " has dtype ", t.dtype(), ", q has ", q.dtype(),
                   ": q, k, v and the gradients must share one dtype");
}

// [batch,] head, token[, head_dim]
template <typename Ref>
Ref ref(const Tensor& t, bool fixed) {
  Ref r{};
  if (!t.defined()) return r;
  r.ptr = t.data_ptr();
  const int h = fixed ? 1 : 0;
  r.stride_batch = fixed ? t.stride(0) : 0;
  r.stride_head = t.stride(h);
  r.stride_token = t.stride(h + 1);
  return r;
}

void poison(const Tensor& t) { t.view(at::kByte).fill_(0xFF); }      // NaN patterns

void check_status(const Tensor& ws, const char* what) {
  const int status = ws.narrow(0, SBA_STATUS_OFFSET, 4).view(at::kInt).item<int>();
  if (status == 0) return;
  static const char* const text[] = {
      "cu_seqlens is not a non-decreasing sequence within [0, total_tokens] (or its leading entry is not 0)",
      "the carry buffer is too small for these sequence lengths (max_seqlens understated?)",
      "one-kernel backward: a workgroup gave up waiting for the key tile below its own",
      "one-kernel backward: the workgroups of a head did not share an XCD"};
  TORCH_CHECK_VALUE(false, what, ": ", status >= 1 && status <= 4 ? text[status - 1] : "unknown status",
                    "; outputs of this call are not valid");
}

// What a call is, apart from q, k and v.
struct Call {
  Tensor cu;      // packed batches only
  bool fixed = false, leading_zero = false, attend_current = false, add_remainder = false;
  int64_t max_seqlen = 0, carry_slots = 0, row_blocks = 0, flags = 0;
  double logit_scale = 0;
};

SbaArgs base_args(const Call& c, const Tensor& q) {
  SbaArgs a{};
  a.dtype = dtype_code(q);
  if (c.fixed) {
    a.num_seqs = (int32_t)q.size(0); a.num_heads = (int32_t)q.size(1); a.total_tokens = q.size(2); a.head_dim = (int32_t)q.size(3);
  } else {
    a.num_heads = (int32_t)q.size(0); a.total_tokens = q.size(1); a.head_dim = (int32_t)q.size(2);
    a.num_seqs = (int32_t)(c.cu.numel() - (c.leading_zero ? 1 : 0));
    a.cu_seqlens = c.cu.data_ptr();
    a.cu_is_int64 = c.cu.scalar_type() == at::kLong;
    a.cu_has_leading_zero = c.leading_zero;
    a.carry_slots = c.carry_slots;
    a.row_blocks = (int32_t)c.row_blocks;
  }
  a.max_seqlen = c.max_seqlen;
  a.logit_scale = (float)c.logit_scale;
  a.attend_current = c.attend_current;
  a.add_remainder = c.add_remainder;
  a.backward_kernels = (int32_t)(c.flags >> kBackwardKernelsShift);
  a.stream = (void*)c10::hip::getCurrentHIPStream(q.device().index()).stream();
  return a;
}

// SbaArgs::row_blocks of these (valid) lengths.
template <typename T>
int64_t row_blocks_of(const T* ends, int64_t n, bool leading_zero) {
  int64_t sum = 0, last = 0;
  for (int64_t i = leading_zero ? 1 : 0; i < n; i++) {
    const int64_t len = (int64_t)ends[i] - last;
    if (len > 256) sum += (len + 255) / 256 * 8;
    last = (int64_t)ends[i];
  }
  return std::max<int64_t>(sum, 1);
}
int64_t row_blocks(const Tensor& host, bool leading_zero) {
  return host.scalar_type() == at::kLong ? row_blocks_of(host.const_data_ptr<int64_t>(), host.numel(), leading_zero)
                                         : row_blocks_of(host.const_data_ptr<int32_t>(), host.numel(), leading_zero);
}

Tensor bytes(size_t n, const Tensor& like) { return at::empty({(int64_t)n}, like.options().dtype(at::kByte)); }
// The least workspace that sba_bwd accepts for these arguments: one head's, in fp32 without the planes of split operands.
size_t least_bytes(const SbaArgs& a) {
  SbaArgs c = a;
  c.num_heads = 1;
  if (c.dtype == SBA_F32) c.backward_kernels = 1;
  size_t n = 0;
  check(sba_workspace_bytes(&c, nullptr, &n, nullptr), "sba_workspace_bytes");
  return n;
}
// The backward's scratch: `n` bytes or, where memory is short, less: what the dQ and dK/dV kernels need (in fp32 without those planes; of what row
// tiles need up to a fifth), then half as much, which takes the heads through in groups, down to the least there can be.
Tensor backward_bytes(const SbaArgs& a, size_t n, const Tensor& like) {
  size_t two_kernels = 0, least = 0;
  for (;;) {
    try {
      return bytes(n, like);
    } catch (const c10::OutOfMemoryError&) {
      if (least == 0) {
        SbaArgs c = a;
        c.backward_kernels = 1;
        check(sba_workspace_bytes(&c, nullptr, &two_kernels, nullptr), "sba_workspace_bytes");
        least = least_bytes(a);
      }
      if (n <= least) throw;
    }
    n = std::max(least, two_kernels < n ? two_kernels : n / 2);
  }
}

struct Outputs {
  Tensor o, rem;
  // Kept for the backward: {schedule (kept_schedule bytes, or none), row_stat, carry}, as far as the backward wants them.
  Tensor state;
  int64_t kept_schedule = 0;
};
size_t align256(size_t n) { return (n + 255) & ~(size_t)255; }
size_t row_stat_bytes(const Tensor& q) { return align256(q.numel() / q.size(-1) * 4); }

// `for_backward`: a backward will follow; `want_carry`: it starts from recorded products instead of rebuilding them.
// The schedule of that backward is prepared (and kept) unless it would go unused, under a workspace limit, or is asked to keep
// little and the schedule has parts per row (the one-kernel backward's tags); tile lists alone are half a byte per token.
Outputs run_forward(const Call& c, const Tensor& q, const Tensor& k, const Tensor& v, bool for_backward, bool want_carry) {
  const c10::DeviceGuard guard(q.device());
  SbaArgs a = base_args(c, q);
  Outputs out;
  out.o = at::empty_like(q);
  if (out.o.stride(-1) != 1) out.o = at::empty(q.sizes(), q.options());
  out.rem = at::empty(q.sizes().slice(0, q.dim() - 1), q.options());
  // No products kept: a backward, if one follows, rebuilds them, and the forward's scheduler checks their capacity as that
  // backward's will (both passes void, or neither).
  a.recompute_carry = !want_carry && a.dtype != SBA_F32;
  sba::Prepared size{};
  bool prepare = for_backward && g_bwd_limit.load(std::memory_order_relaxed) < 0;
  if (for_backward) check(sba::prepared_bytes(&a, &size), "sba_workspace_bytes");
  if (size.row_parts && !want_carry) prepare = false;
  size_t sched = size.schedule;
  if (!prepare) check(sba_workspace_bytes(&a, &sched, nullptr, nullptr), "sba_workspace_bytes");
  const size_t stat = row_stat_bytes(q);
  const bool keep_stat = for_backward && (want_carry || c.add_remainder);
  Tensor scratch;
  size_t kept = 0, used = 0;      // bytes of `state` and of `scratch` so far
  (prepare ? kept : used) += sched;
  (keep_stat ? kept : used) += stat;
  if (used > 0) scratch = bytes(used, q);
  if (for_backward) out.state = bytes(kept + (want_carry ? size.carry : 0), q);
  out.kept_schedule = prepare ? sched : 0;
  if (c.flags & kPoison) {
    if (for_backward) poison(out.state);
    if (used > 0) poison(scratch);
  }
  char* const state = for_backward ? (char*)out.state.data_ptr() : nullptr;
  char* const other = used > 0 ? (char*)scratch.data_ptr() : nullptr;
  a.q = ref<SbaTensor>(q, c.fixed); a.k = ref<SbaTensor>(k, c.fixed); a.v = ref<SbaTensor>(v, c.fixed);
  a.o = ref<SbaTensor>(out.o, c.fixed);
  a.rem = ref<SbaVector>(out.rem, c.fixed);
  a.row_stat = (float*)(keep_stat ? state + out.kept_schedule : other + (prepare ? 0 : sched));
  a.carry = want_carry ? (float*)(state + kept) : nullptr;
  a.workspace = prepare ? state : other;
  a.workspace_bytes = sched;
  check(prepare ? sba::forward_prepared(&a) : for_backward ? sba_fwd(&a) : sba::forward_alone(&a), "sba_fwd");
  if (c.flags & kDebugCheck) check_status(prepare ? out.state : scratch, "sba_fwd");
  return out;
}

// `state` as the forward left it; `fresh`: no backward has run on its schedule yet.  What a saved-tensor hook hands back may lie
// in another place, and in another layout, than what the forward saved.
variable_list run_backward(Call c, Tensor d_o, Tensor d_rem, Tensor q, Tensor k, Tensor v, Tensor state, int64_t kept_schedule,
                           bool have_carry, bool fresh) {
  for (const Tensor* t : {&q, &k, &v, &state}) require_gpu(*t);
  same_dtype(q, k, "k");
  same_dtype(q, v, "v");
  const c10::DeviceGuard guard(q.device());
  q = rows_contiguous(q); k = rows_contiguous(k); v = rows_contiguous(v);
  if (!c.fixed) {
    require_gpu(c.cu);
    c.cu = c.cu.contiguous();
  }
  if (!state.is_contiguous() || ((uintptr_t)state.data_ptr() & 255)) state = state.clone(at::MemoryFormat::Contiguous);
  if (!d_o.defined()) d_o = at::zeros_like(q);
  require_gpu(d_o);
  same_dtype(q, d_o, "do");
  d_o = rows_contiguous(d_o);
  if (d_rem.defined()) {
    require_gpu(d_rem);
    if (d_rem.scalar_type() != q.scalar_type()) d_rem = d_rem.to(q.scalar_type());
  }
  SbaArgs a = base_args(c, q);
  const Tensor dq = at::empty_like(q), dk = at::empty_like(k), dv = at::empty_like(v);
  a.q = ref<SbaTensor>(q, c.fixed); a.k = ref<SbaTensor>(k, c.fixed); a.v = ref<SbaTensor>(v, c.fixed);
  a.d_o = ref<SbaTensor>(d_o, c.fixed);
  a.d_rem = ref<SbaVector>(d_rem, c.fixed);
  a.dq = ref<SbaTensor>(dq, c.fixed); a.dk = ref<SbaTensor>(dk, c.fixed); a.dv = ref<SbaTensor>(dv, c.fixed);
  a.recompute_carry = !have_carry;      // the forward kept no products: rebuild them in the backward's workspace
  sba::Prepared size{};
  check(sba::prepared_bytes(&a, &size), "sba_workspace_bytes");
  const size_t stat = have_carry || c.add_remainder ? row_stat_bytes(q) : 0;
  TORCH_CHECK((size_t)state.numel() == kept_schedule + stat + (have_carry ? size.carry : 0) &&
                  (kept_schedule == 0 || (size_t)kept_schedule == size.schedule),
              "saved state of another size");
  char* const base = (char*)state.data_ptr();
  a.row_stat = stat > 0 ? (float*)(base + kept_schedule) : nullptr;
  a.carry = have_carry ? (float*)(base + kept_schedule + stat) : nullptr;
  const int64_t limit = g_bwd_limit.load(std::memory_order_relaxed);
  // The forward's schedule serves one backward.  Under graph capture it may be replayed more often than the forward.
  const bool prepared = kept_schedule > 0 && fresh && limit < 0 && sba::prepared_fits(&a) &&
                        c10::hip::currentStreamCaptureStatusMayInitCtx() == c10::hip::CaptureStatus::None;
  Tensor ws;
  bool on_schedule = prepared;
  if (prepared) {
    try {
      ws = bytes(size.rest + size.laid, q);
    } catch (const c10::OutOfMemoryError&) {
      on_schedule = false;
    }
    if (!on_schedule && size.laid > 0) {
      try {
        ws = bytes(size.rest, q);
        on_schedule = true;
      } catch (const c10::OutOfMemoryError&) {
      }
    }
  }
  if (!on_schedule) {
    size_t ws_bytes = 0;
    check(sba_workspace_bytes(&a, nullptr, &ws_bytes, nullptr), "sba_workspace_bytes");
    if (limit >= 0 && ws_bytes > (size_t)limit) ws_bytes = std::max((size_t)limit, least_bytes(a));
    ws = backward_bytes(a, ws_bytes, q);
  }
  if (c.flags & kPoison) poison(ws);
  a.workspace = ws.data_ptr();
  a.workspace_bytes = ws.numel();
  check(on_schedule ? sba::backward_prepared(&a, base) : sba_bwd(&a), "sba_bwd");
  if (c.flags & kDebugCheck) check_status(on_schedule ? state : ws, "sba_bwd");
  return {dq, dk, dv};
}

struct StickBreaking : torch::autograd::Function<StickBreaking> {
  static variable_list forward(AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& v, const Call* call,
                               bool save_carry) {
    const Call& c = *call;
    const Outputs out = run_forward(c, q, k, v, true, save_carry);
    ctx->set_materialize_grads(false);
    ctx->save_for_backward({q, k, v, c.cu, out.state});
    ctx->saved_data["fresh"] = true;
    ctx->saved_data["call"] = c10::IValue(std::vector<int64_t>{c.fixed, c.leading_zero, c.attend_current, c.add_remainder,
                                                               c.max_seqlen, c.carry_slots, c.flags, save_carry, out.kept_schedule,
                                                               c.row_blocks});
    ctx->saved_data["scale"] = c.logit_scale;
    return {out.o, out.rem};
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    const variable_list s = ctx->get_saved_variables();
    const std::vector<int64_t> n = ctx->saved_data["call"].toIntVector();
    Call c;
    c.fixed = n[0]; c.leading_zero = n[1]; c.attend_current = n[2]; c.add_remainder = n[3];
    c.max_seqlen = n[4]; c.carry_slots = n[5]; c.flags = n[6]; c.row_blocks = n[9];
    c.logit_scale = ctx->saved_data["scale"].toDouble();
    c.cu = s[3];
    c10::IValue& fresh = ctx->saved_data["fresh"];
    const bool first = fresh.toBool();
    fresh = false;      // (also where the call fails half way through the schedule)
    variable_list g = run_backward(c, grads[0], grads[1], s[0], s[1], s[2], s[4], n[8], n[7], first);
    g.resize(5);      // call, save_carry
    return g;
  }
};

std::tuple<Tensor, Tensor> attention(const Call& c, Tensor q, Tensor k, Tensor v, bool save_carry) {
  dtype_code(q);
  same_dtype(q, k, "k");
  same_dtype(q, v, "v");
  TORCH_CHECK(q.dim() == (c.fixed ? 4 : 3) && k.dim() == q.dim() && v.dim() == q.dim(), "q, k and v must have ", c.fixed ? 4 : 3,
              " dimensions");
  q = rows_contiguous(q); k = rows_contiguous(k); v = rows_contiguous(v);
  if (at::GradMode::is_enabled() && (q.requires_grad() || k.requires_grad() || v.requires_grad())) {
    const variable_list out = StickBreaking::apply(q, k, v, &c, save_carry || q.scalar_type() == at::kFloat);
    return {out[0], out[1]};
  }
  const Outputs out = run_forward(c, q, k, v, false, false);
  return {out.o, out.rem};
}

// Whether a call on these tensors is ordinary eager work.  What records, transforms or replaces operations (a jit trace,
// dispatch modes, torch.func transforms, tensor subclasses and wrappers) and forward-mode derivatives see nothing of what
// happens here: such calls take the Python operators, which record themselves or refuse.
bool ordinary(py::handle q, py::handle k, py::handle v) {
  using c10::DispatchKey;
  static const c10::DispatchKeySet wrapped({DispatchKey::Python, DispatchKey::Functionalize, DispatchKey::FuncTorchBatched,
                                            DispatchKey::FuncTorchGradWrapper, DispatchKey::Batched, DispatchKey::Conjugate,
                                            DispatchKey::Negative, DispatchKey::ZeroTensor});
  if (torch::jit::tracer::isTracing() || c10::impl::TorchDispatchModeTLS::any_modes_set() ||
      c10::impl::tls_is_dispatch_key_included(DispatchKey::FuncTorchDynamicLayerFrontMode))
    return false;
  for (const py::handle h : {q, k, v}) {
    if (!THPVariable_CheckExact(h.ptr())) return false;      // (a tensor or a parameter, and no subclass)
    const Tensor& t = THPVariable_Unpack(h.ptr());
    if (t.key_set().has_any(wrapped) || t._fw_grad(0).defined()) return false;
  }
  return true;
}

double scale_of(const std::optional<double>& inv_temp, const Tensor& q) {
  return inv_temp ? *inv_temp : 1.0 / std::sqrt((double)q.size(-1));
}

// None where the call is not ordinary.  From the first tensor operation on, the interpreter's lock is given up: a device-to-host
// copy of cu_seqlens, a copy of host lengths to the device and an allocator that has to wait all wait for the stream, and another
// Python thread may be the one that what the stream waits for depends on.
std::optional<std::tuple<Tensor, Tensor>> fixed(py::handle hq, py::handle hk, py::handle hv, std::optional<double> inv_temp,
                                                bool attend_current, bool add_remainder, bool save_carry, int64_t flags) {
  if (!ordinary(hq, hk, hv)) return std::nullopt;
  const Tensor q = THPVariable_Unpack(hq.ptr()), k = THPVariable_Unpack(hk.ptr()), v = THPVariable_Unpack(hv.ptr());
  const py::gil_scoped_release unlocked;
  require_gpu(q); require_gpu(k); require_gpu(v);
  Call c;
  c.fixed = true;
  c.attend_current = attend_current; c.add_remainder = add_remainder;
  c.max_seqlen = q.size(2);
  c.flags = flags;
  c.logit_scale = scale_of(inv_temp, q);
  return attention(c, q, k, v, save_carry);
}

std::optional<std::tuple<Tensor, Tensor>> varlen(py::handle hq, py::handle hk, py::handle hv, Tensor cu,
                                                 std::optional<int64_t> max_seqlens, std::optional<double> inv_temp, bool zero_start,
                                                 bool attend_current, bool add_remainder, bool save_carry, int64_t flags) {
  if (!ordinary(hq, hk, hv)) return std::nullopt;
  const Tensor q = THPVariable_Unpack(hq.ptr()), k = THPVariable_Unpack(hk.ptr()), v = THPVariable_Unpack(hv.ptr());
  const py::gil_scoped_release unlocked;
  Call c;
  c.leading_zero = zero_start;
  c.attend_current = attend_current; c.add_remainder = add_remainder;
  c.max_seqlen = max_seqlens.value_or(0);
  c.flags = flags;
  if (cu.scalar_type() != at::kInt && cu.scalar_type() != at::kLong) cu = cu.to(at::kLong);
  // The lengths are on the host when cu_seqlens was given there, or after the one device-to-host copy that stands in for
  // the reference's `assert cu_seqlens[0] == 0`: they are then validated here, the carry buffer is sized exactly, and the
  // longest of them is what the kernels are chosen by, whatever the caller's max_seqlens says.
  Tensor host;
  if (!cu.is_cuda()) host = cu.contiguous();
  else if (zero_start) host = cu.cpu().contiguous();
  if (zero_start) {
    const int64_t first = host.scalar_type() == at::kLong ? *host.const_data_ptr<int64_t>() : *host.const_data_ptr<int32_t>();
    if (first != 0) {
      const py::gil_scoped_acquire locked;
      PyErr_SetString(PyExc_AssertionError, "cu_seqlens[0] must be 0");
      throw py::error_already_set();
    }
  }
  require_gpu(q); require_gpu(k); require_gpu(v);
  if (host.defined()) {
    SbaArgs a{};
    a.total_tokens = q.size(1);
    a.num_seqs = (int32_t)(host.numel() - (zero_start ? 1 : 0));
    a.cu_is_int64 = host.scalar_type() == at::kLong;
    a.cu_has_leading_zero = zero_start;
    SbaPlan plan{};
    check(sba_plan_host(&a, host.const_data_ptr(), &plan), "sba_plan_host");
    TORCH_CHECK_VALUE(plan.status == 0, "cu_seqlens must be non-decreasing sequence ends within [0, total_tokens]");
    c.carry_slots = plan.carry_slots;
    c.row_blocks = row_blocks(host, zero_start);
    c.max_seqlen = std::max(plan.longest, 1);
  }
  if (cu.device() != q.device()) cu = cu.to(q.device());
  c.cu = cu.contiguous();
  c.logit_scale = scale_of(inv_temp, q);
  return attention(c, q, k, v, save_carry);
}

}  // namespace

PYBIND11_MODULE(_sba_torch, m) {
  m.def("ordinary", &ordinary);
  m.def("fixed", &fixed);
  m.def("varlen", &varlen);
  m.def("set_backward_workspace_limit", [](std::optional<int64_t> n) { g_bwd_limit.store(n ? std::max<int64_t>(*n, 0) : -1); });
  // (form, heads of the first pass) of the backward that the SbaArgs at this address describe.
  m.def("backward_route", [](uint64_t args) {
    sba::BackwardRoute r{};
    check(sba::backward_route((const SbaArgs*)(uintptr_t)args, &r), "backward_route");
    return std::make_tuple(r.form, r.heads);
  });
  m.def("backward_with_polls", [](uint64_t args, int32_t polls) { check(sba::backward_with_polls((const SbaArgs*)(uintptr_t)args, polls), "sba_bwd"); });
  m.def("version", &sba_version);
}
