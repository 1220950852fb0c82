// Host side of the operators as a CPython extension: argument checks, output and workspace allocation, launches through
// the C ABI of libfla_hip.so, and the autograd nodes, without a Python frame between a model's call and its launches.
//
// A decode step or a short training step is a handful of launches of a few microseconds each; with ctypes and Python
// autograd functions the host needed 20 us for the former and 170 us for the latter, several times the device.
//
// Every entry takes the operands as a model holds them and returns None where a call needs a conversion first (head-first
// layout, head dims to be padded, fp32 q/k/v, a gradient through a step that has none here): the Python wrappers then take
// their general route.  Sequence-first layout, as in include/fla_hip.h.
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>

#include <map>
#include <mutex>
#include <optional>
#include <vector>

#include "../../include/fla_hip.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

constexpr int64_t BT = 64;

// ---------------------------------------------------------------------------------------------------- helpers
void check(int code, const char* what) {
  TORCH_CHECK(code == 0, what, " failed with code ", code, ": ", fla_error_string(code));
}

bool is16(const Tensor& t) { return t.scalar_type() == at::kBFloat16 || t.scalar_type() == at::kHalf; }
int dt(const Tensor& t) {
  switch (t.scalar_type()) {
    case at::kFloat: return FLA_F32;
    case at::kBFloat16: return FLA_BF16;
    case at::kHalf: return FLA_F16;
    default: TORCH_CHECK_TYPE(false, "fla_amd: unsupported dtype ", t.scalar_type());
  }
}
void* ptr(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }
float* fptr(const Tensor& t) { return (float*)ptr(t); }
fla_stream_t stream_of(const Tensor& t) { return (fla_stream_t)c10::hip::getCurrentHIPStream(t.device().index()).stream(); }
Tensor fresh(at::IntArrayRef sizes, const Tensor& like, at::ScalarType type) { return at::empty(sizes, like.options().dtype(type)); }
Tensor fresh_like(const Tensor& x) { return at::empty(x.sizes(), x.options()); }
Tensor f32(const Tensor& x) {
  if (!x.defined()) return x;
  return (x.scalar_type() == at::kFloat ? x : x.to(at::kFloat)).contiguous();
}
// Whether a call has to go through its autograd node.  An operand with a tangent does too, also where nothing requires a
// gradient: the nodes have no forward-mode derivative and say so, a launch beside them would drop the tangent.
bool has_tangent(std::initializer_list<const Tensor*> ts) {
  for (const Tensor* t : ts)
    if (t->defined() && t->_fw_grad(0).defined()) return true;
  return false;
}
bool wants_grad(std::initializer_list<const Tensor*> ts) {
  if (has_tangent(ts)) return true;
  if (!at::GradMode::is_enabled()) return false;
  for (const Tensor* t : ts)
    if (t->defined() && t->requires_grad()) return true;
  return false;
}
bool on_gpu(std::initializer_list<const Tensor*> ts) {
  for (const Tensor* t : ts)
    if (t->defined() && !t->is_cuda()) return false;
  return true;
}
// grads in the dtype of the operand they belong to
Tensor as(const Tensor& g, at::ScalarType type) { return g.scalar_type() == type ? g : g.to(type); }

// An operand that may be absent, as a node takes it
using Maybe = std::optional<Tensor>;
Maybe maybe(const Tensor& t) { return t.defined() ? Maybe(t) : std::nullopt; }
Tensor given(const Maybe& t) { return t ? *t : Tensor(); }

// Anything a node keeps beside tensors
template <typename X>
struct Held : torch::CustomClassHolder {
  X x;
  explicit Held(X v) : x(std::move(v)) {}
};
template <typename X>
void hold(AutogradContext* ctx, X v) {
  ctx->saved_data["s"] = c10::IValue::make_capsule(c10::make_intrusive<Held<X>>(std::move(v)));
}
template <typename X>
const X& held(AutogradContext* ctx) {
  return static_cast<Held<X>*>(ctx->saved_data["s"].toCapsule().get())->x;
}

// ---------------------------------------------------------------------------------------------------- packed batches
// A pinned host tensor as a device tensor that any stream may read from now on.  The copy goes through a stream of its own
// and is waited for there: the streams that compute go on (a blocking copy would wait for everything queued on its stream:
// a whole forward, where it is a backward's tables).  The memory belongs to that stream: readers call record_stream.
Tensor upload(const Tensor& host, at::Device device) {
  static std::mutex mu;
  static std::map<int, hipStream_t> streams;   // one per device, never destroyed
  c10::DeviceGuard on_device(device);
  std::lock_guard<std::mutex> lock(mu);
  hipStream_t& raw = streams[device.index()];
  if (!raw) TORCH_CHECK(hipStreamCreateWithFlags(&raw, hipStreamNonBlocking) == hipSuccess, "fla_amd: no stream for uploads");
  const auto own = c10::hip::getStreamFromExternal(raw, device.index());
  struct Current {
    c10::hip::HIPStream before;
    ~Current() { c10::hip::setCurrentHIPStream(before); }
  } current{c10::hip::getCurrentHIPStream(device.index())};
  c10::hip::setCurrentHIPStream(own);
  Tensor out = at::empty(host.sizes(), host.options().device(device).pinned_memory(false));
  out.copy_(host, /*non_blocking=*/true);
  own.synchronize();
  return out;
}

struct SplitTables {
  bool cut = false;
  fla_split ints{};
  Tensor tables;   // seg_table, sub_table and sub_base, one behind the other
};
// The device tables of a packed batch, made once per offsets tensor by fla_amd.utils.VarlenPlan.  `offsets` is the caller's
// own tensor where it is int64: a node saves it, so that a backward after it has been written to is refused instead of
// combining the other tables, made from the old boundaries, with the new ones.
struct Plan : torch::CustomClassHolder {
  Tensor offsets, indices, chunk_offsets, seq_order;
  std::vector<int64_t> host;
  int64_t N = 0, NT = 0;
  std::mutex mu;
  std::map<std::tuple<int64_t, int, bool, int>, SplitTables> splits;

  bool covers(int64_t begin, int64_t end) const { return !host.empty() && host.front() == begin && host.back() == end; }

  // The tables of a cut are used by later calls on any stream.  A stream that is being captured takes no copy: a call whose
  // tables are not there yet runs uncut under it.
  SplitTables split(int64_t H, int slabs, bool reverse, int kind) {
    std::lock_guard<std::mutex> lock(mu);
    const auto stream = c10::hip::getCurrentHIPStream(offsets.device().index());
    if (!splits.count({H, slabs, reverse, kind}) &&
        c10::hip::currentStreamCaptureStatusMayInitCtx() != c10::hip::CaptureStatus::None)
      return {};
    auto [it, fresh] = splits.try_emplace({H, slabs, reverse, kind});
    SplitTables& s = it->second;
    if (fresh && N > 0) {
      fla_split sp{};
      auto plan = [&](int32_t* a, int32_t* b, int32_t* c) {
        return fla_scan_split(host.data(), N, 0, H, slabs, reverse, kind, &sp, a, b, c);
      };
      if (plan(nullptr, nullptr, nullptr)) {
        const int64_t sub = 2 * (int64_t)sp.nseg, base = sub + 2 * (int64_t)sp.nsub;
        const Tensor host_tables = at::empty({base + N + 1}, at::TensorOptions().dtype(at::kInt).pinned_memory(true));
        int32_t* h = host_tables.data_ptr<int32_t>();
        plan(h, h + sub, h + base);
        s.tables = upload(host_tables, offsets.device());
        const int32_t* d = s.tables.data_ptr<int32_t>();
        sp.seg_table = d;
        sp.sub_table = d + sub;
        sp.sub_base = d + base;
        s.ints = sp;
        s.cut = true;
      }
    }
    // the plan may be dropped while this stream still reads its tables (tensors of this build call their device CUDA)
    if (s.cut) s.tables.record_stream(c10::Stream(c10::Stream::UNSAFE, offsets.device(), stream.id()));
    return s;
  }
};
using PlanPtr = c10::intrusive_ptr<Plan>;

const int64_t* offs(const PlanPtr& p) { return p ? (const int64_t*)p->offsets.data_ptr() : nullptr; }
const int64_t* idx(const PlanPtr& p) { return p ? (const int64_t*)p->indices.data_ptr() : nullptr; }
const int64_t* coff(const PlanPtr& p) { return p ? (const int64_t*)p->chunk_offsets.data_ptr() : nullptr; }
const int64_t* order(const PlanPtr& p) { return p ? (const int64_t*)p->seq_order.data_ptr() : nullptr; }

// One call's cut: the integers (and tables) of fla_scan_split and the two workspaces.
struct Cut {
  SplitTables tables;   // keeps a packed batch's tables alive
  fla_split s{};
  Tensor states, transitions;
};
std::optional<Cut> cut_scan(const PlanPtr& plan, int64_t N, int64_t T, int64_t H, int slabs, bool reverse, const Tensor& like,
                            int64_t state_elems, int64_t transition_elems, int kind = FLA_SCAN_GLA) {
  Cut c;
  if (plan) {
    c.tables = plan->split(H, slabs, reverse, kind);
    if (!c.tables.cut) return std::nullopt;
    c.s = c.tables.ints;
  } else if (!fla_scan_split(nullptr, N, T, H, slabs, reverse, kind, &c.s, nullptr, nullptr, nullptr)) {
    return std::nullopt;
  }
  c.states = fresh({c.s.slots * H * state_elems}, like, at::kFloat);
  c.transitions = fresh({c.s.slots * H * transition_elems}, like, at::kFloat);
  c.s.states = fptr(c.states);
  c.s.decays = fptr(c.transitions);
  return c;
}

struct Dims {
  int64_t B, T, H, K, V, N, NT, chunks;
};
// q, k [B,T,H,K], v [B,T,H,V] of one 16-bit dtype on one GPU, head dims 64 or 128
bool chunk_operands(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& h0, const PlanPtr& plan, Dims* d) {
  if (!q.defined() || !k.defined() || !v.defined()) return false;
  if (q.dim() != 4 || v.dim() != 4 || q.sizes() != k.sizes() || q.numel() == 0) return false;
  if (!is16(q) || k.scalar_type() != q.scalar_type() || v.scalar_type() != q.scalar_type()) return false;
  if (!on_gpu({&q, &k, &v, &h0})) return false;
  d->B = q.size(0), d->T = q.size(1), d->H = q.size(2), d->K = q.size(3), d->V = v.size(3);
  if (v.size(0) != d->B || v.size(1) != d->T || v.size(2) != d->H) return false;
  if ((d->K != 64 && d->K != 128) || (d->V != 64 && d->V != 128)) return false;
  if (plan && d->B != 1) return false;
  d->N = plan ? plan->N : d->B;
  const int64_t per = (d->T + BT - 1) / BT;
  d->NT = plan ? plan->NT : 0;
  d->chunks = plan ? plan->NT : d->B * per;
  if (h0.defined() && (h0.scalar_type() != at::kFloat || h0.dim() != 4 || h0.size(0) != d->N || h0.size(1) != d->H ||
                       h0.size(2) != d->K || h0.size(3) != d->V))
    return false;
  return true;
}

// ---------------------------------------------------------------------------------------------------- GLA
struct GlaArgs {
  Dims d;
  PlanPtr plan;
  double scale;
  bool want_ht, head_gates;
  int gate_form = 0;
  double normalizer = 1.0;
  std::optional<double> clamp;
};
struct GlaKept {
  Tensor wide, hT, qg, decay;
};

Tensor gla_forward(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& g, const Tensor& h0, const GlaArgs& a,
                   Tensor* ht, GlaKept* kept) {
  const Dims& d = a.d;
  Tensor o = fresh_like(v);
  if (a.want_ht) *ht = fresh({d.N, d.H, d.K, d.V}, q, at::kFloat);
  // the range guard's flags and the states it hands over for flagged chunks
  Tensor wide = fresh({d.chunks, d.H}, q, at::kInt), hwide = fresh({d.chunks, d.H, d.K * d.V}, q, q.scalar_type());
  GlaKept none, &x = kept ? *kept : none;
  if (kept) {
    x.wide = wide;
    x.hT = fresh({d.chunks, d.H, d.K, d.V}, q, q.scalar_type());
    x.qg = fresh_like(q);
    x.decay = fresh({d.chunks, d.H, d.K}, q, at::kFloat);
  }
  const fla_stream_t st = stream_of(q);
  const int form = a.head_gates ? 1 : a.gate_form;
  if (auto c = cut_scan(a.plan, d.N, d.T, d.H, (int)(d.V / 64), false, q, d.K * d.V, d.K)) {
    check(fla_chunk_gla_fwd_fused_split(ptr(q), ptr(k), ptr(v), ptr(g), fptr(h0), ptr(o), fptr(*ht), (int*)ptr(wide),
                                        ptr(hwide), ptr(x.hT), ptr(x.qg), fptr(x.decay), nullptr, nullptr, offs(a.plan),
                                        idx(a.plan), coff(a.plan), &c->s, d.NT, dt(q), dt(g), d.B, d.T, d.H, d.K, d.V, d.N,
                                        (float)a.scale, form, (float)a.normalizer, a.clamp.has_value(),
                                        (float)a.clamp.value_or(0.0), st),
          "fla_chunk_gla_fwd_fused_split");
  } else if (form == 1) {
    check(fla_chunk_simple_gla_fwd_fused(ptr(q), ptr(k), ptr(v), fptr(g), fptr(h0), ptr(o), fptr(*ht), (int*)ptr(wide),
                                         ptr(hwide), ptr(x.hT), ptr(x.qg), fptr(x.decay), nullptr, nullptr, offs(a.plan),
                                         idx(a.plan), coff(a.plan), order(a.plan), d.NT, dt(q), d.B, d.T, d.H, d.K, d.V,
                                         d.N, (float)a.scale, st),
          "fla_chunk_simple_gla_fwd_fused");
  } else if (form == 2) {
    check(fla_chunk_gla_fwd_fused_logits(ptr(q), ptr(k), ptr(v), ptr(g), fptr(h0), ptr(o), fptr(*ht), (int*)ptr(wide),
                                         ptr(hwide), offs(a.plan), idx(a.plan), coff(a.plan), order(a.plan), d.NT, dt(q),
                                         dt(g), d.B, d.T, d.H, d.K, d.V, d.N, (float)a.scale, (float)a.normalizer,
                                         a.clamp.has_value(), (float)a.clamp.value_or(0.0), st),
          "fla_chunk_gla_fwd_fused_logits");
  } else if (kept) {
    check(fla_chunk_gla_fwd_fused_kept(ptr(q), ptr(k), ptr(v), ptr(g), fptr(h0), ptr(o), fptr(*ht), (int*)ptr(wide),
                                       ptr(hwide), ptr(x.hT), ptr(x.qg), fptr(x.decay), nullptr, nullptr, offs(a.plan),
                                       idx(a.plan), coff(a.plan), order(a.plan), d.NT, dt(q), dt(g), d.B, d.T, d.H, d.K,
                                       d.V, d.N, (float)a.scale, st),
          "fla_chunk_gla_fwd_fused_kept");
  } else {
    check(fla_chunk_gla_fwd_fused(ptr(q), ptr(k), ptr(v), ptr(g), fptr(h0), ptr(o), fptr(*ht), (int*)ptr(wide), ptr(hwide),
                                  offs(a.plan), idx(a.plan), coff(a.plan), order(a.plan), d.NT, dt(q), dt(g), d.B, d.T, d.H,
                                  d.K, d.V, d.N, (float)a.scale, st),
          "fla_chunk_gla_fwd_fused");
  }
  return o;
}

struct GlaNode : torch::autograd::Function<GlaNode> {
  struct Rest {
    GlaArgs a;
    at::ScalarType g_type;
    bool has_h0;
  };
  static variable_list forward(AutogradContext* ctx, const Tensor& q_, const Tensor& k_, const Tensor& v_, const Tensor& g_,
                               const Maybe& h0_, const Maybe& offsets, const GlaArgs& a) {
    at::AutoDispatchBelowADInplaceOrView guard;
    const Tensor q = q_.contiguous(), k = k_.contiguous(), v = v_.contiguous();
    const Tensor g = (a.head_gates ? f32(g_) : g_.contiguous());
    const Tensor h0 = h0_ ? h0_->contiguous() : Tensor();
    Tensor ht;
    GlaKept x;
    Tensor o = gla_forward(q, k, v, g, h0, a, &ht, &x);
    ctx->save_for_backward({q, k, v, g, x.wide, x.hT, x.qg, x.decay, given(offsets)});
    ctx->set_materialize_grads(false);
    hold(ctx, Rest{a, g_.scalar_type(), h0.defined()});
    return a.want_ht ? variable_list{o, ht} : variable_list{o};
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    at::AutoDispatchBelowADInplaceOrView guard;
    const auto saved = ctx->get_saved_variables();
    const Rest& rest = held<Rest>(ctx);
    const GlaArgs& a = rest.a;
    const Dims& d = a.d;
    const Tensor &q = saved[0], &k = saved[1], &v = saved[2], &g = saved[3], &wide = saved[4], &hT = saved[5], &qg = saved[6],
                 &decay = saved[7];
    const Tensor dout = grads[0].defined() ? as(grads[0], q.scalar_type()).contiguous() : at::zeros(v.sizes(), v.options());
    const Tensor dht = a.want_ht ? f32(grads[1]) : Tensor();
    Tensor dhtf = fresh_like(hT), dq = fresh_like(q), dk = fresh_like(k), dv = fresh_like(v);
    // per-head gates: rows of a packed batch that belong to no sequence have a gradient of zero
    Tensor dg = !a.head_gates                       ? fresh(q.sizes(), q, at::kFloat)
                : !a.plan || a.plan->covers(0, d.T) ? fresh({d.B, d.T, d.H}, q, at::kFloat)
                                                    : at::zeros({d.B, d.T, d.H}, g.options());
    Tensor dh0 = rest.has_h0 ? fresh({d.N, d.H, d.K, d.V}, q, at::kFloat) : Tensor();
    const fla_stream_t st = stream_of(q);
    // (the reverse scan's workgroups hold 64 x 64 tiles of a state)
    auto c = cut_scan(a.plan, d.N, d.T, d.H, (int)(d.K / 64 * (d.V / 64)), true, q, d.K * d.V, d.K,
                      FLA_SCAN_GLA_GRADIENT);
    if (c) {
      check(fla_chunk_gla_bwd_split(ptr(q), ptr(k), ptr(v), ptr(g), ptr(dout), fptr(dht), ptr(hT), ptr(qg), fptr(decay),
                                    nullptr, nullptr, ptr(dhtf), ptr(dq), ptr(dk), ptr(dv), fptr(dg), fptr(dh0),
                                    (const int*)ptr(wide), offs(a.plan), idx(a.plan), coff(a.plan), &c->s, d.NT, dt(q), dt(g),
                                    d.B, d.T, d.H, d.K, d.V, d.N, (float)a.scale, a.head_gates, st),
            "fla_chunk_gla_bwd_split");
    } else if (a.head_gates) {
      check(fla_chunk_simple_gla_bwd(ptr(q), ptr(k), ptr(v), fptr(g), ptr(dout), fptr(dht), ptr(hT), ptr(qg), fptr(decay),
                                     nullptr, nullptr, ptr(dhtf), ptr(dq), ptr(dk), ptr(dv), fptr(dg), fptr(dh0),
                                     (const int*)ptr(wide), offs(a.plan), idx(a.plan), coff(a.plan), d.NT, dt(q), d.B, d.T,
                                     d.H, d.K, d.V, d.N, (float)a.scale, st),
            "fla_chunk_simple_gla_bwd");
    } else {
      check(fla_chunk_gla_bwd_kept(ptr(q), ptr(k), ptr(v), ptr(g), ptr(dout), fptr(dht), ptr(hT), ptr(qg), fptr(decay),
                                   nullptr, nullptr, ptr(dhtf), ptr(dq), ptr(dk), ptr(dv), fptr(dg), fptr(dh0),
                                   (const int*)ptr(wide), offs(a.plan), idx(a.plan), coff(a.plan), d.NT, dt(q), dt(g), d.B,
                                   d.T, d.H, d.K, d.V, d.N, (float)a.scale, st),
            "fla_chunk_gla_bwd_kept");
    }
    return {dq, dk, dv, as(dg, rest.g_type), dh0, Tensor(), Tensor()};
  }
};

// The forward of chunk_simple_gla that is not differentiated
Tensor simple_gla_scan(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& g, const Tensor& h0, const GlaArgs& a,
                       Tensor* ht) {
  const Dims& d = a.d;
  Tensor o = fresh_like(v);
  if (a.want_ht) *ht = fresh({d.N, d.H, d.K, d.V}, q, at::kFloat);
  if (auto c = cut_scan(a.plan, d.N, d.T, d.H, (int)(d.V / 64), false, q, d.K * d.V, d.K,
                        FLA_SCAN_SIMPLE)) {
    check(fla_chunk_gated_delta_rule_fwd_scan_split(ptr(q), ptr(k), ptr(v), nullptr, fptr(g), nullptr, fptr(h0), ptr(o),
                                                    fptr(*ht), nullptr, nullptr, nullptr, offs(a.plan), coff(a.plan), &c->s,
                                                    dt(q), d.B, d.T, d.H, d.K, d.V, d.N, (float)a.scale, 0.f, stream_of(q)),
          "fla_chunk_gated_delta_rule_fwd_scan_split");
    return o;
  }
  check(fla_chunk_simple_gla_fwd_scan(ptr(q), ptr(k), ptr(v), fptr(g), fptr(h0), ptr(o), fptr(*ht), offs(a.plan),
                                      coff(a.plan), order(a.plan), dt(q), d.B, d.T, d.H, d.K, d.V, d.N, (float)a.scale,
                                      stream_of(q)),
        "fla_chunk_simple_gla_fwd_scan");
  return o;
}

// ---------------------------------------------------------------------------------------------------- delta rule
struct GdrArgs {
  Dims d;
  PlanPtr plan;
  double scale;
  bool want_ht;
  std::optional<double> l2norm_eps;
};
struct GdrKept {
  Tensor gc, AT, Aw, v_new, hT, Aqk, Mt;   // Mt: the segments' transposed transitions where the forward was cut
};

// the kind of a delta-rule scan as fla_scan_split takes it: the same for a forward that keeps its intermediates and its backward
int delta_scan(const Dims& d, bool kept) {
  return (kept ? FLA_SCAN_DELTA_KEPT : FLA_SCAN_DELTA) | (d.K == 64 ? FLA_SCAN_KEYS_64 : 0);
}

Tensor gdr_forward(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& g, const Tensor& beta, const Tensor& h0,
                   const GdrArgs& a, Tensor* ht, GdrKept* kept) {
  const Dims& d = a.d;
  const fla_stream_t st = stream_of(q);
  Tensor AT = fresh({d.chunks, d.H, 10, 16, 16}, q, q.scalar_type());
  Tensor gc = g.defined() ? fresh_like(g) : Tensor();
  Tensor o = fresh_like(v);
  if (a.want_ht) *ht = fresh({d.N, d.H, d.K, d.V}, q, at::kFloat);
  // sequences cut into segments: their K x K transitions take the place of the decays
  auto cut = cut_scan(a.plan, d.N, d.T, d.H, (int)(d.V / 64), false, q, d.K * d.V, d.K * d.K,
                      delta_scan(d, kept));
  auto scan_cut = [&](const Tensor& rstd, const GdrKept& x) {
    check(fla_chunk_gated_delta_rule_fwd_scan_split(ptr(q), ptr(k), ptr(v), ptr(AT), fptr(gc), fptr(rstd), fptr(h0), ptr(o),
                                                    fptr(*ht), ptr(x.v_new), ptr(x.hT), ptr(x.Aqk), offs(a.plan), coff(a.plan),
                                                    &cut->s, dt(q), d.B, d.T, d.H, d.K, d.V, d.N, (float)a.scale,
                                                    (float)a.l2norm_eps.value_or(0.0), st),
          "fla_chunk_gated_delta_rule_fwd_scan_split");
  };
  if (a.l2norm_eps) {
    Tensor rstd = fresh({d.B, d.T, d.H}, q, at::kFloat);
    check(fla_gdr_fwd_prep_l2norm(ptr(k), fptr(beta), fptr(g), 0, fptr(gc), ptr(AT), fptr(rstd), offs(a.plan), idx(a.plan),
                                  d.NT, dt(q), d.B, d.T, d.H, d.K, (float)*a.l2norm_eps, st),
          "fla_gdr_fwd_prep_l2norm");
    if (cut) {
      scan_cut(rstd, {});
      return o;
    }
    check(fla_chunk_gated_delta_rule_fwd_scan_l2norm(ptr(q), ptr(k), ptr(v), ptr(AT), fptr(gc), fptr(rstd), fptr(h0), ptr(o),
                                                     fptr(*ht), offs(a.plan), coff(a.plan), order(a.plan), dt(q), d.B, d.T,
                                                     d.H, d.K, d.V, d.N, (float)a.scale, (float)*a.l2norm_eps, st),
          "fla_chunk_gated_delta_rule_fwd_scan_l2norm");
    return o;
  }
  GdrKept none, &x = kept ? *kept : none;
  if (kept) {
    x.gc = gc;
    x.AT = AT;
    x.Aw = fresh({d.B, d.T, d.H, BT}, q, q.scalar_type());
    x.v_new = fresh_like(v);
    x.hT = fresh({d.chunks, d.H, d.K, d.V}, q, q.scalar_type());
    x.Aqk = fresh_like(AT);
    if (cut) {
      x.Mt = fresh_like(cut->transitions);
      cut->s.transitions_t = fptr(x.Mt);
    }
  }
  if (kept)
    check(fla_gdr_fwd_prep_kept(ptr(k), fptr(beta), fptr(g), 0, fptr(gc), ptr(AT), ptr(x.Aw), offs(a.plan), idx(a.plan),
                                d.NT, dt(q), d.B, d.T, d.H, d.K, st),
          "fla_gdr_fwd_prep_kept");
  else
    check(fla_gdr_fwd_prep(ptr(k), fptr(beta), fptr(g), 0, fptr(gc), ptr(AT), nullptr, nullptr, offs(a.plan), idx(a.plan),
                           d.NT, dt(q), d.B, d.T, d.H, d.K, st),
          "fla_gdr_fwd_prep");
  if (cut) {
    scan_cut({}, x);
    return o;
  }
  check(fla_chunk_gated_delta_rule_fwd_scan(ptr(q), ptr(k), ptr(v), ptr(AT), fptr(gc), fptr(h0), ptr(o), fptr(*ht),
                                            ptr(x.v_new), ptr(x.hT), ptr(x.Aqk), offs(a.plan), coff(a.plan), order(a.plan),
                                            dt(q), d.B, d.T, d.H, d.K, d.V, d.N, (float)a.scale, st),
        "fla_chunk_gated_delta_rule_fwd_scan");
  return o;
}

struct GdrNode : torch::autograd::Function<GdrNode> {
  struct Rest {
    GdrArgs a;
    std::optional<at::ScalarType> g_type;
    at::ScalarType beta_type;
    bool has_h0;
  };
  static variable_list forward(AutogradContext* ctx, const Tensor& q_, const Tensor& k_, const Tensor& v_, const Maybe& g_,
                               const Tensor& beta_, const Maybe& h0_, const Maybe& offsets, const GdrArgs& a) {
    at::AutoDispatchBelowADInplaceOrView guard;
    const Tensor q = q_.contiguous(), k = k_.contiguous(), v = v_.contiguous(), g = f32(given(g_)), beta = f32(beta_);
    const Tensor h0 = h0_ ? h0_->contiguous() : Tensor();
    Tensor ht;
    GdrKept x;
    Tensor o = gdr_forward(q, k, v, g, beta, h0, a, &ht, &x);
    ctx->save_for_backward({q, k, v, beta, x.gc, x.AT, x.Aw, x.v_new, x.hT, x.Aqk, x.Mt, given(offsets)});
    ctx->set_materialize_grads(false);
    Rest r{a, std::nullopt, beta_.scalar_type(), h0.defined()};
    if (g_) r.g_type = g_->scalar_type();
    hold(ctx, std::move(r));
    return a.want_ht ? variable_list{o, ht} : variable_list{o};
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    at::AutoDispatchBelowADInplaceOrView guard;
    const auto saved = ctx->get_saved_variables();
    const Rest& r = held<Rest>(ctx);
    const GdrArgs& a = r.a;
    const Dims& d = a.d;
    const Tensor &q = saved[0], &k = saved[1], &v = saved[2], &beta = saved[3], &gc = saved[4], &AT = saved[5], &Aw = saved[6],
                 &v_new = saved[7], &hT = saved[8], &Aqk = saved[9],
                 &Mt = saved[10];
    const Tensor dout = grads[0].defined() ? as(grads[0], q.scalar_type()).contiguous() : at::zeros(v.sizes(), v.options());
    const Tensor dht = a.want_ht ? f32(grads[1]) : Tensor();
    Tensor dv2 = fresh_like(v), dh = fresh_like(hT);
    Tensor dq = fresh_like(q), dk = fresh_like(k), dv = fresh_like(v);
    Tensor dbeta = fresh({d.B, d.T, d.H}, q, at::kFloat), dg = fresh({d.B, d.T, d.H}, q, at::kFloat);
    Tensor dh0 = r.has_h0 ? fresh({d.N, d.H, d.K, d.V}, q, at::kFloat) : Tensor();
    std::optional<Cut> cut;
    if (Mt.defined())
      cut = cut_scan(a.plan, d.N, d.T, d.H, (int)(d.V / 64), true, q, d.K * d.V, 0, delta_scan(d, true));
    if (cut) cut->s.decays = fptr(Mt);
    check(fla_chunk_gated_delta_rule_bwd_tiles(
              ptr(q), ptr(k), ptr(v), ptr(AT), ptr(v_new), fptr(beta), fptr(gc), ptr(Aw), ptr(dout), fptr(dht), ptr(hT),
              ptr(Aqk), ptr(dv2), ptr(dh), ptr(dq), ptr(dk), ptr(dv), fptr(dbeta), fptr(dg), fptr(dh0), offs(a.plan),
              idx(a.plan), coff(a.plan), cut ? &cut->s : nullptr, d.NT, dt(q), d.B, d.T, d.H, d.K, d.V, d.N, (float)a.scale,
              stream_of(q)),
          "fla_chunk_gated_delta_rule_bwd_tiles");
    return {dq, dk, dv, r.g_type ? as(dg, *r.g_type) : Tensor(), as(dbeta, r.beta_type), dh0, Tensor(), Tensor()};
  }
};

// ---------------------------------------------------------------------------------------------------- layer steps
bool rows_ok(const Tensor& x) {
  return x.defined() && x.is_cuda() && x.dim() >= 1 && x.numel() > 0 && x.size(-1) % 8 == 0 && x.size(-1) <= 2048 &&
         (is16(x) || x.scalar_type() == at::kFloat);
}

// The column sums of per-workgroup partial sums [parts, ...], in the dtype and shape of the weight they belong to
Tensor sum_partials(const Tensor& part, at::IntArrayRef shape, at::ScalarType type) {
  const bool direct = type == at::kFloat || type == at::kBFloat16 || type == at::kHalf;
  Tensor out = fresh(shape, part, direct ? type : at::kFloat);
  check(fla_sum_partials(fptr(part), ptr(out), part.size(0), part.numel() / part.size(0), dt(out), stream_of(part)),
        "fla_sum_partials");
  return as(out, type);
}

struct L2NormNode : torch::autograd::Function<L2NormNode> {
  static Tensor run(const Tensor& x, double eps) {
    Tensor y = fresh_like(x);
    const int64_t D = x.size(-1);
    check(fla_l2norm_fwd(ptr(x), ptr(y), x.numel() / D, D, (float)eps, dt(x), dt(y), stream_of(x)), "fla_l2norm_fwd");
    return y;
  }
  static Tensor forward(AutogradContext* ctx, const Tensor& x_, double eps) {
    at::AutoDispatchBelowADInplaceOrView guard;
    const Tensor x = x_.contiguous();
    ctx->save_for_backward({x});
    hold(ctx, eps);
    return run(x, eps);
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    at::AutoDispatchBelowADInplaceOrView guard;
    const Tensor x = ctx->get_saved_variables()[0], dy = grads[0].contiguous();
    Tensor dx = fresh_like(x);
    const int64_t D = x.size(-1);
    check(fla_l2norm_bwd(ptr(x), ptr(dy), ptr(dx), x.numel() / D, D, (float)held<double>(ctx), dt(x), dt(dy), stream_of(x)),
          "fla_l2norm_bwd");
    return {dx, Tensor()};
  }
};

struct ConvNode : torch::autograd::Function<ConvNode> {
  struct Rest {
    int silu;
    std::vector<int64_t> w_shape;
    at::ScalarType w_type;
    std::optional<at::ScalarType> b_type;
  };
  static Tensor run(const Tensor& x, const Tensor& w, const Tensor& b, int silu) {
    Tensor y = fresh_like(x);
    check(fla_causal_conv1d_fwd(ptr(x), fptr(w), fptr(b), ptr(y), x.size(0), x.size(1), x.size(2), w.size(-1), silu, dt(x),
                                stream_of(x)),
          "fla_causal_conv1d_fwd");
    return y;
  }
  static Tensor forward(AutogradContext* ctx, const Tensor& x_, const Tensor& w_, const Maybe& b_, int silu) {
    at::AutoDispatchBelowADInplaceOrView guard;
    const Tensor x = x_.contiguous(), w = f32(w_), b = f32(given(b_));
    ctx->save_for_backward({x, w, b});
    Rest r{silu, w_.sizes().vec(), w_.scalar_type(), std::nullopt};
    if (b_) r.b_type = b_->scalar_type();
    hold(ctx, std::move(r));
    return run(x, w, b, silu);
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    at::AutoDispatchBelowADInplaceOrView guard;
    const auto saved = ctx->get_saved_variables();
    const Tensor &x = saved[0], &w = saved[1], &b = saved[2];
    const Rest& r = held<Rest>(ctx);
    const int64_t B = x.size(0), T = x.size(1), D = x.size(2), W = w.size(-1);
    const Tensor dy = as(grads[0], x.scalar_type()).contiguous();
    Tensor dx = fresh_like(x);
    const int64_t parts = fla_causal_conv1d_bwd_partials(B, T);
    Tensor dw = fresh({parts, D, W}, x, at::kFloat), db = b.defined() ? fresh({parts, D}, x, at::kFloat) : Tensor();
    check(fla_causal_conv1d_bwd(ptr(x), fptr(w), fptr(b), ptr(dy), ptr(dx), fptr(dw), fptr(db), B, T, D, W, r.silu, dt(x),
                                stream_of(x)),
          "fla_causal_conv1d_bwd");
    return {dx, sum_partials(dw, r.w_shape, r.w_type), b.defined() ? sum_partials(db, {D}, *r.b_type) : Tensor(), Tensor()};
  }
};

struct NormGateNode : torch::autograd::Function<NormGateNode> {
  struct Rest {
    double eps;
    bool rms;
  };
  static Tensor run(const Tensor& x, const Tensor& o, const Tensor& w, const Tensor& b, double eps, bool rms, Tensor* mean,
                    Tensor* rstd) {
    const int64_t D = x.size(-1), M = x.numel() / D;
    Tensor y = fresh_like(x);
    if (!rms) *mean = fresh({M}, x, at::kFloat);
    *rstd = fresh({M}, x, at::kFloat);
    check(fla_norm_swish_gate_fwd(ptr(x), ptr(o), fptr(w), fptr(b), ptr(y), fptr(*mean), fptr(*rstd), M, D, (float)eps, rms,
                                  dt(x), stream_of(x)),
          "fla_norm_swish_gate_fwd");
    return y;
  }
  static Tensor forward(AutogradContext* ctx, const Tensor& x_, const Tensor& o_, const Maybe& w_, const Maybe& b_,
                        double eps, bool rms) {
    at::AutoDispatchBelowADInplaceOrView guard;
    const Tensor w = given(w_), b = given(b_);
    const Tensor x = x_.contiguous(), o = o_.contiguous();
    Tensor mean, rstd;
    Tensor y = run(x, o, f32(w), f32(b), eps, rms, &mean, &rstd);
    ctx->save_for_backward({x, o, w, b, mean, rstd});
    hold(ctx, Rest{eps, rms});
    return y;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    at::AutoDispatchBelowADInplaceOrView guard;
    const auto saved = ctx->get_saved_variables();
    const Tensor &x = saved[0], &o = saved[1], &w = saved[2], &b = saved[3], &mean = saved[4], &rstd = saved[5];
    const Rest& r = held<Rest>(ctx);
    const int64_t D = x.size(-1), M = x.numel() / D;
    const Tensor dy = as(grads[0], x.scalar_type()).contiguous();
    Tensor dx = fresh_like(x), dgate = fresh_like(o);
    const int64_t parts = fla_norm_swish_gate_workgroups(M, D);
    Tensor dw = w.defined() ? fresh({parts, D}, x, at::kFloat) : Tensor();
    Tensor db = b.defined() ? fresh({parts, D}, x, at::kFloat) : Tensor();
    const Tensor w32 = f32(w), b32 = f32(b);
    check(fla_norm_swish_gate_bwd(ptr(dy), ptr(x), ptr(o), fptr(w32), fptr(b32), fptr(mean), fptr(rstd), ptr(dx), ptr(dgate),
                                  fptr(dw), fptr(db), M, D, (float)r.eps, r.rms, dt(x), stream_of(x)),
          "fla_norm_swish_gate_bwd");
    return {dx, dgate, w.defined() ? sum_partials(dw, w.sizes(), w.scalar_type()) : Tensor(),
            b.defined() ? sum_partials(db, b.sizes(), b.scalar_type()) : Tensor(), Tensor(), Tensor()};
  }
};

// ---------------------------------------------------------------------------------------------------- Python entries
Tensor arg_tensor(PyObject* o) {
  if (o == Py_None) return Tensor();
  TORCH_CHECK_TYPE(THPVariable_Check(o), "fla_amd: expected a tensor, got ", Py_TYPE(o)->tp_name);
  return THPVariable_Unpack(o);
}
bool arg_bool(PyObject* o) {
  const int r = PyObject_IsTrue(o);
  if (r < 0) throw python_error();
  return r != 0;
}
double arg_double(PyObject* o) {
  const double r = PyFloat_AsDouble(o);
  if (r == -1.0 && PyErr_Occurred()) throw python_error();
  return r;
}
std::optional<double> arg_opt_double(PyObject* o) {
  if (o == Py_None) return std::nullopt;
  return arg_double(o);
}
constexpr const char* kPlanName = "fla_amd.plan";
PlanPtr arg_plan(PyObject* o) {
  if (o == Py_None) return PlanPtr();
  auto* p = (Plan*)PyCapsule_GetPointer(o, kPlanName);
  if (!p) throw python_error();
  return PlanPtr::reclaim_copy(p);
}
void expect(Py_ssize_t n, Py_ssize_t want) { TORCH_CHECK_TYPE(n == want, "fla_amd: expected ", want, " arguments, got ", n); }
PyObject* none() { Py_RETURN_NONE; }
PyObject* pair(const Tensor& o, const Tensor& ht) {
  PyObject* t = PyTuple_New(2);
  if (!t) throw python_error();
  PyTuple_SET_ITEM(t, 0, THPVariable_Wrap(o));
  if (ht.defined()) {
    PyTuple_SET_ITEM(t, 1, THPVariable_Wrap(ht));
  } else {
    Py_INCREF(Py_None);
    PyTuple_SET_ITEM(t, 1, Py_None);
  }
  return t;
}

void plan_free(PyObject* cap) { PlanPtr::reclaim((Plan*)PyCapsule_GetPointer(cap, kPlanName)); }

// plan(offsets, indices, chunk_offsets, seq_order, host offsets as a CPU int64 tensor)
PyObject* py_plan(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  expect(n, 5);
  auto p = c10::make_intrusive<Plan>();
  p->offsets = arg_tensor(a[0]);
  p->indices = arg_tensor(a[1]);
  p->chunk_offsets = arg_tensor(a[2]);
  p->seq_order = arg_tensor(a[3]);
  const Tensor host = arg_tensor(a[4]).contiguous();
  const int64_t* h = host.data_ptr<int64_t>();
  p->host.assign(h, h + host.numel());
  p->N = host.numel() - 1;
  p->NT = p->indices.size(0);
  return PyCapsule_New(p.release(), kPlanName, plan_free);
  END_HANDLE_TH_ERRORS
}

// chunk_gla(q, k, v, g, scale, h0, want_ht, plan, may_differentiate, normalizer, clamp, offsets)
//   normalizer None: g holds log-gates
PyObject* py_chunk_gla(PyObject*, PyObject* const* p, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  expect(n, 12);
  Tensor q = arg_tensor(p[0]), k = arg_tensor(p[1]), v = arg_tensor(p[2]), g = arg_tensor(p[3]), h0 = arg_tensor(p[5]),
         offsets = arg_tensor(p[11]);
  GlaArgs a{};
  a.plan = arg_plan(p[7]);
  if (!chunk_operands(q, k, v, h0, a.plan, &a.d) || !g.defined() || !g.is_cuda() || g.sizes() != q.sizes()) return none();
  if (g.scalar_type() != at::kFloat && g.scalar_type() != q.scalar_type()) return none();
  const bool grad = wants_grad({&q, &k, &v, &g, &h0});
  const auto normalizer = arg_opt_double(p[9]);
  if (grad && (normalizer || !arg_bool(p[8]))) return none();
  a.scale = p[4] == Py_None ? 1.0 / std::sqrt((double)a.d.K) : arg_double(p[4]);
  if (grad && a.scale == 0.0) return none();
  a.want_ht = arg_bool(p[6]);
  if (normalizer) {
    a.gate_form = 2;
    a.normalizer = *normalizer;
    a.clamp = arg_opt_double(p[10]);
  }
  if (grad) {
    auto out = GlaNode::apply(q, k, v, g, maybe(h0), maybe(offsets), a);
    return pair(out[0], a.want_ht ? out[1] : Tensor());
  }
  at::AutoDispatchBelowADInplaceOrView guard;
  Tensor ht;
  Tensor o = gla_forward(q.contiguous(), k.contiguous(), v.contiguous(), g.contiguous(), h0.defined() ? h0.contiguous() : h0, a,
                         &ht, nullptr);
  return pair(o, ht);
  END_HANDLE_TH_ERRORS
}

// chunk_simple_gla(q, k, v, g, scale, h0, want_ht, plan, may_differentiate, offsets)
PyObject* py_chunk_simple_gla(PyObject*, PyObject* const* p, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  expect(n, 10);
  Tensor q = arg_tensor(p[0]), k = arg_tensor(p[1]), v = arg_tensor(p[2]), g = arg_tensor(p[3]), h0 = arg_tensor(p[5]),
         offsets = arg_tensor(p[9]);
  GlaArgs a{};
  a.plan = arg_plan(p[7]);
  if (!chunk_operands(q, k, v, h0, a.plan, &a.d) || !g.defined() || !g.is_cuda() || g.dim() != 3 || g.size(0) != a.d.B ||
      g.size(1) != a.d.T || g.size(2) != a.d.H || !g.is_floating_point())
    return none();
  const bool grad = wants_grad({&q, &k, &v, &g, &h0});
  if (grad && !arg_bool(p[8])) return none();
  a.scale = p[4] == Py_None ? 1.0 / std::sqrt((double)a.d.K) : arg_double(p[4]);
  if (grad && a.scale == 0.0) return none();
  a.want_ht = arg_bool(p[6]);
  a.head_gates = true;
  if (grad) {
    auto out = GlaNode::apply(q, k, v, g, maybe(h0), maybe(offsets), a);
    return pair(out[0], a.want_ht ? out[1] : Tensor());
  }
  at::AutoDispatchBelowADInplaceOrView guard;
  Tensor ht;
  Tensor o = simple_gla_scan(q.contiguous(), k.contiguous(), v.contiguous(), f32(g), h0.defined() ? h0.contiguous() : h0, a, &ht);
  return pair(o, ht);
  END_HANDLE_TH_ERRORS
}

// chunk_gdr(q, k, v, g | None, beta, scale, h0, want_ht, plan, may_differentiate, l2norm_eps | None, offsets)
PyObject* py_chunk_gdr(PyObject*, PyObject* const* p, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  expect(n, 12);
  Tensor q = arg_tensor(p[0]), k = arg_tensor(p[1]), v = arg_tensor(p[2]), g = arg_tensor(p[3]), beta = arg_tensor(p[4]),
         h0 = arg_tensor(p[6]), offsets = arg_tensor(p[11]);
  GdrArgs a{};
  a.plan = arg_plan(p[8]);
  if (!chunk_operands(q, k, v, h0, a.plan, &a.d) || !beta.defined() || !on_gpu({&g, &beta})) return none();
  auto per_head = [&](const Tensor& t) {
    return t.dim() == 3 && t.size(0) == a.d.B && t.size(1) == a.d.T && t.size(2) == a.d.H && t.is_floating_point();
  };
  if (!per_head(beta) || (g.defined() && !per_head(g))) return none();
  const bool grad = wants_grad({&q, &k, &v, &g, &beta, &h0});
  if (grad && !arg_bool(p[9])) return none();
  a.scale = arg_double(p[5]);
  a.want_ht = arg_bool(p[7]);
  a.l2norm_eps = arg_opt_double(p[10]);
  if (grad) {
    if (a.l2norm_eps) {
      q = L2NormNode::apply(q, *a.l2norm_eps);
      k = L2NormNode::apply(k, *a.l2norm_eps);
      a.l2norm_eps.reset();
    }
    auto out = GdrNode::apply(q, k, v, maybe(g), beta, maybe(h0), maybe(offsets), a);
    return pair(out[0], a.want_ht ? out[1] : Tensor());
  }
  at::AutoDispatchBelowADInplaceOrView guard;
  Tensor ht;
  Tensor o = gdr_forward(q.contiguous(), k.contiguous(), v.contiguous(), f32(g), f32(beta), h0.defined() ? h0.contiguous() : h0, a,
                         &ht, nullptr);
  return pair(o, ht);
  END_HANDLE_TH_ERRORS
}

// The recurrences on equal-length sequences, without gradients.  State in fp32, contiguous where it is updated in place.
bool recurrent_operands(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& h0, bool inplace, Dims* d) {
  if (!q.defined() || !k.defined() || !v.defined() || q.dim() != 4 || v.dim() != 4 || q.sizes() != k.sizes() || q.numel() == 0)
    return false;
  if (!(is16(q) || q.scalar_type() == at::kFloat) || k.scalar_type() != q.scalar_type() || v.scalar_type() != q.scalar_type())
    return false;
  d->B = d->N = q.size(0), d->T = q.size(1), d->H = q.size(2), d->K = q.size(3), d->V = v.size(3);
  if (v.size(0) != d->B || v.size(1) != d->T || v.size(2) != d->H || d->K > 256 || d->V % 4 != 0 || d->V == 0) return false;
  if (inplace && (!h0.defined() || !h0.is_contiguous())) return false;
  return !h0.defined() || (h0.scalar_type() == at::kFloat && h0.dim() == 4 && h0.size(0) == d->N && h0.size(1) == d->H &&
                           h0.size(2) == d->K && h0.size(3) == d->V);
}
Tensor cont(const Tensor& x) { return x.defined() && !x.is_contiguous() ? x.contiguous() : x; }

// recurrent_gla(q, k, v, g | None, gk | None, gv | None, scale, h0, want_ht, reverse, inplace)
PyObject* py_recurrent_gla(PyObject*, PyObject* const* p, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  expect(n, 11);
  Tensor q = arg_tensor(p[0]), k = arg_tensor(p[1]), v = arg_tensor(p[2]), g = arg_tensor(p[3]), gk = arg_tensor(p[4]),
         gv = arg_tensor(p[5]), h0 = arg_tensor(p[7]);
  Dims d{};
  const bool want = arg_bool(p[8]), inplace = arg_bool(p[10]);
  if (wants_grad({&q, &k, &v, &g, &gk, &gv, &h0}) || !on_gpu({&q, &k, &v, &g, &gk, &gv, &h0}) ||
      !recurrent_operands(q, k, v, h0, inplace && want, &d))
    return none();
  at::ScalarType gt = at::kFloat;
  bool have = false;
  for (const Tensor* t : {&g, &gk, &gv}) {
    if (!t->defined()) continue;
    if (have && t->scalar_type() != gt) return none();
    gt = t->scalar_type();
    have = true;
  }
  if (gt != at::kFloat && gt != q.scalar_type()) return none();
  if ((g.defined() && g.numel() != d.B * d.T * d.H) || (gk.defined() && gk.sizes() != k.sizes()) ||
      (gv.defined() && gv.sizes() != v.sizes()))
    return none();
  at::AutoDispatchBelowADInplaceOrView guard;
  q = cont(q), k = cont(k), v = cont(v), g = cont(g), gk = cont(gk), gv = cont(gv), h0 = cont(h0);
  Tensor o = fresh_like(v), ht;
  if (want) ht = inplace ? h0 : fresh({d.N, d.H, d.K, d.V}, q, at::kFloat);
  check(fla_fused_recurrent_fwd(ptr(q), ptr(k), ptr(v), ptr(g), ptr(gk), ptr(gv), ptr(o), fptr(h0), fptr(ht), nullptr, dt(q),
                                gt == at::kFloat ? FLA_F32 : dt(q), dt(o), d.B, d.T, d.H, d.K, d.V, d.N,
                                (float)arg_double(p[6]), arg_bool(p[9]), stream_of(q)),
        "fla_fused_recurrent_fwd");
  return pair(o, ht);
  END_HANDLE_TH_ERRORS
}

// recurrent_gdr(q, k, v, g | None, beta, scale, h0, want_ht, inplace, l2norm_eps | None)
PyObject* py_recurrent_gdr(PyObject*, PyObject* const* p, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  expect(n, 10);
  Tensor q = arg_tensor(p[0]), k = arg_tensor(p[1]), v = arg_tensor(p[2]), g = arg_tensor(p[3]), beta = arg_tensor(p[4]),
         h0 = arg_tensor(p[6]);
  Dims d{};
  const bool want = arg_bool(p[7]), inplace = arg_bool(p[8]);
  if (wants_grad({&q, &k, &v, &g, &beta, &h0}) || !beta.defined() || !on_gpu({&q, &k, &v, &g, &beta, &h0}) ||
      !recurrent_operands(q, k, v, h0, inplace && want, &d))
    return none();
  const bool per_value = beta.dim() == 4;
  if (per_value ? beta.sizes() != v.sizes() : beta.numel() != d.B * d.T * d.H) return none();
  if (g.defined() && g.numel() != d.B * d.T * d.H) return none();
  at::AutoDispatchBelowADInplaceOrView guard;
  q = cont(q), k = cont(k), v = cont(v), h0 = cont(h0), g = f32(g), beta = f32(beta);
  Tensor o = fresh_like(v), ht;
  if (want) ht = inplace ? h0 : fresh({d.N, d.H, d.K, d.V}, q, at::kFloat);
  const float scale = (float)arg_double(p[5]);
  if (const auto eps = arg_opt_double(p[9]))
    check(fla_fused_recurrent_gated_delta_rule_fwd_l2norm(ptr(q), ptr(k), ptr(v), ptr(g), ptr(beta), ptr(o), fptr(h0), fptr(ht),
                                                          nullptr, dt(q), FLA_F32, dt(o), per_value, d.B, d.T, d.H, d.K, d.V,
                                                          d.N, scale, (float)*eps, stream_of(q)),
          "fla_fused_recurrent_gated_delta_rule_fwd_l2norm");
  else
    check(fla_fused_recurrent_gated_delta_rule_fwd(ptr(q), ptr(k), ptr(v), ptr(g), ptr(beta), ptr(o), fptr(h0), fptr(ht),
                                                   nullptr, dt(q), FLA_F32, dt(o), per_value, d.B, d.T, d.H, d.K, d.V, d.N,
                                                   scale, stream_of(q)),
          "fla_fused_recurrent_gated_delta_rule_fwd");
  return pair(o, ht);
  END_HANDLE_TH_ERRORS
}

// l2_norm(x, eps)
PyObject* py_l2_norm(PyObject*, PyObject* const* p, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  expect(n, 2);
  const Tensor x = arg_tensor(p[0]);
  if (!rows_ok(x)) return none();
  const double eps = arg_double(p[1]);
  if (wants_grad({&x})) return THPVariable_Wrap(L2NormNode::apply(x, eps));
  at::AutoDispatchBelowADInplaceOrView guard;
  return THPVariable_Wrap(L2NormNode::run(x.contiguous(), eps));
  END_HANDLE_TH_ERRORS
}

bool conv_weights_ok(const Tensor& w, const Tensor& b, int64_t D) {
  return w.defined() && w.is_cuda() && w.dim() >= 2 && w.size(0) == D && w.size(-1) >= 2 && w.size(-1) <= 4 &&
         w.numel() == D * w.size(-1) && w.is_floating_point() &&
         (!b.defined() || (b.is_cuda() && b.numel() == D && b.is_floating_point()));
}

// causal_conv1d(x [B,T,D], weight, bias | None, silu)
PyObject* py_conv(PyObject*, PyObject* const* p, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  expect(n, 4);
  const Tensor x = arg_tensor(p[0]), w = arg_tensor(p[1]), b = arg_tensor(p[2]);
  if (!x.defined() || !x.is_cuda() || x.dim() != 3 || x.numel() == 0 || x.size(2) % 8 != 0 ||
      !(is16(x) || x.scalar_type() == at::kFloat) || !conv_weights_ok(w, b, x.size(2)))
    return none();
  const int silu = arg_bool(p[3]);
  if (wants_grad({&x, &w, &b})) return THPVariable_Wrap(ConvNode::apply(x, w, maybe(b), silu));
  at::AutoDispatchBelowADInplaceOrView guard;
  return THPVariable_Wrap(ConvNode::run(x.contiguous(), f32(w), f32(b), silu));
  END_HANDLE_TH_ERRORS
}

// causal_conv1d_update(x [B,D], cache [B,D,W], weight, bias | None, silu): the cache is updated in place
// short_conv_step: the same for x [B,1,D], as the module gets it (a squeeze and an unsqueeze around a launch of 2.5 us cost the
// host 2 us)
template <bool STEP>
PyObject* py_conv_update(PyObject*, PyObject* const* p, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  expect(n, 5);
  const Tensor x = arg_tensor(p[0]), cache = arg_tensor(p[1]), w = arg_tensor(p[2]), b = arg_tensor(p[3]);
  if (!x.defined() || !cache.defined() || !x.is_cuda() || !cache.is_cuda() || x.dim() != (STEP ? 3 : 2) || x.numel() == 0 ||
      (STEP && x.size(1) != 1) || !(is16(x) || x.scalar_type() == at::kFloat) || !conv_weights_ok(w, b, x.size(-1)))
    return none();
  if (has_tangent({&x, &cache, &w, &b})) return none();   // (the wrapper refuses it)
  const int64_t B = x.size(0), D = x.size(-1), W = w.size(-1);
  if (cache.dim() != 3 || cache.size(0) != B || cache.size(1) != D || cache.size(2) != W || !cache.is_contiguous() ||
      cache.scalar_type() != x.scalar_type())
    return none();
  at::AutoDispatchBelowADInplaceOrView guard;
  const Tensor xc = x.contiguous(), b32 = f32(b);
  const Tensor wc = w.scalar_type() == x.scalar_type() ? w.contiguous() : f32(w);
  Tensor y = fresh_like(xc);
  check(fla_causal_conv1d_update(ptr(xc), ptr(cache), ptr(wc), fptr(b32), ptr(y), B, D, W, arg_bool(p[4]), dt(xc), dt(wc),
                                 stream_of(xc)),
        "fla_causal_conv1d_update");
  return THPVariable_Wrap(y);
  END_HANDLE_TH_ERRORS
}

// norm_swish_gate(x, gate, weight | None, bias | None, eps, is_rms_norm)
PyObject* py_norm_gate(PyObject*, PyObject* const* p, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  expect(n, 6);
  const Tensor x = arg_tensor(p[0]), o = arg_tensor(p[1]), w = arg_tensor(p[2]), b = arg_tensor(p[3]);
  if (!rows_ok(x) || !o.defined() || !o.is_cuda() || o.sizes() != x.sizes() || o.scalar_type() != x.scalar_type()) return none();
  for (const Tensor* t : {&w, &b})
    if (t->defined() && (!t->is_cuda() || t->numel() != x.size(-1) || !t->is_floating_point())) return none();
  const double eps = arg_double(p[4]);
  const bool rms = arg_bool(p[5]);
  if (wants_grad({&x, &o, &w, &b})) return THPVariable_Wrap(NormGateNode::apply(x, o, maybe(w), maybe(b), eps, rms));
  at::AutoDispatchBelowADInplaceOrView guard;
  Tensor mean, rstd;
  return THPVariable_Wrap(NormGateNode::run(x.contiguous(), o.contiguous(), f32(w), f32(b), eps, rms, &mean, &rstd));
  END_HANDLE_TH_ERRORS
}

#define ENTRY(name, fn) {name, (PyCFunction)(void (*)(void))fn, METH_FASTCALL, nullptr}
PyMethodDef kMethods[] = {
    ENTRY("plan", py_plan),
    ENTRY("chunk_gla", py_chunk_gla),
    ENTRY("chunk_simple_gla", py_chunk_simple_gla),
    ENTRY("chunk_gdr", py_chunk_gdr),
    ENTRY("recurrent_gla", py_recurrent_gla),
    ENTRY("recurrent_gdr", py_recurrent_gdr),
    ENTRY("l2_norm", py_l2_norm),
    ENTRY("causal_conv1d", py_conv),
    ENTRY("causal_conv1d_update", py_conv_update<false>),
    ENTRY("short_conv_step", py_conv_update<true>),
    ENTRY("norm_swish_gate", py_norm_gate),
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_fla_host", nullptr, -1, kMethods};

}  // namespace

PyMODINIT_FUNC PyInit__fla_host(void) {
  PyObject* m = PyModule_Create(&kModule);
  if (m) PyModule_AddIntConstant(m, "ABI_VERSION", FLA_ABI_VERSION);
  return m;
}
