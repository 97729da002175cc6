// The whole MoE layer of two-layer expert MLPs as ONE native autograd node: route ->
// scatter -> linear + activation -> linear -> gather fused with the top-k combine
// (fmoe/layers.py:26-78,281-295 around fmoe/transformer.py:25-33 of the reference),
// optionally with the top-k gate in front of it (fmoe/gates/naive_gate.py:31-38), and
// the mirror image backwards.  Part of the extension (fmoe_cuda_ext.cpp).
//
// Why native: a small layer costs what the host needs to enqueue it (512 tokens,
// 128 -> 256, 4 experts: 377 us per step, of which the GPU worked for about 170).  As a
// torch::autograd::Function neither direction enters Python between two launches, the
// backward needs no interpreter lock, the routing results share one allocation, and a
// forward without gradients saves nothing and keeps no pre-activations.
//
// Expert parameters come as four [E, ...] arrays or as lists of E single-expert tensors
// (the reference's module per expert, fmoe/transformer.py:51-55), whose addresses the
// kernels read from device tables; the gradients of a list are views of one array.
#pragma once
#include <torch/extension.h>

#include <ATen/core/grad_mode.h>
#include <c10/core/InferenceMode.h>

namespace {

using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// Byte offsets of the routing results inside their one allocation.
struct RouteLayout {
  int64_t inv, seg, bytes;   // pos sits at 0
  RouteLayout(int64_t slots, int64_t n_expert)
      : inv(slots * 8), seg(inv + slots * 4), bytes(seg + (n_expert + 1) * 4) {}
};

// Device pointer tables of per-expert parameter lists (w1, b1, w2, b2), rebuilt only when a
// parameter's storage has moved (optimizers update in place, so normally never) or the call
// comes on another stream than the last one (nothing orders it behind the kernel that wrote
// the table).  A call under graph capture gets a table of its own: its writing is a node of
// the graph, so nobody outside may rely on it, and it has to live as long as the graph.
struct ParamTables {
  std::vector<const void*> key;
  Tensor table;   // int64 [4, E]; rows of absent biases stay zero
  void* stream = nullptr;

  Tensor get(const std::vector<Tensor>& params, int64_t n_expert, bool has_b1, bool has_b2) {
    std::vector<const void*> now(4 * n_expert, nullptr);
    const bool present[4] = {true, has_b1, true, has_b2};
    size_t at = 0;
    for (int row = 0; row < 4; ++row)
      if (present[row])
        for (int64_t e = 0; e < n_expert; ++e) now[row * n_expert + e] = params[at++].data_ptr();
    void* on = stream_of(params[0]);
    const bool capturing = is_capturing(on);
    if (capturing || !table.defined() || table.device() != params[0].device() || now != key ||
        on != stream) {
      for (const Tensor& t : params) {
        dev(t, "expert parameter", params[0].scalar_type());
        need(t.device() == params[0].device(), "expert parameters must share their device");
        need((uintptr_t)t.data_ptr() % 16 == 0, "expert parameters must be 16-byte aligned");
      }
      // (a new tensor: kernels of an earlier call may still be reading the old one; an ordinary
      // one also under inference mode, as a later training call saves it for its backward)
      c10::InferenceMode ordinary(false);
      Tensor fresh = torch::empty({4, n_expert}, params[0].options().dtype(at::kLong));
      check(fmoe_pointer_table(now.data(), (int64_t)now.size(), (const void**)fresh.data_ptr(), on),
            "pointer_table");
      if (capturing) return fresh;
      table = fresh;
      key = std::move(now);
      stream = on;
    }
    return table;
  }
};

struct LayerConfig {
  int64_t top_k = 0, act = FMOE_ACT_GELU, n_expert = 0;
  bool gated = false, has_bg = false, has_b1 = false, has_b2 = false, list = false;
  Tensor table;       // list: pointers of w1, b1, w2, b2
  Tensor zero_loss;   // gated: the plain gate's balance loss, written by its kernel

  std::vector<int64_t> ints() const {
    return {top_k, act, n_expert, gated, has_bg, has_b1, has_b2, list};
  }
  static LayerConfig from(const std::vector<int64_t>& v) {
    LayerConfig c;
    c.top_k = v[0]; c.act = v[1]; c.n_expert = v[2];
    c.gated = v[3]; c.has_bg = v[4]; c.has_b1 = v[5]; c.has_b2 = v[6]; c.list = v[7];
    return c;
  }
  int64_t per_kind() const { return list ? n_expert : 1; }   // tensors per parameter kind
};

// One linear layer's parameters as the C ABI takes them.
struct LinearParams {
  const void* w = nullptr;
  const void* const* w_ptrs = nullptr;
  const void* b = nullptr;
  const void* const* b_ptrs = nullptr;
};
struct ExpertParams {
  LinearParams first, second;
};

struct LayerSizes {
  int64_t t, d, h, e, k, n;   // tokens, features, hidden features, experts, top-k, slots
  int dtype;
};

// `params`: w1, b1 (if any), w2, b2 (if any), each one tensor or n_expert of them.
LayerSizes layer_sizes(const LayerConfig& c, const Tensor& x, at::TensorList params) {
  const int64_t per = c.per_kind();
  need(x.dim() == 2, "x must be 2-d");
  need((int64_t)params.size() == per * (2 + c.has_b1 + c.has_b2), "wrong number of expert parameters");
  const Tensor& w1 = params[0];
  const Tensor& w2 = params[per * (1 + c.has_b1)];
  need(w1.dim() == 3 && w2.dim() == 3, "the expert weights must be 3-d");
  LayerSizes s{x.size(0), x.size(1), w1.size(1), c.n_expert, c.top_k, x.size(0) * c.top_k, dt(x, "x")};
  const int64_t lead = c.list ? 1 : s.e;
  size_t at = 0;
  auto kind = [&](const char* name, std::initializer_list<int64_t> shape) {
    for (int64_t i = 0; i < per; ++i) {
      const Tensor& t = params[at++];
      dev(t, name, x.scalar_type());
      need(t.sizes() == at::IntArrayRef(shape), std::string(name) + " has the wrong shape");
    }
  };
  kind("w1", {lead, s.h, s.d});
  if (c.has_b1) kind("b1", {lead, s.h});
  kind("w2", {lead, s.d, s.h});
  if (c.has_b2) kind("b2", {lead, s.d});
  return s;
}

ExpertParams expert_params(const LayerConfig& c, at::TensorList params) {
  ExpertParams p;
  if (c.list) {
    const void* const* base = (const void* const*)c.table.data_ptr();
    p.first.w_ptrs = base;
    if (c.has_b1) p.first.b_ptrs = base + c.n_expert;
    p.second.w_ptrs = base + 2 * c.n_expert;
    if (c.has_b2) p.second.b_ptrs = base + 3 * c.n_expert;
    return p;
  }
  size_t at = 0;
  p.first.w = params[at++].data_ptr();
  if (c.has_b1) p.first.b = params[at++].data_ptr();
  p.second.w = params[at++].data_ptr();
  if (c.has_b2) p.second.b = params[at++].data_ptr();
  return p;
}

// What the backward needs of a forward pass, and the output.
struct LayerPass {
  Tensor y, buf, pre, act, out, score, route;
};

// The routing results of `idx` in one allocation (RouteLayout).  `ws`: scratch of
// fmoe_route_workspace_bytes(), written by one launch and read by the next two.
Tensor route_slots(const LayerSizes& s, const Tensor& idx, const Tensor& ws) {
  const RouteLayout at_(s.n, s.e);
  Tensor route = at::empty({at_.bytes}, idx.options().dtype(at::kByte));
  char* meta = (char*)route.data_ptr();
  check(fmoe_route(idx.data_ptr<int64_t>(), s.n, (int32_t)s.e, nullptr, (int32_t*)(meta + at_.seg),
                   (int64_t*)meta, (int32_t*)(meta + at_.inv), ws.data_ptr(), ws.numel(),
                   stream_of(idx)),
        "route");
  return route;
}

LayerPass experts_forward(const LayerConfig& c, const LayerSizes& s, const ExpertParams& w,
                          const Tensor& x, const Tensor& idx, const Tensor& score, bool train) {
  const auto opts = x.options();
  void* stream = stream_of(x);
  const RouteLayout at_(s.n, s.e);
  LayerPass p;
  p.score = score;
  p.route = route_slots(s, idx, workspace(s.n, s.e, idx));
  const char* meta = (const char*)p.route.data_ptr();
  const int64_t* pos = (const int64_t*)meta;
  const int32_t* inv = (const int32_t*)(meta + at_.inv);
  const int32_t* seg = (const int32_t*)(meta + at_.seg);
  p.buf = at::empty({s.n, s.d}, opts);
  if (s.k >= 4)   // token order: a row is read once for its k copies
    check(fmoe_scatter_tokens(x.data_ptr(), inv, p.buf.data_ptr(), s.t, s.k, s.d, s.dtype, stream),
          "scatter_tokens");
  else
    check(fmoe_local_scatter(x.data_ptr(), pos, p.buf.data_ptr(), s.n, s.d, s.k, seg + s.e, s.dtype,
                             stream),
          "local_scatter");
  // GELU's backward needs the pre-activations, ReLU's the activations, inference neither
  const bool keep_pre = train && c.act == FMOE_ACT_GELU;
  if (keep_pre) p.pre = at::empty({s.n, s.h}, opts);
  p.act = at::empty({s.n, s.h}, opts);
  check(fmoe_expert_linear_fwd(p.buf.data_ptr(), w.first.w, w.first.w_ptrs, w.first.b,
                               w.first.b_ptrs, seg, keep_pre ? p.pre.data_ptr() : nullptr,
                               p.act.data_ptr(), (int)c.act, s.n, s.d, s.h, s.e, s.dtype, stream),
        "expert_linear_fwd");
  p.out = at::empty({s.n, s.d}, opts);
  check(fmoe_expert_linear_fwd(p.act.data_ptr(), w.second.w, w.second.w_ptrs, w.second.b,
                               w.second.b_ptrs, seg, p.out.data_ptr(), nullptr, FMOE_ACT_NONE, s.n,
                               s.h, s.d, s.e, s.dtype, stream),
        "expert_linear_fwd");
  p.y = at::empty({s.t, s.d}, opts);
  check(fmoe_gather_combine_fwd(p.out.data_ptr(), inv, score.data_ptr(), p.y.data_ptr(), s.t, s.k,
                                s.d, s.dtype, stream),
        "gather_combine_fwd");
  return p;
}

// A gate that ran inside the node: its operands in the backward.
struct GateGrad {
  Tensor x, wg, idx;
};
struct LayerGrads {
  Tensor dx, dslot, dscore, dw1, db1, dw2, db2;
};
struct LayerNeeds {
  bool dx, w1, b1, w2, b2;
};

void* out_ptr(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }

// dlogits at the top-k slots, in the accumulation type
Tensor gate_slot_grads(const LayerSizes& s, const Tensor& dscore, const Tensor& score) {
  Tensor dslot = at::empty({s.t, s.k}, score.options().dtype(
      score.scalar_type() == at::kDouble ? at::kDouble : at::kFloat));
  check(fmoe_gate_slot_grad(dscore.data_ptr(), score.data_ptr(), dslot.data_ptr(), s.t, s.k, s.dtype,
                            stream_of(score)),
        "gate_slot_grad");
  return dslot;
}

// Gradients of the gate's weight and bias from the routing results.
std::tuple<Tensor, Tensor> gate_linear_grads(const LayerSizes& s, const Tensor& x,
                                             const Tensor& route, const Tensor& dslot, bool weight,
                                             bool bias) {
  Tensor dwg, dbg;
  if (weight) dwg = at::empty({s.e, s.d}, x.options());
  if (bias) dbg = at::empty({s.e}, x.options());
  const RouteLayout at_(s.n, s.e);
  const char* meta = (const char*)route.data_ptr();
  const int64_t bytes = fmoe_gate_linear_grad_workspace_bytes(x.data_ptr(), s.t, s.k, s.d,
                                                              (int32_t)s.e, s.dtype);
  check(bytes < 0 ? (int)bytes : 0, "gate_linear_grad");
  // (of this call alone: two launches, between which another thread may use the stream)
  Tensor ws = at::empty({bytes}, x.options().dtype(at::kByte));
  check(fmoe_gate_linear_grad(x.data_ptr(), (const int64_t*)meta, (const int32_t*)(meta + at_.seg),
                              dslot.data_ptr(), weight ? dwg.data_ptr() : nullptr,
                              bias ? dbg.data_ptr() : nullptr, s.t, s.k, s.d, (int32_t)s.e,
                              ws.data_ptr(), bytes, s.dtype, stream_of(x)),
        "gate_linear_grad");
  return {dwg, dbg};
}

LayerGrads experts_backward(const LayerConfig& c, const LayerSizes& s, const ExpertParams& w,
                            const LayerPass& p, const Tensor& dy, const LayerNeeds& want,
                            const GateGrad* gate) {
  const auto opts = dy.options();
  void* stream = stream_of(dy);
  const RouteLayout at_(s.n, s.e);
  char* meta = (char*)p.route.data_ptr();
  const int32_t* inv = (const int32_t*)(meta + at_.inv);
  const int32_t* seg = (const int32_t*)(meta + at_.seg);
  LayerGrads g;
  Tensor d_out = at::empty({s.n, s.d}, opts);
  g.dscore = at::empty({s.t, s.k}, opts);
  check(fmoe_gather_combine_bwd(dy.data_ptr(), p.out.data_ptr(), inv, p.score.data_ptr(),
                                d_out.data_ptr(), g.dscore.data_ptr(), s.t, s.k, s.d, s.dtype, stream),
        "gather_combine_bwd");
  if (gate) g.dslot = gate_slot_grads(s, g.dscore, p.score);
  const bool first = want.dx || want.w1 || want.b1;   // whether the first layer has a backward
  Tensor dpre;
  if (first) dpre = at::empty({s.n, s.h}, opts);
  if (want.w2) g.dw2 = at::empty({s.e, s.d, s.h}, opts);
  if (want.b2) g.db2 = at::empty({s.e, s.d}, opts);
  if (first || want.w2 || want.b2)
    check(fmoe_expert_linear_bwd(d_out.data_ptr(), p.act.data_ptr(), w.second.w, w.second.w_ptrs, seg,
                                 p.pre.defined() ? p.pre.data_ptr() : p.act.data_ptr(),
                                 first ? (int)c.act : FMOE_ACT_NONE, out_ptr(dpre), out_ptr(g.dw2),
                                 out_ptr(g.db2), s.n, s.h, s.d, s.e, s.dtype, stream),
          "expert_linear_bwd");
  if (!first) return g;
  Tensor dbuf;
  if (want.dx) dbuf = at::empty({s.n, s.d}, opts);
  if (want.w1) g.dw1 = at::empty({s.e, s.h, s.d}, opts);
  if (want.b1) g.db1 = at::empty({s.e, s.h}, opts);
  check(fmoe_expert_linear_bwd(dpre.data_ptr(), p.buf.data_ptr(), w.first.w, w.first.w_ptrs, seg,
                               nullptr, FMOE_ACT_NONE, out_ptr(dbuf), out_ptr(g.dw1),
                               out_ptr(g.db1), s.n, s.d, s.h, s.e, s.dtype, stream),
        "expert_linear_bwd");
  if (want.dx) {
    g.dx = at::empty({s.t, s.d}, opts);
    if (gate)
      check(fmoe_scatter_reduce_gate(dbuf.data_ptr(), inv, gate->idx.data_ptr<int64_t>(),
                                     g.dslot.data_ptr(), gate->wg.data_ptr(), g.dx.data_ptr(), s.t,
                                     s.k, s.d, (int32_t)s.e, s.dtype, stream),
            "scatter_reduce_gate");
    else
      check(fmoe_scatter_reduce(dbuf.data_ptr(), inv, g.dx.data_ptr(), s.t, s.k, s.d, s.dtype, stream),
            "scatter_reduce");
  }
  return g;
}

// The gate's top-k and softmax.  `zero_loss` (float[1]) is the gate's balance loss, which is
// zero for the plain top-k gate: the kernel writes it, so that it costs no launch of its own.
void gate_topk(const LayerSizes& s, const Tensor& logits, Tensor& idx, Tensor& score,
               const Tensor& zero_loss) {
  need(logits.size(1) == s.e, "the gate must have one output per expert");
  idx = at::empty({s.t, s.k}, logits.options().dtype(at::kLong));
  score = at::empty({s.t, s.k}, logits.options());
  check(fmoe_naive_gate_fwd(logits.data_ptr(), s.t, (int32_t)s.e, (int32_t)s.k,
                            idx.data_ptr<int64_t>(), score.data_ptr(), zero_loss.data_ptr<float>(),
                            s.dtype, stream_of(logits)),
        "naive_gate_fwd");
}

// Forward of the layer.  vars: x, then (wg, bg if any) of a gate to be run here, or (idx,
// score) of a gate that has been run; then the expert parameters.  The gate's linear map
// stays the library call it is in torch.nn.Linear, so the logits (and with them the routing)
// have the bits of the gate module; its gradients come from the top-k slots alone
// (gate_grad.hip).
LayerPass layer_forward(const LayerConfig& c, at::TensorList vars, bool train, Tensor* idx_out) {
  // (a view of the caller's scores is taken where views keep the version of their base: the
  // backward needs the values, so a change in place before it is an error)
  Tensor score = c.gated ? Tensor() : vars[2].reshape({vars[0].size(0), c.top_k});
  at::AutoDispatchBelowADInplaceOrView below;
  const Tensor x = vars[0].contiguous();
  c10::DeviceGuard guard(x.device());
  const at::TensorList params = vars.slice(c.gated ? 2 + c.has_bg : 3);
  const LayerSizes s = layer_sizes(c, x, params);
  Tensor idx;
  if (c.gated) {
    gate_topk(s, at::linear(x, vars[1], c.has_bg ? OptTensor(vars[2]) : OptTensor()), idx, score,
              c.zero_loss);
  } else {
    idx = vars[1];
    score = score.contiguous().to(x.scalar_type());
  }
  LayerPass p = experts_forward(c, s, expert_params(c, params), x, idx, score, train);
  if (idx_out) *idx_out = idx;
  return p;
}

// What a node saves of the plain gate's linear map: as in torch.nn.Linear the input only for the
// parameters' gradients and the weight only for the input's, so that what no gradient needs may
// be written in place before the backward.  (The parameters themselves are kept as well, without
// the check of saved variables: for gradients of higher order.)
void save_gate(AutogradContext* ctx, variable_list& saved, const Tensor& x, const Tensor& wg,
               const Tensor& bg) {
  saved.push_back(wg.requires_grad() || (bg.defined() && bg.requires_grad()) ? x : Tensor());
  saved.push_back(x.requires_grad() ? wg : Tensor());
  ctx->saved_data["gate"] = std::vector<Tensor>{wg, bg};
}
struct GateOperands {
  Tensor x, wg, bg;   // x: undefined where no parameter wants a gradient
};
GateOperands saved_gate(AutogradContext* ctx, const Tensor& x, const Tensor& wg) {
  const std::vector<Tensor> kept = ctx->saved_data["gate"].toTensorVector();
  return {x, wg.defined() ? wg : kept[0], kept[1]};
}

// The gradients of the plain gate's linear map (x, weight, bias) from dscore as torch operations,
// for gradients that will themselves be differentiated.  The softmax over the chosen logits is
// taken at the scores of the forward pass, whatever has become of the bias since; it is a
// constant where the gate is.
variable_list differentiable_gate_grads(const GateOperands& gate, const Tensor& idx,
                                        const Tensor& score, const Tensor& dscore, bool dx,
                                        bool nwg, bool nbg) {
  const auto acc = score.scalar_type() == at::kDouble ? at::kDouble : at::kFloat;
  Tensor p = score.detach().to(acc);
  if (gate.x.defined()) {
    const Tensor chosen =
        at::linear(gate.x, gate.wg, gate.bg.defined() ? OptTensor(gate.bg) : OptTensor())
            .gather(1, idx).to(acc);
    p = at::softmax(chosen + (p.log() - chosen.detach()), -1);
  }
  const Tensor ds = dscore.to(acc);
  const Tensor dchosen = (p * (ds - (ds * p).sum(-1, true))).to(gate.wg.scalar_type());
  const Tensor dlogits =
      at::zeros({idx.size(0), gate.wg.size(0)}, gate.wg.options()).scatter_add(1, idx, dchosen);
  return {dx ? at::mm(dlogits, gate.wg) : Tensor(), nwg ? at::mm(dlogits.t(), gate.x) : Tensor(),
          nbg ? dlogits.sum(0) : Tensor()};
}

struct LayerNode : public torch::autograd::Function<LayerNode> {
  static Tensor forward(AutogradContext* ctx, at::TensorList vars, const LayerConfig& c) {
    Tensor idx;
    LayerPass p = layer_forward(c, vars, true, &idx);
    variable_list saved{p.buf, p.pre, p.act, p.out, p.score, p.route};
    if (c.gated) {
      saved.push_back(idx);
      save_gate(ctx, saved, vars[0], vars[1], c.has_bg ? vars[2] : Tensor());
    } else {
      ctx->saved_data["shape"] = vars[2].sizes();
      ctx->saved_data["dtype"] = (int64_t)vars[2].scalar_type();
    }
    if (c.list) saved.push_back(c.table);
    // the weights (not the biases) are operands of the backward
    const int64_t first = c.gated ? 2 + c.has_bg : 3, per = c.per_kind();
    for (int64_t i = 0; i < per; ++i) saved.push_back(vars[first + i]);
    for (int64_t i = 0; i < per; ++i) saved.push_back(vars[first + per * (1 + c.has_b1) + i]);
    ctx->save_for_backward(std::move(saved));
    ctx->saved_data["c"] = c.ints();
    return p.y;
  }

  // Under create_graph the gate's share is made of torch operations, as where the gate is a
  // module; the experts' kernels have no derivative, so their share is a constant then.
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    LayerConfig c = LayerConfig::from(ctx->saved_data["c"].toIntVector());
    const variable_list v = ctx->get_saved_variables();
    const int64_t per = c.per_kind();
    size_t at = 6 + (c.gated ? 3 : 0);
    if (c.list) c.table = v[at++];
    const at::TensorList weights = at::TensorList(v).slice(at);
    const bool twice = at::GradMode::is_enabled();
    std::optional<at::AutoDispatchBelowADInplaceOrView> below(std::in_place);
    const Tensor dy = grads[0].contiguous();
    c10::DeviceGuard guard(dy.device());
    const LayerPass p{Tensor(), v[0], v[1], v[2], v[3], v[4], v[5]};
    const LayerSizes s{dy.size(0), dy.size(1), weights[0].size(1), c.n_expert, c.top_k,
                       dy.size(0) * c.top_k, dt(dy, "dy")};
    ExpertParams w;
    if (c.list) {
      w = expert_params(c, {});
    } else {
      w.first.w = weights[0].data_ptr();
      w.second.w = weights[1].data_ptr();
    }
    // which gradients are wanted: edges in the order of the forward's tensors
    size_t edge = 0;
    auto any = [&](bool present, int64_t count) {
      bool r = false;
      if (present)
        for (int64_t i = 0; i < count; ++i) r = ctx->needs_input_grad(edge++) || r;
      return r;
    };
    const bool dx = any(true, 1);
    bool nwg = false, nbg = false, ds = false;
    if (c.gated) {
      nwg = any(true, 1);
      nbg = any(c.has_bg, 1);
    } else {
      any(true, 1);   // idx
      ds = any(true, 1);
    }
    const size_t first_param = edge;
    LayerNeeds want{dx, false, false, false, false};
    want.w1 = any(true, per);
    want.b1 = any(c.has_b1, per);
    want.w2 = any(true, per);
    want.b2 = any(c.has_b2, per);
    const bool gate_grads = c.gated && !twice && (dx || nwg || nbg);
    GateGrad gate;
    if (gate_grads) {
      const GateOperands op = saved_gate(ctx, v[7], v[8]);
      gate = {op.x, op.wg.contiguous(), v[6]};
    }
    LayerGrads g = experts_backward(c, s, w, p, dy, want, gate_grads ? &gate : nullptr);
    variable_list out;
    if (c.gated) {
      Tensor dwg, dbg;
      if (gate_grads && (nwg || nbg))
        std::tie(dwg, dbg) = gate_linear_grads(s, gate.x.contiguous(), p.route, g.dslot, nwg, nbg);
      if (twice) {
        below.reset();
        const variable_list own = differentiable_gate_grads(saved_gate(ctx, v[7], v[8]), v[6],
                                                            p.score, g.dscore, dx, nwg, nbg);
        if (dx) g.dx = g.dx + own[0];
        dwg = own[1];
        dbg = own[2];
      }
      out = {g.dx, dwg};
      if (c.has_bg) out.push_back(dbg);
    } else {
      Tensor dscore;
      if (ds)
        dscore = g.dscore.reshape(ctx->saved_data["shape"].toIntVector())
                     .to((at::ScalarType)ctx->saved_data["dtype"].toInt());
      out = {g.dx, Tensor(), dscore};
    }
    auto give = [&](bool present, const Tensor& t) {
      if (!present) return;
      for (int64_t i = 0; i < per; ++i) {
        const bool need_it = t.defined() && ctx->needs_input_grad(out.size());
        out.push_back(!need_it ? Tensor() : c.list ? t.narrow(0, i, 1) : t);
      }
    };
    need(out.size() == first_param, "layer node: gradients out of order");
    give(true, g.dw1);
    give(c.has_b1, g.db1);
    give(true, g.dw2);
    give(c.has_b2, g.db2);
    out.push_back(Tensor());   // the configuration
    return out;
  }
};

bool wants_grad(at::TensorList ts) {
  if (!at::GradMode::is_enabled()) return false;
  for (const Tensor& t : ts)
    if (t.requires_grad()) return true;
  return false;
}

Tensor run_layer(const LayerConfig& c, at::TensorList vars) {
  if (wants_grad(vars)) return LayerNode::apply(vars, c);
  return layer_forward(c, vars, false, nullptr).y;
}

// The expert parameters' share of a call: `params` holds w1, b1, w2, b2 in that order, the
// absent biases left out; one tensor each, or n_expert with `tables`.
void set_experts(LayerConfig& c, const std::vector<Tensor>& params, int64_t n_expert, bool has_b1,
                 bool has_b2, ParamTables* tables) {
  c.n_expert = n_expert;
  c.has_b1 = has_b1;
  c.has_b2 = has_b2;
  c.list = tables != nullptr;
  need((int64_t)params.size() == c.per_kind() * (2 + has_b1 + has_b2),
       "wrong number of expert parameters");
  if (c.list) {
    c10::DeviceGuard guard(params[0].device());
    c.table = tables->get(params, n_expert, has_b1, has_b2);
  }
}

Tensor expert_layer(const Tensor& inp, const Tensor& gate_idx, const Tensor& score,
                    std::vector<Tensor> params, int64_t n_expert, bool has_b1, bool has_b2,
                    int64_t act, ParamTables* tables) {
  need(inp.is_cuda() && gate_idx.is_cuda(), "x and gate_idx must be CUDA tensors");
  need(gate_idx.scalar_type() == at::kLong, "gate_idx has the wrong dtype");
  LayerConfig c;
  c.top_k = gate_idx.dim() >= 2 ? gate_idx.size(-1) : 1;
  c.act = act;
  need(c.top_k >= 1 && c.top_k <= 64 && gate_idx.numel() == inp.size(0) * c.top_k &&
           score.numel() == gate_idx.numel(),
       "gate_idx and score must have tokens * top_k entries");
  set_experts(c, params, n_expert, has_b1, has_b2, tables);
  variable_list vars{inp, gate_idx.contiguous(), score};
  vars.insert(vars.end(), params.begin(), params.end());
  return run_layer(c, vars);
}

// (y, balance loss): the loss is the zero of the plain top-k gate, a leaf that wants a
// gradient as the gate module makes it
std::tuple<Tensor, Tensor> gated_layer(const Tensor& inp, const Tensor& wg, const OptTensor& bg,
                                       std::vector<Tensor> params, int64_t n_expert, bool has_b1,
                                       bool has_b2, int64_t act, int64_t top_k,
                                       ParamTables* tables) {
  need(inp.is_cuda() && inp.dim() == 2, "x must be a 2-d CUDA tensor");
  c10::DeviceGuard guard(inp.device());
  LayerConfig c;
  c.top_k = top_k;
  c.act = act;
  c.gated = true;
  c.has_bg = bg.has_value() && bg->defined();
  c.zero_loss = at::empty({1}, inp.options().dtype(at::kFloat));
  set_experts(c, params, n_expert, has_b1, has_b2, tables);
  variable_list vars{inp, wg};
  if (c.has_bg) vars.push_back(*bg);
  vars.insert(vars.end(), params.begin(), params.end());
  Tensor y = run_layer(c, vars);
  c.zero_loss.set_requires_grad(true);
  return {y, c.zero_loss};
}

// ---------------------------------------------------------------- gates
// fmoe/gates/utils.py:9-26 at one worker in one call: (slots per expert that survive, gate with
// -1 where dropped)
std::tuple<Tensor, Tensor> limit_gate(const Tensor& gate_in, int64_t n_expert, int64_t capacity) {
  const Tensor gate = gate_in.contiguous();
  dev(gate, "gate", at::kLong);
  need(capacity == (int32_t)capacity, "capacity exceeds the range of int32");
  c10::DeviceGuard guard(gate.device());
  Tensor count = at::empty({n_expert}, gate.options()), out = at::empty_like(gate);
  Tensor ws = workspace(gate.numel(), n_expert, gate);
  check(fmoe_limit_gate(gate.data_ptr<int64_t>(), gate.numel(), (int32_t)n_expert, capacity,
                        out.data_ptr<int64_t>(), count.data_ptr<int64_t>(), ws.data_ptr(), ws.numel(),
                        stream_of(gate)),
        "limit_gate");
  return {count, out};
}

// The plain gate as a node of its own (a layer that cannot fold it in: masks, experts of the
// user's), with the kernels and so the bits of the folded one: (idx, score)
struct PlainGateNode : public torch::autograd::Function<PlainGateNode> {
  static variable_list forward(AutogradContext* ctx, const Tensor& x_in, const Tensor& wg,
                               const OptTensor& bg, int64_t top_k) {
    at::AutoDispatchBelowADInplaceOrView below;
    const Tensor x = x_in.contiguous();
    const LayerSizes s{x.size(0), x.size(1), 0, wg.size(0), top_k, x.size(0) * top_k, dt(x, "x")};
    const bool has_bg = bg.has_value() && bg->defined();
    const Tensor logits = at::linear(x, wg, has_bg ? bg : OptTensor());
    Tensor idx = at::empty({s.t, s.k}, logits.options().dtype(at::kLong));
    Tensor score = at::empty({s.t, s.k}, logits.options());
    check(fmoe_topk_softmax_fwd(logits.data_ptr(), s.t, (int32_t)s.e, (int32_t)s.k,
                                idx.data_ptr<int64_t>(), score.data_ptr(), s.dtype, stream_of(x)),
          "topk_softmax_fwd");
    variable_list saved{idx, score};
    save_gate(ctx, saved, x_in, wg, has_bg ? *bg : Tensor());
    ctx->save_for_backward(std::move(saved));
    ctx->mark_non_differentiable({idx});
    ctx->set_materialize_grads(false);
    return {idx, score};
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list v = ctx->get_saved_variables();
    const Tensor &idx = v[0], &score = v[1];
    const GateOperands gate = saved_gate(ctx, v[2], v[3]);
    const bool dx = ctx->needs_input_grad(0), nwg = ctx->needs_input_grad(1),
               nbg = gate.bg.defined() && ctx->needs_input_grad(2);
    if (!grads[1].defined()) return {Tensor(), Tensor(), Tensor(), Tensor()};
    c10::DeviceGuard guard(score.device());
    if (at::GradMode::is_enabled()) {   // gradients that will themselves be differentiated
      variable_list out = differentiable_gate_grads(gate, idx, score, grads[1], dx, nwg, nbg);
      out.push_back(Tensor());
      return out;
    }
    const int64_t d = gate.wg.size(1);
    const LayerSizes s{idx.size(0), d, 0, gate.wg.size(0), idx.size(1), idx.numel(), dt(score, "score")};
    const Tensor dslot = gate_slot_grads(s, grads[1].contiguous(), score);
    Tensor gx, dwg, dbg;
    if (dx) {
      const Tensor w = gate.wg.contiguous();
      gx = at::empty({s.t, s.d}, score.options());
      check(fmoe_scatter_reduce_gate(nullptr, nullptr, idx.data_ptr<int64_t>(), dslot.data_ptr(),
                                     w.data_ptr(), gx.data_ptr(), s.t, s.k, s.d, (int32_t)s.e,
                                     s.dtype, stream_of(score)),
            "scatter_reduce_gate");
    }
    if (nwg || nbg) {
      // (scratch of this call alone: a backward runs without the interpreter lock, so another
      // thread may use the stream's shared buffer between the launches)
      const int64_t bytes = fmoe_route_workspace_bytes(s.n, (int32_t)s.e);
      need(bytes >= 0, "workspace: bad sizes");
      const Tensor ws = at::empty({std::max<int64_t>(bytes, 1)}, idx.options().dtype(at::kByte));
      std::tie(dwg, dbg) =
          gate_linear_grads(s, gate.x.contiguous(), route_slots(s, idx, ws), dslot, nwg, nbg);
    }
    return {gx, dwg, dbg, Tensor()};
  }
};

std::tuple<Tensor, Tensor> plain_gate(const Tensor& x, const Tensor& wg, const OptTensor& bg,
                                      int64_t top_k) {
  need(x.is_cuda() && x.dim() == 2 && wg.dim() == 2, "x must be a 2-d CUDA tensor");
  c10::DeviceGuard guard(x.device());
  variable_list r = PlainGateNode::apply(x, wg, bg, top_k);
  return {r[0], r[1]};
}

// A gate with a balance loss behind its linear map: logits -> (idx limited to the capacity,
// score, loss)
struct BalanceGateNode : public torch::autograd::Function<BalanceGateNode> {
  static variable_list forward(AutogradContext* ctx, const Tensor& logits_in, int64_t kind,
                               int64_t capacity) {
    at::AutoDispatchBelowADInplaceOrView below;
    const Tensor logits = logits_in.contiguous();
    const int64_t t = logits.size(0), e = logits.size(1), k = kind == FMOE_GATE_GSHARD ? 2 : 1;
    Tensor idx = at::empty({t, k}, logits.options().dtype(at::kLong));
    Tensor score = at::empty({t, k}, logits.options());
    const auto f32 = logits.options().dtype(at::kFloat);
    Tensor loss = at::empty({}, f32), coef = at::empty({e}, f32);
    Tensor ws = workspace_of(fmoe_balance_gate_workspace_bytes((int32_t)e), logits);
    check(fmoe_balance_gate_fwd(logits.data_ptr(), t, (int32_t)e, (int)kind, capacity,
                                idx.data_ptr<int64_t>(), score.data_ptr(), loss.data_ptr<float>(),
                                coef.data_ptr<float>(), ws.data_ptr(), ws.numel(),
                                dt(logits, "logits"), stream_of(logits)),
          "balance_gate_fwd");
    Tensor kept = std::get<1>(limit_gate(idx, e, capacity));
    // (Switch's gradient does not need the score, which its caller may then write in place)
    ctx->save_for_backward({logits, coef, kind == FMOE_GATE_GSHARD ? score : Tensor(), idx});
    ctx->saved_data["kind"] = kind;
    ctx->mark_non_differentiable({kept});
    ctx->set_materialize_grads(false);
    return {kept, score, loss};
  }
  // The backward as torch operations, for gradients of higher order and for batches of
  // gradients (torch's vmap over a backward): the loss reaches softmax(logits) with one
  // constant per expert, the scores are the softmax of the chosen logits (GShard) or the
  // chosen values of softmax(logits) (Switch).
  static Tensor differentiable(int64_t kind, const Tensor& logits, const Tensor& coef,
                               const Tensor& idx, const Tensor& dscore, const Tensor& dloss) {
    const Tensor x = logits.to(at::kFloat), p = at::softmax(x, -1);
    Tensor dp = at::zeros_like(p), dx = at::zeros_like(p);
    if (dloss.defined()) dp = dp + coef * dloss;
    if (dscore.defined()) {
      const Tensor ds = dscore.to(at::kFloat);
      if (kind == FMOE_GATE_GSHARD) {
        const Tensor s = at::softmax(x.gather(1, idx), -1);
        dx = dx.scatter_add(1, idx, s * (ds - (ds * s).sum(-1, true)));
      } else {
        dp = dp.scatter_add(1, idx, ds);
      }
    }
    return (dx + p * (dp - (dp * p).sum(-1, true))).to(logits.scalar_type());
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list v = ctx->get_saved_variables();
    const Tensor &logits = v[0], &coef = v[1], &score = v[2], &idx = v[3];
    const Tensor dscore = grads[1].defined() ? grads[1].contiguous() : Tensor();
    const Tensor dloss = grads[2];
    if (!dscore.defined() && !dloss.defined()) return {Tensor(), Tensor(), Tensor()};
    c10::DeviceGuard guard(logits.device());
    // (a batch of gradients has no memory of its own)
    const bool batched = (dscore.defined() && !dscore.has_storage()) ||
                         (dloss.defined() && !dloss.has_storage());
    if (at::GradMode::is_enabled() || batched)
      return {differentiable(ctx->saved_data["kind"].toInt(), logits, coef, idx, dscore, dloss),
              Tensor(), Tensor()};
    Tensor dlogits = at::empty_like(logits);
    check(fmoe_balance_gate_bwd(logits.data_ptr(), coef.data_ptr<float>(),
                                dloss.defined() ? dloss.data_ptr<float>() : nullptr,
                                dscore.defined() ? dscore.data_ptr() : nullptr, out_ptr(score),
                                idx.data_ptr<int64_t>(), dlogits.data_ptr(), logits.size(0),
                                (int32_t)logits.size(1), (int)ctx->saved_data["kind"].toInt(),
                                dt(logits, "logits"), stream_of(logits)),
          "balance_gate_bwd");
    return {dlogits, Tensor(), Tensor()};
  }
};

std::tuple<Tensor, Tensor, Tensor> balance_gate(const Tensor& logits, int64_t kind,
                                                int64_t capacity) {
  need(logits.is_cuda() && logits.dim() == 2, "logits must be a 2-d CUDA tensor");
  c10::DeviceGuard guard(logits.device());
  variable_list r = BalanceGateNode::apply(logits, kind, capacity);
  return {r[0], r[1], r[2]};
}

}  // namespace
