// The whole MoE layer of GELU expert MLPs as ONE native autograd node: route ->
// scatter -> linear + GELU -> linear -> gather fused with the top-k combine
// (fmoe/layers.py:26-78,281-295 around fmoe/transformer.py:25-33 of the reference),
// optionally with the top-k gate in front of it (fmoe/gates/naive_gate.py:31-38), and
// the mirror image backwards.  Part of the extension (fmoe_cuda_ext.cpp).
//
// Why native: a small layer costs what the host needs to enqueue it (512 tokens,
// 128 -> 256, 4 experts: 377 us per step, of which the GPU works for about 170).  As a
// torch::autograd::Function neither direction enters Python between two launches, the
// backward needs no interpreter lock, the routing results share one allocation, and a
// forward without gradients saves nothing.
#pragma once
#include <torch/extension.h>

#include <ATen/core/grad_mode.h>

namespace {

// Byte offsets of the routing results inside their one allocation.
struct RouteLayout {
  int64_t inv, seg, bytes;   // pos sits at 0
  RouteLayout(int64_t slots, int64_t n_expert)
      : inv(slots * 8), seg(inv + slots * 4), bytes(seg + (n_expert + 1) * 4) {}
};

struct LayerSizes {
  int64_t t, d, h, e, k, n;   // tokens, features, hidden features, experts, top-k, slots
  int dtype;
};

LayerSizes layer_sizes(const Tensor& x, const Tensor& w1, const Tensor& b1, const Tensor& w2,
                       const Tensor& b2, int64_t top_k) {
  dev(w1, "w1", x.scalar_type());
  dev(w2, "w2", x.scalar_type());
  need(x.dim() == 2 && w1.dim() == 3 && w2.dim() == 3, "x must be 2-d and the weights 3-d");
  LayerSizes s{x.size(0), x.size(1), w1.size(1), w1.size(0), top_k, x.size(0) * top_k, dt(x, "x")};
  need(w1.size(2) == s.d && w2.size(0) == s.e && w2.size(1) == s.d && w2.size(2) == s.h,
       "the expert weights must be [E, hidden, in] and [E, in, hidden]");
  if (b1.defined()) {
    dev(b1, "b1", x.scalar_type());
    need(b1.numel() == s.e * s.h, "b1 must be [E, hidden]");
  }
  if (b2.defined()) {
    dev(b2, "b2", x.scalar_type());
    need(b2.numel() == s.e * s.d, "b2 must be [E, in]");
  }
  return s;
}

Tensor or_undefined(const OptTensor& t) { return t.has_value() ? *t : Tensor(); }
const void* raw(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }

// What the backward needs of a forward pass, and the output.
struct LayerPass {
  Tensor y, buf, pre, act, out, score, route;
};

LayerPass experts_forward(const LayerSizes& s, const Tensor& x, const Tensor& idx,
                          const Tensor& score, const Tensor& w1, const Tensor& b1,
                          const Tensor& w2, const Tensor& b2) {
  const auto opts = x.options();
  void* stream = stream_of(x);
  const RouteLayout at_(s.n, s.e);
  LayerPass p;
  p.score = score;
  p.route = at::empty({at_.bytes}, opts.dtype(at::kByte));
  char* meta = (char*)p.route.data_ptr();
  int64_t* pos = (int64_t*)meta;
  int32_t* inv = (int32_t*)(meta + at_.inv);
  int32_t* seg = (int32_t*)(meta + at_.seg);
  Tensor ws = workspace(s.n, s.e, x);
  check(fmoe_route(idx.data_ptr<int64_t>(), s.n, (int32_t)s.e, nullptr, seg, pos, inv, ws.data_ptr(),
                   ws.numel(), stream),
        "route");
  p.buf = at::empty({s.n, s.d}, opts);
  if (s.k >= 4)   // token order: a row is read once for its k copies
    check(fmoe_scatter_tokens(x.data_ptr(), inv, p.buf.data_ptr(), s.t, s.k, s.d, s.dtype, stream),
          "scatter_tokens");
  else
    check(fmoe_local_scatter(x.data_ptr(), pos, p.buf.data_ptr(), s.n, s.d, s.k, seg + s.e, s.dtype,
                             stream),
          "local_scatter");
  p.pre = at::empty({s.n, s.h}, opts);
  p.act = at::empty({s.n, s.h}, opts);
  check(fmoe_grouped_linear_fwd_act(p.buf.data_ptr(), w1.data_ptr(), raw(b1), seg, p.pre.data_ptr(),
                                    p.act.data_ptr(), s.n, s.d, s.h, s.e, s.dtype, stream),
        "grouped_linear_fwd_act");
  p.out = at::empty({s.n, s.d}, opts);
  check(fmoe_grouped_linear_fwd(p.act.data_ptr(), w2.data_ptr(), raw(b2), seg, p.out.data_ptr(), s.n,
                                s.h, s.d, s.e, s.dtype, stream),
        "grouped_linear_fwd");
  p.y = at::empty({s.t, s.d}, opts);
  check(fmoe_gather_combine_fwd(p.out.data_ptr(), inv, score.data_ptr(), p.y.data_ptr(), s.t, s.k,
                                s.d, s.dtype, stream),
        "gather_combine_fwd");
  return p;
}

struct LayerGrads {
  Tensor dx, dscore, dw1, db1, dw2, db2;
};
struct LayerNeeds {
  bool dx, w1, b1, w2, b2;
};

LayerGrads experts_backward(const LayerSizes& s, const LayerPass& p, const Tensor& dy,
                            const Tensor& w1, const Tensor& w2, const LayerNeeds& want) {
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
  const bool first = want.dx || want.w1 || want.b1;   // whether the first layer has a backward
  Tensor dpre;
  if (first) dpre = at::empty({s.n, s.h}, opts);
  if (want.w2) g.dw2 = at::empty_like(w2);
  if (want.b2) g.db2 = at::empty({s.e, s.d}, opts);
  void* dw2 = g.dw2.defined() ? g.dw2.data_ptr() : nullptr;
  void* db2 = g.db2.defined() ? g.db2.data_ptr() : nullptr;
  if (first)
    check(fmoe_grouped_linear_bwd_act(d_out.data_ptr(), p.act.data_ptr(), w2.data_ptr(), seg,
                                      p.pre.data_ptr(), dpre.data_ptr(), dw2, db2, s.n, s.h, s.d, s.e,
                                      s.dtype, stream),
          "grouped_linear_bwd_act");
  else if (dw2 || db2)
    check(fmoe_grouped_linear_bwd(d_out.data_ptr(), p.act.data_ptr(), w2.data_ptr(), seg, nullptr,
                                  dw2, db2, s.n, s.h, s.d, s.e, s.dtype, stream),
          "grouped_linear_bwd");
  if (!first) return g;
  Tensor dbuf;
  if (want.dx) dbuf = at::empty({s.n, s.d}, opts);
  if (want.w1) g.dw1 = at::empty_like(w1);
  if (want.b1) g.db1 = at::empty({s.e, s.h}, opts);
  check(fmoe_grouped_linear_bwd(dpre.data_ptr(), p.buf.data_ptr(), w1.data_ptr(), seg,
                                dbuf.defined() ? dbuf.data_ptr() : nullptr,
                                g.dw1.defined() ? g.dw1.data_ptr() : nullptr,
                                g.db1.defined() ? g.db1.data_ptr() : nullptr, s.n, s.d, s.h, s.e,
                                s.dtype, stream),
        "grouped_linear_bwd");
  if (want.dx) {
    g.dx = at::empty({s.t, s.d}, opts);
    check(fmoe_scatter_reduce(dbuf.data_ptr(), inv, g.dx.data_ptr(), s.t, s.k, s.d, s.dtype, stream),
          "scatter_reduce");
  }
  return g;
}

// The gate's top-k and softmax.  `zero_loss` (float[1]) is the gate's balance loss, which is
// zero for the plain top-k gate: the kernel writes it, so that it costs no launch of its own.
void gate_topk(const LayerSizes& s, const Tensor& logits, Tensor& idx, Tensor& score,
               Tensor& zero_loss) {
  idx = at::empty({s.t, s.k}, logits.options().dtype(at::kLong));
  score = at::empty({s.t, s.k}, logits.options());
  check(fmoe_naive_gate_fwd(logits.data_ptr(), s.t, (int32_t)s.e, (int32_t)s.k,
                            idx.data_ptr<int64_t>(), score.data_ptr(), zero_loss.data_ptr<float>(),
                            s.dtype, stream_of(logits)),
        "naive_gate_fwd");
}

// Which of a node's gradients the current backward wants: edges count the node's tensor
// arguments in order, an optional one only where it is given.
struct Edges {
  torch::autograd::AutogradContext* ctx;
  size_t next = 0;
  bool operator()(bool defined) { return defined && ctx->needs_input_grad(next++); }
};

using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// The layer behind any gate: (x, idx, score, w1, b1, w2, b2) -> y
struct ExpertLayerNode : public torch::autograd::Function<ExpertLayerNode> {
  static Tensor forward(AutogradContext* ctx, const Tensor& inp, const Tensor& idx,
                        const Tensor& score_in, const Tensor& w1, const OptTensor& b1_,
                        const Tensor& w2, const OptTensor& b2_, int64_t top_k) {
    const Tensor b1 = or_undefined(b1_), b2 = or_undefined(b2_);
    at::AutoDispatchBelowADInplaceOrView below;
    const Tensor x = inp.contiguous();
    c10::DeviceGuard guard(x.device());
    const LayerSizes s = layer_sizes(x, w1, b1, w2, b2, top_k);
    const Tensor score = score_in.reshape({s.t, s.k}).contiguous().to(x.scalar_type());
    LayerPass p = experts_forward(s, x, idx, score, w1, b1, w2, b2);
    ctx->saved_data["k"] = top_k;
    ctx->saved_data["shape"] = score_in.sizes();
    ctx->saved_data["dtype"] = (int64_t)score_in.scalar_type();
    ctx->saved_data["b1"] = b1.defined();
    ctx->saved_data["b2"] = b2.defined();
    ctx->save_for_backward({p.buf, p.pre, p.act, p.out, p.score, p.route, w1, w2});
    return p.y;
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list v = ctx->get_saved_variables();
    const Tensor &w1 = v[6], &w2 = v[7];
    Edges edge{ctx};
    const bool dx = edge(true);
    edge(true);   // idx
    const bool ds = edge(true), nw1 = edge(true), nb1 = edge(ctx->saved_data["b1"].toBool()),
               nw2 = edge(true), nb2 = edge(ctx->saved_data["b2"].toBool());
    const Tensor dy = grads[0].contiguous();
    c10::DeviceGuard guard(dy.device());
    LayerPass p{Tensor(), v[0], v[1], v[2], v[3], v[4], v[5]};
    const int64_t k = ctx->saved_data["k"].toInt();
    const LayerSizes s{dy.size(0), dy.size(1), w1.size(1), w1.size(0), k, dy.size(0) * k, dt(dy, "dy")};
    LayerGrads g = experts_backward(s, p, dy, w1, w2, {dx, nw1, nb1, nw2, nb2});
    Tensor dscore;
    if (ds)
      dscore = g.dscore.reshape(ctx->saved_data["shape"].toIntVector())
                   .to((at::ScalarType)ctx->saved_data["dtype"].toInt());
    return {g.dx, Tensor(), dscore, g.dw1, g.db1, g.dw2, g.db2, Tensor()};
  }
};

// The layer with the top-k gate in front: (x, wg, bg, w1, b1, w2, b2) -> y.  The gate's
// linear map stays the library call it is in torch.nn.Linear, in both directions, so the
// logits (and with them the routing) and every gradient have the bits of the gate module.
struct GatedLayerNode : public torch::autograd::Function<GatedLayerNode> {
  static Tensor forward(AutogradContext* ctx, const Tensor& inp, const Tensor& wg,
                        const OptTensor& bg_, const Tensor& w1, const OptTensor& b1_,
                        const Tensor& w2, const OptTensor& b2_, int64_t top_k, Tensor zero_loss) {
    const Tensor bg = or_undefined(bg_), b1 = or_undefined(b1_), b2 = or_undefined(b2_);
    at::AutoDispatchBelowADInplaceOrView below;
    const Tensor x = inp.contiguous();
    c10::DeviceGuard guard(x.device());
    const LayerSizes s = layer_sizes(x, w1, b1, w2, b2, top_k);
    const Tensor logits = at::linear(x, wg, bg);
    need(logits.size(1) == s.e, "the gate must have one output per expert");
    Tensor idx, score;
    gate_topk(s, logits, idx, score, zero_loss);
    LayerPass p = experts_forward(s, x, idx, score, w1, b1, w2, b2);
    ctx->saved_data["bg"] = bg.defined();
    ctx->saved_data["b1"] = b1.defined();
    ctx->saved_data["b2"] = b2.defined();
    ctx->save_for_backward({p.buf, p.pre, p.act, p.out, p.score, p.route, w1, w2, x, wg, idx});
    return p.y;
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list v = ctx->get_saved_variables();
    const Tensor &w1 = v[6], &w2 = v[7], &x = v[8], &wg = v[9], &idx = v[10];
    Edges edge{ctx};
    const bool dx = edge(true), nwg = edge(true), nbg = edge(ctx->saved_data["bg"].toBool()),
               nw1 = edge(true), nb1 = edge(ctx->saved_data["b1"].toBool()), nw2 = edge(true),
               nb2 = edge(ctx->saved_data["b2"].toBool());
    at::AutoDispatchBelowADInplaceOrView below;
    const Tensor dy = grads[0].contiguous();
    c10::DeviceGuard guard(dy.device());
    LayerPass p{Tensor(), v[0], v[1], v[2], v[3], v[4], v[5]};
    const int64_t k = idx.size(1);
    const LayerSizes s{dy.size(0), dy.size(1), w1.size(1), w1.size(0), k, dy.size(0) * k, dt(dy, "dy")};
    LayerGrads g = experts_backward(s, p, dy, w1, w2, {dx, nw1, nb1, nw2, nb2});
    Tensor dwg, dbg;
    if (dx || nwg || nbg) {
      Tensor dlogits = at::empty({s.t, s.e}, dy.options());
      check(fmoe_topk_softmax_bwd(g.dscore.data_ptr(), p.score.data_ptr(), idx.data_ptr<int64_t>(),
                                  dlogits.data_ptr(), s.t, (int32_t)s.e, (int32_t)s.k, s.dtype,
                                  stream_of(dy)),
            "topk_softmax_bwd");
      if (nwg) dwg = at::mm(dlogits.t(), x);
      if (nbg) dbg = dlogits.sum(0);
      if (dx) g.dx.add_(at::mm(dlogits, wg));
    }
    return {g.dx, dwg, dbg, g.dw1, g.db1, g.dw2, g.db2, Tensor(), Tensor()};
  }
};

bool wants_grad(std::initializer_list<const Tensor*> ts) {
  if (!at::GradMode::is_enabled()) return false;
  for (const Tensor* t : ts)
    if (t->defined() && t->requires_grad()) return true;
  return false;
}

Tensor expert_layer(const Tensor& inp, const Tensor& gate_idx, const Tensor& score, const Tensor& w1,
                    const OptTensor& b1_, const Tensor& w2, const OptTensor& b2_) {
  need(inp.is_cuda() && gate_idx.is_cuda(), "x and gate_idx must be CUDA tensors");
  need(gate_idx.scalar_type() == at::kLong, "gate_idx has the wrong dtype");
  const Tensor b1 = or_undefined(b1_), b2 = or_undefined(b2_);
  const int64_t k = gate_idx.dim() >= 2 ? gate_idx.size(-1) : 1;
  need(k >= 1 && k <= 64 && gate_idx.numel() == inp.size(0) * k && score.numel() == gate_idx.numel(),
       "gate_idx and score must have tokens * top_k entries");
  const Tensor idx = gate_idx.contiguous();
  if (wants_grad({&inp, &score, &w1, &b1, &w2, &b2}))
    return ExpertLayerNode::apply(inp, idx, score, w1, b1_, w2, b2_, k);
  at::AutoDispatchBelowADInplaceOrView below;
  const Tensor x = inp.contiguous();
  c10::DeviceGuard guard(x.device());
  const LayerSizes s = layer_sizes(x, w1, b1, w2, b2, k);
  return experts_forward(s, x, idx, score.reshape({s.t, s.k}).contiguous().to(x.scalar_type()), w1, b1,
                         w2, b2)
      .y;
}

// (y, balance loss): the loss is the zero of the plain top-k gate, a leaf that wants a
// gradient as the gate module makes it
std::tuple<Tensor, Tensor> gated_layer(const Tensor& inp, const Tensor& wg, const OptTensor& bg_,
                                       const Tensor& w1, const OptTensor& b1_, const Tensor& w2,
                                       const OptTensor& b2_, int64_t top_k) {
  need(inp.is_cuda() && inp.dim() == 2, "x must be a 2-d CUDA tensor");
  const Tensor bg = or_undefined(bg_), b1 = or_undefined(b1_), b2 = or_undefined(b2_);
  c10::DeviceGuard guard(inp.device());
  Tensor loss = at::empty({1}, inp.options().dtype(at::kFloat));
  Tensor y;
  if (wants_grad({&inp, &wg, &bg, &w1, &b1, &w2, &b2})) {
    y = GatedLayerNode::apply(inp, wg, bg_, w1, b1_, w2, b2_, top_k, loss);
  } else {
    at::AutoDispatchBelowADInplaceOrView below;
    const Tensor x = inp.contiguous();
    const LayerSizes s = layer_sizes(x, w1, b1, w2, b2, top_k);
    const Tensor logits = at::linear(x, wg, bg);
    need(logits.size(1) == s.e, "the gate must have one output per expert");
    Tensor idx, score;
    gate_topk(s, logits, idx, score, loss);
    y = experts_forward(s, x, idx, score, w1, b1, w2, b2).y;
  }
  loss.set_requires_grad(true);
  return {y, loss};
}

}  // namespace
