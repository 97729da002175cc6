"""The layer as one native autograd node against the chain of Python nodes it replaces
(which still runs while a per-op event hook is set): the same kernels in the same order,
so the same bits, with and without gradients, for every subset of gradients asked for; only
the gate's own gradients are summed by kernels of their own."""
import copy
import io
import threading

import pytest
import torch

from helpers import DTYPES

pytestmark = pytest.mark.gpu


def _layer(dtype, top_k, gate=None, bias=True, d=64, h=96, activation=None):
    from fastmoe_amd import FMoETransformerMLP, NaiveGate

    torch.manual_seed(3)
    moe = FMoETransformerMLP(6, d, h, top_k=top_k, gate=gate or NaiveGate,
                             activation=activation or torch.nn.GELU())
    if not bias:
        moe.experts.htoh4.bias = moe.experts.h4toh.bias = None
    else:
        torch.nn.init.normal_(moe.experts.htoh4.bias)
        torch.nn.init.normal_(moe.experts.h4toh.bias)
    return moe.to(dtype).cuda()


def _run(moe, x, dy, frozen, watched):
    from fastmoe_amd import fmoe_cuda

    for n, p in moe.named_parameters():
        p.grad = None
        p.requires_grad_(n not in frozen)
    a = x.clone().requires_grad_("x" not in frozen)
    fmoe_cuda.profile_hook = (lambda *args: None) if watched else None
    try:
        out = moe(a)
        out.backward(dy)
        with torch.no_grad():
            assert torch.equal(moe(a), out)
    finally:
        fmoe_cuda.profile_hook = None
    loss = moe.gate.get_loss()
    assert loss.shape == (1,) and loss.item() == 0 and loss.requires_grad and loss.is_leaf
    return [out, a.grad] + [p.grad for p in moe.parameters()]


FROZEN = [(), ("x",), ("gate.gate.weight", "gate.gate.bias", "x"),
          ("experts.htoh4.weight", "experts.h4toh.bias"),
          ("experts.htoh4.weight", "experts.htoh4.bias", "gate.gate.weight", "gate.gate.bias", "x"),
          ("experts.h4toh.weight", "experts.h4toh.bias")]


@pytest.mark.parametrize("dt", ["bf16", "f32"])
@pytest.mark.parametrize("top_k,bias", [(1, True), (2, False), (4, True)])
@pytest.mark.parametrize("frozen", FROZEN, ids=lambda f: "-".join(f) or "none")
def test_native_node_matches_the_chain(dt, top_k, bias, frozen):
    moe = _layer(DTYPES[dt], top_k, bias=bias)
    x = torch.randn(130, 64, device="cuda").to(DTYPES[dt])
    dy = torch.randn(130, 64, device="cuda").to(DTYPES[dt])
    got, want = (_run(moe, x, dy, frozen, w) for w in (False, True))
    names = ["y", "x"] + [n for n, _ in moe.named_parameters()]
    for name, g, w in zip(names, got, want):
        assert (g is None) == (w is None)
        if g is None or not (name == "x" or name.startswith("gate.")):
            assert g is None or torch.equal(g, w)
        else:
            # the chain rounds the logits' gradient to the storage type, which this node keeps
            # in the accumulation type; both round the gate's share of dx, the experts' share
            # and their sum (half an eps each): 2 eps of the gradient's size; f32 sums in
            # another order differ by less than the 130 terms times 2^-24, i.e. 65 eps
            eps = torch.finfo(g.dtype).eps
            bound = (2 if dt == "bf16" else 65) * eps
            assert (g - w).double().norm() <= bound * w.double().norm(), name


def test_gate_hooks_and_no_tokens():
    """A watched gate runs as the module it is; an empty batch is a valid one."""
    moe = _layer(torch.bfloat16, 2)
    x = torch.randn(50, 64, device="cuda", dtype=torch.bfloat16)
    plain, seen = moe(x), []
    hook = moe.gate.register_forward_hook(lambda m, i, o: seen.append(o[0]))
    assert torch.equal(moe(x), plain) and len(seen) == 1
    hook.remove()
    empty = torch.zeros(0, 64, device="cuda", dtype=torch.bfloat16, requires_grad=True)
    out = moe(empty)
    out.sum().backward()
    assert out.shape == (0, 64) and empty.grad.shape == (0, 64)
    assert not any(p.grad.any().item() for p in moe.experts.parameters())


@pytest.mark.parametrize("dt", ["bf16", "f16", "f32"])
@pytest.mark.parametrize("act", [torch.nn.GELU, torch.nn.ReLU])
@pytest.mark.parametrize("gate,top_k", [("NaiveGate", 2), ("GShardGate", 2), ("SwitchGate", 1)])
@pytest.mark.parametrize("fused", [True, False])
def test_gates_activations_and_layouts_match_the_chain(dt, act, gate, top_k, fused):
    """Every gate, activation and expert layout through the native nodes against the Python
    chain with torch's own gate arithmetic.  The routing and the survivors of the capacity are
    the same; values differ by the roundings of the storage type in the gate's loss, whose
    gradient the chain rounds once per torch operation (a few units in the last place of a
    sum over the tokens: 4 roundings of eps each on values of the sum's scale)."""
    import fastmoe_amd
    from fastmoe_amd import FMoETransformerMLP, fmoe_cuda

    dtype = DTYPES[dt]
    torch.manual_seed(11)
    moe = FMoETransformerMLP(8, 64, 96, top_k=top_k, gate=getattr(fastmoe_amd, gate),
                             activation=act(), fused=fused).to(dtype).cuda()
    moe.gate.capacity = (0.9, 0.9)          # some slots are dropped
    moe.gate.random_routing, moe.gate.switch_eps = False, 0.0
    x = torch.randn(500, 64, device="cuda").to(dtype)
    dy = torch.randn(500, 64, device="cuda").to(dtype)
    got = []
    for watched in (False, True):
        fmoe_cuda.profile_hook = (lambda *a: None) if watched else None
        try:
            for p in moe.parameters():
                p.grad = None
            a = x.clone().requires_grad_(True)
            out = moe(a)
            loss = moe.gate.get_loss()
            torch.autograd.backward([out, loss], [dy, None if gate != "NaiveGate" else
                                                  torch.zeros_like(loss)])
            with torch.no_grad():
                idx = moe.gate(x)[0]
        finally:
            fmoe_cuda.profile_hook = None
        got.append([idx, out, loss, a.grad] + [p.grad for p in moe.parameters()])
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])
    assert (got[0][0] == -1).any() or gate == "NaiveGate"
    tol = 4 * torch.finfo(dtype).eps
    for g, w in zip(got[0][2:], got[1][2:]):
        assert (g - w).double().norm() <= tol * w.double().norm()


@pytest.mark.parametrize("n,e,cap", [(0, 4, 2), (0, 513, 2), (100, 4, 0), (4096, 7, 300), (4097, 512, 8),
                                     (9000, 513, 5), (70000, 16, 4000)])
def test_limit_gate_matches_count_limit_prune(n, e, cap):
    from fastmoe_amd import fmoe_cuda
    from fastmoe_amd.gates import limit_by_capacity

    g = torch.Generator().manual_seed(n)
    gate = torch.randint(-1, e, (n, 1), generator=g).cuda()
    new = limit_by_capacity(gate, e, 1, cap)
    fmoe_cuda.profile_hook = lambda *a: None
    try:
        want = limit_by_capacity(gate, e, 1, cap)
    finally:
        fmoe_cuda.profile_hook = None
    for a, b in zip(new, want):
        assert a.dtype == b.dtype and torch.equal(a, b)


@pytest.mark.parametrize("cap", [2 ** 31, -2 ** 31 - 1])
def test_capacity_is_a_number_of_32_bits(cap):
    """Any other is refused: by the helper and, where it comes from the rate, by the gates."""
    from fastmoe_amd import GShardGate, SwitchGate
    from fastmoe_amd.gates import limit_by_capacity

    with pytest.raises(RuntimeError):
        limit_by_capacity(torch.zeros(8, 1, dtype=torch.int64, device="cuda"), 4, 1, cap)
    x = torch.randn(8, 16, device="cuda")
    for gate in (GShardGate(16, 4, 1), SwitchGate(16, 4, 1)):
        gate.capacity = (cap, cap)
        with pytest.raises(RuntimeError):
            gate.cuda()(x)


@pytest.mark.parametrize("dt", ["bf16", "f32"])
@pytest.mark.parametrize("kind,k", [("GATE_GSHARD", 2), ("GATE_SWITCH", 1)])
@pytest.mark.parametrize("t,e", [(1, 2), (33, 16), (500, 17), (300, 64), (700, 65), (9000, 129),
                                 (300, 512)])
def test_balance_gate_against_float64(dt, kind, k, t, e):
    """Indices, scores, loss and the gradient of both outputs against torch in float64 on the
    same rounded logits.  Ties go to the lower expert.  Bounds: one rounding of the storage type
    on the outputs; the loss is a sum of T * E float32 terms (its error stays below
    1e-5 of it)."""
    from fastmoe_amd import fmoe_cuda

    m, dtype = fmoe_cuda.native(), DTYPES[dt]
    g = torch.Generator().manual_seed(t + e)
    logits = torch.randn(t, e, generator=g).to(dtype).cuda()
    cap = max(1, int(1.1 * t * k / e))
    a = logits.clone().requires_grad_(True)
    idx, score, loss = m.balance_gate(a, getattr(m, kind), cap)
    ds = torch.randn(t, k, generator=g).to(dtype).cuda()
    torch.autograd.backward([score, loss], [ds, torch.tensor(3.0, device="cuda")])
    ref = logits.double().requires_grad_(True)
    p = torch.softmax(ref, -1)
    order = torch.argsort(logits.double(), dim=-1, descending=True, stable=True)[:, :k]
    chosen = torch.gather(ref, 1, order)
    want = torch.softmax(chosen, -1) if k == 2 else torch.gather(p, 1, order)
    count = torch.bincount(order[:, 0], minlength=e).double()
    if k == 2:
        want_loss = (count / t * p.mean(0)).mean() * e ** 2
    else:
        kept = count.clamp(max=cap)
        want_loss = (kept / kept.sum() * p.sum(0) / kept.sum()).sum() * e
    torch.autograd.backward([want, want_loss],
                            [ds.double(), torch.tensor(3.0, device="cuda", dtype=torch.float64)])
    live = m.limit_gate(order.contiguous(), e, cap)[1]
    assert torch.equal(idx, live)
    eps = torch.finfo(dtype).eps
    assert (score.double() - want).abs().max() <= eps
    assert abs(loss.item() - want_loss.item()) <= 1e-5 * abs(want_loss.item())
    assert (a.grad.double() - ref.grad).abs().max() <= 4 * eps * ref.grad.abs().max()


def _replace_forward(module, seen):
    """`module` wrapped in place: its calls are counted and their first result doubled."""
    inner = module.forward

    def forward(*args):
        seen.append(module)
        out = inner(*args)
        return (out[0], out[1] * 2) if isinstance(out, tuple) else out * 2

    module.forward = forward


@pytest.mark.parametrize("fused", [True, False])
@pytest.mark.parametrize("act", [torch.nn.GELU, torch.nn.ReLU])
@pytest.mark.parametrize("where", ["gate", "gate.gate", "experts", "htoh4", "h4toh", "activation"])
@pytest.mark.parametrize("how", ["instance", "class"])
def test_modules_with_another_forward_are_called(fused, act, where, how):
    """A `forward` set on an instance or by a subclass is what runs, wherever in the layer: twice
    the logits, hidden values or scores there change the output, and the module is counted."""
    from fastmoe_amd import FMoETransformerMLP

    torch.manual_seed(4)
    moe = FMoETransformerMLP(4, 32, 48, top_k=2, activation=act(), fused=fused).cuda()
    x = torch.randn(60, 32, device="cuda", requires_grad=True)
    want, seen = moe(x), []
    if where.startswith("gate"):
        modules = [moe.get_submodule(where)]
    else:
        experts = [moe.experts] if fused else list(moe.experts)
        modules = experts if where == "experts" else [getattr(e, where) for e in experts]
    for m in set(modules):
        if how == "instance":
            _replace_forward(m, seen)
        else:
            def forward(self, *args, _parent=type(m)):
                seen.append(self)
                out = _parent.forward(self, *args)
                return (out[0], out[1] * 2) if isinstance(out, tuple) else out * 2

            m.__class__ = type("Other", (type(m),), {"forward": forward})
    got = moe(x)
    got.sum().backward()
    assert set(seen) == set(modules) and not torch.allclose(got, want, rtol=1e-2)
    assert x.grad is not None and x.grad.any()


@pytest.mark.parametrize("fused", [True, False])
def test_hooks_on_all_modules_see_relu_experts(fused):
    """A hook on every module (as profilers and loggers set) sees the gate's linear map, the
    activation and, where it holds all experts, the expert module called; the output stays."""
    from fastmoe_amd import FMoETransformerMLP

    torch.manual_seed(4)
    moe = FMoETransformerMLP(4, 32, 48, top_k=2, activation=torch.nn.ReLU(), fused=fused).cuda()
    x, seen = torch.randn(60, 32, device="cuda"), []
    want = moe(x)
    hook = torch.nn.modules.module.register_module_forward_hook(lambda m, *_: seen.append(m))
    try:
        got = moe(x)
    finally:
        hook.remove()
    called = [moe, moe.gate, moe.gate.gate] + ([moe.experts, moe.experts.activation] if fused
                                               else [moe.experts[0].activation])
    assert all(any(m is s for s in seen) for m in called)
    assert (got - want).norm() <= 65 * torch.finfo(x.dtype).eps * want.norm()


def _gate(d, e, k, dtype=torch.float32):
    from fastmoe_amd import NaiveGate

    torch.manual_seed(2)
    return NaiveGate(d, e, 1, k).to(dtype).cuda()


def test_gate_backward_leaves_the_shared_routing_scratch_alone():
    """The backward of the gate module runs without the interpreter lock, so what it routes
    with has to be its own: no scratch of its size stays behind for the stream (512 experts and
    a million slots: a megabyte; the first, small call sets up the stream's other buffers)."""
    gate, stream = _gate(8, 512, 8), torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        for tokens in (64, 1 << 17):
            torch.cuda.synchronize()
            before = torch.cuda.memory_allocated()
            x = torch.randn(tokens, 8, device="cuda", requires_grad=True)
            score = gate(x)[1]
            grads = torch.autograd.grad(score, [gate.gate.weight, gate.gate.bias],
                                        torch.ones_like(score))
            torch.cuda.synchronize()
            assert all(g.shape[0] == 512 for g in grads)
            del x, score, grads
    assert torch.cuda.memory_allocated() - before < 1 << 16


def test_two_threads_on_one_stream():
    """One thread differentiates a gate while another routes on the same stream, both with
    slots enough for three launches each: everybody gets what they get alone, bit for bit."""
    gate, moe = _gate(64, 16, 2), _layer(torch.float32, 2)
    x, y = torch.randn(6000, 64, device="cuda"), torch.randn(9000, 64, device="cuda")

    def differentiate():
        a = x.clone().requires_grad_(True)
        score = gate(a)[1]
        return torch.autograd.grad((score * score).sum(), [a, gate.gate.weight, gate.gate.bias])

    def forward():
        with torch.no_grad():
            return (moe(y),)

    want, failed = {f: f() for f in (differentiate, forward)}, []

    def loop(f):
        for _ in range(40):
            if not all(torch.equal(g, w) for g, w in zip(f(), want[f])):
                failed.append(f.__name__)

    threads = [threading.Thread(target=loop, args=(f,)) for f in want]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed


@pytest.mark.parametrize("alone", [True, False])
def test_gate_bias_may_change_before_the_backward(alone):
    """No gradient depends on the value of the gate's bias, so updating it in place (as balancing
    without a loss does) between the forward and the backward pass is allowed."""
    gate, moe = _gate(64, 6, 2), _layer(torch.float32, 2)
    if not alone:
        gate = moe.gate
    x, got = torch.randn(70, 64, device="cuda"), []
    for change in (False, True):
        a = x.clone().requires_grad_(True)
        out = gate(a)[1] if alone else moe(a)
        if change:
            with torch.no_grad():
                gate.gate.bias.add_(0.5 * torch.randn_like(gate.gate.bias))
        got.append(torch.autograd.grad((out * out).sum(), [a, gate.gate.weight, gate.gate.bias]))
    assert all(torch.equal(p, q) for p, q in zip(*got))


@pytest.mark.parametrize("alone", [True, False])
@pytest.mark.parametrize("what", ["weight", "x"])
def test_what_no_gradient_needs_may_change_before_the_backward(alone, what):
    """As in torch.nn.Linear: the gate's weight where x wants no gradient, x where the gate is
    frozen.  Where they are needed, the change is an error."""
    gate, moe = _gate(64, 6, 2), _layer(torch.float32, 2)
    if not alone:
        gate = moe.gate
    x, got = torch.randn(70, 64, device="cuda"), []
    gate.requires_grad_(what == "weight")
    for change in (False, True):
        a = (x.clone().requires_grad_(True) * 1) if what == "x" else x.clone()
        out = gate(a)[1] if alone else moe(a)
        wanted = a if what == "x" else gate.gate.weight
        if change:
            with torch.no_grad():
                (a if what == "x" else gate.gate.weight).add_(1.0)
        got.append(torch.autograd.grad((out * out).sum(), wanted)[0])
    assert torch.equal(*got)
    gate.requires_grad_(True)
    a = x.clone().requires_grad_(True) * 1
    out = gate(a)[1] if alone else moe(a)
    with torch.no_grad():
        (a if what == "x" else gate.gate.weight).add_(1.0)
    with pytest.raises(RuntimeError, match="inplace"):
        (out * out).sum().backward()


def _list_layer():
    from fastmoe_amd import FMoETransformerMLP

    torch.manual_seed(5)
    return FMoETransformerMLP(4, 64, 96, top_k=2, fused=False).cuda()


@pytest.mark.parametrize("fused", [True, False])
@pytest.mark.parametrize("shape", [(70, 2), (140,)])
def test_scores_may_not_change_before_the_backward(fused, shape):
    """The gradients need the scores that the forward used, so changing a user's gate's scores in
    place between the two is an error, whatever shape they come in."""
    from fastmoe_amd import FMoETransformerMLP

    moe = FMoETransformerMLP(6, 64, 96, top_k=2, fused=fused).cuda()
    idx = torch.randint(0, 6, (70, 2), device="cuda")
    score = torch.rand(shape, device="cuda", requires_grad=True) * 1
    moe.gate.forward = lambda x: (idx, score)
    out = moe(torch.randn(70, 64, device="cuda"))
    with torch.no_grad():
        score.mul_(2)
    with pytest.raises(RuntimeError, match="inplace"):
        out.sum().backward()


def test_list_layer_copies_and_pickles_after_a_call():
    """A layer that has run is still one that can be copied and saved; its copy reads its own
    parameters."""
    moe = _list_layer()
    x = torch.randn(50, 64, device="cuda")
    want = moe(x).detach()
    twin = copy.deepcopy(moe)
    file = io.BytesIO()
    torch.save(moe, file)
    file.seek(0)
    for other in (twin, torch.load(file, weights_only=False)):
        assert torch.equal(other(x), want)
        with torch.no_grad():
            for p in other.experts.parameters():
                p.zero_()
        assert not other(x).any() and torch.equal(moe(x), want)


@pytest.mark.parametrize("dt", ["bf16", "f32"])
def test_switch_score_may_change_before_the_backward(dt):
    """Its gradient depends on the logits alone, so a caller may scale the score in place: the
    gradients are those of a scaled copy."""
    from fastmoe_amd import SwitchGate

    torch.manual_seed(5)
    gate = SwitchGate(16, 4, 1).to(DTYPES[dt]).cuda().eval()
    x = torch.randn(40, 16, device="cuda", dtype=DTYPES[dt])

    def grads(in_place):
        _, score = gate(x)
        score = score.mul_(2) if in_place else score * 2
        return torch.autograd.grad(score.float().square().sum() + gate.get_loss(),
                                   list(gate.parameters()))

    for a, b in zip(grads(True), grads(False)):
        assert torch.equal(a, b)


@pytest.mark.parametrize("name", ["htoh4.weight", "htoh4.bias", "h4toh.weight", "h4toh.bias"])
def test_relu_experts_with_parameters_in_another_layout(name):
    """A parameter whose memory is not in [E, out, in] order: the same values and gradients, up
    to the order in which 70 tokens are summed (fewer than 65 units)."""
    moe = _layer(torch.float32, 2, activation=torch.nn.ReLU())
    x, got = torch.randn(70, 64, device="cuda"), []
    p = moe.experts.get_parameter(name)
    for other in (False, True):
        if other:
            p.data = p.data.transpose(0, -1).contiguous().transpose(0, -1)
            assert not p.is_contiguous()
        for q in moe.parameters():
            q.grad = None
        out = moe(x)
        out.sum().backward()
        got.append([out.detach()] + [q.grad for q in moe.parameters()])
    for a, b in zip(*got):
        assert (a - b).norm() <= 65 * torch.finfo(a.dtype).eps * a.norm()


@pytest.mark.parametrize("fused", [True, False])
@pytest.mark.parametrize("act", [torch.nn.GELU, torch.nn.ReLU])
def test_experts_whose_output_has_another_width(fused, act):
    """An FMoE layer of experts 32 -> 48 -> 40 against the sum over the experts in float64."""
    from fastmoe_amd import FMoE
    from fastmoe_amd.linear import FMoELinear
    from fastmoe_amd.transformer import _Expert

    def expert(n):
        e = _Expert(n, 32, 48, activation)
        e.h4toh = FMoELinear(n, 48, 40)
        return e

    torch.manual_seed(6)
    activation = act()
    moe = FMoE(4, 32, top_k=2, expert=None if fused else lambda d: expert(1))
    if fused:
        moe.experts = expert(4)
    moe.cuda()
    x = torch.randn(60, 32, device="cuda", requires_grad=True)
    out = moe(x)
    out.sum().backward()
    idx, score = moe.gate(x)
    want = torch.zeros(60, 40, dtype=torch.float64, device="cuda")
    for e in range(4):
        m = moe.experts[e]
        w = [t.double()[0] for t in (m.htoh4.weight, m.htoh4.bias, m.h4toh.weight, m.h4toh.bias)]
        y = torch.nn.functional.linear(activation(torch.nn.functional.linear(
            x.double(), w[0], w[1])), w[2], w[3])
        want = want + y * (score.double() * (idx == e)).sum(1, keepdim=True)
    # (sums of 32 and 48 products in float32)
    assert out.shape == (60, 40) and (out - want).norm() <= 1e-6 * want.norm()
    assert x.grad.any() and all(p.grad is not None for p in moe.parameters())


@pytest.mark.parametrize("fused", [True, False])
@pytest.mark.parametrize("outputs", [5, 9])
def test_gate_with_more_or_fewer_outputs_than_experts(fused, outputs):
    """A gate may choose among more numbers than there are experts (a choice of none: the slot is
    dropped) or never choose some of them."""
    from fastmoe_amd import FMoETransformerMLP, fmoe_cuda

    torch.manual_seed(6)
    moe = FMoETransformerMLP(6, 64, 96, top_k=2, fused=fused).cuda()
    moe.gate.gate = torch.nn.Linear(64, outputs).cuda()
    x, got = torch.randn(130, 64, device="cuda"), []
    for watched in (False, True):
        fmoe_cuda.profile_hook = (lambda *a: None) if watched else None
        try:
            for p in moe.parameters():
                p.grad = None
            a = x.clone().requires_grad_(True)
            out = moe(a)
            out.sum().backward()
        finally:
            fmoe_cuda.profile_hook = None
        got.append([out, a.grad] + [p.grad for p in moe.parameters()])
    assert torch.equal(got[0][0], got[1][0]) and moe.gate(x)[0].max() == outputs - 1
    # (the gate's gradients are sums of 130 terms in another order: 65 units)
    for g, w in zip(got[0][1:], got[1][1:]):
        assert (g - w).norm() <= 65 * torch.finfo(g.dtype).eps * w.norm()


@pytest.mark.parametrize("container", [list, tuple])
@pytest.mark.parametrize("act", [torch.nn.GELU, torch.nn.ReLU])
def test_experts_in_a_plain_container(container, act):
    """Experts kept in a Python list or tuple instead of a ModuleList: the same layer."""
    from fastmoe_amd import FMoETransformerMLP

    torch.manual_seed(5)
    moe = FMoETransformerMLP(4, 64, 96, top_k=2, fused=False, activation=act()).cuda()
    x, got = torch.randn(50, 64, device="cuda"), []
    experts = moe.experts
    for holder in (experts, container(experts)):
        del moe.experts
        moe.experts = holder
        for p in experts.parameters():
            p.grad = None
        out = moe(x)
        out.sum().backward()
        got.append([out.detach()] + [p.grad for p in experts.parameters()])
    assert all(torch.equal(a, b) for a, b in zip(*got))


@pytest.mark.parametrize("watched", [True, False])
def test_list_layer_trains_after_inference_mode(watched):
    """The table of the experts' addresses made by a call under inference mode serves a training
    call as well, through the native node and through the chain."""
    from fastmoe_amd import fmoe_cuda

    moe, x = _list_layer(), torch.randn(50, 64, device="cuda")
    fmoe_cuda.profile_hook = (lambda *a: None) if watched else None
    try:
        with torch.inference_mode():
            want = moe(x)
        out = moe(x)
        out.sum().backward()
    finally:
        fmoe_cuda.profile_hook = None
    assert torch.equal(out, want) and all(p.grad.any() for p in moe.experts.parameters())


def test_list_layer_first_called_under_capture_or_on_another_stream():
    """The table of the experts' addresses is written by the stream that reads it: a graph
    that has not run yet leaves nothing behind for eager calls, nor do calls on one stream
    for those on another."""
    moe, x = _list_layer(), torch.randn(50, 64, device="cuda")
    with torch.no_grad():
        want = copy.deepcopy(moe)(x)
        warm = torch.cuda.Stream()
        warm.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(warm):
            copy.deepcopy(moe)(x)
        torch.cuda.current_stream().wait_stream(warm)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = moe(x)
        assert torch.equal(moe(x), want)          # before the first replay
        other = torch.cuda.Stream()
        other.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(other):
            assert torch.equal(moe(x), want)
        torch.cuda.synchronize()
        for _ in range(3):
            out.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, want) and torch.equal(moe(x), want)


@pytest.mark.parametrize("gate,top_k", [("GShardGate", 2), ("SwitchGate", 1)])
def test_balance_loss_differentiates_twice_and_forwards(gate, top_k):
    """The gradient of a balance loss has a gradient of its own, and the Switch gate takes
    forward-mode tangents, as the torch operations that the gates consist of do.  Against the
    gate run operation by operation in float32: sums of 200 x 8 terms, 1e-5 of their size."""
    import fastmoe_amd
    from fastmoe_amd import fmoe_cuda
    from torch.autograd import forward_ad

    torch.manual_seed(9)
    layer = getattr(fastmoe_amd, gate)(32, 8, 1, topk=top_k).cuda()
    layer.random_routing, layer.switch_eps = False, 0.0
    x = torch.randn(200, 32, device="cuda")
    got = []
    for watched in (False, True):
        fmoe_cuda.profile_hook = (lambda *a: None) if watched else None
        try:
            a = x.clone().requires_grad_(True)
            _, score = layer(a)
            loss = layer.get_loss() + (score[:, 0] ** 2).sum() * (gate == "SwitchGate")
            (da,) = torch.autograd.grad(loss, a, create_graph=True)
            (dda,) = torch.autograd.grad((da ** 2).sum(), a)
        finally:
            fmoe_cuda.profile_hook = None
        got.append((da.detach(), dda))
    for g, w in zip(*got):
        assert w.any() and (g - w).norm() <= 1e-5 * w.norm()
    if gate == "SwitchGate":
        with forward_ad.dual_level():
            layer(forward_ad.make_dual(x, torch.ones_like(x)))
            assert forward_ad.unpack_dual(layer.get_loss()).tangent is not None


@pytest.mark.parametrize("bias", [True, False])
@pytest.mark.parametrize("alone", [True, False])
def test_plain_gate_differentiates_twice(alone, bias):
    """The gradient of the plain gate has a gradient of its own, as a module and folded into the
    layer (where the gradient of the scores and the experts' share count as constants).  Against
    torch in float64: sums of up to 300 float32 terms, off by at most 300 units of 2^-24 each
    time, a handful in a row: 1e-4 of the norm."""
    from fastmoe_amd import FMoETransformerMLP

    torch.manual_seed(12)
    moe = FMoETransformerMLP(6, 64, 96, top_k=2, gate_bias=bias).cuda()
    lin = moe.gate.gate
    x = torch.randn(300, 64, device="cuda", requires_grad=True)
    c = torch.randn(300, 2 if alone else 64, device="cuda")
    idx, score = moe.gate(x)
    params = [p for p in (lin.weight, lin.bias) if p is not None]
    ref = [t.detach().double().requires_grad_(True) for t in (x, *params)]
    want = torch.softmax(torch.nn.functional.linear(*ref).gather(1, idx), -1)
    if alone:
        dscore, share = c.double(), 0.0
        out = score
    else:
        out = moe(x)
        rows = [moe.experts[e].h4toh(moe.experts.activation(moe.experts[e].htoh4(x, torch.tensor([300]))),
                                     torch.tensor([300])) for e in range(6)]
        y = torch.stack(rows, 1).gather(1, idx[..., None].expand(-1, -1, 64))     # [T, k, d]
        dscore = (y.detach().double() * c.double()[:, None]).sum(-1)
        share = torch.autograd.grad((y * score.detach()[..., None]).sum(1), x, c)[0].double()
    once = torch.autograd.grad(out, [x, *params], c, create_graph=True)
    g = torch.autograd.grad(want, ref, dscore, create_graph=True)
    g = [g[0] + share, *g[1:]]
    for a, b in zip(once, g):
        assert (a - b).norm() <= 1e-4 * b.norm()
    twice = torch.autograd.grad(sum((t ** 2).sum() for t in once), [x, *params])
    want2 = torch.autograd.grad(sum((t ** 2).sum() for t in g), ref)
    for a, b in zip(twice, want2):
        assert b.any() and (a - b).norm() <= 1e-4 * b.norm()
    plain = torch.autograd.grad(moe(x) if not alone else moe.gate(x)[1], [x, *params], c)
    for a, b in zip(once, plain):
        assert (a - b).norm() <= 1e-6 * b.norm()


@pytest.mark.parametrize("dt", ["bf16", "f16"])
def test_relu_in_the_tiles_of_a_large_product(dt):
    """More than 4 Mi values behind the first layer: ReLU forward and backward inside the
    products' tiles against torch's.  The same sums, a ReLU is exact: the same bits forward; the
    chain's gradients pass through the same roundings (bounds as above)."""
    from fastmoe_amd import fmoe_cuda

    dtype = DTYPES[dt]
    moe = _layer(dtype, 2, d=64, h=1032, activation=torch.nn.ReLU())
    x = torch.randn(2100, 64, device="cuda").to(dtype)
    dy = torch.randn(2100, 64, device="cuda").to(dtype)
    got = []
    for watched in (False, True):
        fmoe_cuda.profile_hook = (lambda *a: None) if watched else None
        try:
            for p in moe.parameters():
                p.grad = None
            a = x.clone().requires_grad_(True)
            out = moe(a)
            out.backward(dy)
        finally:
            fmoe_cuda.profile_hook = None
        got.append([out, a.grad] + [p.grad for p in moe.parameters()])
    assert torch.equal(got[0][0], got[1][0])
    for g, w in zip(got[0][1:], got[1][1:]):
        assert (g - w).double().norm() <= 4 * torch.finfo(dtype).eps * w.double().norm()
