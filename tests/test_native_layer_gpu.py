"""The layer as one native autograd node against the chain of Python nodes it replaces
(which still runs while a per-op event hook is set): the same kernels in the same order,
so the same bits, with and without gradients, for every subset of gradients asked for."""
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
    for g, w in zip(got, want):
        assert (g is None) == (w is None)
        assert g is None or torch.equal(g, w)


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
