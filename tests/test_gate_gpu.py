"""Fused top-k + softmax gate kernels against the CPU checker and against the
torch.topk + softmax formulation of the reference's NaiveGate."""
import numpy as np
import pytest
import torch
import torch.nn.functional as F

from helpers import DTYPES
from oracle import moe_oracle as O

pytestmark = pytest.mark.gpu

CASES = [  # tokens, experts, top_k
    (1, 1, 1),
    (5, 2, 2),
    (33, 16, 2),        # config 2 shape
    (100, 8, 2),
    (257, 128, 8),      # config 5 shape
    (64, 64, 1),
    (19, 100, 16),      # largest supported top_k
    (7, 4096, 3),
    (1000, 7, 7),       # every expert chosen
    (50, 256, 8),       # up to 512 experts: logits held in registers (8 per lane here)
    (33, 300, 4),       # 32 lanes per token, ragged last register
    (20, 512, 16),
    (40, 17, 3),
    (40, 40, 5),
    (9, 513, 2),        # above 512: sorted lists over 32 lanes
]
SCORE_TOL = {"f64": 1e-12, "f32": 2e-6, "f16": 2e-3, "bf16": 1.6e-2}


@pytest.mark.parametrize("dt", ["f32", "f64", "f16", "bf16"])
@pytest.mark.parametrize("t,e,k", CASES)
def test_forward_and_backward(dt, t, e, k):
    from fastmoe_amd import fmoe_cuda

    dtype = DTYPES[dt]
    rng = np.random.default_rng(t * 131 + e)
    # a permutation of a grid per token: distinct values in float64; the narrow
    # dtypes round the widest cases to ties, which must then go by index
    logits = np.stack([rng.permutation(e) for _ in range(t)]).astype(np.float64)
    logits = (logits - e / 2) / max(e / 8, 1.0)
    lt = torch.from_numpy(logits).to(dtype)
    exact = lt.double().numpy()                       # what the kernel really sees
    idx, score = fmoe_cuda.topk_softmax_fwd(lt.cuda(), k)
    want_idx, want_score = O.topk_softmax(exact, k)
    assert idx.dtype == torch.int64 and score.dtype == dtype
    assert (idx.cpu().numpy() == want_idx).all()
    assert np.abs(score.double().cpu().numpy() - want_score).max() <= SCORE_TOL[dt]
    dscore = torch.from_numpy(rng.standard_normal((t, k))).to(dtype)
    dl = fmoe_cuda.topk_softmax_bwd(dscore.cuda(), score, idx, e)
    want_dl = O.topk_softmax_backward(dscore.double().numpy(), score.double().cpu().numpy(),
                                      want_idx, e)
    assert dl.shape == (t, e) and dl.dtype == dtype
    assert np.abs(dl.double().cpu().numpy() - want_dl).max() <= 4 * SCORE_TOL[dt]
    # zero outside the chosen experts, exactly
    mask = np.ones((t, e), dtype=bool)
    np.put_along_axis(mask, want_idx, False, axis=1)
    assert not dl.double().cpu().numpy()[mask].any()


def test_ties_and_minus_infinity():
    from fastmoe_amd import fmoe_cuda

    lt = torch.tensor([[1.0, 3.0, 3.0, float("-inf"), 3.0],
                       [0.0, 0.0, 0.0, 0.0, 0.0],
                       [float("-inf"), float("-inf"), 2.0, float("-inf"), 1.0]])
    idx, score = fmoe_cuda.topk_softmax_fwd(lt.cuda(), 2)
    assert idx.cpu().tolist() == [[1, 2], [0, 1], [2, 4]]
    want = O.topk_softmax(lt.double().numpy(), 2)[1]
    assert np.abs(score.double().cpu().numpy() - want).max() <= 1e-6


def test_ties_and_minus_infinity_in_a_wide_expert_set():
    from fastmoe_amd import fmoe_cuda

    e = 70
    lt = torch.full((3, e), float("-inf"))
    lt[0, [5, 40, 69]] = torch.tensor([2.0, 2.0, 2.0])       # three-way tie
    lt[1, 33] = 1.0                                           # one finite logit, k = 3
    lt[2] = 0.5                                               # all equal
    idx, score = fmoe_cuda.topk_softmax_fwd(lt.cuda(), 3)
    assert idx.cpu().tolist() == [[5, 40, 69], [33, 0, 1], [0, 1, 2]]
    want = O.topk_softmax(lt.double().numpy(), 3)[1]
    assert np.abs(score.double().cpu().numpy() - want).max() <= 1e-6


def test_nan_logits_rank_first_as_in_torch_topk():
    """torch.topk ranks NaN above every number (naive_gate.py:31-38 inherits that):
    a NaN logit is selected and the token's scores become NaN, for both the
    register-resident (<= 512 experts) and the sorted-list kernels."""
    from fastmoe_amd import fmoe_cuda

    nan, ninf = float("nan"), float("-inf")
    for e in (6, 600):
        lt = torch.zeros(4, e)
        lt[0, :6] = torch.tensor([1.0, nan, 3.0, ninf, 2.0, 0.5])
        lt[1, :6] = torch.tensor([nan, nan, nan, 1.0, ninf, 0.0])     # fewer numbers than k
        lt[2, :6] = torch.tensor([ninf, ninf, 1.0, ninf, ninf, ninf])
        lt[3, :6] = torch.tensor([5.0, 4.0, 3.0, 2.0, 1.0, 0.5])
        lt[:, 6:] = -10.0
        idx, score = fmoe_cuda.topk_softmax_fwd(lt.cuda(), 3)
        tval, tidx = torch.topk(lt, 3, dim=-1)
        idx, score = idx.cpu(), score.cpu()
        assert idx[0].tolist() == [1, 2, 4] and idx[1].tolist() == [0, 1, 2]
        assert idx[2, 0].item() == 2 and idx[3].tolist() == [0, 1, 2]
        for r in range(4):                      # same experts as torch.topk picks
            assert sorted(idx[r].tolist()) == sorted(tidx[r].tolist()) or r == 2
        assert idx.min().item() >= 0 and idx.max().item() < e
        assert torch.isnan(score[0]).all() and torch.isnan(score[1]).all()
        want = F.softmax(tval[3].double(), dim=-1)
        assert (score[3].double() - want).abs().max().item() <= 1e-6
        assert not torch.isnan(score[2:]).any()


def test_autograd_matches_torch_formulation():
    """The fused op inside autograd against torch.topk + softmax (no ties)."""
    from fastmoe_amd.functions import topk_softmax

    torch.manual_seed(3)
    logits = torch.randn(513, 32, device="cuda")
    a = logits.clone().requires_grad_(True)
    b = logits.clone().requires_grad_(True)
    idx, score = topk_softmax(a, 4)
    val, tidx = torch.topk(b, 4, dim=-1, largest=True, sorted=True)
    tscore = F.softmax(val, dim=-1)
    assert (idx == tidx).all()
    assert (score - tscore).abs().max().item() <= 2e-6
    g = torch.randn_like(score)
    score.backward(g)
    tscore.backward(g)
    assert (a.grad - b.grad).abs().max().item() <= 2e-6


def test_naive_gate_uses_the_kernel_and_errors():
    from fastmoe_amd import fmoe_cuda
    from fastmoe_amd.gates import NaiveGate

    gate = NaiveGate(24, 6, 1, top_k=2).cuda()
    x = torch.randn(50, 24, device="cuda")
    seen = []
    fmoe_cuda.profile_hook = lambda name, a, b: seen.append(name)
    try:
        idx, score = gate(x)
    finally:
        fmoe_cuda.profile_hook = None
    assert "topk_softmax_fwd" in seen
    logits = gate.gate(x)
    want_idx, want_score = O.topk_softmax(logits.double().cpu().detach().numpy(), 2)
    assert (idx.cpu().numpy() == want_idx).all()
    assert np.abs(score.double().cpu().detach().numpy() - want_score).max() <= 2e-6
    with pytest.raises(RuntimeError):
        fmoe_cuda.topk_softmax_fwd(torch.zeros(4, 3, device="cuda"), 4)      # k > experts
    with pytest.raises(RuntimeError):
        fmoe_cuda.topk_softmax_fwd(torch.zeros(4, 40, device="cuda"), 17)    # k > supported


@pytest.mark.parametrize("dt", ["bf16", "f16", "f32", "f64"])
@pytest.mark.parametrize("t,e,k,d", [(1, 1, 1, 1), (33, 4, 2, 7), (500, 5, 2, 264), (700, 130, 8, 520),
                                     (5000, 3, 2, 1032), (4096, 16, 1, 4100)])
def test_gate_gradients_from_slots(dt, t, e, k, d):
    """The plain gate's gradients from its top-k slots (one slot in eight dropped, expert 0
    popular) against the dense products in float64.  A sum of n products in the accumulation
    type is off by at most (n + 8) units of the sum of their magnitudes (8: the gradient of the
    slot itself), the result by one rounding of the storage type."""
    from fastmoe_amd import _lib, fmoe_cuda

    lib, dtype = _lib.load(), DTYPES[dt]
    acc = torch.float64 if dt == "f64" else torch.float32
    g = torch.Generator().manual_seed(t + d)
    idx = torch.argsort(torch.rand(t, e, generator=g) - torch.eye(1, e) * 0.4, 1)[:, :k]
    idx[torch.rand(t, k, generator=g) < 0.125] = -1
    rnd = lambda *s: torch.randn(*s, generator=g, dtype=torch.float64).to(dtype)
    x, wg, dbuf, dscore = rnd(t, d), rnd(e, d), rnd(t * k, d), rnd(t, k)
    score = torch.softmax(rnd(t, k).double(), 1).to(dtype)
    c = {n: v.cuda().contiguous() for n, v in dict(idx=idx, x=x, wg=wg, dbuf=dbuf, dscore=dscore,
                                                   score=score).items()}
    pos, _, seg, inv = fmoe_cuda.route(c["idx"], e)
    code = {"f32": 0, "f64": 1, "f16": 2, "bf16": 3}[dt]
    stream = torch.cuda.current_stream().cuda_stream
    dl = torch.empty(t, k, device="cuda", dtype=acc)
    dx, dwg = torch.empty_like(c["x"]), torch.empty_like(c["wg"])
    dbg = torch.empty(e, device="cuda", dtype=dtype)
    n = lib.fmoe_gate_linear_grad_workspace_bytes(c["x"].data_ptr(), t, k, d, e, code)
    ws = torch.empty(n, device="cuda", dtype=torch.uint8)
    p = lambda a: a.data_ptr()
    assert lib.fmoe_gate_slot_grad(p(c["dscore"]), p(c["score"]), p(dl), t, k, code, stream) == 0
    assert lib.fmoe_scatter_reduce_gate(p(c["dbuf"]), p(inv), p(c["idx"]), p(dl), p(c["wg"]), p(dx),
                                        t, k, d, e, code, stream) == 0
    assert lib.fmoe_gate_linear_grad(p(c["x"]), p(pos), p(seg), p(dl), p(dwg), p(dbg), t, k, d, e,
                                     p(ws), n, code, stream) == 0
    s, ds = score.double(), dscore.double()
    want_dl = s * (ds - (ds * s).sum(1, keepdim=True))
    mag_dl = s * (ds.abs() + (ds * s).abs().sum(1, keepdim=True))
    rows = inv.cpu().view(t, k).long()
    live = (idx >= 0)[..., None].double()
    moved = dbuf.double()[rows.clamp(min=0)] * live
    alone = torch.empty_like(dx)      # the gate's share without rows of the experts
    assert lib.fmoe_scatter_reduce_gate(None, None, p(c["idx"]), p(dl), p(c["wg"]), p(alone), t, k,
                                        d, e, code, stream) == 0
    dense = torch.zeros(t, e, dtype=torch.float64).scatter_add_(1, idx.clamp(min=0), want_dl * live[..., 0])
    mags = torch.zeros(t, e, dtype=torch.float64).scatter_add_(1, idx.clamp(min=0), mag_dl * live[..., 0])
    unit, eps = torch.finfo(acc).eps, torch.finfo(dtype).eps
    for got, want, mag, terms in (
            (dx, moved.sum(1) + dense @ wg.double(), moved.abs().sum(1) + mags @ wg.double().abs(), 2 * k),
            (alone, dense @ wg.double(), mags @ wg.double().abs(), k),
            (dwg, dense.t() @ x.double(), mags.t() @ x.double().abs(), t),
            (dbg, dense.sum(0), mags.sum(0), t)):
        err = (got.double().cpu() - want).abs()
        # (f16 below its smallest normal number: half a step of 2^-24)
        if got is dx:   # either share is rounded before the addition
            err = err - eps * (moved.sum(1).abs() + (dense @ wg.double()).abs())
        assert (err <= eps * want.abs() + unit * (terms + 8 + k) * mag + (2 ** -25 if dt == "f16" else 0)).all()


def test_gate_over_more_experts_than_can_be_routed():
    """Choosing needs no routing, so a gate module may have more outputs than a layer may have
    experts, and differentiate.  Against torch's own operations: sums of 50 terms in float32."""
    from fastmoe_amd import NaiveGate

    torch.manual_seed(8)
    gate = NaiveGate(16, 5000, 1, 2).cuda()
    x = torch.randn(50, 16, device="cuda", requires_grad=True)
    params = [x, gate.gate.weight, gate.gate.bias]
    idx, score = gate(x)
    got = torch.autograd.grad((score * score).sum(), params)
    val, want_idx = torch.topk(gate.gate(x), 2)
    want = torch.autograd.grad((torch.softmax(val, -1) ** 2).sum(), params)
    assert torch.equal(idx, want_idx)
    for g, w in zip(got, want):
        assert (g - w).norm() <= 1e-5 * w.norm()


def test_gshard_indices_keep_the_leading_dimensions():
    """On a [S, B, d] input the choices come as [S, B, 2], the scores as [S * B, 2], as those of
    the plain gate."""
    from fastmoe_amd import GShardGate, NaiveGate

    torch.manual_seed(3)
    gate = GShardGate(16, 4, 1, capacity=(8.0, 8.0), random_routing=False).cuda()
    plain = NaiveGate(16, 4, 1, 2).cuda()
    plain.load_state_dict(gate.state_dict())
    x = torch.randn(10, 6, 16, device="cuda")
    idx, score = gate(x)
    want_idx, want = plain(x)
    assert idx.shape == (10, 6, 2) and torch.equal(score, want)
    assert ((idx == want_idx) | (idx == -1)).all() and (idx >= 0).any()


@pytest.mark.parametrize("gate", ["GShardGate", "SwitchGate"])
def test_balance_gates_refuse_another_number_of_outputs(gate):
    """Their loss has one term per expert: a linear map with more outputs is an error, not a
    loss over something else."""
    import fastmoe_amd

    layer = getattr(fastmoe_amd, gate)(16, 4, 1).cuda()
    layer(torch.randn(50, 16, device="cuda"))
    layer.gate = torch.nn.Linear(16, 6).cuda()
    with pytest.raises(RuntimeError, match="size"):
        layer(torch.randn(50, 16, device="cuda"))


@pytest.mark.parametrize("which", ["score", "loss"])
def test_batches_of_gradients_through_the_balance_gates(which):
    """Several gradients at once (is_grads_batched) are those taken one by one, up to the 20 or
    so roundings of each way to them."""
    from fastmoe_amd import GShardGate, SwitchGate

    torch.manual_seed(5)
    gates = [SwitchGate(16, 4, 1).cuda()]
    if which == "loss":   # (GShard's scores have no batched gradient)
        gates.append(GShardGate(16, 4, 1, random_routing=False).cuda())
    for gate in gates:
        x = torch.randn(50, 16, device="cuda", requires_grad=True)
        score = gate(x)[1]
        out = score if which == "score" else gate.get_loss()
        dy = torch.randn((3,) + out.shape, device="cuda")
        got = torch.autograd.grad(out, x, dy, is_grads_batched=True, retain_graph=True)[0]
        for g, d in zip(got, dy):
            want = torch.autograd.grad(out, x, d, retain_graph=True)[0]
            assert want.any() and (g - want).norm() <= 20 * torch.finfo(g.dtype).eps * want.norm()
