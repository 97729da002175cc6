"""HIP-graph capture and replay of the whole layer (forward + backward).  Kept
in a file of its own that pytest collects last."""
import os
import subprocess
import sys

import pytest
import torch

from conftest import ROOT
from test_layer_gpu import _make

pytestmark = pytest.mark.gpu


def test_forward_and_backward_replay_from_a_hip_graph():
    """The fused layer enqueues without reading anything back to the host, so
    forward + backward can be captured once and replayed on new data whose
    routing differs.  Every replay is checked against the eager layer, with
    eager work and synchronisations between the replays."""
    dtype = torch.bfloat16
    moe = _make(8, 128, 256, 2, dtype, seed=5, scale=0.05)
    g = torch.Generator().manual_seed(21)
    xs = [torch.randn(300, 128, generator=g).to(dtype).cuda() for _ in range(4)]
    dys = [torch.randn(300, 128, generator=g).to(dtype).cuda() for _ in range(4)]
    params = list(moe.parameters())

    def eager(x, dy):
        for p in params:
            p.grad = None
        xi = x.clone().requires_grad_(True)
        out = moe(xi)
        out.backward(dy)
        return [out.detach().clone(), xi.grad.clone()] + [p.grad.clone() for p in params]

    want = [eager(x, dy) for x, dy in zip(xs, dys)]    # also warms every kernel up
    static_x = xs[0].clone().requires_grad_(True)
    static_dy = dys[0].clone()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):                      # warm-up on the capture stream
        for _ in range(2):
            for p in params:
                p.grad = None
            static_x.grad = None
            moe(static_x).backward(static_dy)
    torch.cuda.current_stream().wait_stream(side)
    for p in params:
        p.grad = None
    static_x.grad = None
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        static_out = moe(static_x)
        static_out.backward(static_dy)
    # the tensors the graph writes (eager steps below rebind p.grad to new ones)
    got = [static_out, static_x.grad] + [p.grad for p in params]
    for i in (1, 2, 3, 0, 2):
        with torch.no_grad():
            static_x.copy_(xs[i])
            static_dy.copy_(dys[i])
        graph.replay()
        torch.cuda.synchronize()
        for a, b in zip(got, want[i]):
            assert torch.equal(a, b)
        _ = eager(xs[(i + 1) % 4], dys[(i + 1) % 4])   # eager work between replays
        torch.cuda.synchronize()


def test_make_graphed_callables_replays_the_layer():
    """fastmoe_amd.graphed (torch.cuda.make_graphed_callables behind the library's
    set-up) captures the layer's forward and backward in two graphs behind an ordinary
    autograd interface.  The graphed layer gives the bits of an eager twin on new data
    with other routings, with eager work and synchronisations between its calls."""
    import copy

    import fastmoe_amd

    dtype = torch.bfloat16
    moe = _make(8, 128, 256, 2, dtype, seed=5, scale=0.05)
    twin = copy.deepcopy(moe)
    g = torch.Generator().manual_seed(22)
    xs = [torch.randn(300, 128, generator=g).to(dtype).cuda() for _ in range(4)]
    dys = [torch.randn(300, 128, generator=g).to(dtype).cuda() for _ in range(4)]

    def run(layer, x, dy):
        params = list(layer.parameters())
        for p in params:
            p.grad = None
        xi = x.clone().requires_grad_(True)
        out = layer(xi)
        out.backward(dy)
        return [out.detach().clone(), xi.grad.clone()] + [p.grad.clone() for p in params]

    want = [run(twin, x, dy) for x, dy in zip(xs, dys)]
    graphed = fastmoe_amd.graphed(moe, xs[0].clone().requires_grad_(True))
    for i in (1, 2, 3, 0, 2):
        got = run(graphed, xs[i], dys[i])
        torch.cuda.synchronize()
        for a, b in zip(got, want[i]):
            assert torch.equal(a, b)
        _ = run(twin, xs[(i + 1) % 4], dys[(i + 1) % 4])
        torch.cuda.synchronize()


FIRST_RELU = """
import sys, torch
sys.path.insert(0, {tests!r}); sys.path.insert(0, {root!r})
from helpers import DTYPES, randn
from fastmoe_amd import _lib
lib, dtype, code = _lib.load(), DTYPES[{dt!r}], {{"f16": 2, "bf16": 3}}[{dt!r}]
counts, n_in, n_out = [300, 0, 257, 70], 64, 96
n, e = sum(counts), len(counts)
x, w, dy = (randn(s, dtype, i, 0.3).cuda() for i, s in enumerate([(n, n_in), (e, n_out, n_in), (n, n_in)]))
seg = torch.tensor([0] + counts).cumsum(0).int().cuda()
a, dpre = (torch.empty(n, n_out, dtype=dtype, device="cuda") for _ in range(2))
w2, dw2 = randn((e, n_in, n_out), dtype, 4, 0.3).cuda(), torch.empty(e, n_in, n_out, dtype=dtype, device="cuda")
assert lib.fmoe_set_gemm_path({path}) == 0
def call():
    s = torch.cuda.current_stream().cuda_stream
    for rc in (lib.fmoe_expert_linear_fwd(x.data_ptr(), w.data_ptr(), None, None, None, seg.data_ptr(), None,
                                          a.data_ptr(), 2, n, n_in, n_out, e, code, s),
               lib.fmoe_expert_linear_bwd(dy.data_ptr(), a.data_ptr(), w2.data_ptr(), None, seg.data_ptr(),
                                          a.data_ptr(), 2, dpre.data_ptr(), dw2.data_ptr(), None, n, n_out,
                                          n_in, e, code, s)):
        assert rc == 0, lib.fmoe_last_error()
graph = torch.cuda.CUDAGraph()
with torch.cuda.graph(graph):
    call()
got = []
for _ in range(3):
    a.zero_(), dpre.zero_(), dw2.zero_()
    graph.replay()
    torch.cuda.synchronize()
    got.append([t.clone() for t in (a, dpre, dw2)])
call()
torch.cuda.synchronize()
for r in got:
    assert all(torch.equal(p, q) for p, q in zip(r, (a, dpre, dw2)))
assert a.any() and dpre.any() and (a == 0).any()
print("captured")
"""


@pytest.mark.parametrize("dt", ["bf16", "f16"])
@pytest.mark.parametrize("path", [0, 2])
def test_the_first_relu_of_a_process_can_be_captured(dt, path):
    """A ReLU needs no table, so nothing has to be set up outside the graph: in a process of its
    own, on the small tiles and on the 256-row ones."""
    code = FIRST_RELU.format(root=ROOT, tests=os.path.join(ROOT, "tests"), dt=dt, path=path)
    res = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=100)
    assert res.returncode == 0 and "captured" in res.stdout, (res.stdout + res.stderr)[-2000:]
