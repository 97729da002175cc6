"""The plain-pipeline matrix-core GEMMs (f32 of any shape; bf16 / f16 of even feature
sizes): every tile shape forced at sizes on and around the edges of its tiles and K
slices, against float64; the f32 activation inside the tiles against the activation
kernel, bit for bit."""
import numpy as np
import pytest
import torch

from helpers import DTYPES, TOL, max_rel_err, randn
from test_linear_gpu import _run

pytestmark = pytest.mark.gpu

# counts per expert, in_feat, out_feat
EDGES = [
    ([1], 2, 2),
    ([64, 65, 0, 127, 129], 62, 66),
    ([63, 128, 1, 0, 200], 130, 126),
    ([33, 31, 0, 2], 258, 34),
    ([70, 300], 36, 300),
]


@pytest.mark.parametrize("dt", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("tile", [0, 1, 2])
@pytest.mark.parametrize("counts,in_f,out_f", EDGES)
def test_every_tile_shape_at_its_edges(dt, tile, counts, in_f, out_f):
    _run(counts, in_f, out_f, DTYPES[dt], True, tile + 1 if tile else 0, extra_rows=3)


@pytest.mark.parametrize("tile", [0, 1, 2])
@pytest.mark.parametrize("counts,in_f,out_f", [([64, 65, 0, 127], 64, 68), ([130, 5], 132, 128)])
def test_f32_sixteen_byte_rows(tile, counts, in_f, out_f):
    _run(counts, in_f, out_f, torch.float32, True, tile + 1 if tile else 0, extra_rows=1)


@pytest.mark.parametrize("in_f,out_f", [(64, 132), (38, 66)])
def test_f32_activation_inside_the_tiles(in_f, out_f):
    from fastmoe_amd import fmoe_cuda

    counts = [70, 0, 129, 3]
    seg = torch.from_numpy(np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)).cuda()
    n, e = sum(counts), len(counts)
    x, w, b = (randn(s, torch.float32, i, 0.5).cuda()
               for i, s in enumerate([(n, in_f), (e, out_f, in_f), (e, out_f)]))
    y, a = fmoe_cuda.grouped_linear_fwd(x, seg, w, b, with_gelu=True)
    assert torch.equal(y, fmoe_cuda.grouped_linear_fwd(x, seg, w, b))
    assert torch.equal(a, fmoe_cuda.gelu_fwd(y))
    dy = randn((n, out_f), torch.float32, 7).cuda()
    pre = randn((n, in_f), torch.float32, 8).cuda()
    dx, dw, db = fmoe_cuda.grouped_linear_bwd(dy, x, seg, w, act_pre=pre)
    dh, dw0, db0 = fmoe_cuda.grouped_linear_bwd(dy, x, seg, w)
    assert torch.equal(dw, dw0) and torch.equal(db, db0)
    assert torch.equal(dx, fmoe_cuda.gelu_bwd(dh, pre))
    # each product alone runs the same tiles
    for kw, want in (({"need_dw": False, "need_bias": False}, (dh, None, None)),
                     ({"need_dx": False}, (None, dw, db))):
        for got, ref in zip(fmoe_cuda.grouped_linear_bwd(dy, x, seg, w, **kw), want):
            assert (got is None) == (ref is None)
            assert got is None or max_rel_err(got, ref) <= TOL[torch.float32]


@pytest.mark.parametrize("dt", ["bf16", "f16"])
@pytest.mark.parametrize("counts,in_f,out_f", [([1], 8, 8), ([128, 129, 0, 31, 32], 256, 128),
                                               ([127, 0, 300], 264, 136), ([33, 5, 97], 520, 248)])
def test_wide_column_tiles(dt, counts, in_f, out_f):
    """The backward's 128 x 256 tiles: edges of tiles, of K slices of 32 and of the three
    stages."""
    _run(counts, in_f, out_f, DTYPES[dt], True, 9, extra_rows=3)


@pytest.mark.parametrize("dt", ["bf16", "f16"])
@pytest.mark.parametrize("path", [3, 4, 8, 9])
@pytest.mark.parametrize("counts,in_f,out_f", [([1, 1], 8, 8), ([64, 65, 0, 127], 64, 72),
                                               ([129, 63, 128, 1], 136, 256), ([200], 200, 56)])
def test_sixteen_bit_rows_of_sixteen_bytes(dt, path, counts, in_f, out_f):
    """All four kinds of small tiles at the edges of each, with one and with several experts, an
    odd number of them among others."""
    _run(counts, in_f, out_f, DTYPES[dt], True, path, extra_rows=3)


@pytest.mark.parametrize("dt", ["bf16", "f16"])
@pytest.mark.parametrize("counts,in_f,out_f", [([1], 8, 8), ([32, 33, 0, 31, 1], 136, 72),
                                               ([0, 0, 150, 0, 0, 0, 2, 1], 264, 128),
                                               ([65, 63, 0, 64, 1, 33], 136, 264),
                                               ([0, 0, 300, 3, 0, 0], 520, 136),
                                               ([3, 0, 40, 1, 9], 200, 3328),
                                               ([40, 64, 0, 33, 65, 38] * 85, 64, 136)])
def test_tiles_of_few_rows_per_expert(dt, counts, in_f, out_f):
    """The forward as the average number of rows chooses it, experts far above the average among
    them: 32 x 64 tiles, 64 x 64 ones for few tiles (the fourth and fifth), 64 x 128 ones for many
    (the last); each kind at its edges is below."""
    _run(counts, in_f, out_f, DTYPES[dt], True, 0, extra_rows=3)


def _bits(t):
    return t.view(torch.int16)


# rows at the edges of 32, 64 and 128, columns at those of 64 and 128, and K slices of 64 from one
# to more than twice round a ring of six stages, with and without a tail
LOW_TILES = [([1], 8, 8), ([32, 33, 0, 31, 1], 384, 72), ([64, 65, 0, 63, 2], 392, 128),
             ([128, 129, 0, 127, 30], 776, 136), ([0, 0, 300, 3, 96, 97], 1032, 264),
             ([3, 0, 40, 1, 9], 448, 3328),
             # long experts: few tiles of them, and enough to be cut higher; also above 64 experts
             ([70, 1, 20, 33, 0], 136, 3464), ([70, 1, 200, 33, 0], 136, 11016),
             ([0, 1, 33, 130, 96] * 14, 72, 200), ([0, 1, 33, 130, 96] * 14, 72, 808)]


@pytest.mark.parametrize("dt", ["bf16", "f16"])
@pytest.mark.parametrize("path", [11, 12])
@pytest.mark.parametrize("counts,in_f,out_f", LOW_TILES)
def test_every_tile_of_few_rows(dt, path, counts, in_f, out_f):
    """Forward tiles of few rows against float64 and, bit for bit, against the 128 x 128 ones:
    with and without a bias, weights behind pointer tables, both activations, and a ReLU whose
    argument is not kept."""
    from fastmoe_amd import _lib, fmoe_cuda
    from test_fused_act_gpu import _expert_linear

    dtype = DTYPES[dt]
    for with_bias in (True, False):
        _run(counts, in_f, out_f, dtype, with_bias, path, extra_rows=3)
    n, e = sum(counts), len(counts)
    seg = torch.tensor([0] + counts).cumsum(0).int().cuda()
    x, w, b = (randn(s, dtype, i, 0.3).cuda()
               for i, s in enumerate([(n + 3, in_f), (e, out_f, in_f), (e, out_f)]))
    got = {}
    for p in (path, 3):
        fmoe_cuda.set_gemm_path(p)
        try:
            y, a = fmoe_cuda.grouped_linear_fwd(x, seg, w, b, with_gelu=True)
            apart = [[t[i:i + 1].clone() for i in range(e)] for t in (w, b)]
            z = fmoe_cuda.grouped_linear_fwd_ptrs(x, seg, *map(fmoe_cuda.pointer_table, apart),
                                                  out_f)
            relu = _expert_linear(_lib.load(), dtype, counts, in_f, out_f, p)[1]
            got[p] = [y[:n], a[:n], fmoe_cuda.grouped_linear_fwd(x, seg, w, None)[:n],
                      relu(2, True)[1], relu(2, False)[1]]
            assert torch.equal(_bits(z[:n]), _bits(y[:n]))
        finally:
            fmoe_cuda.set_gemm_path(0)
    assert all(torch.equal(_bits(g), _bits(h)) for g, h in zip(got[path], got[3]))


def test_all_rows_on_one_of_many_experts():
    """The choice of tiles sees the average number of rows, 16 here; an expert that holds all of
    them is cut into higher tiles.  Tiles of 128 rows, which know no average, are the measure
    (129 us where tiles of 32 rows took 250; 1.3 times that is the expectation)."""
    from fastmoe_amd import fmoe_cuda

    e, n, in_f, out_f = 64, 1024, 4096, 14336
    w = randn((1, 112, 8), torch.bfloat16, 1, 0.02).cuda().repeat(1, out_f // 112, in_f // 8)
    x = randn((n, in_f), torch.bfloat16, 2).cuda()
    seg = torch.tensor([0] * 21 + [n] * (e + 1 - 21), dtype=torch.int32).cuda()
    table = fmoe_cuda.pointer_table([w] * e)
    best = {0: float("inf"), 3: float("inf")}
    for _ in range(6):
        for path in best:
            fmoe_cuda.set_gemm_path(path)
            try:
                start, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
                start.record()
                for _ in range(10):
                    fmoe_cuda.grouped_linear_fwd_ptrs(x, seg, table, None, out_f)
                end.record()
                end.synchronize()
            finally:
                fmoe_cuda.set_gemm_path(0)
            best[path] = min(best[path], start.elapsed_time(end))
    assert best[0] <= 1.6 * best[3], best
