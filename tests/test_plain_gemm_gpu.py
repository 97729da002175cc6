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
                                               ([3, 0, 40, 1, 9], 200, 3328)])
def test_tiles_of_few_rows_per_expert(dt, counts, in_f, out_f):
    """The forward's 32- and 64-row tiles, which the average number of rows chooses: edges of
    tiles, of K slices of 64 and of the stages (six with up to 256 tiles, three beyond), and
    experts far above the average."""
    _run(counts, in_f, out_f, DTYPES[dt], True, 0, extra_rows=3)
