"""GPU tests of the gate+up launch that applies the activation itself (ext.MMA_SILU_PAIRS through QVBandMLPV8): against the float64
chain and the separate calls, at row counts and shapes where tiles, waves and the two ways of joining partial sums change."""
import copy

import numpy as np
import pytest
import torch
import torch.nn.functional as F

from oracle import qvb8_oracle as O
from qvb8_amd import ext_qvb8 as ext
from qvb8_amd.formats.qvb8.mlp import QVBandMLPV8, tiles_of_pairs, unit_order
from tests import helpers as H
from tests.test_gpu_mlp import _build

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

SHAPES = [  # hidden, inter, out, rows of several widths
    (128, 128, 128, False),        # one step, eight units
    (1024, 2048, 256, True),
    (4096, 12288, 512, False),     # three tiles per workgroup: one pass over sixteen lanes an output
    (5120, 1536, 256, True),       # rows of 40 steps
    (8192, 384, 256, False),       # two panels
]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_activated_rows_against_the_chain(shape, dtype):
    hidden, inter, out, spread = shape
    mlp, Ws = _build(hidden, inter, out, seed=7 * hidden + inter, spread=spread)
    step = 2.0 ** -7 if dtype == torch.bfloat16 else 2.0 ** -10
    for M in (1, 2, 5, 8, 9, 16):
        x = torch.randn(M, hidden, generator=torch.Generator().manual_seed(M)).to(dtype).to(DEV)
        print("silu pairs", shape, dtype, M, flush=True)
        h = mlp._activated(x)
        assert h is not None and h.dtype == dtype and h.shape == (M, inter)
        xs = O.sat_half(x.float().cpu().numpy())
        g_ref, u_ref = O.linear_f64(xs, Ws[0]), O.linear_f64(xs, Ws[1])
        h_ref = O.silu(g_ref) * u_ref
        # each product's bound and one rounding step of g, u, silu(g) and h (|silu'| <= 1.1)
        dg = H.gemv_tolerance(g_ref, Ws[0], xs) + step * np.abs(g_ref)
        du = H.gemv_tolerance(u_ref, Ws[1], xs) + step * np.abs(u_ref)
        bound = 1.1 * dg * np.abs(u_ref) + du * np.abs(O.silu(g_ref)) + 2 * step * np.abs(h_ref) + 1e-7
        gap = np.abs(h.float().cpu().numpy().astype(np.float64) - h_ref)
        assert np.all(gap <= bound), (M, float((gap / bound).max()))
        # the separate calls: the same sums in another order of joining, the same roundings
        gu = mlp.gate_up(x)
        chain = F.silu(gu[..., :inter]) * gu[..., inter:]
        assert (h != chain).float().mean().item() < 5e-3
        assert torch.equal(mlp.separate(x), mlp.down(h))


def test_what_takes_the_separate_calls():
    mlp, _ = _build(512, 768, 512, seed=3)
    x = torch.randn(17, 512, device=DEV).to(torch.bfloat16)
    assert mlp._activated(x) is None and mlp._activated(x[:4].float()) is None and mlp._activated(x[:8:2]) is None
    assert mlp.separate(x).shape == (17, 512)
    seen = []
    hook = mlp.gate_up.register_forward_hook(lambda m, a, y: seen.append(y.shape))
    mlp(x[:2])
    hook.remove()
    assert seen == [(2, 1536)]
    gu = mlp.gate_up
    perm, rowinfo, layout = gu._mma_order()
    args = (gu.ids, gu.min_s, gu.nbits, gu.bit_off, 512, gu.tau_s, None, None)
    kw = dict(perm=perm, rowinfo=rowinfo, planes=gu._planes, silu_pairs=True)
    for bad in (dict(out_dtype=None, layout=layout), dict(out_dtype=torch.bfloat16, layout=None)):
        with pytest.raises(RuntimeError):
            ext.mma_tiles(x[:2], *args, **kw, **bad)
    with pytest.raises(RuntimeError):
        ext.mma_tiles(x, *args, **kw, out_dtype=torch.bfloat16, layout=layout)


def _other_order(gu):
    """The rows in unit_order's own order (16 gate rows, then their 16 up rows): no tile holds both rows of an output."""
    assert gu.store_in_order(*unit_order(gu.nbits, gu.out_features // 2))


def test_rows_that_are_no_pairs_give_nan():
    mlp, _ = _build(512, 256, 512, seed=4)
    gu = mlp.gate_up
    _other_order(gu)
    perm, rowinfo, layout = gu._mma_order()
    x = torch.randn(2, 512, device=DEV).to(torch.bfloat16)
    h = ext.mma_tiles(x, gu.ids, gu.min_s, gu.nbits, gu.bit_off, 512, gu.tau_s, None, None, perm=perm, rowinfo=rowinfo, layout=layout,
                      out_dtype=torch.bfloat16, planes=gu._planes, silu_pairs=True)
    assert bool(torch.isnan(h.float()).all())


def test_gate_up_in_another_order_or_replaced_takes_the_separate_calls():
    """The order the launch needs is a fact of gate_up's rows, and gate_up may be stored again, replaced, wrapped, copied and moved."""
    for M in (1, 7, 16):
        mlp, _ = _build(512, 256, 512, seed=4)
        x = torch.randn(M, 512, generator=torch.Generator().manual_seed(M)).to(torch.bfloat16).to(DEV)
        gu = mlp.gate_up

        def chain():
            y = mlp.gate_up(x)
            return mlp.down(F.silu(y[:, :256]) * y[:, 256:])

        moved = copy.deepcopy(mlp).cpu().to(DEV)                       # the same bytes in the same order
        for m in (mlp, moved):
            assert m._activated(x) is not None
        assert torch.equal(moved(x), mlp(x))
        gu.forward = lambda rows: torch.zeros(rows.shape[0], 512, dtype=rows.dtype, device=rows.device)
        assert mlp._activated(x) is None and not mlp(x).any()
        del gu.forward
        other, _ = _build(512, 256, 512, seed=5)
        _other_order(other.gate_up)
        mlp.gate_up = other.gate_up
        assert mlp._activated(x) is None and torch.equal(mlp(x), chain()) and torch.isfinite(mlp(x)).all()
        mlp.gate_up = gu
        assert mlp._activated(x) is not None
        _other_order(gu)
        assert mlp._activated(x) is None and torch.equal(mlp(x), chain()) and torch.isfinite(mlp(x)).all()


def test_tiles_of_pairs():
    perm, _ = unit_order(torch.tensor([6] * 64, dtype=torch.uint8), 32)
    tiles = tiles_of_pairs(perm).view(-1, 2, 8)
    assert bool((tiles[:, 1] == tiles[:, 0] + 32).all()) and sorted(tiles[:, 0].reshape(-1).tolist()) == list(range(32))


def test_activated_rows_in_a_graph():
    mlp, _ = _build(1024, 2048, 1024, seed=21)
    x = torch.zeros(1, 1024, dtype=torch.bfloat16, device=DEV)
    mlp(x)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = mlp(x)
    for i in range(4):
        x.copy_(torch.randn(1, 1024, generator=torch.Generator().manual_seed(i)).to(torch.bfloat16))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, mlp(x.clone()))
