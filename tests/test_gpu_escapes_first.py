"""16-bit results of a weight with escapes: corrected in fp32, then rounded, in one launch behind the kernels (ext.mma_tiles with
escapes_first)."""
import pytest
import torch

from qvb8_amd import ext_qvb8 as ext
from qvb8_amd.formats.qvb8 import pack as PK
from qvb8_amd.formats.qvb8.module import QVBandLinearV8
from tests import helpers as H

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _sorted_pack(Q, P, seed):
    d = H.mixed_width_pack(Q, P, [7, 6, 5], seed=seed)
    d["tau_s"] = d["tau_s"] * (1.0 / 64)
    ids, min_s, nbits, bit_off, P, tau_s, _, _ = H.to_device_args(d, DEV)
    perm = torch.argsort(nbits.to(torch.int16), stable=True).to(torch.int32)
    ids, bit_off, layout = ext.sort_rows_by_width(ids, nbits, bit_off, P, perm)
    rowinfo = ext.mma_prepare(nbits, bit_off, tau_s, min_s, P, ids.numel(), perm)
    return (ids, min_s, nbits, bit_off, P, tau_s), dict(perm=perm, rowinfo=rowinfo, layout=layout)


def _escapes(positions, seed):
    at = torch.tensor(sorted(set(positions)), dtype=torch.int64)
    return at.to(DEV), torch.randn(at.numel(), generator=torch.Generator().manual_seed(seed)).to(DEV)


@pytest.mark.parametrize("M", [1, 7, 16, 17, 64, 256])
@pytest.mark.parametrize("x_dtype,out_dtype", [(torch.bfloat16, torch.bfloat16), (torch.float16, torch.float16), (torch.bfloat16, torch.float16)])
def test_same_values_as_rounding_the_corrected_fp32_results(M, x_dtype, out_dtype):
    """Bit for bit, with escapes in the first and the last place of a row and of the 64 rows a workgroup takes, a row full of them,
    none in whole workgroups, one in 29 columns, and Q that ends inside a workgroup."""
    for Q, P in ((300, 768), (129, 2048)):
        pack, order = _sorted_pack(Q, P, seed=M + Q)
        x = torch.randn(M, P, generator=torch.Generator().manual_seed(M)).to(x_dtype).to(DEV)
        edges = [0, P - 1, P, 63 * P, 64 * P - 1, 64 * P, 64 * P + P - 1, 128 * P + 5, Q * P - 1]
        everywhere = list(range(0, Q * P, 29))
        for positions in ([Q * P - 1], edges, edges + list(range(70 * P, 71 * P)), everywhere):
            esc = _escapes(positions, seed=M)
            for saturate in (True, False):
                y32 = ext.mma_tiles(x, *pack, *esc, saturate=saturate, **order)
                y16 = ext.mma_tiles(x, *pack, *esc, saturate=saturate, out_dtype=out_dtype, escapes_first=True, **order)
                assert y16.dtype == out_dtype and torch.equal(y16, y32.to(out_dtype)), (Q, P, len(positions), saturate)


@pytest.mark.parametrize("M", [1, 4, 5, 63, 64, 65, 130])
def test_rows_of_many_escapes(M):
    """Rows that go on when their neighbours have ended: the last few of a wave are prepared by all its lanes, 64 escapes at a time.
    Runs of 16 (a lane does them alone), 17, 64 + 16, 64 + 17, 128 + 16 and whole rows; two, six, seven and all rows of a wave; the list's end."""
    Q, P = 200, 768
    pack, order = _sorted_pack(Q, P, seed=M)
    x = torch.randn(M, P, generator=torch.Generator().manual_seed(M)).to(torch.bfloat16).to(DEV)
    run = lambda row, n, at=0: list(range(row * P + at, row * P + at + n))                           # noqa: E731
    lists = [run(3, 16) + run(4, 17) + run(40, 80) + run(63, P), run(Q - 1, 144, P - 144), sum((run(r, 81, 7 * r % 600) for r in range(6)), []) + [70 * P],
             sum((run(r, 82 + r, 3) for r in range(64, 71)), []), sum((run(r, 12 + r % 9, r) for r in range(Q)), [])]
    for positions in lists:
        esc = _escapes(positions, seed=M)
        for x_in, out_dtype, saturate in ((x, torch.bfloat16, True), (x.half(), torch.float16, True), (x, torch.bfloat16, False)):
            y32 = ext.mma_tiles(x_in, *pack, *esc, saturate=saturate, **order)
            y16 = ext.mma_tiles(x_in, *pack, *esc, saturate=saturate, out_dtype=out_dtype, escapes_first=True, **order)
            assert torch.equal(y16, y32.to(out_dtype)), (len(positions), saturate)


@pytest.mark.parametrize("M", [1, 16, 64])
def test_corrected_results_in_a_graph(M):
    """The fp32 results between the two launches live in the graph's own memory; every replay against the eager call, with eager calls between."""
    enc = PK.encode_tensor(H.synth_weight(300, 1024, seed=5).to(DEV), 1e-3, restore="fp16", force_escapes=torch.arange(0, 300 * 1024, 997))
    lin = QVBandLinearV8.from_encoded(enc).prepare()
    x = torch.zeros(M, 1024, dtype=torch.bfloat16, device=DEV)
    lin(x)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = lin(x)
    for i in range(4):
        x.copy_(torch.randn(M, 1024, generator=torch.Generator().manual_seed(i)).to(torch.bfloat16))
        graph.replay()
        torch.cuda.synchronize()
        assert y.dtype == torch.bfloat16 and torch.equal(y, lin(x.clone()))


@pytest.mark.parametrize("n_esc", [256, 257, 65536, 65537, 70000])
def test_long_lists_through_the_module(n_esc):
    """One search step more from 257 and from 65537 escapes on; the module against fp32 results rounded by torch."""
    Q, P = 192, 1024
    enc = PK.encode_tensor(H.synth_weight(Q, P, seed=3).to(DEV), 1e-3, restore="fp16")
    enc["esc_idx"], enc["esc_vals"] = _escapes(torch.randperm(Q * P, generator=torch.Generator().manual_seed(n_esc))[:n_esc].tolist(), seed=4)
    x = torch.randn(5, P, generator=torch.Generator().manual_seed(1)).to(torch.float16).to(DEV)
    lin = QVBandLinearV8.from_encoded(enc)
    y = lin(x)
    perm, rowinfo, layout = lin._mma_order()
    y32 = ext.mma_tiles(x, *H.pack_args(dict(enc, ids=lin.ids, nbits=lin.nbits, bit_off=lin.bit_off)), perm=perm, rowinfo=rowinfo, layout=layout, planes=lin._planes)
    assert y.dtype == torch.float16 and torch.equal(y, y32.to(torch.float16))


@pytest.mark.parametrize("M", [1, 20])
def test_a_list_that_does_not_ascend_stays_inside_its_rows(M):
    """Against its documented order the correction may miss a row, and never reads a column of another one: rows 5 and 7 are followed by
    rows before them, row 0 comes last."""
    Q, P = 100, 768
    pack, order = _sorted_pack(Q, P, seed=2)
    x = torch.randn(M, P, generator=torch.Generator().manual_seed(M)).to(torch.bfloat16).to(DEV)
    positions = [5 * P + 3, 5 * P + 700, 2 * P + 1, 7 * P, 6 * P + 5, 9 * P + 767, 0]
    vals = torch.randn(len(positions), generator=torch.Generator().manual_seed(3)).to(DEV)
    at = torch.tensor(positions, dtype=torch.int64)
    by_row = torch.argsort(at)
    whole = ext.mma_tiles(x, *pack, at[by_row].to(DEV), vals[by_row.to(DEV)], **order).to(torch.bfloat16)
    none = ext.mma_tiles(x, *pack, None, None, **order).to(torch.bfloat16)
    y = ext.mma_tiles(x, *pack, at.to(DEV), vals, out_dtype=torch.bfloat16, escapes_first=True, **order)
    assert torch.equal(y[:, 5], whole[:, 5]) and torch.equal(y[:, 7], whole[:, 7]) and torch.equal(y[:, 9], whole[:, 9])
    rest = [q for q in range(Q) if q not in (0, 2, 5, 6, 7, 9)]
    assert torch.equal(y[:, rest], none[:, rest])
    for q in (0, 2, 6):
        assert torch.equal(y[:, q], whole[:, q]) or torch.equal(y[:, q], none[:, q])
