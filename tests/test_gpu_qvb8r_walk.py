"""GPU tests of the QVB8R walk where its window of words moves most often and tiles of a wave differ: nearly uniform symbols (ten bits
each, so a pair of steps takes some 20 of the 64 words kept ahead), rows of one step group and of many, tiles with fewer rows
than their neighbour, blocks that are not full."""
import numpy as np
import pytest
import torch

from oracle import qvb8_oracle as O
from oracle import qvb8r_oracle as R
from qvb8_amd import ext_qvb8r as ext
from qvb8_amd.formats.qvb8 import pack as PK
from qvb8_amd.formats.qvb8r import pack as RP
from qvb8_amd.formats.qvb8r.module import QVBandLinearV8R
from tests import helpers as H

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("Q,P,kw", [(5, 128, dict(rows_per_tile=2)), (67, 384, dict(rows_per_tile=5, n_classes=3)), (130, 640, dict(rows_per_tile=1)),
                                     (33, 2176, dict(rows_per_tile=4)), (19, 8192, dict())])
def test_window_of_words(Q, P, kw):
    g = torch.Generator().manual_seed(Q * P)
    W = (0.1 * (2.0 * torch.rand(Q, P, generator=g) - 1.0)).to(torch.bfloat16).to(DEV)
    enc = PK.encode_tensor(W, 1.3e-4, keep_ids=True)
    d = RP.transcode(enc, **kw)
    want = enc["ids_dense"].cpu().numpy().astype(np.int64)
    assert np.array_equal(R.ids(d), want) and 32 * len(d["words"]) > 7 * Q * P
    lin = QVBandLinearV8R(d, device=DEV)
    assert np.array_equal(ext.ids(P, *lin._core(), T=lin.T).cpu().numpy().astype(np.int64), want)
    Wr = R.reconstruct(d, enc["esc_idx"].cpu().numpy(), enc["esc_vals"].cpu().numpy())
    assert np.array_equal(lin.dense(torch.float32).cpu().numpy().view(np.uint32), Wr.view(np.uint32))
    for dtype in (torch.float32, torch.float16, torch.bfloat16):
        for M in (1, 5, 33):
            x = torch.randn(M, P, generator=torch.Generator().manual_seed(M)).to(dtype).to(DEV)
            xs = x.float().cpu().numpy()
            ref = O.linear_f64(xs, Wr)
            eps = {torch.float32: 0.0, torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}[dtype]
            tol = H.gemv_tolerance(ref, Wr, xs) + eps * np.abs(ref)
            diff = np.abs(lin(x).float().cpu().numpy().astype(np.float64) - ref)
            assert np.all(diff <= tol), (dtype, M, float((diff / tol).max()))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_results_in_the_callers_type(dtype):
    """Rounded by the kernel where nothing is added afterwards: the values of casting the fp32 results, both sides bit for bit."""
    enc = PK.encode_tensor(H.synth_weight(70, 512, seed=4).to(DEV), 2e-3, keep_ids=True)
    assert enc["esc_idx"].numel() == 0
    lin = QVBandLinearV8R(RP.transcode(enc, rows_per_tile=3), device=DEV)
    for M in (1, 2, 17, 48):
        x = torch.randn(M, 512, generator=torch.Generator().manual_seed(M)).to(dtype).to(DEV)
        x[0, 7] = 3.0e4
        y = lin(x)
        assert y.dtype == dtype and torch.equal(y, ext.multi(x, *lin._core(), T=lin.T).to(dtype))
    lin.bias = torch.nn.Parameter(torch.ones(70, device=DEV), requires_grad=False)
    assert torch.equal(lin(x), (ext.multi(x, *lin._core(), T=lin.T) + 1.0).to(dtype))


def test_whole_weight_in_one_chunk_and_in_several():
    """More than 48 rows: the weight restored at once in its rows' own order, or chunk by chunk in the stream's."""
    Q, P, M = 150, 512, 60
    enc = PK.encode_tensor(H.synth_weight(Q, P, seed=9).to(DEV), 2e-3, force_escapes=torch.tensor([3, 700, P * Q - 1]), keep_ids=True)
    d = RP.transcode(enc, rows_per_tile=3)
    lin, several = QVBandLinearV8R(d, device=DEV), type("Several", (QVBandLinearV8R,), dict(CHUNK_BYTES=2 * P * 40))(d, device=DEV)
    assert len(lin.chunks) == 1 and len(several.chunks) > 1
    Wr = O.narrow_fp16(R.reconstruct(d, enc["esc_idx"].cpu().numpy(), enc["esc_vals"].cpu().numpy())).astype(np.float32)
    for dtype in (torch.float32, torch.float16, torch.bfloat16):
        x = torch.randn(M, P, generator=torch.Generator().manual_seed(1)).to(dtype).to(DEV)
        x[2, 5] = 7.0e4 if dtype != torch.float16 else float("inf")                    # becomes 65504
        xs = O.sat_half(x.float().cpu().numpy())
        ref = O.linear_f64(xs, Wr)
        eps = {torch.float32: 0.0, torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}[dtype]
        tol = H.gemv_tolerance(ref, Wr, xs) + eps * np.abs(ref)
        for m in (lin, several):
            diff = np.abs(m(x).float().cpu().numpy().astype(np.float64) - ref)
            finite = np.abs(ref) < (6.5e4 if dtype == torch.float16 else 1e30)
            assert np.all(diff[finite] <= tol[finite]), (dtype, float((diff / tol)[finite].max()))


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
def test_rows_that_want_a_gradient_stay_in_the_graph(dtype):
    """The dense product has no derivative.  A backward through it is refused, as for a call that is part of a larger graph: the rest of
    the graph must not be answered without this product's part.  The values are those of a call without a gradient."""
    lin = QVBandLinearV8R(RP.transcode(PK.encode_tensor(H.synth_weight(64, 256, seed=3).to(DEV), 2e-3, keep_ids=True)), device=DEV)
    x = torch.randn(70, 256, generator=torch.Generator().manual_seed(2)).to(dtype).to(DEV)
    x[1, 2] = 7.0e4
    with torch.no_grad():
        want = lin(x)
    x.requires_grad_()
    y = lin(x)
    assert torch.equal(y.detach(), want) and y.requires_grad
    with pytest.raises(RuntimeError, match="not implemented"):
        (y.float().sum() + x.float().sum()).backward()


@pytest.mark.parametrize("P", [128, 640, 2176, 5120])
def test_sums_of_one_fp32_row_are_taken_in_pairs(P):
    """A weight of one symbol, a power of two, has exact products: each lane adds its columns one by one to the product's sum, and in pairs
    to the sum of x; the lanes meet in a tree.  Bit for bit, so that the error against 64 bits stays what it was."""
    Q = 24
    W = torch.linspace(-0.05, 0.05, Q).to(torch.bfloat16).view(Q, 1).expand(Q, P).contiguous().to(DEV)
    lin = QVBandLinearV8R(RP.transcode(PK.encode_tensor(W, 2e-3, keep_ids=True)), device=DEV)
    ts, dr, mn = (t.cpu().numpy().astype(np.float64) for t in (lin.tau_s, lin.drow, lin.min_s))
    symbols = ext.ids(P, *lin._core(), T=lin.T).cpu().numpy() - dr.reshape(Q, 1)
    c = np.float32(symbols[0, 0])
    assert (symbols == c).all() and (c == 0 or np.log2(c) % 1 == 0)

    def tree(v):
        while v.size > 1:
            v = v[0::2] + v[1::2]
        return np.float64(v[0])

    for seed in range(4):
        x = torch.randn(1, P, generator=torch.Generator().manual_seed(seed)) * 3.0
        sx, acc = np.zeros(32, np.float32), np.zeros(32, np.float32)
        for first, second in x.numpy().reshape(P // 64, 2, 32):          # (pair of steps, step, lane)
            acc = (acc + c * first) + c * second
            sx = sx + (first + second)
        assert sx.dtype == acc.dtype == np.float32
        a, b = tree(acc), tree(sx)
        want = (ts * (a + dr * b) + mn * b).astype(np.float32)
        got = ext.multi(x.to(DEV), *lin._core(), T=lin.T).cpu().numpy()[0]
        # (the double expression may be contracted: its last bit, relative to its largest term)
        room = 2.0 ** -50 * (np.abs(ts) * (abs(a) + np.abs(dr * b)) + np.abs(mn * b))
        lo, hi = ((ts * (a + dr * b) + mn * b + s * room).astype(np.float32) for s in (-1, 1))
        assert np.all((got >= np.minimum(lo, want)) & (got <= np.maximum(hi, want))), (P, seed)


@pytest.mark.parametrize("levels", [6, 256, 257, 700])
@pytest.mark.parametrize("Q,P,T", [(19, 640, 2), (3, 1024, 1), (70, 1152, 3), (9, 4224, 1)])
def test_one_row_of_16_bits_and_symbols_around_a_byte(Q, P, T, levels):
    """A large enough launch on rows of 1024 columns and more takes a class's least symbol off all of them and treats those that fit a byte
    then apart.  Large by a schedule that lists its blocks over and over.  Bound: fp32 sums of P / 32 terms a lane, a tree over the lanes."""
    g = torch.Generator().manual_seed(levels)
    level = torch.randint(0, levels, (Q, P), generator=g)
    level[:, 0], level[:, 1] = 0, levels - 1
    W = (level.float() / levels).to(DEV)
    lin = QVBandLinearV8R(RP.transcode(PK.encode_tensor(W, 0.5 / levels, keep_ids=True), rows_per_tile=T, n_classes=1), device=DEV)
    core = list(lin._core())
    ids = ext.ids(P, *core, T=lin.T).cpu().numpy().astype(np.float64)
    ts, mn = (t.cpu().numpy().astype(np.float64) for t in (lin.tau_s, lin.min_s))
    dense = mn[:, None] + ts[:, None] * ids
    blocks, enough = core[4], 2 ** 17 * torch.cuda.get_device_properties(0).multi_processor_count // (8 * T * P) + 1
    for dtype in (torch.float16, torch.bfloat16):
        x = (torch.randn(1, P, generator=g) + 0.5).to(dtype).to(DEV)
        xs = x.double().cpu().numpy()[0]
        for core[4] in (blocks, blocks.repeat(-(-enough // blocks.shape[0]), 1)):
            got = ext.multi(x, *core, T=lin.T).double().cpu().numpy()[0]
            size = np.abs(xs).sum() * (ts * 2048.0 + np.abs(mn))
            assert np.all(np.abs(got - dense @ xs) <= (P / 32 + 8) * 2.0 ** -24 * size + 2.0 ** -24 * np.abs(got)), (dtype, core[4].shape)
