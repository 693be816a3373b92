"""The dense restore along the row records and the activation narrowing, bit for bit against what they stand for."""
import numpy as np
import pytest
import torch

from oracle import qvb8_oracle as O
from qvb8_amd import ext_qvb8 as ext
from qvb8_amd.formats.qvb8 import pack as PK
from qvb8_amd.formats.qvb8.module import QVBandLinearV8
from tests.helpers import mixed_width_pack, oracle_ids, to_device_args

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# whole tiles in planes and rows that are not (rest of a run, widths 3 and 9, 14), one step and several chunks of columns
@pytest.mark.parametrize("Q,P,widths,planes", [(16, 128, [7], True), (47, 384, [4, 6, 8], True), (200, 2176, [5, 7], True), (33, 256, [3, 5, 9, 14, 8], False),
                                               (1, 128, [6], True), (130, 4096, [8, 7, 6], True)])
def test_restore_by_row_records(Q, P, widths, planes):
    d = mixed_width_pack(Q, P, widths, seed=Q)
    ids, mn, nb, off, _, ts, ei, ev = to_device_args(d, DEV)
    perm = torch.argsort(nb.to(torch.int16), stable=True).to(torch.int32)
    if planes:
        ids, off, _ = ext.sort_rows_by_width(ids, nb, off, P, perm, planes=True)
    rowinfo = ext.mma_prepare(nb, off, ts, mn, P, ids.numel(), perm)
    W = O.reconstruct(d["min_s"], d["tau_s"], oracle_ids(d), d["esc_idx"], d["esc_vals"])
    want = torch.from_numpy(np.ascontiguousarray(W))
    got = ext.decode(ids, mn, nb, off, P, ts, ei, ev, rowinfo).cpu()
    assert torch.equal(got.view(torch.int16), want.to(torch.float16).view(torch.int16))
    got = ext.decode_bf16(ids, mn, nb, off, P, ts, ei, ev, rowinfo).cpu()
    assert torch.equal(got.view(torch.int16), want.to(torch.bfloat16).view(torch.int16))
    bad = off.clone()
    bad[Q // 2] = 8 * ids.numel()                                 # metadata outside the buffer: that row is NaN, the others are not touched
    got = ext.decode(ids, mn, nb, bad, P, ts, ei, ev, ext.mma_prepare(nb, bad, ts, mn, P, ids.numel(), perm)).cpu()
    assert bool(got[Q // 2].isnan().all()) and int(got.isnan().any(1).sum()) == 1


@pytest.mark.parametrize("n,skip", [(1, 0), (7, 0), (8, 0), (2049, 0), (4096, 1), (5000, 8)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
def test_narrowing_of_any_length_and_alignment(n, skip, dtype):
    x = (torch.randn(n + skip, generator=torch.Generator().manual_seed(n)) * 3e4).to(dtype)
    x[skip:][::5] = torch.tensor([float("nan"), float("inf"), -float("inf"), 65519.0, -7e4]).to(dtype).repeat(-(-n // 5) // 5 + 1)[:-(-n // 5)]
    got = ext.saturating_half(x.to(DEV)[skip:]).cpu()
    want = x[skip:] if dtype == torch.float16 else x[skip:].float().clamp(-65504, 65504).half()
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.nan_to_num(), want.nan_to_num())


@pytest.mark.parametrize("x", [torch.float16, torch.bfloat16])
def test_constants_rewritten_after_prepare_are_honoured(x):
    """More than 256 rows restore the weight: row constants changed in place since prepare() count, as they do when the
    weight has no row records."""
    Q, P, M = 272, 1024, 300
    enc = PK.encode_tensor((0.02 * torch.randn(Q, P, generator=torch.Generator().manual_seed(1))).to(torch.bfloat16).to(DEV), 1e-3)
    mod = QVBandLinearV8.from_encoded(enc).prepare()
    assert mod._planes
    X = torch.randn(M, P, generator=torch.Generator().manual_seed(2)).to(x).to(DEV)
    other = QVBandLinearV8.from_encoded(dict(enc, min_s=enc["min_s"] - 0.01, tau_s=enc["tau_s"] * 1.5))
    assert other.__dict__.get("_mma_cache") is None              # restored row by row
    before = mod(X)
    with torch.no_grad():
        mod.min_s.sub_(0.01), mod.tau_s.mul_(1.5)
    now = mod(X)
    assert not torch.equal(now, before) and torch.equal(now, other(X))
