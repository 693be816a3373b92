"""GPU tests of the one-call attention (qvb8_attend): the queries prepared where they are read, the splits joined in one pass -- against
the separate calls on the same splits and the CPU's combination, for every kernel and query type."""
import ctypes

import numpy as np
import pytest
import torch

from oracle import kv_attn_oracle as A
from qvb8_amd import _lib
from qvb8_amd.kv import fused_attn as FA
from tests.test_gpu_kv_attn import DEV, to_device
from tests.test_oracle_kv_attn import make_layout

pytestmark = pytest.mark.gpu


def _lay(lay, dl, wide):
    seg = [int(n) for n in np.bincount(lay["tseg"], weights=lay["tl"]).astype(int)]
    return FA.QVLayout(dl["ki"], dl["vi"], dl["kmid"], dl["kstep"], dl["vmid"], dl["vstep"], seg, DEV, kc=dl["kc"], vc=dl["vc"])


@pytest.mark.parametrize("D,Hkv,G,MQ,seg_len,bits", [(128, 2, 4, 1, [70, 33], 6), (256, 2, 6, 4, [300], 7), (256, 1, 6, 9, [200, 17], 6),
                                                      (128, 2, 8, 40, [500], 7), (256, 1, 4, 2, [90], 11), (128, 1, 1, 1, [1], 6)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
def test_one_call_is_the_separate_calls(D, Hkv, G, MQ, seg_len, bits, dtype):
    lay = make_layout(D + MQ, seg_len, Hkv, D, bits=bits)
    lq = _lay(lay, to_device(lay, wide=bits > 8), bits > 8)
    n, scale = sum(seg_len), D ** -0.5
    q = torch.randn(MQ, Hkv * G, D, generator=torch.Generator().manual_seed(n)).to(dtype).to(DEV)
    q[0, 0, 3] = 60000.0
    if dtype != torch.float16:
        q[0, 0, 5] = 3.0e7                                             # saturates once the scale is in
    for n_splits in (None, 1, 3):
        out, lse = FA.attend(q, lq, n - MQ, scale, n_splits=n_splits)
        tps, S = FA.plan_splits(lq.n_tiles, Hkv, MQ * G, DEV, d=D, wide=bits > 8) if n_splits is None else (-(-lq.n_tiles // n_splits), None)
        S = S or -(-lq.n_tiles // tps)
        q16 = torch.empty(q.shape, dtype=torch.float16, device=DEV)
        lib = _lib.load()
        _lib._check(lib.qvb8_scale_sat_half(q.data_ptr(), _lib.dtype_code(dtype), q.numel(), scale, q16.data_ptr(), _lib.stream_of(q)), lib)
        o = torch.empty(S, Hkv, MQ * G, D, device=DEV)
        m, l = torch.empty(S, Hkv, MQ * G, device=DEV), torch.empty(S, Hkv, MQ * G, device=DEV)
        FA.fwd(q16, lq.ki, lq.vi, lq.kmin, lq.kstep, lq.vmin, lq.vstep, lq.kc, lq.vc, lq.t_start, lq.t_len, lq.t_seg, o, m, l, n - MQ, tps, 1.0, G)
        want, want_lse = FA.combine_splits(o, m, l, G)
        assert torch.equal(out, want) and torch.equal(lse, want_lse)
        ref, ref_lse = A.combine(o.cpu().numpy(), m.cpu().numpy(), l.cpu().numpy(), MQ, G)
        assert np.allclose(out.cpu().numpy(), ref, rtol=1e-5, atol=1e-5) and np.allclose(lse.cpu().numpy(), ref_lse, rtol=1e-5, atol=1e-5)
    # a view that is not aligned to four elements, and one with other strides
    flat = torch.empty(q.numel() + 1, dtype=dtype, device=DEV)
    flat[1:] = q.reshape(-1)
    odd = flat[1:].view(q.shape)
    turned = q.transpose(0, 1).contiguous().transpose(0, 1)
    for view in (odd, turned):
        assert torch.equal(FA.attend(view, lq, n - MQ, scale, n_splits=3)[0], out)


# (a thread, a wave and four waves a unit; one split too few, exact and one too many for each way of taking them)
@pytest.mark.parametrize("S,rows", [(1, 6), (8, 6), (9, 6), (64, 6), (65, 6), (256, 6), (257, 6), (700, 6), (18, 63), (65, 63), (24, 160), (64, 160), (65, 160), (129, 160),
                                    (17, 150), (18, 150), (29, 330), (7, 660), (64, 660)])
def test_splits_joined_in_one_pass(S, rows):
    """Rows without a visible key in some splits and in all, partial results a few powers of e apart."""
    g = torch.Generator().manual_seed(S)
    h, d, G = 2, 256 if rows == 63 else 128, 1 if rows % 3 else 3
    o, m = torch.randn(S, h, rows, d, generator=g), 20 * torch.randn(S, h, rows, generator=g)
    l = torch.rand(S, h, rows, generator=g) + 0.5
    m[S // 2:, 0, 1], l[S // 2:, 0, 1], o[S // 2:, 0, 1] = -float("inf"), 0, 0
    m[:, 1, 2], l[:, 1, 2], o[:, 1, 2] = -float("inf"), 0, 0
    out, lse = (t.cpu().numpy() for t in FA.combine_splits(o.to(DEV), m.to(DEV), l.to(DEV), G))
    ref, ref_lse = A.combine(o.double().numpy(), m.double().numpy(), l.double().numpy(), rows // G, G)
    assert np.array_equal(np.isneginf(lse), np.isneginf(ref_lse))
    assert np.allclose(out, ref, rtol=1e-5, atol=2e-5) and np.allclose(lse[np.isfinite(lse)], ref_lse[np.isfinite(ref_lse)], rtol=1e-5, atol=1e-5)


def test_refusals():
    lay = make_layout(3, [64], 1, 128)
    dl = to_device(lay)
    lq = _lay(lay, dl, False)
    q = torch.zeros(1, 2, 128, device=DEV)
    lib = _lib.load()
    ws = torch.empty(4096, device=DEV)
    args = [q.data_ptr(), 0, 1.0, 256, 128, lq.ki.data_ptr(), lq.vi.data_ptr(), 1, lq.ki.stride(0), lq.ki.stride(1),
            *[p.data_ptr() for p in (lq.kmin, lq.kstep, lq.vmin, lq.vstep, lq.kc, lq.vc, lq.t_start, lq.t_len, lq.t_seg)], 2, 2, 2, 1, 128, 63, 1, 2,
            ws.data_ptr(), ws.data_ptr(), ws.data_ptr(), ws.numel() * 4, _lib.stream_of(q)]
    for at, bad in ((1, 7), (0, q.data_ptr() + 4), (23, 64), (30, 100), (29, None)):
        wrong = list(args)
        wrong[at] = bad
        assert lib.qvb8_attend(*wrong) != 0 and ctypes.string_at(lib.qvb8_last_error())
