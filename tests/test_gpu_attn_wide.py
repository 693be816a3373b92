"""Attention of many query rows over the banded KV cache (the kernel of 128 or 256 rows per workgroup) against the oracle, at the sizes
where its tiles change: the fewest rows it takes, one row more than a wave and a workgroup hold, tokens cut across both, key
tiles of one key and of none a row sees, segment changes, 16-bit ids, scores that keep rising (a rescale at every tile) or jump."""
import numpy as np
import pytest
import torch

from oracle import kv_attn_oracle as A
from tests.test_gpu_kv_attn import DEV, check_split_outputs, run_fwd, to_device, vmax
from tests.test_oracle_kv_attn import make_layout
from qvb8_amd import _lib
from qvb8_amd.kv import fused_attn as FA

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,Hkv,G,MQ,seg_len,q_pos0,bits,tps,amp", [
    (256, 2, 6, 6, [33, 1, 70], 98, 6, 2, 1.0), (128, 1, 3, 11, [40], 5, 8, 1, 1.0), (256, 1, 8, 16, [300], 284, 7, 4, 1.0),
    (128, 2, 1, 129, [200, 31], 102, 6, 3, 1.0), (256, 1, 6, 43, [500, 17], -3, 6, 100, 1.0), (128, 3, 8, 33, [64, 64, 3], 98, 11, 2, 1.0),
    (256, 1, 4, 40, [130], 90, 10, 3, 1.0), (128, 4, 6, 24, [321], 297, 7, 2, 40.0), (256, 1, 5, 30, [257], 227, 6, 9, 40.0)])
def test_wide_rows_match_the_oracle(D, Hkv, G, MQ, seg_len, q_pos0, bits, tps, amp):
    lay = make_layout(D + MQ + G, seg_len, Hkv, D, bits=bits)
    rng = np.random.default_rng(MQ)
    q = (rng.normal(0, amp, (MQ, Hkv * G, D)) * D ** -0.5).astype(np.float16)
    want = A.fwd_split(q, lay["ki"], lay["vi"], lay["kmid"], lay["kstep"], lay["vmid"], lay["vstep"], lay["kc"], lay["vc"],
                       lay["ts"], lay["tl"], lay["tseg"], q_pos0, tps, 1.0, G)
    dl = to_device(lay, wide=bits > 8, slack=MQ % 3)
    got = run_fwd(lay, dl, torch.from_numpy(q).to(DEV), q_pos0, tps, G)
    check_split_outputs(got, want, lay)
    ref, ref_lse = A.combine(*want, MQ, G)
    out, lse = (t.cpu().numpy() for t in FA.combine_splits(*[torch.from_numpy(t).to(DEV) for t in got], G))
    assert np.all(np.abs(out - ref) <= 1e-3 * vmax(lay) + 1e-6)
    assert np.array_equal(np.isneginf(lse), np.isneginf(ref_lse))
    seen = np.isfinite(ref_lse)
    assert np.all(np.abs(lse[seen] - ref_lse[seen]) <= 1e-3 * np.abs(ref_lse[seen]) + 1e-3)


@pytest.mark.parametrize("D,Hkv,G,MQ,seg_len,q_pos0,bits,tps,scale", [
    (256, 1, 8, 26, [33, 1, 70], 78, 6, 2, 1.0), (128, 2, 5, 51, [300], 249, 7, 4, 1.0), (256, 2, 8, 32, [40, 64], -3, 6, 1, 1.0), (128, 1, 1, 257, [90], 20, 8, 3, 1.0),
    (256, 1, 6, 72, [130, 31], 89, 8, 100, 0.4), (128, 1, 8, 64, [64, 64, 3], 67, 6, 2, 1.0), (256, 1, 4, 64, [97], 33, 7, 2, -0.5), (256, 1, 8, 27, [45], 18, 6, 1, 0.0)])
def test_workgroups_of_256_rows_match_the_oracle(D, Hkv, G, MQ, seg_len, q_pos0, bits, tps, scale):
    """208 (the fewest of them), 216, 255, 256 and 257 (too few for two) rows, blocks with empty waves, rows that see no key, one split of
    every tile; a scale that is not positive is multiplied before the maximum is taken.  Splits without a tile make up the number of
    workgroups from which that kernel takes over; once without them, for the other kernel."""
    lay = make_layout(D + MQ + G, seg_len, Hkv, D, bits=bits)
    rng = np.random.default_rng(MQ)
    q = (rng.normal(0, 1, (MQ, Hkv * G, D)) * D ** -0.5).astype(np.float16)
    want = A.fwd_split(q, lay["ki"], lay["vi"], lay["kmid"], lay["kstep"], lay["vmid"], lay["vstep"], lay["kc"], lay["vc"],
                       lay["ts"], lay["tl"], lay["tseg"], q_pos0, tps, scale, G)
    dl, q16 = to_device(lay, slack=MQ % 3), torch.from_numpy(q).to(DEV)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    for empty in (512 // Hkv, 0):
        block = _lib.load().qvb8_attn_rows_per_workgroup(MQ * G, want[0].shape[0] + empty, Hkv, 1, cus)
        assert block == (256 if empty and MQ * G != 257 else 128)
        o, m, l = (torch.full((w.shape[0] + empty,) + w.shape[1:], float("nan"), device=DEV) for w in want)
        FA.fwd(q16, dl["ki"], dl["vi"], dl["kmid"], dl["kstep"], dl["vmid"], dl["vstep"], dl["kc"], dl["vc"], dl["ts"], dl["tl"], dl["tseg"], o, m, l, q_pos0, tps, scale, G)
        S = want[0].shape[0]
        check_split_outputs((o[:S].cpu().numpy(), m[:S].cpu().numpy(), l[:S].cpu().numpy()), want, lay)
        assert torch.isneginf(m[S:]).all() and (l[S:] == 0).all() and (o[S:] == 0).all()


def test_combining_many_rows_is_combining_few():
    """3 splits of 300 rows x 4 heads (a thread per four channels) against the CPU's combination, rows without a key among them."""
    g = torch.Generator().manual_seed(2)
    S, h, rows, d, G = 3, 4, 300, 256, 6
    o, m = torch.randn(S, h, rows, d, generator=g), 3 * torch.randn(S, h, rows, generator=g)
    l = torch.rand(S, h, rows, generator=g) + 0.5
    m[0, 1], l[0, 1], o[0, 1] = -float("inf"), 0, 0
    m[:, 2, 7:19], l[:, 2, 7:19], o[:, 2, 7:19] = -float("inf"), 0, 0
    out, lse = FA.combine_splits(o.to(DEV), m.to(DEV), l.to(DEV), G)
    ref, ref_lse = A.combine(o.numpy(), m.numpy(), l.numpy(), rows // G, G)
    assert np.allclose(out.cpu().numpy(), ref, rtol=1e-5, atol=1e-5) and np.allclose(lse.cpu().numpy(), ref_lse, rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("D,Hkv,G,MQ,n,bits", [(256, 2, 6, 40, 4000, 7), (128, 2, 8, 32, 3000, 6), (256, 1, 6, 6, 2500, 10)])
def test_no_further_from_64_bits_than_the_row_block_kernel(D, Hkv, G, MQ, n, bits, monkeypatch):
    """One long split, so that the running maximum keeps rising.  Both kernels round keys, values and probabilities to fp16 and
    sum in fp32; with every probability rounded relative to the same running maximum their errors (5.6e-4 here) differ by the fp32
    order of sums only, 1e-6 of the result = 2e-3 of the error at most.  A maximum that lags behind costs 1 .. 2.5 % of it."""
    lay = make_layout(7 * D + MQ, [n], Hkv, D, bits=bits)
    rng = np.random.default_rng(n)
    q = (rng.normal(0, 1, (MQ, Hkv * G, D)) * D ** -0.5).astype(np.float16)
    dl = to_device(lay, wide=bits > 8)
    K, V = ((lay[m][0][None].astype(np.float64) + lay[s][0][None] * (lay[i].astype(np.float64) - lay[c][0][None, :, None]))
            for i, m, s, c in (("ki", "kmid", "kstep", "kc"), ("vi", "vmid", "vstep", "vc")))
    exact = np.empty((MQ, Hkv * G, D))
    for h in range(Hkv * G):
        s = q[:, h].astype(np.float64) @ K[:, h // G].T
        s[np.arange(n)[None] > n - MQ + np.arange(MQ)[:, None]] = -np.inf
        p = np.exp(s - s.max(1, keepdims=True))
        exact[:, h] = p @ V[:, h // G] / p.sum(1, keepdims=True)

    def error():
        got = run_fwd(lay, dl, torch.from_numpy(q).to(DEV), n - MQ, 1 << 20, G)
        out, _ = FA.combine_splits(*[torch.from_numpy(t).to(DEV) for t in got], G)
        return np.linalg.norm(out.cpu().numpy() - exact) / np.linalg.norm(exact)

    wide = error()
    monkeypatch.setenv("QVB8_ATTN_ROW_BLOCKS", "1")
    assert wide <= 1.002 * error()
