"""The kernel of 17..64 rows of X whose waves take columns of their own (csrc/qvb8_columns.hip), at the sizes where it can go wrong: against the
oracle in float64, and bit for bit between the ways a weight's rows can be stored."""
import numpy as np
import pytest
import torch

from oracle import qvb8_oracle as O
from qvb8_amd import ext_qvb8 as ext
from tests import helpers as H
from tests.test_gpu_qvb8_mma import _sorted_pack, _sorted_planes, _x

pytestmark = pytest.mark.gpu

# rows of X at the edges of the token tiles; Q: a tile, whole tiles, a rest of 1 or 15 rows, runs that start inside a tile; P: one
# step, fewer steps than waves, an odd number of rounds, the most steps; more rows of X than 32 with column ranges (17000 x 4096, 64 rows)
SIZES = [(17, 16, 128, [7]), (32, 31, 1024, [4]), (33, 17, 1152, [8]), (48, 1000, 384, [5, 6, 7]), (49, 257, 2304, [6, 7]), (64, 333, 4096, [4, 6, 8]),
         (40, 95, 3328, [5]), (20, 4111, 256, [6, 7]), (64, 6145, 512, [7]), (31, 12300, 128, [6, 7]), (64, 17000, 4096, [7])]


def _float64(d, x, saturate):
    W = O.reconstruct(d["min_s"], d["tau_s"], d["ids_dense"], d["esc_idx"], d["esc_vals"])
    xs = x.float().cpu().numpy()
    xs = O.sat_half(xs) if saturate else xs
    return O.linear_f64(xs, W), W, xs


@pytest.mark.parametrize("M,Q,P,widths", SIZES)
def test_products_against_float64_and_across_storages(M, Q, P, widths):
    d = H.mixed_width_pack(Q, P, widths, seed=Q + P)
    d["tau_s"] = d["tau_s"] * (1.0 / 64)
    packs = [_sorted_pack(d), _sorted_planes(d)]
    for dtype in (torch.float16, torch.bfloat16):
        x = _x(M, P, dtype, M)
        got = [ext.mma_tiles(x, *args, perm=perm, rowinfo=rowinfo, layout=layout, planes=planes)
               for planes, (args, perm, rowinfo, layout) in enumerate(packs)]
        assert torch.equal(*got)
        ref, W, xs = _float64(d, x, dtype == torch.bfloat16)
        assert np.all(np.abs(got[0].cpu().numpy().astype(np.float64) - ref) <= H.gemv_tolerance(ref, W, xs))


def test_values_outside_fp16_and_nan_stay_in_their_row():
    d = H.mixed_width_pack(272, 1024, [6, 7], seed=3)
    args, perm, rowinfo, layout = _sorted_planes(d)
    x = _x(40, 1024, torch.bfloat16, 5)
    x[3, 100], x[17, 5], x[39, 1023] = 1e38, float("-inf"), float("nan")
    y = ext.mma_tiles(x, *args, perm=perm, rowinfo=rowinfo, layout=layout, planes=True).cpu()
    ref, W, xs = _float64(d, x[:39], True)
    assert bool(y[39].isnan().all()) and np.all(np.abs(y[:39].numpy().astype(np.float64) - ref) <= H.gemv_tolerance(ref, W, xs))


def test_a_run_of_a_large_weight_is_whole_workgroups():
    from qvb8_amd.formats.qvb8.module import QVBandLinearV8, _run_multiple
    from qvb8_amd.formats.qvb8 import pack as PK
    assert [_run_multiple(q) for q in (100, 8191, 8192, 12288, 40000)] == [16, 16, 32, 192, 192]
    enc = PK.encode_tensor(H.synth_weight(12299, 128, seed=1).cuda(), 1e-3)
    dense = ext.decode_f32(*H.pack_args(enc))
    lin = QVBandLinearV8.from_encoded(enc).prepare()
    layout = lin._mma_order()[2]
    assert all(int(layout.first_pos[c]) % 192 == 0 for c in range(int(layout.n_classes)))
    assert torch.equal(dense, ext.decode_f32(lin.ids, lin.min_s, lin.nbits, lin.bit_off, 128, lin.tau_s, lin.esc_idx, lin.esc_vals))
