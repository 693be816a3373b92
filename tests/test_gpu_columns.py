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

# rows of X at the edges of the token tiles; Q: a tile, whole tiles, a rest of 1 or 15 rows, runs that start inside a tile (no lane's row is where its
# tile says); P: one step, fewer steps than waves, an odd number of rounds, the most steps
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


def _cost(units, token_tiles, group, steps):
    """What csrc/qvb8_columns.hip reckons a call takes with `group` row tiles a workgroup."""
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    rounds = -(-units // cus)
    return rounds * (700 + -(-steps // 8) * max(68 * group * min(units, rounds * cus) // (rounds * cus), 62 * token_tiles, 22 * group + 6 * group * token_tiles))


def _instance(M, P, runs):
    """(token tiles, row tiles a workgroup) of the kernel that takes such runs of whole tiles in planes."""
    MT = 2 if M <= 32 else 3 if M <= 48 else 4
    groups = [g for g in (1, 2, 3, 4, 6, 8) if g <= (8 if MT == 2 else 6)]
    units = {g: sum(-(-(n // 16) // g) for n in runs) + (sum(runs) % 16 > 0) for g in groups}
    return MT, min(groups, key=lambda g: _cost(units[g], MT, g, P // 128))


# Rows as a loaded weight has them: every run but the last whole tiles, so that the tiles' places follow from their numbers; one size for each
# instance of the kernel, with one step a wave and with a second for some of them
RUNS = [((2, 1), 25, 1152, [16, 16, 4]), ((2, 2), 17, 384, [6720, 1152, 145]), ((2, 3), 32, 384, [1872, 1680, 4475]), ((2, 4), 17, 384, [4288, 1792, 2234]),
        ((2, 6), 32, 384, [8032, 848, 3359]), ((2, 8), 32, 384, [1360, 7904, 7034]), ((3, 1), 48, 1152, [16, 16, 2]), ((3, 2), 48, 384, [6512, 784, 721]),
        ((3, 3), 47, 384, [880, 3504, 3761]), ((3, 4), 47, 384, [7936, 1472, 1801]), ((3, 6), 48, 384, [11088, 1232, 2008]), ((4, 1), 57, 512, [16, 16, 4]),
        ((4, 2), 49, 512, [1968, 1248, 881]), ((4, 3), 49, 512, [3312, 3536, 1297]), ((4, 4), 49, 512, [9568, 2080, 553]), ((4, 6), 57, 512, [10192, 1040, 5027])]


@pytest.mark.parametrize("instance,M,P,runs", RUNS)
def test_runs_of_whole_tiles_in_planes(instance, M, P, runs, monkeypatch):
    assert _instance(M, P, runs) == instance
    widths = {1: (5, 6, 7), 2: (4, 7, 8), 3: (5, 6, 8), 4: (6, 7, 8), 6: (4, 5, 6), 8: (5, 7, 8)}[instance[1]]
    rows = np.random.default_rng(M).permutation(np.repeat(widths, runs))
    d = H.mixed_width_pack(len(rows), P, rows.tolist(), seed=P)
    d["tau_s"] = d["tau_s"] * (1.0 / 64)
    x = _x(M, P, torch.bfloat16, M)
    packs = [_sorted_pack(d), _sorted_planes(d)]
    call = lambda pack, planes, **kw: ext.mma_tiles(x, *pack[0], perm=pack[1], rowinfo=pack[2], layout=pack[3], planes=planes, **kw)   # noqa: E731
    assert [packs[1][3].first_pos[c] for c in range(3)] == [0, runs[0], runs[0] + runs[1]]
    got = call(packs[1], True)
    assert torch.equal(got, call(packs[0], False))
    assert torch.equal(got.half(), call(packs[1], True, out_dtype=torch.float16))
    ref, W, xs = _float64(d, x, True)
    far = lambda y: np.linalg.norm(y.cpu().numpy().astype(np.float64) - ref) / np.linalg.norm(ref)                # noqa: E731
    assert np.all(np.abs(got.cpu().numpy().astype(np.float64) - ref) <= H.gemv_tolerance(ref, W, xs))
    # the kernels it stands in for answer otherwise, and no nearer to 64 bits
    monkeypatch.setenv("QVB8_COLUMNS", "0")
    other = call(packs[1], True)
    assert not torch.equal(other, got) and far(got) < far(other)


@pytest.mark.parametrize("M", [17, 40, 64])
def test_a_weight_as_it_is_loaded(M, monkeypatch):
    """Rows of three widths, widened to whole workgroups at load, some with escapes: in planes, and back to back as they came (a widened row's
    middle is another one, so sums round differently), the products of the restored weight in float64."""
    from qvb8_amd.formats.qvb8.module import QVBandLinearV8
    from qvb8_amd.formats.qvb8 import pack as PK
    Q, P = 12299, 1280
    gen = torch.Generator(device="cuda").manual_seed(3)
    scale = torch.tensor([0.007, 0.014, 0.027], device="cuda")[torch.arange(Q, device="cuda") % 3, None]
    enc = PK.encode_tensor((scale * torch.randn(Q, P, device="cuda", generator=gen)).bfloat16(), 1e-3, force_escapes=[5, Q * P // 2, Q * P - 1])
    W = ext.decode_f32(*H.pack_args(enc)).double()
    x = _x(M, P, torch.float16, M)
    want = x.double() @ W.t()
    for planes in ("1", "0"):
        monkeypatch.setenv("QVB8_PLANES", planes)
        lin = QVBandLinearV8.from_encoded(enc).prepare()
        layout = lin._mma_order()[2]
        assert lin._planes == (planes == "1") and int(layout.n_classes) == 3
        assert float((lin(x).double() - want).norm() / want.norm()) < 2 ** -11          # one rounding to fp16


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
