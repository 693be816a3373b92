"""Host logic of the banded KV cache on the CPU: the codec (bit packing, widths, certificate, truncation) and the id layout
with its tile table, against the oracle's restatement.  No kernel is called."""
import numpy as np
import pytest
import torch

from oracle import kv_attn_oracle as A
from qvb8_amd.kv import codec as C
from qvb8_amd.kv import fused_attn as FA


@pytest.mark.parametrize("bits,n", [(1, 9), (4, 64), (6, 1000), (7, 77), (8, 5), (11, 333), (16, 40)])
def test_pack_ids_is_lsb_first_and_round_trips(bits, n):
    g = torch.Generator().manual_seed(bits * 100 + n)
    ids = torch.randint(0, 1 << bits, (n,), generator=g)
    packed = C.pack_ids(ids, bits)
    assert packed.dtype == torch.uint8 and packed.numel() == (n * bits + 7) // 8
    assert torch.equal(C.unpack_ids(packed, bits, n), ids)
    # the same bytes as the weight format's bit packing of one row (LSB first, fields back to back)
    from oracle import qvb8_oracle as O
    want = O.pack_bits_rows(ids.numpy()[None, :], np.array([bits]))
    buf = want[0] if isinstance(want, tuple) else want
    assert np.array_equal(packed.numpy(), np.asarray(buf)[:packed.numel()])


def test_known_bytes_of_three_bit_ids():
    ids = torch.tensor([1, 2, 3, 4, 5, 6, 7, 0])
    assert C.pack_ids(ids, 3).tolist() == [0xD1, 0x58, 0x1F]


def test_band_kv_heads_matches_the_oracle_codec_on_the_cpu():
    torch.manual_seed(4)
    x = (torch.randn(3, 50, 32) * torch.rand(3, 1, 32) * 4).to(torch.bfloat16)
    x[1, :, 5] = 0.75                                                # a constant channel
    for bits, tau in ((6, 0.0), (4, 0.05), (6, 0.003)):
        got = C.band_kv_heads(x, torch.bfloat16, bits, tau=tau)
        want = A.band_kv(x.float().numpy(), bits, tau, "bf16")
        for h, (bk, (ids, mn, step, b)) in enumerate(zip(got, want)):
            assert bk.bits == b and bk.orig_shape == (50, 32) and bk.orig_dtype == torch.bfloat16
            assert np.array_equal(bk.min_s.numpy(), mn) and np.array_equal(bk.tau_s.numpy(), step)
            assert np.array_equal(bk.ids().numpy(), ids)
            assert bk.nbytes() == (50 * 32 * b + 7) // 8 + 8 * 32
            if tau > 0:
                assert float((bk.decode_all_torch(dtype=torch.bfloat16).float() - x[h].float()).abs().max()) <= tau
            assert np.array_equal(bk.decode_all_torch().numpy(), A.decode_kv(ids, mn, step))
            cut = bk.truncate(7)
            assert cut.orig_shape == (7, 32) and torch.equal(cut.ids(), bk.ids()[:7]) and bk.truncate(50) is bk
            with pytest.raises(ValueError):
                bk.truncate(0)
    assert got[1].ids()[:, 5].abs().max() == 0
    with pytest.raises(C.KVCertificateError):
        C.band_kv_heads(torch.tensor([[[0.0], [1.1], [3e4]]]), torch.float32, 6, tau=1e-9)       # 16 bits: steps of 0.46


def test_layout_and_tile_table_from_segments():
    torch.manual_seed(6)
    seg_len = [40, 9, 64]
    segs_k = [C.band_kv_heads(torch.randn(2, sl, 128).to(torch.bfloat16), torch.bfloat16, 6, tau=0.1) for sl in seg_len]
    segs_v = [C.band_kv_heads(torch.randn(2, sl, 128).to(torch.bfloat16), torch.bfloat16, 5) for sl in seg_len]
    lay = FA.layout_from_segments(segs_k, segs_v, seg_len, "cpu")
    assert lay.ki.shape == (113, 2, 128) and lay.ki.dtype == torch.uint8 and lay.n == 113
    ts, tl, tseg = A.tile_table(seg_len)
    assert np.array_equal(lay.t_start.numpy(), ts) and np.array_equal(lay.t_len.numpy(), tl) and np.array_equal(lay.t_seg.numpy(), tseg)
    assert lay.n_tiles == 2 + 1 + 2 and int(lay.t_len.max()) <= FA.BLOCK_N
    pos = 0
    for si, sl in enumerate(seg_len):
        for h in range(2):
            bk = segs_k[si][h]
            mid, step, c = A.centre_form(bk.min_s.numpy(), bk.tau_s.numpy(), bk.bits)
            assert np.array_equal(lay.kmin[si, h].numpy(), mid) and np.array_equal(lay.kstep[si, h].numpy(), step) and float(lay.kc[si, h]) == c
            assert torch.equal(lay.ki[pos:pos + sl, h].to(torch.int64), bk.ids())
            assert float(lay.vc[si, h]) == (2 ** segs_v[si][h].bits - 1) / 2
        pos += sl
    with pytest.raises(ValueError):
        FA.QVLayout(lay.ki, lay.vi, lay.kmin, lay.kstep, lay.vmin, lay.vstep, seg_len, "cpu", block_n=64)
    # more than 8 bits: no byte layout; on request 16-bit patterns in int16
    tight = C.band_kv_heads((torch.randn(1, 16, 128) * 4).to(torch.bfloat16), torch.bfloat16, 6, tau=0.004)
    assert tight[0].bits > 8 and FA.layout_from_segments([tight], [tight], [16], "cpu") is None
    wide = FA.layout_from_segments([tight], [tight], [16], "cpu", allow_wide=True)
    assert wide.ki.dtype == torch.int16
    assert torch.equal(wide.ki[:, 0].to(torch.int64) & 0xFFFF, tight[0].ids())


def test_split_planner_rules():
    assert FA.rows_per_workgroup(6, 256) == 16 and FA.rows_per_workgroup(24, 256) == 32 and FA.rows_per_workgroup(96, 256) == 32
    assert FA.rows_per_workgroup(96, 128) == 64 and FA.rows_per_workgroup(17, 128) == 32


def test_take_rows_and_unband_keep_every_value():
    torch.manual_seed(8)
    x = torch.randn(2, 30, 16).to(torch.bfloat16)
    heads = C.band_kv_heads(x, torch.bfloat16, 6, tau=0.1)
    full = C.unband_kv_4d(heads, 1, 2)
    assert full.shape == (1, 2, 30, 16) and full.dtype == torch.bfloat16
    assert float((full[0].float() - x.float()).abs().max()) <= 0.1
    rows = torch.tensor([0, 3, 4, 29])
    sub = heads[0].take_rows(rows)
    assert sub.orig_shape == (4, 16) and sub.bits == heads[0].bits and sub.min_s is heads[0].min_s
    assert torch.equal(sub.decode_all(), heads[0].decode_all()[rows])          # the same values, bit for bit
    assert torch.equal(heads[0].decode_row(3), heads[0].decode_all()[3])
    assert heads[0].take_rows(torch.arange(30)) is heads[0] and heads[0].outlier_count == 0
    with pytest.raises(ValueError):
        heads[0].take_rows(torch.tensor([30]))
    assert C.unband_kv_4d([], 1, 2).shape == (1, 2, 0, 0)


def test_only_whole_heads_go_to_the_unpacking_kernel():
    """The kernel reads seq * dim * bits bits and dim constants without looking at lengths: a head that holds fewer, or in
    another type, must not reach it (the general path refuses a short stream)."""
    import dataclasses
    import types
    g = torch.Generator().manual_seed(3)
    bk = C.band_kv_heads(torch.randn(1, 40, 32, generator=g), torch.float32, 6)[0]
    here = types.SimpleNamespace(index=-1)                       # what get_device() says of a CPU tensor
    reads = lambda **change: FA._kernel_reads(dataclasses.replace(bk, **change), 40, 32, here)       # noqa: E731
    assert reads()
    assert not reads(packed=bk.packed[:-1].clone()) and not reads(bits=7) and not reads(bits=0)
    assert not reads(packed=bk.packed.to(torch.int32)) and not reads(packed=torch.cat([bk.packed] * 2)[::2])
    assert not reads(min_s=bk.min_s[:-1].clone()) and not reads(tau_s=bk.tau_s.double()) and not reads(tau_s=bk.tau_s[:1].expand(32))
    assert not FA._kernel_reads(bk, 41, 32, here) and not FA._kernel_reads(bk, 40, 33, here)
    short = dataclasses.replace(bk, packed=bk.packed[:-1].clone())
    with pytest.raises(RuntimeError):
        FA.layout_from_segments([[short]], [[bk]], [40], "cpu")


def lengths_and_segments_must_match(device):
    seg = C.band_kv_heads(torch.randn(2, 40, 32, generator=torch.Generator().manual_seed(3)).to(device), torch.float32, 6)
    two = [seg, seg]
    for k, v, lens in ((two, two, [40]), (two, [seg], [40, 40]), ([seg], [seg], [40, 40]), (two, two, [])):
        with pytest.raises(IndexError):
            FA.layout_from_segments(k, v, lens, device)
    whole = FA.layout_from_segments(two, two, [40, 40], device)
    padded = FA.layout_from_segments(two, two, [40, 40, 0], device)              # an empty segment more: no tiles
    assert whole.n == 80 and torch.equal(padded.ki, whole.ki) and torch.equal(padded.t_seg, whole.t_seg) and padded.n_tiles == whole.n_tiles


def test_lengths_and_segments_must_match():
    lengths_and_segments_must_match("cpu")


def test_split_plans(monkeypatch):
    """As many splits as workgroups fit the card at once, by the kernel that takes the rows; a forced row-block kernel is planned
    for as such."""
    import types
    monkeypatch.setattr(torch.cuda, "get_device_properties", lambda device: types.SimpleNamespace(multi_processor_count=256))
    monkeypatch.delenv("QVB8_ATTN_WG_PER_CU", raising=False)
    monkeypatch.delenv("QVB8_ATTN_ROW_BLOCKS", raising=False)
    plan = lambda rows, **kw: FA.plan_splits(4096, 4, rows, "cuda", **kw)                  # noqa: E731
    assert plan(16) == (22, 187) and plan(32) == (32, 128)                       # 3 and 2 workgroups on each of 256 CUs, over 4 heads
    assert plan(33) == plan(128) == (32, 128) and plan(129) == (64, 64)          # 128 rows share a workgroup
    assert plan(33, d=128) == (22, 187) and plan(33, wide=True) == (64, 64)
    short = lambda rows: FA.plan_splits(188, 2, rows, "cuda")[0]                 # noqa: E731
    assert short(512) == short(520) == 8 and short(120) == 3                     # short splits: no step where a fifth row block begins
    monkeypatch.setenv("QVB8_ATTN_ROW_BLOCKS", "1")
    assert plan(33) == (64, 64) and plan(96) == (128, 32)                        # 16 rows: 3 and 6 row blocks
    monkeypatch.setenv("QVB8_ATTN_ROW_BLOCKS", "4")
    assert plan(33, d=128) == (32, 128) and plan(33) == (64, 64)                 # 64 rows; 256 channels: 32 at most


@pytest.mark.parametrize("cus", [256, 64, 304])
def test_plans_are_for_the_workgroups_the_library_will_launch(cus, monkeypatch):
    """plan_splits asks the library how many rows a workgroup will serve, then changes the splits, on which that answer depends: the final
    splits have to get the answer that they were planned for."""
    from types import SimpleNamespace
    from qvb8_amd import _lib
    lib = _lib.load()
    monkeypatch.setattr(torch.cuda, "get_device_properties", lambda device: SimpleNamespace(multi_processor_count=cus))
    for name in ("QVB8_ATTN_ROW_BLOCKS", "QVB8_ATTN_WG_PER_CU"):
        monkeypatch.delenv(name, raising=False)

    def planned_for(answer, *args, **kw):
        with monkeypatch.context() as m:
            m.setattr(_lib, "load", lambda: SimpleNamespace(qvb8_attn_rows_per_workgroup=lambda *a: answer))
            return FA.plan_splits(*args, **kw)

    seen = set()
    for rows in (33, 128, 129, 207, 208, 256, 257, 400, 415, 416, 512, 630, 720, 768, 1100, 2048):
        for hkv in (1, 2, 3, 4, 8, 16, 96):
            for d in (128, 256):
                for n_tiles in (*range(1, 140), 500, 511, 513, 2048, 4096):
                    for wide in (False, True):
                        args, kw = (n_tiles, hkv, rows, "cuda"), dict(d=d, wide=wide)
                        tps, splits = FA.plan_splits(*args, **kw)
                        block = lib.qvb8_attn_rows_per_workgroup(rows, splits, hkv, 2 if wide else 1, cus)
                        assert (tps, splits) == planned_for(block, *args, **kw), (rows, hkv, d, n_tiles, wide, block)
                        seen.add((block, wide))
    assert seen == {(128, False), (256, False), (128, True)}
    assert lib.qvb8_attn_rows_per_workgroup(32, 4, 4, 1, cus) == 0


@pytest.mark.parametrize("wrong", [dict(n_splits=0), dict(n_splits=-3), dict(G=0), dict(n_rows=65), dict(n_kv_heads=0), dict(n_rows=-2), dict(head_dim=0)])
def test_attend_refuses_bad_sizes_before_its_first_launch(wrong):
    """The preparation of many queries is a launch ahead of the attention kernel's own checks: with no splits it would be asked for no
    workspace and write in front of it, with rows that are no whole tokens read queries that are not there."""
    import ctypes
    from qvb8_amd import _lib
    lib = _lib.load()
    size = dict(n_rows=64, n_splits=2, n_kv_heads=4, head_dim=128, G=2)
    size.update(wrong)
    here = ctypes.create_string_buffer(64)
    at = (ctypes.addressof(here) + 15) & ~15
    d, g, heads = size["head_dim"], size["G"], size["n_kv_heads"]
    rc = lib.qvb8_attend(at, _lib.F16, 1.0, heads * g * d, d, at, at, 1, heads * d, d, *[at] * 9, 4, size["n_splits"], size["n_rows"], heads, d, 0, 2, g,
                         at, at, at, 1 << 40, None)
    assert rc == -1 and "bad size" in lib.qvb8_last_error().decode()
