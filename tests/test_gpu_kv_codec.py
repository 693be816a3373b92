"""The banded KV codec's kernels against the same codec on the CPU (torch operations, pinned by the oracle): streams, constants
and widths bit for bit, and the id layout built from them."""
import pytest
import torch

from qvb8_amd.kv import codec as C
from qvb8_amd.kv import fused_attn as FA
from tests.test_kv_host import lengths_and_segments_must_match

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _values(heads, seq, dim, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(heads, seq, dim, generator=g) * torch.exp(torch.randn(heads, 1, dim, generator=g)) + torch.randn(heads, 1, dim, generator=g)
    x[:, :, dim // 2] = 0.75                                     # a constant channel
    if seq > 3:
        x[0, 1, 0], x[0, 2, 1], x[0, 3, 0] = float("nan"), float("inf"), float("-inf")
    return x.to(dtype)


# tau small enough for bf16 that the first width leaves a rounding too much and has to rise; none at all; and wide fp32 ids: the
# widest channel spans about 72, so 16 bits reach 72 / 65535 / 2 = 5.5e-4 and a bound of 1e-3 is within them
@pytest.mark.parametrize("heads,seq,dim,dtype,bits,tau", [
    (1, 1, 8, torch.float32, 1, 0.0), (3, 17, 64, torch.bfloat16, 5, 0.03), (2, 70, 100, torch.float16, 6, 0.01), (5, 9, 33, torch.bfloat16, 7, 0.5),
    (4, 513, 256, torch.bfloat16, 6, 0.25), (2, 1025, 128, torch.float32, 4, 0.001), (3, 31, 2048, torch.float16, 16, 0.0), (32, 40, 96, torch.bfloat16, 3, 0.1)])
def test_bands_are_those_of_the_cpu_codec(heads, seq, dim, dtype, bits, tau):
    x = _values(heads, seq, dim, dtype, seed=seq + dim)
    if tau and dtype == torch.bfloat16:
        x = x.clamp(-12, 12)                                     # what bf16 can certify
    want = C.band_kv_heads(x, dtype, bits, tau=tau)
    got = C.band_kv_heads(x.to(DEV), dtype, bits, tau=tau)
    for w, g in zip(want, got):
        assert g.bits == w.bits and g.orig_shape == w.orig_shape and g.orig_dtype == w.orig_dtype
        for name in ("min_s", "tau_s", "packed"):
            assert torch.equal(getattr(g, name).cpu(), getattr(w, name)), name
    wide = any(b.bits > 8 for b in want)
    want_lay = FA.layout_from_segments([want, want], [want, want], [seq, seq], "cpu", allow_wide=True)
    got_lay = FA.layout_from_segments([got, got], [got, got], [seq, seq], DEV, allow_wide=True)
    assert got_lay.ki.dtype == (torch.int16 if wide else torch.uint8)
    for name in ("ki", "vi", "kmin", "kstep", "vmin", "vstep", "kc", "vc", "t_start", "t_len", "t_seg"):
        assert torch.equal(getattr(got_lay, name).cpu(), getattr(want_lay, name)), name


@pytest.mark.parametrize("heads,seq,dim,dtype", [(1, 4101, 8, torch.float32), (1, 201, 2048, torch.bfloat16), (2, 83, 2047, torch.float16), (2, 270, 1000, torch.float32),
                                                 (32, 129, 16, torch.bfloat16), (4, 1500, 58, torch.float16), (3, 497, 72, torch.bfloat16)])
def test_chunks_that_end_inside_a_batch_of_rows(heads, seq, dim, dtype):
    """Several rows are loaded at once, the last one again where a chunk ends, and channels past the first pass follow behind."""
    x = _values(heads, seq, dim, dtype, seed=seq).clamp(-12, 12)
    want = C.band_kv_heads(x, dtype, 5, tau=0.06)
    got = C.band_kv_heads(x.to(DEV), dtype, 5, tau=0.06)
    for w, g in zip(want, got):
        assert g.bits == w.bits
        for name in ("min_s", "tau_s", "packed"):
            assert torch.equal(getattr(g, name).cpu(), getattr(w, name)), name


def test_a_bound_that_sixteen_bits_miss_is_refused():
    x = torch.tensor([[[0.0], [1.1], [3e4]]])
    for dev in ("cpu", DEV):
        with pytest.raises(C.KVCertificateError):
            C.band_kv_heads(x.to(dev), torch.float32, 6, tau=1e-9)


def test_lengths_and_segments_must_match_on_the_gpu():
    """The kernel path paired segments with lengths until one of the two ran out: the rest was dropped without a word."""
    lengths_and_segments_must_match(DEV)


@pytest.mark.parametrize("n_seg", [1, 256, 257, 600])
def test_tile_tables_of_many_segments(n_seg):
    """The table is filled 256 segments a launch: empty segments and ones of a single key among them."""
    lens = [(7 * i) % 90 for i in range(n_seg - 1)] + [33]
    parts = [torch.zeros(n_seg, 1, 128) for _ in range(4)]
    ids = torch.zeros(sum(lens), 1, 128, dtype=torch.uint8)
    want, got = (FA.QVLayout(ids.to(d), ids.to(d), *[p.to(d) for p in parts], lens, d) for d in ("cpu", DEV))
    for name in ("t_start", "t_len", "t_seg"):
        assert torch.equal(getattr(got, name).cpu(), getattr(want, name)), name


@pytest.mark.parametrize("heads,seq,dim,dtype", [(1, 1, 3, torch.float32), (2, 16, 64, torch.bfloat16), (3, 17, 40, torch.float16), (32, 511, 8, torch.bfloat16),
                                                 (2, 512, 256, torch.bfloat16), (1, 4096, 2048, torch.bfloat16)])
@pytest.mark.parametrize("bits,tau", [(7, 0.25), (3, 0.01)])
def test_figures_for_the_waiting_host_are_the_checks(heads, seq, dim, dtype, bits, tau):
    """qvb8_kv_measure + qvb8_kv_wait (partial ranges joined by every workgroup, three words a head) against qvb8_kv_range + qvb8_kv_check."""
    from qvb8_amd import _lib
    lib, code = _lib.load(), {torch.float32: 0, torch.float16: 1, torch.bfloat16: 2}[dtype]
    x = _values(heads, seq, dim, dtype, seed=seq).to(DEV)
    s, chunks = _lib.stream_of(x), lib.qvb8_kv_chunks(heads, seq)
    partial, both = torch.empty(heads * chunks * 2 * dim, device=DEV), torch.empty(2, 2, heads, dim, device=DEV)
    report = torch.empty(heads, 2 + chunks, pin_memory=True)
    _lib._check(lib.qvb8_kv_range(x.data_ptr(), code, heads, seq, dim, partial.data_ptr(), chunks, s), lib)
    _lib._check(lib.qvb8_kv_check(x.data_ptr(), code, heads, seq, dim, partial.data_ptr(), chunks, code, bits, tau, None, both[0, 0].data_ptr(), both[0, 1].data_ptr(),
                                  report.data_ptr(), s), lib)
    scratch, found = torch.empty(lib.qvb8_kv_measure_floats(heads, seq, dim), device=DEV), torch.empty(heads, 3, pin_memory=True)
    for _ in range(3):                                           # the words the workgroups meet in are cleared by every call
        _lib._check(lib.qvb8_kv_measure(x.data_ptr(), code, heads, seq, dim, code, bits, tau, scratch.data_ptr(), both[1, 0].data_ptr(), both[1, 1].data_ptr(),
                                        found.data_ptr(), s), lib)
        _lib._check(lib.qvb8_kv_wait(found.data_ptr(), heads, s), lib)
        assert torch.equal(both[0].view(torch.int32), both[1].view(torch.int32))
        assert torch.equal(found, torch.cat([report[:, :2], report[:, 2:].amax(1, keepdim=True)], 1))


@pytest.mark.parametrize("risen", [[0], [2], [5], [1, 4], [0, 5], [0, 1, 2, 3, 4, 5]])
@pytest.mark.parametrize("seq,dim", [(300, 64), (77, 30), (16, 7)])
def test_heads_that_need_more_are_packed_again_and_no_others(risen, seq, dim, monkeypatch):
    """Single heads, heads with others between them, all heads: the CPU codec's bits, and a second launch over those heads only."""
    from qvb8_amd import _lib
    x = _values(6, seq, dim, torch.bfloat16, seed=dim).clamp(-8, 8)
    for n, i in enumerate(risen):
        x[i, n, n] = 100.0 * (n + 1)
    want = C.band_kv_heads(x, x.dtype, 7, tau=0.25)
    assert [i for i, b in enumerate(want) if b.bits > 7] == risen
    lib, packed = _lib.load(), []

    class Watched:
        def __getattr__(self, name):
            if name == "qvb8_kv_pack":
                return lambda *a: (packed.append((a[2], bytes(a[7]))), lib.qvb8_kv_pack(*a))[1]
            return getattr(lib, name)

    monkeypatch.setattr(_lib, "load", Watched)
    got = C.band_kv_heads(x.to(DEV), x.dtype, 7, tau=0.25)
    assert packed == [(6, bytes([7] * 6)), (risen[-1] + 1 - risen[0], bytes(b.bits for b in want[risen[0]:risen[-1] + 1]))]
    for w, g in zip(want, got):
        assert g.bits == w.bits
        for name in ("min_s", "tau_s", "packed"):
            assert torch.equal(getattr(g, name).cpu(), getattr(w, name)), name
