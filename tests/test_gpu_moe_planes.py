"""Expert stacks whose tiles are stored in planes: every path gives, bit for bit, what it gives with the rows back to back."""
import pytest
import torch

from qvb8_amd import ext_qvb8 as ext
from qvb8_amd.formats.qvb8 import backends_experts as BE
from qvb8_amd.formats.qvb8 import pack as PK
from qvb8_amd.formats.qvb8.module import QVBandLinearV8

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _experts(E, hidden, inter, tau):
    gen = torch.Generator(device=DEV).manual_seed(7)
    pack = lambda Q, P: QVBandLinearV8.from_encoded(PK.encode_tensor((0.02 * torch.randn(Q, P, device=DEV, generator=gen)).bfloat16(), tau))   # noqa: E731
    return [pack(2 * inter, hidden) for _ in range(E)], [pack(hidden, inter) for _ in range(E)]


ROUTED = [(1, 2, torch.bfloat16), (5, 2, torch.float16), (8, 2, torch.bfloat16), (16, 3, torch.float16), (3, 2, torch.float32),
          (17, 2, torch.float32), (40, 3, torch.bfloat16), (150, 4, torch.bfloat16)]


@pytest.mark.parametrize("tau,growth", [(2e-3, 0.25), (1e-3, 0.25), (4e-4, 0.25)])            # 6, 7 and 8 bits a weight
@pytest.mark.parametrize("T,k,dtype", ROUTED)
def test_planes_change_no_result(T, k, dtype, tau, growth, monkeypatch):
    _same_in_planes(T, k, dtype, 384, 128, tau, growth, monkeypatch)


# one dword in the second plane and none (rows long enough that their ranges, and so their widths, differ little); rows of more than 2048 columns
@pytest.mark.parametrize("hidden,inter,tau,bits", [(512, 512, 3e-3, 5), (512, 512, 5.6e-3, 4), (2304, 256, 2e-3, 6), (256, 2176, 2e-3, 6)])
@pytest.mark.parametrize("T,k,dtype", ROUTED)
def test_planes_of_narrow_and_of_long_rows_change_no_result(T, k, dtype, hidden, inter, tau, bits, monkeypatch):
    _same_in_planes(T, k, dtype, hidden, inter, tau, 0.25, monkeypatch, bits)


def _same_in_planes(T, k, dtype, hidden, inter, tau, growth, monkeypatch, bits=None):
    E = 5
    monkeypatch.setenv("QVB8_MOE_ONE_WIDTH_GROWTH", str(growth))
    g = torch.Generator(device=DEV).manual_seed(T)
    x = torch.randn(T, hidden, device=DEV, generator=g).to(dtype)
    w, idx = torch.softmax(torch.randn(T, E, device=DEV, generator=g), -1).topk(k, -1)
    out, one = [], []
    for least in (1 << 40, 0):
        monkeypatch.setattr(BE, "PLANES_FROM_BYTES", least)
        gu, dn = _experts(E, hidden, inter, tau)
        mod = BE.QVBandExpertsV8(gu, dn, num_experts=E).prepare()
        assert [s["planes"] for s in mod._stk] == [least == 0] * 2 and bits in (None, int(mod._stk[0]["nbits"][0, 0]))
        out.append(mod(x, idx, w))
        one += [ext.decode_f32(m.ids, m.min_s, m.nbits, m.bit_off, m.in_features, m.tau_s, m.esc_idx, m.esc_vals) for m in (gu[3], dn[1])]
        one[-2:] = [*one[-2:], gu[2](x), dn[4](gu[0](x)[:, :inter])]
    assert torch.equal(*out)
    for a, b in zip(one[:4], one[4:]):                  # the experts' own modules read their rows where they are now
        assert torch.equal(a, b)


def _ops(s):
    return s["ids"], s["min_s"], s["tau_s"], s["nbits"], s["bit_off"], s["Q"], s["P"]


def _two_stacks(monkeypatch, E, hidden, inter, gated):
    """The same experts as stacks back to back and in planes, (up, down) each."""
    monkeypatch.setattr(BE, "PLANES_FROM_BYTES", 0)
    out = []
    for planes in (False, True):
        gu, dn = _experts(E, hidden, inter, 2e-3)
        up = gu if gated else [m.row_subset(torch.arange(inter, device=DEV)) for m in gu]
        out.append((BE.stack_projection(up, 2 if gated else 1, planes=planes), BE.stack_projection(dn, planes=planes)))
        assert [s["planes"] for s in out[-1]] == [planes] * 2 and all(s["regular"] for s in out[-1])
    return out


CALLS = [(1, torch.bfloat16), (5, torch.float16), (8, torch.bfloat16), (16, torch.float16), (3, torch.float32), (40, torch.bfloat16)]


@pytest.mark.parametrize("gated", [True, False])
def test_every_entry_point_reads_a_stack_in_planes_or_says_nan(gated, monkeypatch):
    E, hidden, inter = 3, 256, 384
    plain, planes = _two_stacks(monkeypatch, E, hidden, inter, gated)
    for a, b in zip(plain, planes):                     # restored and looked up through the stack's own table
        assert ext.rows_in_planes(b["bit_off"]) and not ext.rows_in_planes(a["bit_off"])
        rows = [(s["ids"], s["min_s"].reshape(-1), s["nbits"].reshape(-1), s["bit_off"].reshape(-1), s["P"], s["tau_s"].reshape(-1), None, None) for s in (a, b)]
        assert torch.equal(*(ext.decode_f32(*r) for r in rows))
        some = torch.tensor([0, 17, a["Q"], E * a["Q"] - 1], device=DEV)
        assert torch.equal(*(ext.lookup_rows(some, *r) for r in rows))
    fn = ext.moe_experts if gated else ext.moe_experts_relu2
    off_a_dword = [dict(s, bit_off=s["bit_off"] + 8) for s in planes]
    unmarked = [dict(p, bit_off=s["bit_off"]) for s, p in zip(plain, planes)]
    for T, dtype in CALLS:
        g = torch.Generator(device=DEV).manual_seed(T)
        x = torch.randn(T, hidden, device=DEV, generator=g).to(dtype)
        w, idx = torch.softmax(torch.randn(T, E, device=DEV, generator=g), -1).topk(2, -1)
        yes = dict(regular=(True, True))
        want, got = fn(x, idx, w, *_ops(plain[0]), *_ops(plain[1]), **yes), fn(x, idx, w, *_ops(planes[0]), *_ops(planes[1]), **yes, planes=(True, True))
        assert bool(want.isfinite().all())
        assert torch.equal(got, want)
        # one projection at a time: marked and not said so, regular or not; said to be in planes and not marked; off a dword
        for stack, regular, said in ((planes, True, False), (planes, False, False), (unmarked, True, True), (off_a_dword, True, True)):
            for bad in (0, 1):
                ops = [*_ops((stack if bad == 0 else planes)[0]), *_ops((stack if bad == 1 else planes)[1])]
                flags = dict(regular=(bad == 1 or regular, bad == 0 or regular), planes=(bad == 1 or said, bad == 0 or said))
                assert bool(fn(x, idx, w, *ops, **flags).isnan().all()), (T, dtype, bad, regular, said)


@pytest.mark.parametrize("T,k,dtype", [(1, 2, torch.float32), (9, 3, torch.float32), (2, 9, torch.bfloat16), (6, 10, torch.float16), (20, 2, torch.bfloat16)])
@pytest.mark.parametrize("hidden,inter,tau", [(2048, 2176, 2e-3), (4224, 128, 3e-3), (1024, 1920, 6e-3)])        # 6, 5 and 4 bits
def test_the_general_kernel_reads_planes(T, k, dtype, hidden, inter, tau, monkeypatch):
    """Rows of a part of 64 slices, of exactly 64 and of more; what it computes is, bit for bit, what it computes with rows back to back, H in fp32."""
    monkeypatch.setenv("QVB8_MOE_ONE_WIDTH_GROWTH", "0.5")
    monkeypatch.setenv("QVB8_MOE_GROUPED", "0")
    E = 10
    g = torch.Generator(device=DEV).manual_seed(T)
    x = torch.randn(T, hidden, device=DEV, generator=g).to(dtype)
    w, idx = torch.softmax(torch.randn(T, E, device=DEV, generator=g), -1).topk(k, -1)
    out = []
    for least in (1 << 40, 0):
        monkeypatch.setattr(BE, "PLANES_FROM_BYTES", least)
        gu, dn = _experts(E, hidden, inter, tau)
        mod = BE.QVBandExpertsV8(gu, dn, num_experts=E).prepare()
        assert [s["planes"] for s in mod._stk] == [least == 0] * 2 and int(mod._stk[0]["nbits"].max()) <= 6
        if least:
            W = [[ext.decode_f32(m.ids, m.min_s, m.nbits, m.bit_off, m.in_features, m.tau_s, m.esc_idx, m.esc_vals).double() for m in ms] for ms in (gu, dn)]
        out.append(mod(x, idx, w))
    assert torch.equal(*out)
    want = torch.zeros(T, hidden, dtype=torch.float64, device=DEV)
    for t in range(T):
        for e, s in zip(idx[t].tolist(), w[t].tolist()):
            h = W[0][e] @ x[t].half().double()
            want[t] += s * (W[1][e] @ (torch.nn.functional.silu(h[:inter]) * h[inter:]))
    # fp32 sums of some thousand products that cancel: about 1e-6 of the norm; one rounding of the result
    assert float((out[0].double() - want).norm() / want.norm()) < (4e-6 if dtype == torch.float32 else 2 ** -8)


def test_a_stack_is_back_to_back_unless_planes_are_asked_for(monkeypatch):
    monkeypatch.setattr(BE, "PLANES_FROM_BYTES", 0)
    gu, dn = _experts(2, 256, 128, 2e-3)
    for s in (BE.stack_projection(gu), BE.stack_projection(dn)):
        assert not s["planes"] and not ext.rows_in_planes(s["bit_off"])


@pytest.mark.parametrize("hidden,inter", [(256, 96), (96, 256), (256, 128)])
def test_planes_are_for_stacks_of_whole_steps(hidden, inter, monkeypatch):
    monkeypatch.setattr(BE, "PLANES_FROM_BYTES", 0)
    monkeypatch.setenv("QVB8_MOE_ONE_WIDTH_GROWTH", "0.25")
    gu, dn = _experts(2, hidden, inter, 2e-3)
    mod = BE.QVBandExpertsV8(gu, dn, num_experts=2).prepare()
    assert [s["planes"] for s in mod._stk] == [hidden % 128 == 0 and inter % 128 == 0] * 2


def test_an_expert_in_planes_is_restored_tile_by_tile(monkeypatch):
    """More than 256 rows, the first call of a module that has no row records of its own: by the tiles' order, the values of rows back to back."""
    x = torch.randn(300, 256, device=DEV, generator=torch.Generator(device=DEV).manual_seed(1))
    out, orders = [], []
    for name in ("decode", "decode_bf16"):
        real = getattr(ext, name)
        monkeypatch.setattr(ext, name, lambda *a, real=real: (orders.append(a[8] if len(a) > 8 else None), real(*a))[1])
    for least in (1 << 40, 0):
        monkeypatch.setattr(BE, "PLANES_FROM_BYTES", least)
        gu, dn = _experts(3, 256, 128, 2e-3)
        BE.QVBandExpertsV8(gu, dn, num_experts=3).prepare()
        for dtype in (torch.float32, torch.float16, torch.bfloat16):
            orders.clear()
            out.append(gu[1](x.to(dtype)))
            assert len(orders) == 1 and (orders[0] is not None) == (least == 0)
        assert gu[1].__dict__.get("_mma_cache") is None
    for a, b in zip(out[:3], out[3:]):
        assert torch.equal(a, b)


def test_a_second_stack_of_the_same_experts(monkeypatch):
    """Built from modules that lie in the planes of an earlier one: as large, and the same results."""
    monkeypatch.setattr(BE, "PLANES_FROM_BYTES", 0)
    gu, dn = _experts(4, 256, 384, 2e-3)
    x, idx, w = torch.randn(9, 256, device=DEV).half(), torch.arange(18, device=DEV).view(9, 2) % 4, torch.full((9, 2), 0.5, device=DEV)
    out, size = [], []
    for _ in range(2):
        mod = BE.QVBandExpertsV8(gu, dn, num_experts=4).prepare()
        assert all(s["planes"] for s in mod._stk)
        out.append(mod(x, idx, w))
        size.append([s["ids"].numel() for s in mod._stk])
    assert torch.equal(*out) and size[0] == size[1]


def test_planes_without_what_they_need_are_refused():
    E, hidden, inter = 2, 256, 128
    gu, dn = _experts(E, hidden, inter, 2e-3)
    g, d = BE.stack_projection(gu, 2), BE.stack_projection(dn)
    x, idx, w = torch.randn(3, hidden, device=DEV), torch.zeros(3, 1, dtype=torch.int64, device=DEV), torch.ones(3, 1, device=DEV)
    with pytest.raises(RuntimeError, match="regular"):
        ext.moe_experts(x, idx, w, *_ops(g), *_ops(d), planes=(True, False))
