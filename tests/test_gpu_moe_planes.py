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


@pytest.mark.parametrize("tau,growth", [(2e-3, 0.25), (1e-3, 0.25), (4e-4, 0.25)])            # 6, 7 and 8 bits a weight
@pytest.mark.parametrize("T,k,dtype", [(1, 2, torch.bfloat16), (5, 2, torch.float16), (8, 2, torch.bfloat16), (16, 3, torch.float16), (3, 2, torch.float32),
                                       (17, 2, torch.float32), (40, 3, torch.bfloat16), (150, 4, torch.bfloat16)])
def test_planes_change_no_result(T, k, dtype, tau, growth, monkeypatch):
    E, hidden, inter = 5, 384, 128
    monkeypatch.setenv("QVB8_MOE_ONE_WIDTH_GROWTH", str(growth))
    g = torch.Generator(device=DEV).manual_seed(T)
    x = torch.randn(T, hidden, device=DEV, generator=g).to(dtype)
    w, idx = torch.softmax(torch.randn(T, E, device=DEV, generator=g), -1).topk(k, -1)
    out, one = [], []
    for least in (1 << 40, 0):
        monkeypatch.setattr(BE, "PLANES_FROM_BYTES", least)
        gu, dn = _experts(E, hidden, inter, tau)
        mod = BE.QVBandExpertsV8(gu, dn, num_experts=E).prepare()
        assert [s["planes"] for s in mod._stk] == [least == 0] * 2
        out.append(mod(x, idx, w))
        one += [ext.decode_f32(m.ids, m.min_s, m.nbits, m.bit_off, m.in_features, m.tau_s, m.esc_idx, m.esc_vals) for m in (gu[3], dn[1])]
        one[-2:] = [*one[-2:], gu[2](x), dn[4](gu[0](x)[:, :inter])]
    if dtype == torch.float32 and T <= 16:
        # rows back to back go through the general kernel, whose fp32 products are no closer to 64 bits than the others
        assert float((out[0] - out[1]).norm() / out[0].norm()) < 2e-6
    else:
        assert torch.equal(*out)
    for a, b in zip(one[:4], one[4:]):                  # the experts' own modules read their rows where they are now
        assert torch.equal(a, b)


def test_planes_without_what_they_need_are_refused():
    E, hidden, inter = 2, 256, 128
    gu, dn = _experts(E, hidden, inter, 2e-3)
    g, d = BE.stack_projection(gu, 2), BE.stack_projection(dn)
    x, idx, w = torch.randn(3, hidden, device=DEV), torch.zeros(3, 1, dtype=torch.int64, device=DEV), torch.ones(3, 1, device=DEV)
    ops = lambda s: (s["ids"], s["min_s"], s["tau_s"], s["nbits"], s["bit_off"], s["Q"], s["P"])       # noqa: E731
    with pytest.raises(RuntimeError, match="regular"):
        ext.moe_experts(x, idx, w, *ops(g), *ops(d), planes=(True, False))
