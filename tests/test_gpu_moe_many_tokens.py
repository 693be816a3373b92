"""GPU parity of the many-token expert kernels (more than 16 tokens, rows of whole 128-column steps): the sizes at which their
tiles change -- 16, 32, 48, 64 and 65 pairs of an expert, one step and several chunks of columns -- with every width of
row, against the oracle and run to run."""
import numpy as np
import pytest
import torch

from oracle import qvb8_oracle as O
from qvb8_amd import ext_qvb8 as ext
from qvb8_amd.formats.qvb8 import pack as PK
from qvb8_amd.formats.qvb8.backends_experts import stack_projection
from qvb8_amd.formats.qvb8.module import QVBandLinearV8
from tests.test_gpu_moe import _check, _hand_made_stack

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("T,pairs,hidden,inter,gated,dtype", [
    (17, 16, 128, 128, True, torch.bfloat16), (17, 17, 384, 256, False, torch.float16), (40, 33, 1152, 128, True, torch.float32),
    (70, 48, 256, 640, False, torch.bfloat16), (70, 65, 640, 384, True, torch.float16), (140, 129, 2176, 128, True, torch.bfloat16)])
def test_many_tokens(T, pairs, hidden, inter, gated, dtype):
    """Expert 1 is chosen by `pairs` of the T tokens, the rest is spread; one expert is chosen by nobody."""
    E, k = 6, 2
    Qup = 2 * inter if gated else inter
    up, Wup = _hand_made_stack(E, Qup, hidden, [6] * 16 + [7, 5, 6] + [4] * 13 + list(range(1, 15)) + [8] * 18, seed=40)
    dn, Wdn = _hand_made_stack(E, hidden, inter, [5] * 16 + [4, 5, 6, 7, 8, 11, 3], seed=80)
    rng = np.random.default_rng(T)
    idx = np.stack([rng.permutation([0, 2, 3, 4])[:k] for _ in range(T)]).astype(np.int64)          # 5 is never chosen
    idx[rng.permutation(T)[:pairs], 0] = 1
    w = rng.uniform(0.1, 1.0, (T, k)).astype(np.float32)
    x = torch.randn(T, hidden, generator=torch.Generator().manual_seed(T)).to(dtype)
    fn = ext.moe_experts if gated else ext.moe_experts_relu2
    args = (x.to(DEV), torch.from_numpy(idx).to(DEV), torch.from_numpy(w).to(DEV), *up, Qup, hidden, *dn, hidden, inter)
    out = fn(*args)
    assert out.dtype == dtype and out.shape == (T, hidden)
    _check(out, O.moe_reference(x.float().numpy(), idx, w, Wup, Wdn, act="silu" if gated else "relu2"), dtype)
    assert torch.equal(out, fn(*args))
    bad = args[1].clone()
    bad[3, 1] = E
    assert bool(torch.isnan(fn(args[0], bad, *args[2:]).float()).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_tokens_that_start_off_a_16_byte_line(dtype):
    """Activations that are a view one element into a buffer: the same bits as from a buffer of their own."""
    E, k, T, hidden, inter = 3, 2, 37, 256, 128
    up, _ = _hand_made_stack(E, 2 * inter, hidden, [6, 7, 5, 8], seed=4)
    dn, _ = _hand_made_stack(E, hidden, inter, [5, 6], seed=8)
    g = torch.Generator().manual_seed(1)
    idx = torch.stack([torch.randperm(E, generator=g)[:k] for _ in range(T)]).to(DEV)
    w = torch.rand(T, k, generator=g).to(DEV)
    buf = torch.randn(T * hidden + 1, generator=g).to(dtype).to(DEV)
    x = buf[1:].view(T, hidden)
    rest = (idx, w, *up, 2 * inter, hidden, *dn, hidden, inter)
    assert torch.equal(ext.moe_experts(x, *rest), ext.moe_experts(x.clone(), *rest))


@pytest.mark.parametrize("T,E,hidden,inter,gated", [(17, 4, 2048, 768, True), (64, 6, 1152, 512, True), (40, 3, 640, 896, False)])
def test_no_further_from_64_bits_than_the_general_path(T, E, hidden, inter, gated, monkeypatch):
    """fp32 activations that fp16 holds exactly and fp32 results: what is left is the arithmetic.  The general path multiplies
    and adds in fp32; the matrix-core kernels have to be as exact on weights whose rows lie unevenly around zero in their width."""
    k, Qup = 2, 2 * inter if gated else inter
    up, dn = (_packed_stack(E, Q, P, seed) for Q, P, seed in ((Qup, hidden, 1), (hidden, inter, 2)))
    g = torch.Generator().manual_seed(T)
    idx = torch.stack([torch.randperm(E, generator=g)[:k] for _ in range(T)])
    w = torch.rand(T, k, generator=g).half().float()
    x = torch.randn(T, hidden, generator=g).half().float()
    exact = torch.zeros(T, hidden, dtype=torch.float64)
    for e in range(E):
        t, c = (idx == e).nonzero(as_tuple=True)
        h = x[t].double() @ up[1][e].T
        h = torch.relu(h) ** 2 if not gated else h[:, :inter] * torch.sigmoid(h[:, :inter]) * h[:, inter:]
        exact.index_add_(0, t, (h @ dn[1][e].T) * w[t, c, None].double())
    fn = ext.moe_experts if gated else ext.moe_experts_relu2

    def error():
        out = fn(x.to(DEV), idx.to(DEV), w.to(DEV), *up[0], Qup, hidden, *dn[0], hidden, inter)
        return float((out.cpu().double() - exact).norm() / exact.norm())

    grouped = error()
    monkeypatch.setenv("QVB8_MOE_GROUPED", "0")
    assert grouped <= error()


def _packed_stack(E, Q, P, seed):
    """E packed experts of N(0.003, 0.02) weights (several widths, no row centred in its own) and what they stand for in 64 bits."""
    gen = torch.Generator().manual_seed(seed)
    enc = [PK.encode_tensor((0.02 * torch.randn(Q, P, generator=gen) + 0.003).to(torch.bfloat16).to(DEV), 2e-3) for _ in range(E)]
    stk = stack_projection([QVBandLinearV8.from_encoded(e) for e in enc])
    exact = []
    for e in range(E):
        row = [stk[n][e] for n in ("nbits", "bit_off", "min_s", "tau_s")]
        ids = ext.decode_f32(stk["ids"], torch.zeros_like(row[2]), row[0], row[1], P, torch.ones_like(row[3]), *(enc[0][n] for n in ("esc_idx", "esc_vals")))
        exact.append((ids.double() * row[3].double()[:, None] + row[2].double()[:, None]).cpu())
    return tuple(stk[n] for n in ("ids", "min_s", "tau_s", "nbits", "bit_off")), exact


@pytest.mark.parametrize("T", [17, 40, 70])
def test_infinities_among_fp16_activations(T):
    """Narrowed to +-65504 like every value fp16 cannot hold (what O.moe_reference does); on request they stay, and only the
    tokens that hold one are lost."""
    E, k, hidden, inter = 3, 2, 256, 128
    up, Wup = _hand_made_stack(E, 2 * inter, hidden, [6, 7, 5, 8, 11], seed=4)
    dn, Wdn = _hand_made_stack(E, hidden, inter, [5, 6, 3], seed=8)
    g = torch.Generator().manual_seed(T)
    idx = torch.stack([torch.randperm(E, generator=g)[:k] for _ in range(T)])
    w = torch.rand(T, k, generator=g)
    x = (1e-3 * torch.randn(T, hidden, generator=g)).half()
    x[3, 5], x[T - 1, 200] = float("inf"), -float("inf")
    args = (x.to(DEV), idx.to(DEV), w.to(DEV), *up, 2 * inter, hidden, *dn, hidden, inter)
    clamped = torch.equal(ext.moe_experts(*args), ext.moe_experts(x.clamp(-65504, 65504).to(DEV), *args[1:]))
    assert clamped
    kept = ext.moe_experts(*args, keep_inf=True).isfinite().all(1).cpu()
    assert kept.tolist() == [t not in (3, T - 1) for t in range(T)]


@pytest.mark.parametrize("T", [17, 70])
def test_rows_that_claim_to_lie_in_planes_are_nan(T):
    """Stacks hold their rows back to back; a plane mark (bit 62 of the offset) puts a row outside the buffer on every path."""
    E, k, hidden, inter = 4, 2, 256, 128
    up, _ = _hand_made_stack(E, 2 * inter, hidden, [6] * 16 + [7, 5], seed=4)
    dn, _ = _hand_made_stack(E, hidden, inter, [5, 6], seed=8)
    g = torch.Generator().manual_seed(T)
    idx = torch.stack([torch.randperm(E, generator=g)[:k] for _ in range(T)])
    marked = up[4].clone()
    marked[2, 5] |= 1 << 62
    out = ext.moe_experts(torch.randn(T, hidden, generator=g).to(DEV), idx.to(DEV), torch.rand(T, k, generator=g).to(DEV), *up[:4], marked,
                          2 * inter, hidden, *dn, hidden, inter)
    assert torch.equal(out.isnan().all(1).cpu(), (idx == 2).any(1)) and torch.equal(out.isnan().any(1).cpu(), (idx == 2).any(1))


# 1024 threads place the pairs: one round of them and a ragged second one, more than the four rounds that are kept in registers,
# more experts than the table of counts takes (turns), with more than a round of pairs there too, and one expert that gets all
@pytest.mark.parametrize("T,E,k", [(550, 6, 2), (2100, 6, 2), (2049, 3, 2), (40, 513, 3), (700, 520, 2), (2100, 600, 2), (1100, 1, 1)])
def test_routing_plans_of_many_pairs(T, E, k):
    hidden = inter = 128
    made = min(E, 8)
    up, Wup = _hand_made_stack(made, 2 * inter, hidden, [6, 7, 5, 8], seed=4)
    dn, Wdn = _hand_made_stack(made, hidden, inter, [5, 6], seed=8)
    same = torch.arange(E, device=DEV) % made                    # expert e holds the rows of expert e % 8
    up, dn = ((s[0], *[t[same].contiguous() for t in s[1:]]) for s in (up, dn))
    g = torch.Generator().manual_seed(T + E)
    idx = torch.rand(T, E, generator=g).topk(k, 1).indices
    w = torch.rand(T, k, generator=g) + 0.1
    x = torch.randn(T, hidden, generator=g).half()
    out = ext.moe_experts(x.to(DEV), idx.to(DEV), w.to(DEV), *up, 2 * inter, hidden, *dn, hidden, inter, checked=True)
    _check(out, O.moe_reference(x.float().numpy(), (idx % made).numpy(), w.numpy(), Wup, Wdn), torch.float16)
