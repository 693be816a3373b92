"""QVBandExpertsV8 with more than FUSED_MAX_TOKENS tokens: the routed kernels where they do what the per-expert loop does, the loop
for every other call."""
import pytest
import torch

from oracle import qvb8_oracle as O
from qvb8_amd.formats.qvb8 import pack as PK
from qvb8_amd.formats.qvb8.backends_experts import QVBandExpertsV8
from qvb8_amd.formats.qvb8.module import QVBandLinearV8
from tests import helpers as H
from tests.test_gpu_moe import _check, _experts

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
E, K, HIDDEN, INTER = 4, 2, 256, 128


def _module(tau=2e-3, restore="fp16", hidden=HIDDEN, inter=INTER):
    made = lambda Q, P, seed: QVBandLinearV8.from_encoded(PK.encode_tensor(H.synth_weight(Q, P, seed=seed).to(DEV), tau, restore=restore))     # noqa: E731
    return QVBandExpertsV8([made(2 * inter, hidden, 2 * e) for e in range(E)], [made(hidden, inter, 2 * e + 1) for e in range(E)], num_experts=E)


def _call(T, dtype=torch.bfloat16, seed=0, hidden=HIDDEN):
    g = torch.Generator().manual_seed(seed + T)
    idx = torch.stack([torch.randperm(E, generator=g)[:K] for _ in range(T)])
    return torch.randn(T, hidden, generator=g).to(dtype).to(DEV), idx.to(DEV), torch.rand(T, K, generator=g).to(DEV)


def _apart(a, b):
    """How far two fp32 results of the same tokens may lie apart when the tokens come in other blocks: the sum of a pair's
    activations is then cut into other parts.  Each result is within 5e-7 of its norm from 64 bits (3.3e-7 measured)."""
    return float((a.double() - b.double()).norm() / b.double().norm()) > 1e-6


def _spy(mod, monkeypatch):
    """Counts the calls the loop answers."""
    calls, loop = [], mod._forward_loop
    monkeypatch.setattr(mod, "_forward_loop", lambda *a: (calls.append(1), loop(*a))[1], raising=False)
    return calls


@pytest.mark.parametrize("T", [65, 300])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_many_tokens_match_the_oracle(T, dtype, monkeypatch):
    gu, dn, Wgu, Wdn = _experts(E, HIDDEN, INTER, 2e-3, seed=7)
    mod = QVBandExpertsV8(gu, dn, num_experts=E)
    calls = _spy(mod, monkeypatch)
    x, idx, w = _call(T, dtype)
    out = mod(x, idx, w)
    assert not calls and out.dtype == dtype
    _check(out, O.moe_reference(x.float().cpu().numpy(), idx.cpu().numpy(), w.cpu().numpy(), Wgu, Wdn), dtype)
    assert torch.equal(mod(x, idx.to(torch.int32), w), out)                     # any integer routing, as the loop takes it
    assert torch.equal(mod(x, idx.to(torch.uint8), w.to(torch.float64)), out) and not calls


def test_calls_the_loop_answers(monkeypatch):
    mod, T = _module(), 70
    x, idx, w = _call(T)
    mod(x, idx, w)
    calls = _spy(mod, monkeypatch)
    w.requires_grad_()
    out = mod(x, idx, w)                                                         # routing weights that want a gradient
    out.float().pow(2).sum().backward()
    assert len(calls) == 1 and w.grad is not None and bool((w.grad != 0).any())
    with torch.no_grad():
        mod(x, idx, w)
    assert len(calls) == 1
    w = w.detach()
    fired = []
    hook = mod.down_experts[2].register_forward_hook(lambda *a: fired.append(1))
    mod(x, idx, w)
    assert len(calls) == 2 and fired
    hook.remove()
    more = torch.cat([x, x[:3]])                                                 # rows that no routing row names give zeros
    assert torch.equal(mod(more, idx, w)[:T], mod._forward_loop(x, idx, w)) and len(calls) == 4
    mod(x, idx, w)
    assert len(calls) == 4


def test_bf16_certified_experts_multiply_bf16_activations_as_they_are(monkeypatch):
    mod = _module(restore="fp16+bf16")
    if any(m.esc_idx_bf16.numel() for m in [*mod.gate_up_experts, *mod.down_experts]):
        pytest.skip("this pack has bf16 escapes: never stacked")
    x, idx, w = _call(80)
    x[5, 7] = 1e6                                                                # beyond fp16, within bf16
    assert torch.equal(mod(x, idx, w), mod._forward_loop(x, idx, w))
    calls = _spy(mod, monkeypatch)
    mod(x.clamp(-1e4, 1e4).half(), idx, w)
    assert not calls


@pytest.mark.parametrize("T", [65, 300])
def test_expert_numbers_outside_the_stack(T):
    """Past the end: refused, by the call that has them.  Negative ones count from the end, as in any list."""
    mod = _module()
    x, idx, w = _call(T)
    want = mod(x, idx, w)
    for at, bad in (((T - 1, 1), E), ((0, 0), 1 << 40), ((T // 2, 0), -E - 1)):
        wrong = idx.clone()
        wrong[at] = bad
        with pytest.raises(IndexError):
            mod(x, wrong, w)
    back = torch.where(torch.arange(T, device=DEV)[:, None] % 3 == 0, idx - E, idx)
    assert torch.equal(mod(x, back, w), mod._forward_loop(x, back, w))
    assert torch.equal(mod(x, idx, w), want)


@pytest.mark.parametrize("loop_is_faster", [False, True])
def test_many_tokens_inside_a_graph(loop_is_faster, monkeypatch):
    """Captured and replayed with other inputs in the same buffers, eager calls between the replays -- also where the loop, which
    cannot be captured, would be the faster one."""
    mod = _module()
    x, idx, w = _call(90)
    mod(x, idx, w)
    torch.cuda.synchronize()
    limit = QVBandExpertsV8.LOOP_FROM_PAIRS
    if loop_is_faster:
        monkeypatch.setattr(QVBandExpertsV8, "LOOP_FROM_PAIRS", 1)
        monkeypatch.setattr(QVBandExpertsV8, "LOOP_FROM_PRODUCTS", 0)
    graph = torch.cuda.CUDAGraph()
    with torch.no_grad(), torch.cuda.graph(graph):
        out = mod(x, idx, w)
    monkeypatch.setattr(QVBandExpertsV8, "LOOP_FROM_PAIRS", limit)
    for seed in range(3):
        nx, nidx, nw = _call(90, seed=10 + seed)
        x.copy_(nx), idx.copy_(nidx), w.copy_(nw)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, mod(nx, nidx, nw))


def test_the_loop_takes_what_it_is_faster_at(monkeypatch):
    """The rule by pairs per expert and weights per expert, at its edges; and that a call follows it."""
    mod = _module()
    x, idx, w = _call(100)
    mod(x, idx, w)
    weights = 3 * HIDDEN * INTER
    monkeypatch.setattr(QVBandExpertsV8, "LOOP_FROM_PRODUCTS", 50 * weights)
    assert not mod._loop_is_faster(512 * E - 1) and mod._loop_is_faster(512 * E)
    monkeypatch.setattr(QVBandExpertsV8, "LOOP_FROM_PRODUCTS", 600 * weights)
    assert not mod._loop_is_faster(600 * E - 1) and mod._loop_is_faster(600 * E)
    monkeypatch.setattr(QVBandExpertsV8, "LOOP_FROM_PAIRS", 100)
    monkeypatch.setattr(QVBandExpertsV8, "LOOP_FROM_PRODUCTS", 0)
    calls = _spy(mod, monkeypatch)
    mod(x, idx, w)                                                               # 50 pairs per expert
    assert not calls
    mod(x.repeat(2, 1), idx.repeat(2, 1), w.repeat(2, 1))
    assert len(calls) == 1
    monkeypatch.setenv("QVB8_MOE_GROUPED", "0")
    mod(x, idx, w)
    assert len(calls) == 2


def test_stacks_with_rows_read_id_by_id(monkeypatch):
    mod = _module(tau=2e-4)
    x, idx, w = _call(100)
    mod.prepare()
    assert int(mod._stk[0]["nbits"].max()) > 8 and not mod._stk[0]["sliced"]
    calls = _spy(mod, monkeypatch)
    out = mod(x, idx, w)                                                         # 50 pairs per expert of 98304 weights
    assert not calls
    monkeypatch.setattr(QVBandExpertsV8, "ODD_ROWS_MAX_PAIRS", 49)
    loop = mod(x, idx, w)
    monkeypatch.setattr(QVBandExpertsV8, "ODD_ROWS_MAX_PAIRS", 75)
    monkeypatch.setattr(QVBandExpertsV8, "ODD_ROWS_MAX_WEIGHTS", 98303)
    assert torch.equal(mod(x, idx, w), loop) and len(calls) == 2
    assert float((out.float() - loop.float()).norm() / loop.float().norm()) <= 1e-2      # (the loop rounds to bf16 four times)


@pytest.mark.parametrize("T,slices", [(66, 1), (130, 2), (131, 2), (700, 5)])
def test_tokens_in_slices(T, slices, monkeypatch):
    """Bounded scratch: the tokens in equal slices, with the results of the whole; an expert number outside the stack in
    the last one is still refused."""
    mod = _module()
    x, idx, w = _call(T, torch.float32)
    want = mod(x, idx, w)
    monkeypatch.setattr(QVBandExpertsV8, "SCRATCH_BYTES", -(-T // slices) * 4 * K * (HIDDEN + INTER))
    sizes, routed = [], mod._routed
    monkeypatch.setattr(mod, "_routed", lambda *a: (sizes.append(a[0].shape[0]), routed(*a))[1], raising=False)
    assert not _apart(mod(x, idx, w), want)
    assert len(sizes) == slices and sum(sizes) == T and min(sizes) > mod.FUSED_MAX_TOKENS and max(sizes) - min(sizes) <= 1
    idx[T - 1, 0] = E
    with pytest.raises(IndexError):
        mod(x, idx, w)


def test_more_tokens_than_a_grid_has_rows():
    """70000 tokens of one slice: as the first 300 of them alone."""
    mod = _module(hidden=128, inter=128)
    x, idx, w = _call(300, torch.float32, hidden=128)
    want = mod(x, idx, w)
    n = 70000
    many = [t.repeat(-(-n // 300), 1)[:n] for t in (x, idx, w)]
    out = mod._routed(*many[:2], many[2].float(), True) if mod.build_stack() else None
    assert not _apart(out, want.repeat(-(-n // 300), 1)[:n])
    assert not _apart(out[65500:65600], want.repeat(-(-n // 300), 1)[65500:65600]) and not _apart(out[-100:], want.repeat(-(-n // 300), 1)[n - 100:n])
