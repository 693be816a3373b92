"""QVBandExpertsV8: MoE expert stack on packed QVB8 experts.

Same class name, constructor, `from_packfiles`, `build_stack` layout and `forward(hidden_states, top_k_index,
top_k_weights)` as the reference (src/qv_band/formats/qvb8/backends_experts.py:91-272).  The routed decode path is
ext.moe_experts (four launches, no host round trip, each selected expert read once for all the tokens that chose it), for
any number of tokens when the rows are whole 128-column steps; stacks with escapes, other activations, and more than
FUSED_MAX_TOKENS tokens of other shapes, or of calls that need what only the loop does (_many_as_the_loop), take the
per-expert loop over QVBandLinearV8 modules, which still runs on the GPU library.  There is no CPU reader here (the reference's QVBandLinearCPUV8 is its
CPU-only dense path; this build's CPU restatement lives with the tests and is not a product path).
"""
from __future__ import annotations

import os

import torch
import torch.nn as nn
from torch.nn.modules.module import _has_any_global_hook

from qvb8_amd import ext_qvb8 as ext
from .module import QVBandLinearV8

_KERNEL_DTYPES = (torch.float32, torch.float16, torch.bfloat16)
_INDEX_DTYPES = (torch.int64, torch.int32, torch.int16, torch.int8, torch.uint8)


# Stacks of at least this many bytes store the tiles of a regular stack in planes: a wave's request is then one contiguous run, in operand
# order.  Smaller ones lie in the last-level cache, where rows of a tile apart cost little.
PLANES_FROM_BYTES = 16 << 20


def stack_projection(mods, halves: int = 1, planes: bool = False) -> dict:
    """One projection of every expert as ONE launch operand: the experts' packed ids back to back in a single buffer
    (each part starting on a 16-byte boundary, 64 spare bytes at the end), the row vectors as (experts, Q) tables, bit
    offsets counted from the start of the shared buffer.  `halves`: 2 where a projection's rows are gate rows and up rows.  `planes`: the
    tiles of a large regular stack may be stored in planes; the result's "planes" says whether they are, and a call has to be told so
    (ext.moe_experts).  Every module is re-pointed at the shared buffer (its own bit_off moved accordingly), so the separate copies can be
    freed and the modules keep working.
    Layout of the reference's stacked call (src/qv_band/formats/qvb8/backends_experts.py:145-195).
    Unlike the reference's build_stack, which only re-points the experts' ids, this one may store the rows again: wider
    fields for some rows (every row of a 16-row tile in the tile's widest width, or every row of the stack in one width when
    that costs at most QVB8_MOE_ONE_WIDTH_GROWTH = 4 % more bytes), tiles in planes, all others' rows back to back.  The
    experts' nbits / ids / bit_off change with it (their values do not), so a footprint taken before the stack is built
    differs from one taken after by up to that growth."""
    uniform = os.environ.get("QVB8_MOE_UNIFORM_TILES", "1") != "0"
    # The routed kernels take 16 consecutive rows of an expert as one matrix-core tile and decode a tile once per width
    # found in it.  So every row of a tile is stored in the tile's largest width (same ids, same values: rows of
    # neighbouring widths mixed at random grow a weight by a few per cent and halve the decode work) -- or, when that
    # costs at most 4 % more (QVB8_MOE_ONE_WIDTH_GROWTH), every row of the stack in ONE width: the stack is then regular (a row's place follows from
    # its expert and row number) and the kernels are told so.
    targets = [None] * len(mods)
    one_width = None
    if uniform:
        targets = [ext.tile_uniform_widths(m.nbits) for m in mods]
        widths = torch.cat([(m.nbits if t is None else t).reshape(-1) for m, t in zip(mods, targets)]).to(torch.int64)
        lo, hi, mean = int(widths.min()), int(widths.max()), float(widths.float().mean())
        growth = float(os.environ.get("QVB8_MOE_ONE_WIDTH_GROWTH", "0.04"))
        if lo >= 4 and hi <= 8 and hi <= (1.0 + growth) * mean and all(m.in_features % 8 == 0 for m in mods):
            one_width = hi
    for m, wider in zip(mods, targets):                  # the routed kernels read rows stored back to back only
        if m._planes or ext.rows_in_planes(m.bit_off):
            # (the module's own rows alone: an expert of an earlier stack in planes reads a buffer that holds all of them)
            m.ids, m.bit_off = ext.repack_rows(m.ids, m.nbits, m.bit_off, m.in_features, m.nbits)
            m._planes = False
            m.__dict__.pop("_mma_cache", None)
        if one_width is not None:
            in_place = m.bit_off[0] + torch.arange(m.out_features, device=m.bit_off.device) * (m.in_features * one_width)
            if bool((m.nbits != one_width).any()) or not bool((m.bit_off == in_place).all()):
                wider = torch.full_like(m.nbits, one_width)          # rows in row order, back to back, one width
        if wider is not None:
            packed = ext.repack_rows(m.ids, m.nbits, m.bit_off, m.in_features, wider)
            if packed is not None:
                m.ids, m.bit_off = packed
                m.nbits = wider
                m.__dict__.pop("_mma_cache", None)
                m.__dict__.pop("_sorted_layout", None)
    sizes = torch.tensor([m.ids.numel() for m in mods], dtype=torch.int64)
    starts = torch.zeros_like(sizes)
    starts[1:] = torch.cumsum((sizes[:-1] + 15) // 16 * 16, 0)
    total = int(starts[-1] + (sizes[-1] + 15) // 16 * 16) + 64
    shared = torch.zeros(total, dtype=torch.uint8, device=mods[0].ids.device)
    for m, at, n in zip(mods, starts.tolist(), sizes.tolist()):
        shared[at:at + n] = m.ids
        m.bit_off = m.bit_off + 8 * at
        m.ids = shared
        m.__dict__.pop("_mma_cache", None)               # launch data built for the old buffer is void
        m.__dict__.pop("_sorted_layout", None)
    table = {name: torch.stack([getattr(m, name) for m in mods]).contiguous() for name in ("min_s", "tau_s", "nbits", "bit_off")}
    regular = uniform and ext.stack_is_regular(table["nbits"], table["bit_off"], mods[0].in_features)
    sliced = bool(((table["nbits"] >= 4) & (table["nbits"] <= 8) & (table["bit_off"] % 32 == 0)).all())       # no row is read id by id
    P, Q = int(mods[0].in_features), int(mods[0].out_features)
    planes = (planes and regular and sliced and total >= PLANES_FROM_BYTES and P % 128 == 0 and Q % (16 * halves) == 0
              and bool((table["bit_off"][:, 0] % 128 == 0).all()) and os.environ.get("QVB8_PLANES", "1") != "0")
    if planes:
        table["bit_off"] = ext.stack_in_planes(shared, table["bit_off"], P, int(table["nbits"][0, 0]))
        # an expert's rows in row order, for all of them: what a dense restore needs to take whole tiles (the loop, from 257 rows on)
        in_order = ext.mma_prepare(*(table[name][0] for name in ("nbits", "bit_off", "tau_s", "min_s")), P, shared.numel())
        for m, off in zip(mods, table["bit_off"]):           # the modules' own offsets say where their rows are now
            m.bit_off = off.clone()
            m._planes, m._rows_in_order = True, in_order
    return dict(ids=shared, Q=Q, P=P, regular=regular, sliced=sliced, planes=planes, **table)


def _stackable(mods) -> bool:
    """Experts the routed kernels can read as one stack: on the GPU, one shape, no escapes, no bias, P % 32 == 0."""
    first = mods[0] if mods else None
    if first is None or not first.ids.is_cuda or first.in_features % 32:
        return False
    for m in mods:
        if (m.out_features, m.in_features) != (first.out_features, first.in_features):
            return False
        if m.bias is not None or m.esc_idx.numel() or m.esc_idx_bf16.numel():
            return False
    return True


class QVBandExpertsV8(nn.Module):
    # Up to this many tokens the routed kernels run whatever the shape; above it only stacks whose rows are whole 128-column
    # steps (the matrix-core kernels), the others take the per-expert loop.
    FUSED_MAX_TOKENS = 64
    # Above it the loop also takes calls it is faster at.  It restores an expert once and multiplies with a library GEMM, where the
    # routed kernels decode it again for every 64 of its pairs: that pays from 512 pairs per expert on, if the expert is large
    # enough for its product to outlast the ten or so launches it costs (products of pairs and weights per expert; measured,
    # us, routed / loop).  8 experts of 4096/14336 (176 M weights): 256 pairs 2239 / 2855, 512 pairs 3591 / 3583, 1024 pairs
    # 6609 / 4886, 2048 pairs 12697 / 8312.  50 M weights: 512 pairs 2137 / 2897 (16 experts of 4096/4096) and 653 / 883 (4 of
    # 2048/8192), 1024 pairs 3874 / 3826 and 1157 / 1182, 2048 pairs 7558 / 5945 and 2082 / 1716.  2048/768 (4.7 M weights): 8192 pairs
    # 3531 / 4634 (16 experts), 512 pairs 1996 / 19906 (128 experts).  That was with rows back to back.  Stacks in planes would have the
    # line at about 1e11 products: 8 experts of 4096/14336, 512 pairs 2700 / 3125, 768 pairs 3850 / 3805, 1024 pairs 5325 / 4520; 16 of
    # 4096/4096, 1024 pairs 3005 / 3590, 2048 pairs 6020 / 5740; 4 of 2048/8192, 1024 pairs 880 / 1075, 2048 pairs 1620 / 1605.
    LOOP_FROM_PAIRS, LOOP_FROM_PRODUCTS = 512, 5e10
    # Rows the kernels read id by id (width outside 4..8 or off a dword): for each pair again, while the loop restores them once
    # from 97 rows of activations on and is slow below that only where experts are small.  32 experts of 2048/768, a third of
    # the rows 9 bits wide: 16 pairs 4049 / 17287, 75 pairs 15259 / 81750, 150 pairs 19489 / 5636; 8 of 4096/4096, three quarters:
    # 16 pairs 24125 / 14425, 64 pairs 73024 / 48029, 150 pairs 104639 / 1548.
    ODD_ROWS_MAX_PAIRS, ODD_ROWS_MAX_WEIGHTS = 75, 2 ** 23
    # The routed kernels keep H and the down results of all pairs of a call in fp32: tokens go through them in slices whose
    # share stays below this (5957 tokens of a 2048/768 layer with 8 experts each).
    SCRATCH_BYTES = 512 << 20

    def __init__(self, gate_up_experts, down_experts, *, num_experts: int, act_fn=None):
        super().__init__()
        self.num_experts = int(num_experts)
        for what, mods in (("gate_up_proj", gate_up_experts), ("down_proj", down_experts)):
            mods = list(mods)
            if len(mods) != self.num_experts:
                raise ValueError(f"expected {num_experts} {what} experts, got {len(mods)}")
            setattr(self, "gate_up_experts" if what == "gate_up_proj" else "down_experts", nn.ModuleList(mods))
        self.act_fn = nn.SiLU() if act_fn is None else act_fn
        self._stk = None                      # None = not built yet, False = this stack cannot use the routed kernels

    @classmethod
    def from_packfiles(cls, gate_up_packfiles: dict, down_packfiles: dict, *, num_experts: int, act_fn=None,
                       device: str = "cuda", tau: float | None = None) -> "QVBandExpertsV8":
        """One pack file per expert and projection (dicts expert number -> path); every expert must be there.  `tau` is
        accepted for call-site compatibility and ignored (every pack carries its own certified tau)."""
        del tau
        absent = {what: [e for e in range(num_experts) if e not in files]
                  for what, files in (("gate_up", gate_up_packfiles), ("down", down_packfiles))}
        if absent["gate_up"] or absent["down"]:
            raise ValueError("QVBandExpertsV8 requires every expert packed -- missing gate_up: "
                             f"{absent['gate_up'][:10]}, down: {absent['down'][:10]}")
        load = lambda files: [QVBandLinearV8.from_packfile(files[e], device=device) for e in range(num_experts)]
        return cls(load(gate_up_packfiles), load(down_packfiles), num_experts=num_experts, act_fn=act_fn)

    def _act_code(self):
        return 0 if "silu" in type(self.act_fn).__name__.lower() else None

    def build_stack(self) -> bool:
        """Prepares the two stacked operands of the routed kernels (stack_projection) on first use.  False, and the loop
        path stays in use, for an activation the kernels do not know, experts that cannot be stacked, or shapes that
        are not gate+up (2I, H) / down (H, I)."""
        if self._stk is None:
            gu, dn = list(self.gate_up_experts), list(self.down_experts)
            ok = (self._act_code() is not None and _stackable(gu) and _stackable(dn)
                  and gu[0].out_features == 2 * dn[0].in_features and gu[0].in_features == dn[0].out_features)
            # planes for both projections or for neither: the matrix-core kernels want whole steps of both, and the general kernel, which
            # then takes every call, gains nothing by them (32 experts of 2048/736, us a call, neither / up alone in planes: 1 token
            # 31.2 / 32.7, 8 tokens 109 / 109, 40 tokens 326 / 333)
            whole = ok and self._whole_steps()
            self._stk = (stack_projection(gu, 2, planes=whole), stack_projection(dn, planes=whole)) if ok else False
        return self._stk is not False

    def _whole_steps(self) -> bool:
        return self.gate_up_experts[0].in_features % 128 == 0 and self.down_experts[0].in_features % 128 == 0

    def prepare(self) -> "QVBandExpertsV8":
        """Builds the stacks now (at load) instead of on the first routed call: the experts' rows are re-stored then, so
        footprints read afterwards are the ones that stay, and a first call inside a graph capture finds them built.
        Returns self."""
        if self.gate_up_experts[0].ids.is_cuda:
            self.build_stack()
        return self

    def _loop_is_faster(self, n_pairs: int) -> bool:
        """Whether a call of so many (token, choice) pairs is the loop's, going by the pairs an expert gets on average.  Never
        inside a graph capture: the loop reads the routing back."""
        if torch.cuda.is_current_stream_capturing():
            return False
        g, d = self._stk
        pairs, weights = n_pairs / self.num_experts, g["Q"] * g["P"] + d["Q"] * d["P"]
        if os.environ.get("QVB8_MOE_GROUPED", "1") == "0":           # the kernels are switched off
            return True
        if not (g["sliced"] and d["sliced"]) and (pairs > self.ODD_ROWS_MAX_PAIRS or weights > self.ODD_ROWS_MAX_WEIGHTS):
            return True
        return pairs >= self.LOOP_FROM_PAIRS and pairs * weights >= self.LOOP_FROM_PRODUCTS

    def _many_as_the_loop(self, x: torch.Tensor, idx: torch.Tensor, w: torch.Tensor) -> bool:
        """Whether the routed kernels do for more than FUSED_MAX_TOKENS tokens what the per-expert loop does.  They see neither
        autograd nor the experts' hooks; activations are narrowed to fp16, which the loop does not do to bf16 ones of packs
        certified for it; and calls of other types or layouts are the loop's, to answer or to refuse."""
        if x.dtype not in _KERNEL_DTYPES or idx.dtype not in _INDEX_DTYPES or not w.is_floating_point():
            return False
        if x.dim() != 2 or idx.dim() != 2 or w.shape != idx.shape or x.shape != (idx.shape[0], self.gate_up_experts[0].in_features):
            return False
        if idx.device != x.device or w.device != x.device or self.gate_up_experts[0].ids.device != x.device or not self._whole_steps():
            return False
        if torch.is_grad_enabled() and (x.requires_grad or w.requires_grad):
            return False
        if _has_any_global_hook() or getattr(self.act_fn, "_forward_hooks", None) or getattr(self.act_fn, "_forward_pre_hooks", None):
            return False
        bf16, fp16 = x.dtype == torch.bfloat16, x.dtype == torch.float16
        for stack in (self.gate_up_experts, self.down_experts):
            for m in stack._modules.values():
                if m._forward_hooks or m._forward_pre_hooks or (bf16 and m.bf16_certified) or (fp16 and m.fp16_table_missing):
                    return False
        return True

    def forward(self, hidden_states: torch.Tensor, top_k_index: torch.Tensor, top_k_weights: torch.Tensor) -> torch.Tensor:
        many = top_k_index.shape[0] > self.FUSED_MAX_TOKENS
        if hidden_states.is_cuda and (not many or self._many_as_the_loop(hidden_states, top_k_index, top_k_weights)) and self.build_stack():
            if not many:
                return self._routed(hidden_states, top_k_index, top_k_weights, False)
            if not self._loop_is_faster(top_k_index.numel()):
                out = self._routed_in_slices(hidden_states, top_k_index.to(torch.int64), top_k_weights)
                if out is not None:
                    return out
        return self._forward_loop(hidden_states, top_k_index, top_k_weights)

    def _routed_in_slices(self, x: torch.Tensor, idx: torch.Tensor, w: torch.Tensor):
        """_routed of many tokens, in equal slices of at most SCRATCH_BYTES of fp32 results (never as few tokens as the other
        kernels take)."""
        n_tok, per_token = idx.shape[0], 4 * idx.shape[1] * (self._stk[1]["P"] + self._stk[1]["Q"])
        n = -(-n_tok // max(self.FUSED_MAX_TOKENS + 1, self.SCRATCH_BYTES // per_token))
        while n > 1 and n_tok // n <= self.FUSED_MAX_TOKENS:
            n -= 1
        if n == 1:
            return self._routed(x, idx, w, True)
        out, at = [], 0
        for i in range(n):
            end = n_tok * (i + 1) // n
            part = self._routed(x[at:end], idx[at:end], w[at:end], True)
            if part is None:
                return None
            out.append(part)
            at = end
        return torch.cat(out)

    def _routed(self, x: torch.Tensor, idx: torch.Tensor, w: torch.Tensor, many: bool):
        """The routed kernels.  With more than FUSED_MAX_TOKENS tokens, None where an expert number lies outside 0..E-1: the loop
        counts negative ones from the end and refuses the others (inside a graph capture nothing can be read back: NaN)."""
        g, d = self._stk
        return ext.moe_experts(x.contiguous(), idx.contiguous(), w.float(),
                               g["ids"], g["min_s"], g["tau_s"], g["nbits"], g["bit_off"], g["Q"], g["P"],
                               d["ids"], d["min_s"], d["tau_s"], d["nbits"], d["bit_off"], d["Q"], d["P"],
                               regular=(g["regular"], d["regular"]), planes=(g["planes"], d["planes"]), keep_inf=many, checked=many and not torch.cuda.is_current_stream_capturing())

    def _forward_loop(self, hidden_states: torch.Tensor, top_k_index: torch.Tensor, top_k_weights: torch.Tensor) -> torch.Tensor:
        """The (token, choice) pairs sorted by expert once, then one pass per expert that was chosen: its tokens through
        its own gate+up and down modules, scaled by the routing weights and added to their rows in the hidden dtype
        (what the reference's loop computes, backends_experts.py:228-272).  One host sync, for the segment lengths."""
        top_k = top_k_index.shape[1]
        expert_of_pair, by_expert = torch.sort(top_k_index.reshape(-1), stable=True)
        chosen, n_pairs = torch.unique_consecutive(expert_of_pair, return_counts=True)
        token_of_pair = torch.div(by_expert, top_k, rounding_mode="floor")
        weight_of_pair = top_k_weights.reshape(-1)[by_expert]
        out = torch.zeros_like(hidden_states)
        at = 0
        for e, n in zip(chosen.tolist(), n_pairs.tolist()):
            rows = token_of_pair[at:at + n]
            gate, up = self.gate_up_experts[e](hidden_states[rows]).chunk(2, dim=-1)
            y = self.down_experts[e](self.act_fn(gate) * up)
            out.index_add_(0, rows, (y * weight_of_pair[at:at + n, None].to(y.dtype)).to(out.dtype))
            at += n
        return out
