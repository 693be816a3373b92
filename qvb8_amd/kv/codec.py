"""Per-channel affine KV codec (reference: src/qv_band/kv/codec.py): fixed bits per element of a (seq, head_dim)
segment of one kv head, one (min_s, tau_s) per channel,

    id = round((x - min_c) / step_c),  step_c = (max_c - min_c) / (2^B - 1),  recon = min_c + id * step_c,

no escapes (minimum and maximum cover every value).  On the GPU the encoder is three launches of the HIP library (a fourth
packs the heads that need more than the width asked for, one more checks each time a head still misses its bound), on the CPU torch
ops; both give the same bits.  The ids are kept bit-packed, LSB first,
row-major (codec.py:53-82), as the cache stores them between attention calls.
"""
from __future__ import annotations

import ctypes
import math
from dataclasses import dataclass

import torch

from qvb8_amd import _lib

STEP_FLOOR = 1e-12
MAX_BITS = 16


class KVCertificateError(ValueError):
    """tau is below what 16 bits per element can certify for a head (codec.py:171-172)."""


def pack_ids(ids: torch.Tensor, bits: int) -> torch.Tensor:
    """Flat ids (< 2^bits) -> uint8, fields LSB first and bit-contiguous (codec.py:53-68)."""
    n = ids.numel()
    shifts = torch.arange(bits, device=ids.device, dtype=torch.int64)
    stream = ((ids.reshape(-1, 1).to(torch.int64) >> shifts) & 1).to(torch.uint8).reshape(-1)
    pad = (-stream.numel()) % 8
    if pad:
        stream = torch.cat([stream, stream.new_zeros(pad)])
    weights = (1 << torch.arange(8, device=ids.device, dtype=torch.int64)).to(torch.uint8)
    out = (stream.reshape(-1, 8) * weights).sum(dim=1, dtype=torch.int64).to(torch.uint8)
    assert out.numel() == (n * bits + 7) // 8
    return out


def unpack_ids(packed: torch.Tensor, bits: int, n: int) -> torch.Tensor:
    """Inverse of pack_ids: int64[n] (codec.py:71-82)."""
    shifts = torch.arange(8, device=packed.device, dtype=torch.int64)
    stream = ((packed.reshape(-1, 1).to(torch.int64) >> shifts) & 1).reshape(-1)[: n * bits].reshape(n, bits)
    return (stream << torch.arange(bits, device=packed.device, dtype=torch.int64)).sum(dim=1)


@dataclass(eq=False)
class BandedKV:
    """One kv head of one segment (codec.py:99-166)."""
    packed: torch.Tensor            # uint8, bits * seq * head_dim bits, row-major
    min_s: torch.Tensor             # (head_dim,) fp32
    tau_s: torch.Tensor             # (head_dim,) fp32 step per channel
    bits: int
    orig_shape: tuple               # (seq, head_dim)
    orig_dtype: torch.dtype
    tau: float

    def nbytes(self) -> int:
        return int(self.packed.numel() + 4 * (self.min_s.numel() + self.tau_s.numel()))

    @property
    def max_error(self) -> float:
        return float(self.tau_s.max()) * 0.5

    def ids(self) -> torch.Tensor:
        seq, hd = self.orig_shape
        return unpack_ids(self.packed, self.bits, seq * hd).reshape(seq, hd)

    def decode_all_torch(self, device=None, dtype=torch.float32) -> torch.Tensor:
        """min_s + id * tau_s in fp32, rounded once to `dtype` (codec.py:117-118)."""
        dev = self.packed.device if device is None else torch.device(device)
        ids = self.ids().to(dev)
        return (self.min_s.to(dev) + ids.to(torch.float32) * self.tau_s.to(dev)).to(dtype)

    def truncate(self, n_rows: int) -> "BandedKV":
        """The first n_rows tokens, not re-quantised: a byte prefix of `packed` (codec.py:120-139)."""
        seq, hd = self.orig_shape
        if not 0 < n_rows <= seq:
            raise ValueError(f"truncate({n_rows}) outside 1..{seq}")
        if n_rows == seq:
            return self
        nbytes = (n_rows * hd * self.bits + 7) // 8
        return BandedKV(self.packed[:nbytes].clone(), self.min_s, self.tau_s, self.bits, (n_rows, hd), self.orig_dtype, self.tau)


    def take_rows(self, rows: torch.Tensor) -> "BandedKV":
        """Only the given token rows (indices inside 0..seq-1), not re-quantised: the ids are unpacked, selected and
        packed again at the same width with the same constants (codec.py:141-158)."""
        seq, hd = self.orig_shape
        rows = rows.to(torch.int64)
        if rows.numel() == 0 or int(rows.min()) < 0 or int(rows.max()) >= seq:
            raise ValueError(f"take_rows indices must lie in 0..{seq - 1} and be non-empty")
        if rows.numel() == seq and bool((rows == torch.arange(seq, device=rows.device)).all()):
            return self
        kept = self.ids()[rows.to(self.packed.device)]
        return BandedKV(pack_ids(kept.reshape(-1), self.bits), self.min_s, self.tau_s, self.bits, (int(rows.numel()), hd),
                        self.orig_dtype, self.tau)

    def decode_all(self) -> torch.Tensor:
        return self.decode_all_torch("cpu", torch.float32)

    def decode_row(self, row_idx: int) -> torch.Tensor:
        return self.decode_all()[row_idx]

    outlier_count = property(lambda s: 0)           # minimum and maximum cover every value: there are no escapes
    outlier_ratio = property(lambda s: 0.0)


def unband_kv_4d(banded: list, batch: int, heads: int, device="cpu") -> torch.Tensor:
    """(batch, heads, seq, head_dim) in the cache's dtype from one BandedKV per head (codec.py:252-262)."""
    if not banded:
        return torch.empty(batch, heads, 0, 0, device=device)
    seq, dim = banded[0].orig_shape
    mats = [bk.decode_all_torch(device, banded[0].orig_dtype) for bk in banded]
    return torch.stack(mats, dim=0).reshape(batch, heads, seq, dim)


def _channel_grid(x, lo, span, widths):
    """Nearest point of each channel's grid of 2^w - 1 intervals over [lo, lo + span] (w per head): (ids, step)."""
    levels = torch.tensor([float((1 << w) - 1) for w in widths], device=x.device).view(-1, 1, 1)
    step = (span / levels).clamp_min(STEP_FLOOR)
    return torch.minimum(torch.round((x - lo) / step).clamp_(min=0), levels), step


def _first_width(widest: float, bits: int, tau: float) -> int:
    """The least width that puts half a step of the widest channel within tau, `bits` at least."""
    return min(MAX_BITS, max(bits, math.ceil(math.log2(widest / (2.0 * tau) + 1.0)))) if widest > 0 else bits


def _next_width(head: int, width: int, off: float, tau: float, orig_dtype) -> int:
    if width >= MAX_BITS:
        raise KVCertificateError(f"head {head}: at {MAX_BITS} bits the per-channel grid is still {off:.4g} off, "
                                 f"tau = {tau:g} cannot be certified for values stored as {orig_dtype}")
    return width + 1


_KV_MAX_DIM = 2048                         # channels per head the kernels take
_STORED_DTYPES = (torch.float32, torch.float16, torch.bfloat16)


def _band_on_gpu(t, orig_dtype, bits: int, tau: float, certify: bool) -> list:
    """band_kv_heads on the HIP library: ranges, and the least widths with the error they leave; while those figures are on their way to
    the host, the ids are packed at the width asked for.  Heads that need more are checked again, one bit wider while they still miss
    tau, and packed again.  Keys of 4 heads x 4096 x 256: 38 us a call as asked, 44 when one head needs more, 48 when all do (65 in each
    case with the widths awaited before the first id is packed); 32 heads x 4096 x 128: 113, 122, 166 (178)."""
    heads, seq, dim = t.shape
    x = t.detach()
    x = (x if x.dtype in _STORED_DTYPES else x.to(torch.float32)).contiguous()
    lib, dev, dt, odt = _lib.load(), x.device, _lib.dtype_code(x.dtype), _lib.dtype_code(orig_dtype)
    certifying = bool(certify and tau > 0)
    with _lib.on_device_of(x):
        stream, x_at = _lib.stream_of(x), x.data_ptr()
        grid = torch.empty((3, heads, dim), dtype=torch.float32, device=dev)                          # minima, steps, spans
        lo_at, step_at, span_at = (grid.data_ptr() + 4 * heads * dim * i for i in range(3))

        def pack(packed, widths, x_at=x_at, skip=0):
            """Some neighbouring heads into their streams, the first one's values at x_at, its constants `skip` bytes into theirs."""
            n = len(packed)
            where = (ctypes.c_void_p * n)(*[p.data_ptr() for p in packed])
            _lib._check(lib.qvb8_kv_pack(x_at, dt, n, seq, dim, lo_at + skip, span_at + skip, bytes(widths), step_at + skip, where, stream), lib)

        widths, stored = [bits] * heads, (seq * dim * bits + 7) // 8
        if not certifying:
            chunks = lib.qvb8_kv_chunks(heads, seq)
            partial = torch.empty(heads * chunks * 2 * dim, dtype=torch.float32, device=dev)
            _lib._check(lib.qvb8_kv_range(x_at, dt, heads, seq, dim, partial.data_ptr(), chunks, stream), lib)
            _lib._check(lib.qvb8_kv_check(x_at, dt, heads, seq, dim, partial.data_ptr(), chunks, odt, bits, float(tau), None, lo_at, span_at, None, stream), lib)
            packed = [torch.empty(stored, dtype=torch.uint8, device=dev) for _ in widths]
            pack(packed, widths)
            los, steps = (g.unbind(0) for g in grid[:2].unbind(0))
        else:
            scratch = torch.empty(lib.qvb8_kv_measure_floats(heads, seq, dim), dtype=torch.float32, device=dev)
            shown = torch.empty(3 * heads, dtype=torch.float32, pin_memory=True)
            _lib._check(lib.qvb8_kv_measure(x_at, dt, heads, seq, dim, odt, bits, float(tau), scratch.data_ptr(), lo_at, span_at, shown.data_ptr(), stream), lib)
            try:
                packed = [torch.empty(stored, dtype=torch.uint8, device=dev) for _ in widths]
                pack(packed, widths)
                los, steps = (g.unbind(0) for g in grid[:2].unbind(0))
            finally:
                _lib._check(lib.qvb8_kv_wait(shown.data_ptr(), heads, stream), lib)       # the figures are written whatever happened since
            found = shown.tolist()
            widths = [_first_width(found[3 * i], bits, tau) for i in range(heads)]
            errors = found[2::3]

            def check():
                chunks = lib.qvb8_kv_chunks(heads, seq)
                report = torch.empty((heads, 2 + chunks), dtype=torch.float32, pin_memory=True)
                _lib._check(lib.qvb8_kv_check(x_at, dt, heads, seq, dim, scratch.data_ptr(), chunks, odt, bits, float(tau), bytes(widths), lo_at, span_at,
                                              report.data_ptr(), stream), lib)
                torch.cuda.current_stream().synchronize()
                return report[:, 2:].amax(1).tolist()

            if widths != [int(w) for w in found[1::3]]:          # a span on the edge of a power of two: the host's logarithm decides
                errors = check()
            while not all(e <= tau for e in errors):
                widths = [w if e <= tau else _next_width(i, w, e, tau, orig_dtype) for i, (w, e) in enumerate(zip(widths, errors))]
                errors = check()
            if widths != [bits] * heads:                         # one launch over the heads that rose and what lies between (the same bytes again)
                risen = [i for i, w in enumerate(widths) if w != bits]
                for i in risen:
                    packed[i] = torch.empty((seq * dim * widths[i] + 7) // 8, dtype=torch.uint8, device=dev)
                a, b = risen[0], risen[-1] + 1
                pack(packed[a:b], widths[a:b], x_at + a * seq * dim * x.element_size(), 4 * dim * a)
    return [BandedKV(p, m, s, w, (seq, dim), orig_dtype, tau) for p, m, s, w in zip(packed, los, steps, widths)]


def band_kv_heads(t: torch.Tensor, orig_dtype: torch.dtype, bits: int, tau: float = 0.0, certify: bool = True) -> list:
    """(heads, seq, head_dim) -> one BandedKV per head (codec.py:175-241).  With certify and tau > 0, `bits` is a floor:
    a head's width rises (to 16 at most) until the decoder's own expression, rounded to `orig_dtype`, is within tau of
    every element; KVCertificateError when 16 bits do not reach it.  Heads are independent: only the heads that still
    miss tau are quantised again, one host read per round."""
    heads, seq, dim = t.shape
    if t.is_cuda and 0 < heads <= _lib.KV_MAX_HEADS and seq > 0 and 0 < dim <= _KV_MAX_DIM and seq * dim < 1 << 31 and 1 <= bits <= MAX_BITS \
            and orig_dtype in _STORED_DTYPES:
        return _band_on_gpu(t, orig_dtype, bits, tau, certify)
    x = torch.nan_to_num(t.detach().to(torch.float32), nan=0.0, posinf=0.0, neginf=0.0)
    lo = x.amin(1, keepdim=True)
    span = x.amax(1, keepdim=True) - lo
    widths = [bits] * heads
    open_heads = []
    if certify and tau > 0:
        open_heads = list(range(heads))
        for i, widest in enumerate(span.amax((1, 2)).cpu().tolist()):     # first guess: half a step within tau
            widths[i] = _first_width(widest, bits, tau)
    ids, step = _channel_grid(x, lo, span, widths)
    while open_heads:
        sel = torch.tensor(open_heads, device=x.device)
        shown = (lo[sel] + ids[sel] * step[sel]).to(orig_dtype).to(torch.float32)      # what the decoder will hand out
        miss = (shown - x[sel]).abs().amax((1, 2)).cpu().tolist()
        open_heads = [i for i, e in zip(open_heads, miss) if e > tau]
        if not open_heads:
            break
        worst = dict(zip(sel.tolist(), miss))
        for i in open_heads:
            widths[i] = _next_width(i, widths[i], worst[i], tau, orig_dtype)
        sel = torch.tensor(open_heads, device=x.device)
        ids[sel], step[sel] = _channel_grid(x[sel], lo[sel], span[sel], [widths[i] for i in open_heads])
    return [BandedKV(pack_ids(ids[i].to(torch.int64).reshape(-1), widths[i]), lo[i, 0].contiguous(), step[i, 0].contiguous(),
                     widths[i], (seq, dim), orig_dtype, tau) for i in range(heads)]
