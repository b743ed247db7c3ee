"""Segment attention: the functional entry to the HIP attention kernels.

``segment_attention`` computes ``softmax(q k^T * scale) v`` for a selection of
token-major query rows over an ordered table of slot segments (no mask), as
``torch.nn.functional.scaled_dot_product_attention(..., is_causal=False)``
does over the concatenated K/V in the reference
(src/taomate_hd/streaming/attention_hook.py:100-115).  ``backend="i8qk"`` runs
the SageAttention-style variant (smooth-K, per-128-block INT8 Q/K, bf16 P.V;
ref attention_hook.py:335-371, inference/sage_value_padding.py:79-97).
"""

from __future__ import annotations

import ctypes
from dataclasses import dataclass
from typing import Any, Sequence

from . import _native
from .profiling import ComponentTimer, maybe_region
from .slots import KV_TILE, KVSlot, SlotView, round_up, vt_columns

BACKENDS = ("bf16", "i8qk")


class QKQuantWorkspace:
    """Grow-only INT8-QK operand storage, keyed by (device, stream).

    Work on one stream is ordered, so a call may reuse the buffers of the
    previous call on that stream without synchronising.  ``nbytes`` reports
    what it holds and ``release`` returns it to the allocator.
    """

    def __init__(self, torch: Any) -> None:
        self._torch = torch
        self._buffers: dict[tuple[Any, ...], dict[str, Any]] = {}

    @property
    def nbytes(self) -> int:
        return sum(int(t.numel()) * t.element_size() for store in self._buffers.values() for t in store.values())

    def release(self) -> None:
        self._buffers.clear()

    def _grow(self, store: dict[str, Any], name: str, numel: int, dtype: Any, device: Any) -> Any:
        buf = store.get(name)
        if buf is None or buf.numel() < numel:
            buf = self._torch.empty(max(numel, 1), dtype=dtype, device=device)
            store[name] = buf
        return buf

    def quant_struct(self, *, heads: int, head_dim: int, lq: int, tokens: Sequence[int], device: Any) -> tuple[Any, dict[str, Any]]:
        structs, views = self.quant_structs(heads=heads, head_dim=head_dim, calls=[(lq, tokens)], device=device,
                                            with_views=True)
        return structs[0], views[0]

    def quant_structs(self, *, heads: int, head_dim: int, calls: Sequence[tuple[int, Sequence[int]]], device: Any,
                      with_views: bool = False) -> tuple[Any, list[dict[str, Any]]]:
        """The operands of ``calls`` (query rows, segment tokens) side by side in
        this stream's buffers: an array of structs, and with ``with_views`` a
        dict of tensors per call."""
        torch = self._torch
        key = (str(device), _native.stream_ptr(torch, device))
        store = self._buffers.setdefault(key, {})
        # 256-byte aligned carve-out offsets inside the int8 and fp32 buffers
        plan, q_total, qs_total, k_total, ks_total = [], 0, 0, 0, 0
        for lq, tokens in calls:
            qcap = round_up(max(lq, 1), _native.QUERY_TILE)
            segs = []
            for t in tokens:
                cap = round_up(t, KV_TILE)
                nblk = round_up(cap, _native.QUANT_BLOCK) // _native.QUANT_BLOCK
                segs.append((cap, nblk, k_total, ks_total))
                k_total += round_up(heads * cap * head_dim, 256)
                ks_total += round_up(heads * nblk, 64)
            plan.append((qcap, q_total, qs_total, segs))
            q_total += heads * qcap * head_dim
            qs_total += round_up(heads * (qcap // _native.QUANT_BLOCK), 64)
        n = len(plan)
        width = heads * head_dim
        q_i8 = self._grow(store, "q_i8", q_total, torch.int8, device)
        q_scale = self._grow(store, "q_scale", qs_total, torch.float32, device)
        k_i8 = self._grow(store, "k_i8", k_total, torch.int8, device)
        k_scale = self._grow(store, "k_scale", ks_total, torch.float32, device)
        k_mean = self._grow(store, "k_mean", n * width, torch.bfloat16, device)
        q_at, qs_at, k_at, ks_at, mean_at = (_native.ptr(t) for t in (q_i8, q_scale, k_i8, k_scale, k_mean))
        structs = (_native.QKQuant * n)()
        views = []
        for i, (qcap, q_off, qs_off, segs) in enumerate(plan):
            qq = structs[i]
            qq.q_i8 = q_at + q_off
            qq.q_scale = qs_at + 4 * qs_off
            qq.q_head_stride = qcap * head_dim
            qq.q_scale_head_stride = qcap // _native.QUANT_BLOCK
            for j, (cap, nblk, k_off, s_off) in enumerate(segs):
                qq.k_i8[j] = k_at + k_off
                qq.k_scale[j] = ks_at + 4 * s_off
                qq.k_head_stride[j] = cap * head_dim
                qq.k_scale_head_stride[j] = nblk
            qq.k_mean = mean_at + 2 * i * width
            if with_views:
                views.append({
                    "q_i8": q_i8[q_off : q_off + heads * qcap * head_dim].view(heads, qcap, head_dim),
                    "q_scale": q_scale[qs_off : qs_off + heads * (qcap // _native.QUANT_BLOCK)].view(heads, -1),
                    "k_mean": k_mean[i * width : (i + 1) * width].view(heads, head_dim),
                    "k_i8": [k_i8[o : o + heads * c * head_dim].view(heads, c, head_dim) for c, _, o, _ in segs],
                    "k_scale": [k_scale[o : o + heads * b].view(heads, b) for _, b, _, o in segs],
                })
        return structs, views


_SPLIT_WORKSPACES: dict[tuple[Any, ...], Any] = {}


def split_workspace(torch: Any, device: Any, head_dim: int) -> Any:
    """Scratch for the key-range split of an attention call's last round.

    One uint8 buffer per (device, stream), grown to what the library asks for
    on that device; calls on one stream are ordered, so they share it.
    """
    need = int(_native.load().tmhd_attn_split_workspace_bytes(int(head_dim)))
    key = (str(device), _native.stream_ptr(torch, device))
    buf = _SPLIT_WORKSPACES.get(key)
    if buf is None or buf.numel() < need:
        buf = torch.empty(max(need, 1), dtype=torch.uint8, device=device)
        _SPLIT_WORKSPACES[key] = buf
    return buf


def split_workspace_bytes() -> int:
    """Bytes held by the split workspaces of every (device, stream) so far."""
    return sum(int(buf.numel()) for buf in _SPLIT_WORKSPACES.values())


def release_split_workspaces() -> None:
    """Return the split workspaces to the allocator (the next call regrows its own)."""
    _SPLIT_WORKSPACES.clear()


def _validate_tokens_major(torch: Any, tensor: Any, name: str) -> None:
    _native.require_device_tensor(torch, tensor, name)
    if tensor.dtype != torch.bfloat16 or tensor.ndim != 3 or tensor.stride(2) != 1:
        raise ValueError(f"{name} must be a [tokens, heads, dim] bf16 view with unit dim stride")


def _row_list(torch: Any, rows: Any, device: Any, limit: int, name: str, checked: bool) -> Any:
    """A row list as a contiguous int32 tensor on ``device`` with entries in
    [0, limit).  The range check reads the list's min / max back (one sync);
    callers whose lists are valid by construction pass ``checked``."""
    if not torch.is_tensor(rows) or rows.device != torch.device(device):
        raise ValueError(f"{name} must be a tensor on the GPU of the rows it indexes")
    if rows.dtype not in (torch.int32, torch.int64):
        raise ValueError(f"{name} must be an int32 or int64 tensor")
    rows = rows.reshape(-1)
    if not checked and rows.numel():
        # on the list as given: an int64 entry past 2^31 must not wrap into range
        lo, hi = (int(v) for v in torch.aminmax(rows))
        if lo < 0 or hi >= limit:
            raise ValueError(f"{name} entries must lie in [0, {limit})")
    return rows.to(torch.int32).contiguous()


def _key_sums(torch: Any, segments: Sequence[SlotView], stream: int, qq: Any, out: Any, base: int,
              new: dict[tuple[KVSlot, tuple[int, int, int]], Any]) -> None:
    """Where the exact fixed-point key sums of each segment (the smooth-K mean's
    terms) are or go, memoised on its slot per (row0, tokens, stream): a cached
    block's keys are summed once, not on every call.  The slot drops the memo
    whenever it is written.  Sums that this batch takes go to ``new``: the
    caller memoises them once their kernels are queued (a refused batch must
    not leave unfilled ones behind)."""
    for j, view in enumerate(segments):
        slot = view.slot
        key = (int(view.row0), int(view.tokens), int(stream))
        hit = slot.key_sums.get(key)
        if hit is None:
            hit = new.get((slot, key))
        if hit is None:
            hit = new[slot, key] = torch.empty((slot.heads, slot.head_dim), dtype=torch.int64, device=slot.device)
            out[base + j] = _native.ptr(hit)  # summed by this batch
        else:
            qq.k_sum[j] = _native.ptr(hit)


def _coalesce_segments(torch: Any, segments: list[SlotView], limit: int) -> list[SlotView]:
    """One launch takes at most ``limit`` segments; the reference has no such
    bound (it concatenates every part).  With more, the oldest segments are
    copied, in order, into one temporary slot: their keys stay the same keys,
    so the result is the attention over the same set (the INT8-QK key blocks
    then run over the merged rows, as they run over any segment)."""
    n_merge = len(segments) - limit + 1
    head, rest = segments[:n_merge], segments[n_merge:]
    keys, values = [], []
    for view in head:
        slot, r0, n = view.slot, int(view.row0), int(view.tokens)
        keys.append(slot.k[:, r0 : r0 + n, :].permute(1, 0, 2))
        cols = r0 + vt_columns(torch, n, slot.device)  # r0 is a multiple of 64: whole 16-token groups
        values.append(slot.vt.index_select(2, cols).permute(2, 0, 1))
    key, value = torch.cat(keys, 0).contiguous(), torch.cat(values, 0).contiguous()
    first = head[0].slot
    merged = KVSlot(torch, heads=first.heads, head_dim=first.head_dim, capacity=int(key.shape[0]), device=first.device)
    merged.pack(key, value)
    return [merged.view(), *rest]


def segment_attention(
    torch: Any,
    query: Any,
    segments: Sequence[SlotView],
    *,
    scale: float,
    backend: str = "bf16",
    q_rows: Any | None = None,
    q_row0: int = 0,
    lq: int | None = None,
    out: Any | None = None,
    o_rows: Any | None = None,
    o_row0: int = 0,
    workspace: QKQuantWorkspace | None = None,
    split: bool = True,
    return_quant: bool = False,
    timer: ComponentTimer | None = None,
    rows_checked: bool = False,
) -> Any:
    """Attention of the selected query rows over ``segments`` (in place, no mask).

    Query row ``i`` is ``query[q_rows[i]]`` (or ``query[q_row0 + i]``); its
    output goes to ``out[o_rows[i]]`` (or ``out[o_row0 + i]``).  Without
    ``out`` a new ``[lq, H, D]`` tensor is returned.  ``split`` lets the
    library run the items of a partial last round as key ranges (merged on
    the same stream); results agree with the unsplit run to fp32 rounding.
    Row lists are device tensors; their range is checked (one sync) unless
    ``rows_checked`` says the caller built them in range.
    """
    outs, views = segment_attention_batch(
        torch,
        [AttentionCall(query, segments, q_rows=q_rows, q_row0=q_row0, lq=lq, out=out, o_rows=o_rows, o_row0=o_row0,
                       rows_checked=rows_checked)],
        scale=scale, backend=backend, workspace=workspace, split=split, return_quant=return_quant, timer=timer,
    )
    return (outs[0], views[0]) if return_quant and backend == "i8qk" else outs[0]


@dataclass
class AttentionCall:
    """One call of ``segment_attention_batch``: the arguments of
    ``segment_attention`` that belong to a single call."""

    query: Any
    segments: Sequence[SlotView]
    q_rows: Any | None = None
    q_row0: int = 0
    lq: int | None = None
    out: Any | None = None
    o_rows: Any | None = None
    o_row0: int = 0
    rows_checked: bool = False


def _call_args(torch: Any, call: AttentionCall, args: Any, scale: float, keep: list[Any]) -> tuple[Any, list[SlotView]]:
    """Check one call and fill its C arguments; returns its output and segments."""
    query, out, q_rows, o_rows, lq = call.query, call.out, call.q_rows, call.o_rows, call.lq
    q_row0, o_row0 = int(call.q_row0), int(call.o_row0)
    _validate_tokens_major(torch, query, "query")
    rows_in, heads, head_dim = query.shape
    if q_rows is not None:
        q_rows = _row_list(torch, q_rows, query.device, rows_in, "q_rows", call.rows_checked)
        keep.append(q_rows)
        n = int(q_rows.numel())
        if lq is not None and int(lq) != n:
            raise ValueError("lq differs from the query row list")
        lq = n
    elif lq is None:
        lq = rows_in - q_row0
    lq = int(lq)
    if out is None:
        out = torch.empty((lq, heads, head_dim), dtype=torch.bfloat16, device=query.device)
        o_rows, o_row0 = None, 0
    _validate_tokens_major(torch, out, "out")
    if tuple(out.shape[1:]) != (heads, head_dim):
        raise ValueError("out heads/dim differ from query")
    if o_rows is not None:
        o_rows = _row_list(torch, o_rows, out.device, int(out.shape[0]), "o_rows", call.rows_checked)
        keep.append(o_rows)
        if int(o_rows.numel()) != lq:
            raise ValueError("output row list length differs from the query rows")
    elif not (0 <= o_row0 and o_row0 + lq <= int(out.shape[0])):
        raise ValueError(f"output rows [{o_row0}, {o_row0 + lq}) outside out ({int(out.shape[0])} rows)")
    if q_rows is None and not (0 <= q_row0 and q_row0 + lq <= rows_in):
        raise ValueError(f"query rows [{q_row0}, {q_row0 + lq}) outside query ({rows_in} rows)")
    segments = [s for s in call.segments if s.tokens > 0]
    if not segments:
        raise ValueError("attention needs at least one key/value token")
    for s in segments:
        if s.slot.heads != heads or s.slot.head_dim != head_dim or s.slot.device != query.device:
            raise ValueError("segment heads/dim/device differ from the query")
    if len(segments) > _native.MAX_SEGMENTS:
        segments = _coalesce_segments(torch, segments, _native.MAX_SEGMENTS)
        keep.append(segments)
    args.q = _native.ptr(query)
    args.q_token_stride = query.stride(0)
    args.q_head_stride = query.stride(1)
    args.q_rows = _native.ptr(q_rows) if q_rows is not None and lq else None
    args.q_row0 = q_row0
    args.lq = lq
    args.o = _native.ptr(out)
    args.o_token_stride = out.stride(0)
    args.o_head_stride = out.stride(1)
    args.o_rows = _native.ptr(o_rows) if o_rows is not None and lq else None
    args.o_row0 = o_row0
    args.heads = heads
    args.head_dim = head_dim
    args.scale = scale
    args.n_segments = len(segments)
    for i, s in enumerate(segments):
        s.fill_segment(args.seg[i])
    return out, segments


def segment_attention_batch(
    torch: Any,
    calls: Sequence[AttentionCall],
    *,
    scale: float,
    backend: str = "bf16",
    workspace: QKQuantWorkspace | None = None,
    split: bool = True,
    return_quant: bool = False,
    timer: ComponentTimer | None = None,
) -> tuple[list[Any], list[dict[str, Any]]]:
    """Independent ``segment_attention`` calls in one kernel launch (see
    ``tmhd_attn_fwd_bf16_batch``): a hook call's condition, media and padding
    attention, or a packed sequence's documents, none of which alone fills the
    GPU's last round of workgroups.  The calls share heads, head_dim and the
    query and output strides; their output rows must not overlap.  Returns
    their outputs, and with ``return_quant`` the INT8-QK operand views."""
    if backend not in BACKENDS:
        raise ValueError(f"unknown attention backend {backend!r}")
    if not calls:
        return [], []
    keep: list[Any] = []  # row lists and merged slots, alive until the launches are queued
    args = (_native.AttnArgs * len(calls))()
    outs, segments = [], []
    for i, call in enumerate(calls):
        out, segs = _call_args(torch, call, args[i], float(scale), keep)
        outs.append(out)
        segments.append(segs)
    device, heads, head_dim = calls[0].query.device, args[0].heads, args[0].head_dim
    if any(call.query.device != device or out.device != device for call, out in zip(calls, outs)):
        raise ValueError("the queries and outputs of a batch must share one GPU")
    lib = _native.load()
    stream = _native.stream_ptr(torch, device)
    if split and any(a.lq for a in args):
        ws = split_workspace(torch, device, head_dim)
        args[0].split_workspace = _native.ptr(ws)
        args[0].split_workspace_bytes = int(ws.numel())
    if backend == "bf16":
        with maybe_region(timer, "attention"):
            status = lib.tmhd_attn_fwd_bf16_batch(args, len(calls), stream)
        _native.check(status, "tmhd_attn_fwd_bf16")
        return outs, []
    if workspace is None:
        workspace = QKQuantWorkspace(torch)
    quants, views = workspace.quant_structs(
        heads=heads, head_dim=head_dim, calls=[(a.lq, [s.tokens for s in segs]) for a, segs in zip(args, segments)],
        device=device, with_views=return_quant,
    )
    with maybe_region(timer, "qk_quant"):
        sums = (ctypes.c_void_p * (_native.MAX_SEGMENTS * len(calls)))()
        new_sums: dict[tuple[KVSlot, tuple[int, int, int]], Any] = {}
        for i, segs in enumerate(segments):
            _key_sums(torch, segs, stream, quants[i], sums, i * _native.MAX_SEGMENTS, new_sums)
        status = lib.tmhd_qk_smooth_quant_batch(args, quants, sums, len(calls), stream)
    _native.check(status, "tmhd_qk_smooth_quant")
    for (slot, key), value in new_sums.items():
        slot.key_sums[key] = value
    with maybe_region(timer, "attention"):
        status = lib.tmhd_attn_fwd_i8qk_batch(args, quants, len(calls), stream)
    _native.check(status, "tmhd_attn_fwd_i8qk")
    return outs, views
