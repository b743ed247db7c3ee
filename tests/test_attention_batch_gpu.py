"""The dealing of a last, partial round of attention items to workgroups: calls
whose items are cut into ranges that do not divide evenly, so that a
workgroup's share begins in one item and ends in another."""

from __future__ import annotations

import pytest

from oracle import attention as oatt
from oracle import bf16
from tests.helpers import err_stats, key_offset, randn_bf16, to_dev

pytestmark = pytest.mark.gpu


def _slots(torch, dev, k, v, splits):
    from taomate_hd_amd import KVSlot

    views, off = [], 0
    for n in splits:
        slot = KVSlot(torch, heads=k.shape[1], head_dim=k.shape[2], capacity=n, device=dev)
        slot.pack(to_dev(k[off : off + n], dev), to_dev(v[off : off + n], dev))
        views.append(slot.view())
        off += n
    return views


@pytest.mark.parametrize("backend", ["bf16", "i8qk"])
@pytest.mark.parametrize(
    "heads,dim,lq,splits",
    [
        (14, 128, 2717, [331, 3000, 1]),  # 154 items of 54 key tiles: shares of several ranges of two items
        (3, 128, 130, [2000]),  # 3 items: every one cut into many ranges
        (37, 128, 2049, [1500, 37]),  # 333 items: a whole round, then 77 (the last query tile of one row)
        (8, 64, 256, [768, 256]),  # 8 items of 16 key tiles
        (45, 64, 1025, [700, 900]),  # 225 items, most of a round
    ],
)
def test_shared_out_ranges_match_whole_items(torch_mod, dev, backend, heads, dim, lq, splits):
    torch = torch_mod
    from taomate_hd_amd import segment_attention

    n = sum(splits)
    q = randn_bf16((lq, heads, dim), 140)
    k = randn_bf16((n, heads, dim), 141, offset=key_offset(heads, dim, 143))
    v = randn_bf16((n, heads, dim), 142)
    views = _slots(torch, dev, k, v, splits)
    qd = to_dev(q, dev)
    whole = segment_attention(torch, qd, views, scale=dim ** -0.5, backend=backend, split=False)
    split = segment_attention(torch, qd, views, scale=dim ** -0.5, backend=backend)
    torch.cuda.synchronize()
    a, b = bf16.from_torch(whole), bf16.from_torch(split)
    # same scores and probabilities, other summation order: outputs below 4 in
    # magnitude, so one bf16 step is at most 1.6e-2
    mx, mean = err_stats(b, a)
    assert mx <= 1.6e-2 and mean <= 2e-4, (mx, mean)
    if backend == "bf16":
        hs = [0, heads // 2, heads - 1]
        want = oatt.attention_fp64(q[:, hs], k[:, hs], v[:, hs], dim ** -0.5)
        mx, mean = err_stats(b[:, hs], want)
        assert mx <= 2e-2 and mean <= 1e-3, (mx, mean)


@pytest.mark.parametrize("backend", ["bf16", "i8qk"])
@pytest.mark.parametrize(
    "heads,dim,docs,shared",
    [
        (14, 128, [300, 1, 64, 65, 513], True),  # a shared segment in front of every document's own
        (3, 64, [33, 257, 256, 0, 700], False),  # a call without queries
        (2, 128, list(range(1, 20)), True),  # more calls and segments than one launch takes (16, 24)
    ],
)
def test_batch_matches_single_calls(torch_mod, dev, backend, heads, dim, docs, shared):
    """A batch gives what its calls give alone: for INT8-QK the same operands bit
    for bit (with the key sums taken in the batch), and outputs that differ only
    by where the ranges of the last round are cut; one call reads its rows
    through a row list."""
    torch = torch_mod
    from taomate_hd_amd import KVSlot, segment_attention
    from taomate_hd_amd.attention import AttentionCall, QKQuantWorkspace, segment_attention_batch
    from taomate_hd_amd.slots import PackRows, SlotView, round_up

    lengths = [max(n, 1) for n in docs]  # keys of each document; docs: its queries
    total = sum(lengths)
    q = to_dev(randn_bf16((total, heads, dim), 150), dev)
    k = to_dev(randn_bf16((total, heads, dim), 151, offset=key_offset(heads, dim, 153)), dev)
    v = to_dev(randn_bf16((total, heads, dim), 152), dev)
    slot = KVSlot(torch, heads=heads, head_dim=dim, capacity=sum(round_up(n, 64) for n in lengths), device=dev)
    alone = KVSlot(torch, heads=heads, head_dim=dim, capacity=slot.capacity, device=dev)
    for s in (slot, alone):
        s.k.fill_(9.0)
        s.vt.fill_(9.0)
    at, row, ranges, starts = 0, 0, [], []
    for n in lengths:
        starts.append((row, at))
        rows = torch.arange(row, row + n, device=dev) if n % 2 else None
        ranges.append(PackRows(rows, row, n, at))
        alone.pack(k, v, row0=row, count=n, dst=at)
        row, at = row + n, at + round_up(n, 64)
    slot.pack_ranges(k, v, ranges)
    torch.cuda.synchronize()
    assert torch.equal(slot.k.view(torch.int16), alone.k.view(torch.int16))
    assert torch.equal(slot.vt.view(torch.int16), alone.vt.view(torch.int16))
    assert slot.tokens == alone.tokens
    first = SlotView(slot, lengths[0], 0)

    def views(i):
        own = SlotView(slot, lengths[i], starts[i][1])
        return [first, own] if shared and i else [own]

    out = torch.full_like(q, 7.0)
    calls = []
    for i, n in enumerate(docs):
        rows = dict(q_row0=starts[i][0], lq=n, o_row0=starts[i][0])
        if i == 1:
            index = torch.arange(starts[i][0], starts[i][0] + n, device=dev, dtype=torch.int32)
            rows = dict(q_rows=index, o_rows=index)
        calls.append(AttentionCall(q, views(i), out=out, **rows))
    outs, quants = segment_attention_batch(torch, calls, scale=dim ** -0.5, backend=backend,
                                           workspace=QKQuantWorkspace(torch), return_quant=True)
    assert all(o is out for o in outs)
    torch.cuda.synchronize()
    for i, n in enumerate(docs):
        ref = torch.full_like(q, 7.0)
        got = segment_attention(torch, q, [SlotView(alone, x.tokens, x.row0) for x in views(i)], scale=dim ** -0.5,
                                backend=backend, q_row0=starts[i][0], lq=n, out=ref, o_row0=starts[i][0],
                                workspace=QKQuantWorkspace(torch), return_quant=backend == "i8qk")
        torch.cuda.synchronize()
        rows = slice(starts[i][0], starts[i][0] + n)
        if backend == "i8qk":
            want = got[1]
            nq = round_up(n, 256)
            assert torch.equal(quants[i]["k_mean"].view(torch.int16), want["k_mean"].view(torch.int16)), i
            assert torch.equal(quants[i]["q_i8"][:, :nq], want["q_i8"][:, :nq]), i
            assert torch.equal(quants[i]["q_scale"][:, : nq // 128], want["q_scale"][:, : nq // 128]), i
            for a, b in zip(quants[i]["k_i8"] + quants[i]["k_scale"], want["k_i8"] + want["k_scale"]):
                assert torch.equal(a, b), i
        if n:
            # outputs below 4 in magnitude: one bf16 step is at most 1.6e-2
            mx, mean = err_stats(bf16.from_torch(out[rows]), bf16.from_torch(ref[rows]))
            assert mx <= 1.6e-2 and mean <= 2e-4, (i, mx, mean)
        else:
            assert torch.equal(out[rows], ref[rows])


@pytest.mark.parametrize("backend", ["bf16", "i8qk"])
@pytest.mark.parametrize("dim,lq,n", [(128, 300, 200), (64, 70, 130), (128, 257, 2000)])
def test_output_rows_aligned_to_8_bytes(torch_mod, dev, backend, dim, lq, n):
    """Output rows that 16-byte stores do not fit (8-byte aligned base and
    strides), whole items and cut ones (the last shape), with output rows in
    reverse order: the values of the aligned output, nothing else touched."""
    torch = torch_mod
    from taomate_hd_amd import segment_attention

    heads = 3
    q = to_dev(randn_bf16((lq, heads, dim), 160), dev)
    views = _slots(torch, dev, randn_bf16((n, heads, dim), 161), randn_bf16((n, heads, dim), 162), [n])
    ref = segment_attention(torch, q, views, scale=dim ** -0.5, backend=backend)
    base = torch.full((lq + 2, heads, dim + 12), 7.0, dtype=torch.bfloat16, device=dev)
    out = base[:, :, 4 : 4 + dim]
    order = torch.arange(lq, 0, -1, device=dev, dtype=torch.int32)
    segment_attention(torch, q, views, scale=dim ** -0.5, backend=backend, out=out, o_rows=order)
    torch.cuda.synchronize()
    assert torch.equal(out[1 : lq + 1].flip(0).view(torch.int16), ref.view(torch.int16))
    assert bool((base[:, :, :4] == 7.0).all()) and bool((base[:, :, 4 + dim :] == 7.0).all())
    assert bool((base[0] == 7.0).all()) and bool((base[lq + 1] == 7.0).all())
