"""K/V ranges packed by one call: one range (arguments of its own size), two, a
full launch and one range more, with a row list and empty ranges among them,
against the copies that they stand for."""

import pytest

from tests.helpers import randn_bf16, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("ranges", [1, 2, 32, 33])
def test_pack_ranges(torch_mod, dev, dim, ranges):
    torch = torch_mod
    from taomate_hd_amd import KVSlot
    from taomate_hd_amd.slots import PackRows, vt_columns

    heads, total = 3, 400
    k, v = (to_dev(randn_bf16((total, heads, dim), seed), dev) for seed in (190, 191))
    counts = [0 if i == 1 else (1, 63, 64, 65, 100)[i % 5] for i in range(ranges)]
    items, at = [], 0
    for i, n in enumerate(counts):
        rows = torch.arange(n, device=dev) * 3 % total if i % 3 == 0 else None
        items.append(PackRows(rows=rows, row0=7 * i, count=n, dst=at) if rows is None else PackRows(rows=rows, dst=at))
        at += (n + 63) // 64 * 64
    slot = KVSlot(torch, heads=heads, head_dim=dim, capacity=at, device=dev)
    slot.k.fill_(9.0)
    slot.vt.fill_(9.0)
    slot.pack_ranges(k, v, items)
    want_k = torch.zeros(at, heads, dim, dtype=torch.bfloat16, device=dev)
    want_v = torch.zeros_like(want_k)
    for item, n in zip(items, counts):
        src = item.rows if item.rows is not None else torch.arange(item.row0, item.row0 + n, device=dev)
        want_k[item.dst : item.dst + n], want_v[item.dst : item.dst + n] = k[src], v[src]
    got_v = slot.vt.index_select(2, vt_columns(torch, at, dev)).permute(2, 0, 1)
    assert torch.equal(slot.k.permute(1, 0, 2), want_k) and torch.equal(got_v, want_v)
    assert slot.tokens == items[-1].dst + counts[-1]
