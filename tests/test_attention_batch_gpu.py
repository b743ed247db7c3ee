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
