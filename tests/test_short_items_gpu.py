"""Attention items of few query rows, whose results go out straight from the
registers: bit for bit the rows of a full item, which go through LDS, and no
other row written."""

from __future__ import annotations

import pytest

from tests.helpers import key_offset, randn_bf16, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("backend", ["bf16", "i8qk"])
@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("lead", [0, 256])
@pytest.mark.parametrize("rows", ["range", "list", "unaligned"])
def test_rows_of_a_short_item(torch_mod, dev, backend, dim, lead, rows):
    torch = torch_mod
    from taomate_hd_amd import KVSlot, segment_attention

    heads, n, full = 3, 150, lead + 256
    q = randn_bf16((full, heads, dim), 180)
    q[::128, :, 0] = 8.0  # the same largest query of every 128-row block, however few of its rows a call has
    slot = KVSlot(torch, heads=heads, head_dim=dim, capacity=n, device=dev)
    slot.pack(to_dev(randn_bf16((n, heads, dim), 181, offset=key_offset(heads, dim, 183)), dev),
              to_dev(randn_bf16((n, heads, dim), 182), dev))
    qd = to_dev(q, dev)

    def attend(lq):
        pad = 4 if rows == "unaligned" else 0  # rows aligned to 8 bytes only
        out = torch.full((full + 7, heads, dim + pad), 7.0, dtype=torch.bfloat16, device=dev)
        at = torch.randperm(full + 7, generator=torch.Generator().manual_seed(lq))[:lq].sort().values.to(dev)
        kwargs = {"o_rows": at} if rows == "list" else {}
        segment_attention(torch, qd, [slot.view()], scale=dim ** -0.5, backend=backend, split=False, lq=lq,
                          out=out[:, :, :dim], **kwargs)
        if rows == "list":
            rest = torch.ones(full + 7, dtype=torch.bool, device=dev)
            rest[at] = False
            return out[at][:, :, :dim], out[rest], out[:, :, dim:]
        return out[:lq, :, :dim], out[lq:], out[:, :, dim:]

    want, _, _ = attend(full)
    for tail in (1, 31, 32, 33, 64, 65, 128, 191, 192, 193, 255):
        got, other, padding = attend(lead + tail)
        assert torch.equal(got.contiguous().view(torch.int16), want[: lead + tail].contiguous().view(torch.int16)), tail
        assert bool((other == 7.0).all()) and bool((padding == 7.0).all()), tail
