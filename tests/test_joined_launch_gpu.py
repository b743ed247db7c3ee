"""Norm + RoPE with the V rows in the same launch, where the V part's blocks end:
heads that do not fill a workgroup, one token, ranges that end inside a
64-position block, ranks that hold only padding. Bit-equal to the separate calls."""

import numpy as np
import pytest

from oracle import bf16
from tests.helpers import randn_bf16, to_dev

pytestmark = pytest.mark.gpu


def _inputs(dev, tokens, heads, dim):
    import torch

    rng = np.random.default_rng(tokens + heads)
    x = to_dev(randn_bf16((tokens, 3 * heads * dim), 7), dev)
    w = [bf16.to_torch(bf16.round_f32(1.0 + 0.1 * rng.standard_normal(dim).astype(np.float32)), dev) for _ in range(2)]
    table = to_dev(randn_bf16((64, 64), 8), dev)
    return x, (*w, table, torch.from_numpy(rng.integers(0, 64, tokens)).to(dev), 1e-6)


@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("tokens,heads,row0,count,dst", [(1, 1, 0, 1, 0), (66, 5, 1, 65, 64), (130, 7, 0, 128, 64), (9, 3, 8, 1, 192)])
def test_stage(torch_mod, dev, tokens, heads, row0, count, dst, dim):
    torch = torch_mod
    from taomate_hd_amd import fused_qkv_qk_norm_rope_, fused_qkv_qk_norm_rope_stage_
    from taomate_hd_amd.slots import KVSlot

    x, args = _inputs(dev, tokens, heads, dim)
    slots = []
    for _ in range(2):
        s = KVSlot(torch, heads=heads, head_dim=dim, capacity=dst + count + 70, device=dev)
        s.k.fill_(3.0), s.vt.fill_(5.0)  # stale rows
        slots.append(s)
    a, b, width = x.clone(), x.clone(), heads * dim
    fused_qkv_qk_norm_rope_(a, *args)
    k, v = (a[:, i * width : (i + 1) * width].view(tokens, heads, dim) for i in (1, 2))
    slots[0].pack(k, v, row0=row0, count=count, dst=dst)
    fused_qkv_qk_norm_rope_stage_(b, *args, slots[1], row0=row0, count=count, dst=dst)
    torch.cuda.synchronize()
    assert torch.equal(a.view(torch.int16), b.view(torch.int16))
    assert torch.equal(slots[0].k.view(torch.int16), slots[1].k.view(torch.int16))
    assert torch.equal(slots[0].vt.view(torch.int16), slots[1].vt.view(torch.int16))


@pytest.mark.parametrize("token_major", [False, True])
@pytest.mark.parametrize("tokens,heads,dim,world", [(1, 5, 128, 4), (5, 5, 64, 4), (3, 17, 128, 2), (4, 3, 64, 8)])
def test_send(torch_mod, dev, tokens, heads, dim, world, token_major):
    torch = torch_mod
    from taomate_hd_amd import fused_qkv_qk_norm_rope_, ulysses

    x, args = _inputs(dev, tokens, heads, dim)
    fused = ulysses.qkv_norm_rope_send_layout(x, *args, world_size=world, token_major=token_major)
    fused_qkv_qk_norm_rope_(x, *args)
    plain = ulysses.qkv_send_layout(x, num_heads=heads, head_dim=dim, world_size=world, token_major=token_major)
    torch.cuda.synchronize()
    assert torch.equal(fused.view(torch.int16), plain.view(torch.int16))
