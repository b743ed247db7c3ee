"""The memo of a slot's key sums holds only sums that a successful call has
queued: a refused INT8-QK call leaves none behind (with a stand-in for the
library on the CPU, with a refused query on the GPU)."""

from __future__ import annotations

import pytest
import torch

from taomate_hd_amd import KVSlot, _native
from taomate_hd_amd.attention import AttentionCall, QKQuantWorkspace, segment_attention, segment_attention_batch
from taomate_hd_amd.slots import SlotView
from tests.helpers import key_offset, randn_bf16, to_dev


class _Library:
    """Records the key sums each quantization call is given and asked for."""

    def __init__(self):
        self.quant_status, self.attn_status, self.given, self.asked = [], [], [], []

    def tmhd_qk_smooth_quant_batch(self, args, quants, sums, n, stream):
        per = _native.MAX_SEGMENTS
        self.given.append([[quants[i].k_sum[j] for j in range(args[i].n_segments)] for i in range(n)])
        self.asked.append([[sums[i * per + j] for j in range(args[i].n_segments)] for i in range(n)])
        return self.quant_status.pop(0)

    def tmhd_attn_fwd_i8qk_batch(self, args, quants, n, stream):
        return self.attn_status.pop(0)

    def tmhd_last_error(self):
        return b"refused"


@pytest.mark.parametrize("status,error", [(_native.TMHD_ERR_INVALID, ValueError), (_native.TMHD_ERR_HIP, RuntimeError)])
def test_refused_call_leaves_no_memo(monkeypatch, status, error):
    lib = _Library()
    monkeypatch.setattr(_native, "load", lambda: lib)
    monkeypatch.setattr(_native, "stream_ptr", lambda torch, device: 0)
    monkeypatch.setattr(_native, "require_device_tensor", lambda torch, tensor, name: None)
    slots = [KVSlot(torch, heads=2, head_dim=64, capacity=128, device="cpu") for _ in range(2)]
    query = torch.zeros(8, 2, 64, dtype=torch.bfloat16)
    views = [SlotView(slots[0], 70), SlotView(slots[1], 5)]
    calls = [AttentionCall(query, [views[0]]), AttentionCall(query, views)]

    def attend():
        segment_attention_batch(torch, calls, scale=0.125, backend="i8qk", split=False)

    lib.quant_status, lib.attn_status = [status, _native.TMHD_OK, _native.TMHD_OK], [status, _native.TMHD_OK]
    with pytest.raises(error):
        attend()
    assert not any(slot.key_sums for slot in slots)
    # the next call sums every segment once, also the one that two calls share; its
    # sums stay, even if the attention that follows is refused
    with pytest.raises(error):
        attend()
    shared, own = lib.asked[1][0][0], lib.asked[1][1][1]
    assert shared and own and shared != own
    assert lib.asked[1] == [[shared], [None, own]] and lib.given[1] == [[None], [shared, None]]
    assert [t.data_ptr() for slot in slots for t in slot.key_sums.values()] == [shared, own]
    attend()
    assert lib.asked[2] == [[None], [None, None]] and lib.given[2] == [[shared], [shared, own]]


@pytest.mark.gpu
def test_call_after_a_refused_one(torch_mod, dev):
    heads, dim, lq, n = 3, 128, 70, 200
    k = randn_bf16((n, heads, dim), 171, offset=key_offset(heads, dim, 173))
    v = randn_bf16((n, heads, dim), 172)
    q = to_dev(randn_bf16((lq, heads, dim), 170), dev)
    base = torch.empty(q.numel() + 4, dtype=torch.bfloat16, device=dev)
    unaligned = base[4:].view(lq, heads, dim)  # 8-byte aligned: refused on the host
    unaligned.copy_(q)

    def slot():
        s = KVSlot(torch, heads=heads, head_dim=dim, capacity=n, device=dev)
        s.pack(to_dev(k, dev), to_dev(v, dev))
        return s

    def attend(s, query):
        return segment_attention(torch, query, [s.view()], scale=dim ** -0.5, backend="i8qk", return_quant=True,
                                 workspace=QKQuantWorkspace(torch))

    fresh, used = slot(), slot()
    want, quants = attend(fresh, q)
    with pytest.raises(ValueError, match="16-byte aligned"):
        attend(used, unaligned)
    assert not used.key_sums
    got, again = attend(used, q)
    torch.cuda.synchronize()
    assert torch.equal(again["k_mean"].view(torch.int16), quants["k_mean"].view(torch.int16))
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))
    (key, value), = used.key_sums.items()
    assert torch.equal(value, fresh.key_sums[key])
