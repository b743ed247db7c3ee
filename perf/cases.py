"""The work a streaming session and its DiT block give this package, as timed cases.

Kinds of case, by the public entry points they go through:

* ``hook``     one layer call of the streaming attention hook (``StreamingAttentionHook``): the live
               document's condition queries over the condition rows, its media queries over [condition,
               cached history, own media], and a padding document over itself; noisy steps read the cache,
               ``commit`` steps also write the chunk's block into it (and take it back, so that a pass can
               be repeated);
* ``packed``   ``packed_sdpa`` over the documents of a packed sequence (token refiner, non-streamed forward);
* ``front``    what stands before the hook: the W8A8 QKV projection of the hidden rows, then Q/K RMSNorm +
               RoPE in place with the K/V staged into a slot;
* ``fc1``      the MLP's W8A8 FC1 with SwiGLU (``cutlass_w8a8_linear_swiglu``);
* ``linear``   one W8A8 projection with a bf16 bias (``cutlass_w8a8_linear`` with a workspace);
* ``rows``     the block's row ops (``fused_*`` of the residual stream) before or after an attention call;
* ``ulysses``  Q/K RMSNorm + RoPE into the sequence -> heads send buffer.

Inputs are synthetic: bf16 activations ~ N(0, 1), keys with a per-(head, channel) offset ~ N(0, 0.5), W8A8
activations with 1% outlier channels, weights ~ N(0, 0.02), AdaLN tables as strided chunks of one projection.
"""

import sys
from pathlib import Path

import torch

# the package of the repository this runs in (its root is the working folder)
sys.path.insert(1, str(Path("taomate-hd_amd").resolve()))

import taomate_hd_amd as tm  # noqa: E402
from taomate_hd_amd import ulysses  # noqa: E402

DEV = "cuda:0"
LAYER = "blocks.0.attn"
EPS = 1e-6
ROTARY = 96  # rotary span of a 128-channel head
TABLE_ROWS = 4096  # positions of the cos / sin cache
AUDIO_TAG = 2


class _Attention:
    def __init__(self, head_dim):
        self.softmax_scale = head_dim ** -0.5


def listed():
    return [
        # the smallest hook call: a 256-token chunk over 768 cached tokens on 8 heads of 64; host path and launches
        {"name": "hook_first_chunk", "kind": "hook", "backend": "sdpa", "heads": 8, "dim": 64, "media": 256,
         "history": 768, "blocks": 1, "condition": 0, "pad": 0, "commit": False},
        # the 480p stage's layer call, serial (BF16) mode: chunk of 4,836 over 11,232 cached tokens
        {"name": "hook_480p", "kind": "hook", "backend": "sdpa", "heads": 40, "dim": 128, "media": 4836,
         "history": 11232, "blocks": 3, "condition": 0, "pad": 0, "commit": False},
        # the 768p stage's layer call, serial mode: the largest work of a session
        {"name": "hook_768p", "kind": "hook", "backend": "sdpa", "heads": 40, "dim": 128, "media": 12252,
         "history": 28536, "blocks": 3, "condition": 0, "pad": 0, "commit": False},
        # the 768p call of one rank of a TP 2 x Ulysses 2 group (14 local heads) in accelerated (INT8-QK) mode,
        # with the prompt's condition rows and the packed sequence's padding document
        {"name": "hook_i8qk_768p_rank", "kind": "hook", "backend": "sage_attn", "heads": 14, "dim": 128,
         "media": 10434, "history": 33252, "blocks": 3, "condition": 331, "pad": 91, "commit": False},
        # a low-stage denoise step of the same rank, serial mode: ragged chunk, condition rows, padding document
        {"name": "hook_low_rank", "kind": "hook", "backend": "sdpa", "heads": 14, "dim": 128, "media": 2717,
         "history": 5590, "blocks": 2, "condition": 331, "pad": 91, "commit": False},
        # the clean pass that writes a chunk into the cache (once per chunk), accelerated mode
        {"name": "hook_commit", "kind": "hook", "backend": "sage_attn", "heads": 14, "dim": 128, "media": 4836,
         "history": 11232, "blocks": 3, "condition": 331, "pad": 0, "commit": True},
        # token refiner: a packed batch of ragged text / media documents, all heads of a rank
        {"name": "packed_documents", "kind": "packed", "heads": 28, "dim": 128, "documents": 6, "longest": 1337,
         "shortest": 77},
        # QKV projection + Q/K norm + RoPE + K/V staging of the 480p chunk on one rank (28 heads of TP 2)
        {"name": "front_480p", "kind": "front", "rows": 4836, "hidden": 5376, "heads": 28},
        # FC1 + SwiGLU of the 768p chunk, full MLP width
        {"name": "fc1_768p", "kind": "fc1", "rows": 12252, "hidden": 5376, "ffn": 14336},
        # a projection of the prompt's rows alone: few rows, the weight is what is read
        {"name": "linear_prompt", "kind": "linear", "rows": 331, "cols": 5120, "out": 13824},
        # residual gate + RMSNorm + AdaLN of the 768p chunk: memory-bound
        {"name": "rows_768p", "kind": "rows", "op": "residual", "rows": 12252, "cols": 5376},
        # Ulysses send of one rank's 768p shard (group of 4)
        {"name": "ulysses_768p", "kind": "ulysses", "tokens": 3063, "heads": 40, "world": 4, "token_major": True},
    ]


def _log_int(rng, low, high):
    return max(low, min(high, round(low * (high / low) ** rng.random())))


def draw(rng):
    kind = rng.choice(("hook", "hook", "hook", "packed", "front", "fc1", "linear", "rows", "ulysses"))
    if kind == "hook":
        commit = rng.random() < 0.2
        case = {"kind": "hook", "backend": rng.choice(("sdpa", "sage_attn")), "heads": rng.choice((8, 14, 20, 40)),
                "dim": 64 if rng.random() < 0.15 else 128, "media": _log_int(rng, 130, 12252), "history": 0,
                "blocks": rng.choice((1, 2, 3)), "condition": 0 if rng.random() < 0.4 else _log_int(rng, 16, 512),
                "pad": 0 if rng.random() < 0.5 else rng.randint(1, 255), "commit": commit}
        case["history"] = max(case["blocks"] * 8, round(case["media"] * rng.uniform(0.3, 3.2)))
        most = 40 * 12252 * 40000  # no larger than the largest listed call
        while case["heads"] * case["media"] * (case["history"] + case["media"]) > most:
            case["media"] = case["media"] * 3 // 4
            case["history"] = case["history"] * 3 // 4
        return case
    if kind == "packed":
        return {"kind": "packed", "heads": rng.choice((8, 14, 28, 40)), "dim": 64 if rng.random() < 0.15 else 128,
                "documents": rng.randint(1, 12), "longest": _log_int(rng, 64, 6000), "shortest": rng.randint(1, 63)}
    if kind == "front":
        return {"kind": "front", "rows": _log_int(rng, 60, 12252), "hidden": 5376, "heads": rng.choice((14, 28, 40))}
    if kind == "fc1":
        return {"kind": "fc1", "rows": _log_int(rng, 60, 12252), "hidden": 5376, "ffn": rng.choice((7168, 14336))}
    if kind == "linear":
        return {"kind": "linear", "rows": _log_int(rng, 16, 12252), "cols": rng.choice((5120, 5376)),
                "out": rng.choice((5376, 10752, 13824))}
    if kind == "rows":
        return {"kind": "rows", "op": rng.choice(("residual", "norm_modulate", "norm", "gate", "swiglu")),
                "rows": _log_int(rng, 16, 12252), "cols": rng.choice((1024, 2688, 5376))}
    return {"kind": "ulysses", "tokens": _log_int(rng, 60, 12252), "heads": rng.choice((14, 28, 40, 56)),
            "world": rng.choice((2, 4, 8)), "token_major": rng.random() < 0.7}


# ---- inputs


def _generator(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _randn(g, *shape, std=1.0):
    return (torch.randn(*shape, generator=g, device=DEV) * std).to(torch.bfloat16)


def _tags(n):
    """Token tags of a media block: audio rows first, then video."""
    tags = torch.zeros(n, dtype=torch.long, device=DEV)
    tags[: max(1, n // 80)] = AUDIO_TAG
    return tags


def _history_blocks(case):
    """Token counts of the cached blocks: an anchor, then chunks."""
    n = case["blocks"]
    base = case["history"] // n
    return [case["history"] - base * (n - 1)] + [base] * (n - 1)


def _keys(g, n, offset):
    heads, dim = offset.shape
    return (torch.randn(n, heads, dim, generator=g, device=DEV) + offset).to(torch.bfloat16)


def _hook_tensors(case, seed):
    """(history [(k, v)], q, k, v) of a hook case; rows of q / k / v: condition, media, padding."""
    g = _generator(seed)
    heads, dim = case["heads"], case["dim"]
    offset = torch.randn(heads, dim, generator=g, device=DEV) * 0.5
    history = [(_keys(g, n, offset), _randn(g, n, heads, dim)) for n in _history_blocks(case)]
    total = case["condition"] + case["media"] + case["pad"]
    # the hook reads the thirds of a merged projection in place
    merged = torch.empty(total, 3, heads, dim, dtype=torch.bfloat16, device=DEV)
    merged[:, 0] = _randn(g, total, heads, dim)
    merged[:, 1] = _keys(g, total, offset)
    merged[:, 2] = _randn(g, total, heads, dim)
    return history, merged[:, 0], merged[:, 1], merged[:, 2]


def _prepare_hook(case, seed):
    history, q, k, v = _hook_tensors(case, seed)
    contract = tm.KVContract(layer_names=(LAYER,), local_heads=case["heads"], head_dim=case["dim"])
    cache = tm.HeadMajorRingKVCache(contract)
    for block, (hk, hv) in enumerate(history):
        n = int(hk.shape[0])
        cache.begin_clean_commit(block)
        cache.stage(LAYER, hk, hv, _tags(n), torch.ones(n, dtype=torch.bool, device=DEV))
        cache.commit()
    live = case["condition"] + case["media"]
    total = live + case["pad"]
    mask = torch.zeros(total, dtype=torch.bool, device=DEV)
    mask[case["condition"] : live] = True
    tags = torch.ones(total, dtype=torch.long, device=DEV)
    tags[case["condition"] : live] = _tags(case["media"])
    bounds = (0, live, total) if case["pad"] else (0, live)
    hook = tm.StreamingAttentionHook(cache, attention_backend=case["backend"])
    if not case["commit"]:
        hook.activate(mode=tm.HookMode.NOISY, block_index=cache.committed_blocks)
    call = dict(attention=_Attention(case["dim"]), layer_name=LAYER, query=q, key=k, value=v, token_tags=tags,
                commit_mask=mask, cu_seqlens=torch.tensor(bounds, dtype=torch.int32, device=DEV),
                cu_seqlens_host=bounds, max_seqlen=max(live, case["pad"]), live_documents_hint=(0,))
    return {"kind": "hook", "commit": case["commit"], "cache": cache, "hook": hook, "call": call}


def _run_hook(s):
    hook, cache = s["hook"], s["cache"]
    if not s["commit"]:
        return hook(**s["call"])
    cache.begin_clean_commit(cache.committed_blocks)
    hook.activate(mode=tm.HookMode.CLEAN_COMMIT, block_index=cache.committed_blocks)
    out = hook(**s["call"])
    slot = cache.staged_view(LAYER).slot  # the block as written: keys and transposed values
    hook.deactivate()
    cache.rollback()
    return out, slot.k, slot.vt


def _documents(case):
    n = case["documents"]
    low, high = min(case["shortest"], case["longest"]), case["longest"]
    return [low + (high - low) * ((i * 5 + 2) % n + 1) // n for i in range(n)]


def _prepare_packed(case, seed):
    g = _generator(seed)
    lengths = _documents(case)
    bounds = [0]
    for n in lengths:
        bounds.append(bounds[-1] + n)
    qkv = _randn(g, bounds[-1], 3, case["heads"], case["dim"])
    return {"kind": "packed", "q": qkv[:, 0], "k": qkv[:, 1], "v": qkv[:, 2], "bounds": tuple(bounds),
            "longest": max(lengths), "scale": case["dim"] ** -0.5,
            "cu": torch.tensor(bounds, dtype=torch.int32, device=DEV)}


def _activations(g, rows, cols):
    x = torch.randn(rows, cols, generator=g, device=DEV)
    x[:, torch.randperm(cols, generator=g, device=DEV)[: max(1, cols // 100)]] *= 20.0
    return x.to(torch.bfloat16)


def _rope_inputs(g, tokens, dim):
    rotary = min(ROTARY, dim)
    angle = torch.randn(TABLE_ROWS, rotary // 2, generator=g, device=DEV)
    table = torch.cat([angle.cos(), angle.sin()], -1).to(torch.bfloat16)
    qw = (1.0 + 0.1 * torch.randn(dim, generator=g, device=DEV)).to(torch.bfloat16)
    kw = (1.0 + 0.1 * torch.randn(dim, generator=g, device=DEV)).to(torch.bfloat16)
    return qw, kw, table, torch.arange(tokens, device=DEV) % TABLE_ROWS


def _front_tensors(case, seed):
    g = _generator(seed)
    x = _randn(g, case["rows"], case["hidden"])
    w = _randn(g, 3 * case["heads"] * 128, case["hidden"], std=0.02)
    return x, w, _rope_inputs(g, case["rows"], 128)


def _prepare_front(case, seed):
    x, w, rope = _front_tensors(case, seed)
    qw, sw = tm.quantize_cutlass_w8a8_weight(torch, w)
    slot = tm.KVSlot(torch, heads=case["heads"], head_dim=128, capacity=case["rows"], device=torch.device(DEV))
    return {"kind": "front", "x": x, "w": qw, "ws": sw, "wt": qw.t(), "wst": sw.t(), "rope": rope, "slot": slot,
            "workspace": tm.W8A8Workspace(torch)}


def _fc1_tensors(case, seed):
    g = _generator(seed)
    return _randn(g, case["rows"], case["hidden"]), _randn(g, 2 * case["ffn"], case["hidden"], std=0.02)


def _prepare_fc1(case, seed):
    x, w = _fc1_tensors(case, seed)
    qw, sw = tm.quantize_cutlass_w8a8_swiglu_weight(torch, w)
    return {"kind": "fc1", "x": x, "w": qw, "ws": sw, "workspace": tm.W8A8Workspace(torch)}


def _linear_tensors(case, seed):
    g = _generator(seed)
    x = _activations(g, case["rows"], case["cols"])
    return x, _randn(g, case["out"], case["cols"], std=0.02), _randn(g, case["out"], std=0.02)


def _prepare_linear(case, seed):
    x, w, bias = _linear_tensors(case, seed)
    qw, sw = tm.quantize_cutlass_w8a8_weight(torch, w)
    return {"kind": "linear", "x": x, "w": qw, "ws": sw, "wt": qw.t(), "wst": sw.t(), "bias": bias,
            "workspace": tm.W8A8Workspace(torch)}


def _prepare_rows(case, seed):
    g = _generator(seed)
    rows, cols = case["rows"], case["cols"]
    s = {"kind": "rows", "op": case["op"]}
    if case["op"] == "swiglu":
        s["x"] = _randn(g, rows, 2 * cols)
        return s
    proj = _randn(g, 2, 6 * cols, std=0.3)  # the AdaLN projection of two timesteps: shift, scale, gate twice
    s.update(x=_randn(g, rows, cols), branch=_randn(g, rows, cols),
             w=(1.0 + 0.1 * torch.randn(cols, generator=g, device=DEV)).to(torch.bfloat16),
             tables=[proj[:, i * cols : (i + 1) * cols] for i in range(6)],
             index=(torch.arange(rows, device=DEV) >= rows // 2).long())
    return s


def _run_rows(s):
    op = s["op"]
    if op == "swiglu":
        return tm.fused_swiglu(s["x"])
    t = s["tables"]
    if op == "residual":
        return tm.fused_residual_gate_rms_norm_modulate(s["x"], s["branch"], t[2], s["w"], t[4], t[3], s["index"], EPS)
    if op == "norm_modulate":
        return tm.fused_rms_norm_modulate(s["x"], s["w"], t[1], t[0], s["index"], EPS)
    if op == "norm":
        return tm.fused_rms_norm(s["x"], s["w"], EPS)
    return tm.fused_gate_add(s["x"], t[5], s["branch"], s["index"])


def _prepare_ulysses(case, seed):
    g = _generator(seed)
    qkv = _randn(g, case["tokens"], 3 * case["heads"] * 128)
    return {"kind": "ulysses", "qkv": qkv, "rope": _rope_inputs(g, case["tokens"], 128), "world": case["world"],
            "token_major": case["token_major"]}


def prepare(case, seed):
    return {"hook": _prepare_hook, "packed": _prepare_packed, "front": _prepare_front, "fc1": _prepare_fc1,
            "linear": _prepare_linear, "rows": _prepare_rows, "ulysses": _prepare_ulysses}[case["kind"]](case, seed)


def run(s):
    kind = s["kind"]
    if kind == "hook":
        return _run_hook(s)
    if kind == "packed":
        return tm.packed_sdpa(s["q"], s["k"], s["v"], cu_seqlens=s["cu"], cu_seqlens_host=s["bounds"],
                              max_seqlen=s["longest"], scale=s["scale"])
    if kind == "front":
        qkv = tm.cutlass_w8a8_linear(torch, s["x"], s["w"], s["ws"], bias=None, workspace=s["workspace"],
                                     weight_t=s["wt"], weight_scale_t=s["wst"])
        qw, kw, table, positions = s["rope"]
        tm.fused_qkv_qk_norm_rope_stage_(qkv, qw, kw, table, positions, EPS, s["slot"])
        return qkv, s["slot"].k, s["slot"].vt
    if kind == "fc1":
        return tm.cutlass_w8a8_linear_swiglu(torch, s["x"], s["w"], s["ws"], workspace=s["workspace"])
    if kind == "linear":
        return tm.cutlass_w8a8_linear(torch, s["x"], s["w"], s["ws"], bias=s["bias"], workspace=s["workspace"],
                                      weight_t=s["wt"], weight_scale_t=s["wst"])
    if kind == "rows":
        return _run_rows(s)
    qw, kw, table, positions = s["rope"]
    return ulysses.qkv_norm_rope_send_layout(s["qkv"], qw, kw, table, positions, EPS, world_size=s["world"],
                                             token_major=s["token_major"])


# ---- what a pass cannot do without


def work(case):
    kind = case["kind"]
    if kind == "hook":
        hd, cond, media, pad = case["heads"] * case["dim"], case["condition"], case["media"], case["pad"]
        pairs = media * (cond + media + case["history"]) + cond * cond + pad * pad
        rows = cond + media + pad
        moved = 2 * hd * (4 * rows + 2 * case["history"])  # q, k, v, o of the sequence; cached k, v
        if case["commit"]:
            moved += 2 * hd * 2 * media  # the block written
        return {"bytes": moved, "flops": 4 * hd * pairs}
    if kind == "packed":
        hd, lengths = case["heads"] * case["dim"], _documents(case)
        return {"bytes": 2 * hd * 4 * sum(lengths), "flops": 4 * hd * sum(n * n for n in lengths)}
    if kind == "front":
        m, k, n = case["rows"], case["hidden"], 3 * case["heads"] * 128
        return {"bytes": 2 * m * k + n * k + 4 * n + 2 * m * n + 2 * m * n * 2 // 3, "flops": 2 * m * n * k}
    if kind == "fc1":
        m, k, f = case["rows"], case["hidden"], case["ffn"]
        return {"bytes": 2 * m * k + 2 * f * k + 8 * f + 2 * m * f, "flops": 4 * m * f * k}
    if kind == "linear":
        m, k, n = case["rows"], case["cols"], case["out"]
        return {"bytes": 2 * m * k + n * k + 6 * n + 2 * m * n, "flops": 2 * m * n * k}
    if kind == "rows":
        per = {"residual": 4, "norm_modulate": 2, "norm": 2, "gate": 3, "swiglu": 3}[case["op"]]
        return {"bytes": 2 * per * case["rows"] * case["cols"], "flops": 10 * case["rows"] * case["cols"]}
    local = -(-case["heads"] // case["world"])
    sent = case["world"] * case["tokens"] * 3 * local * 128
    return {"bytes": 2 * (case["tokens"] * 3 * case["heads"] * 128 + sent), "flops": 20 * sent}


def tolerance(case):
    # against float64 the paths are off by 2.9e-3 (attention; 1.3e-2 with INT8 scores, nearly all of it the
    # quantization, whose operands are fixed by formula), 2.8e-3 (chains of bf16 roundings) and 3.7e-3 or less
    # (row ops, projections): two correct implementations differ by no more than the roundings of both
    if case["kind"] in ("hook", "packed"):
        return {"rel": 1e-2}
    return {"rel": 6e-3}


# ---- the same results in 64 bits


def _attend64(q, k, v, scale):
    """softmax(q k^T scale) v per head in float64; q / k / v [T, H, D]."""
    out = torch.empty(q.shape, dtype=torch.float64, device=q.device)
    step = max(256, 1 << 28 >> max(1, int(k.shape[0]).bit_length()))  # rows of scores at a time
    for h in range(q.shape[1]):
        kh, vh = k[:, h].double().t().contiguous(), v[:, h].double()
        for r in range(0, q.shape[0], step):
            scores = (q[r : r + step, h].double() * scale) @ kh
            out[r : r + step, h] = torch.softmax(scores, dim=-1) @ vh
            del scores
    return out


def _slot64(k, v):
    """Head-major keys [H, cap, D] and transposed values [H, D, cap] of a slot holding k / v [n, H, D]."""
    n, heads, dim = k.shape
    cap = (n + 63) // 64 * 64
    sk = torch.zeros(heads, cap, dim, dtype=torch.float64, device=k.device)
    sv = torch.zeros(heads, dim, cap, dtype=torch.float64, device=k.device)
    sk[:, :n] = k.double().transpose(0, 1)
    at = torch.tensor([tm.vt_position(t) for t in range(cap)], device=k.device)
    sv[:, :, at[:n]] = v.double().permute(1, 2, 0)
    return sk, sv


def _exact_hook(case, seed):
    history, q, k, v = _hook_tensors(case, seed)
    cond, live = case["condition"], case["condition"] + case["media"]
    scale = case["dim"] ** -0.5
    out = torch.empty(q.shape, dtype=torch.float64, device=q.device)
    if cond:
        out[:cond] = _attend64(q[:cond], k[:cond], v[:cond], scale)
    keys = torch.cat([hk for hk, _ in history] + [k[:live]])
    values = torch.cat([hv for _, hv in history] + [v[:live]])
    out[cond:live] = _attend64(q[cond:live], keys, values, scale)
    if case["pad"]:
        out[live:] = _attend64(q[live:], k[live:], v[live:], scale)
    if not case["commit"]:
        return out
    return (out, *_slot64(k[cond:live], v[cond:live]))


def _scaled_mm64(x, w):
    """Per-token INT8 x times per-channel INT8 w, in float64 from the quantized values."""
    x, w = x.float(), w.float()
    ax = x.abs().amax(1, keepdim=True)
    xq = torch.clamp(torch.round(x * torch.where(ax > 0, 127.0 / ax, torch.zeros_like(ax))), -128, 127).double()
    sw = torch.clamp(w.abs().amax(1, keepdim=True) / 127.0, min=1e-12)
    wq = torch.clamp(torch.round(w / sw), -127, 127)
    out = torch.empty(x.shape[0], w.shape[0], dtype=torch.float64, device=x.device)
    for r in range(0, w.shape[0], 4096):
        out[:, r : r + 4096] = xq @ wq[r : r + 4096].double().t()
    return out * (ax / 127.0).double() * sw.double().t()


def _bf16(x):
    return x.to(torch.bfloat16).double()


def _norm64(x, w):
    return x / torch.sqrt(x.square().mean(-1, keepdim=True) + EPS) * w.double()


def _norm_rope64(qkv, heads, rope):
    """Q/K RMSNorm + RoPE of a merged projection [T, 3 H 128] held in float64 -> [T, 3, H, 128]."""
    qw, kw, table, positions = rope
    t = qkv.shape[0]
    x = qkv.view(t, 3, heads, 128).clone()
    half = table.shape[1] // 2
    cos = table[positions, :half].double()[:, None]
    sin = table[positions, half:].double()[:, None]
    for part, w in ((0, qw), (1, kw)):
        n = _norm64(x[:, part], w)
        a, b = n[..., :half].clone(), n[..., half : 2 * half].clone()
        n[..., :half] = a * cos - b * sin
        n[..., half : 2 * half] = b * cos + a * sin
        x[:, part] = n
    return x


def exact(case, seed):
    kind = case["kind"]
    if kind == "hook":
        # float64 softmax on the GPU: about 1e9 (query, key) pairs a second and head of 128
        hd = case["heads"] * case["dim"]
        return None if hd * case["media"] * (case["media"] + case["history"]) > 4e11 else _exact_hook(case, seed)
    if kind == "packed":
        s = _prepare_packed(case, seed)
        return torch.cat([_attend64(s["q"][a:b], s["k"][a:b], s["v"][a:b], s["scale"])
                          for a, b in zip(s["bounds"], s["bounds"][1:])])
    if kind == "front":
        x, w, rope = _front_tensors(case, seed)
        qkv = _norm_rope64(_bf16(_scaled_mm64(x, w)), case["heads"], rope)
        return (qkv.reshape(qkv.shape[0], -1), *_slot64(qkv[:, 1], qkv[:, 2]))
    if kind == "fc1":
        x, w = _fc1_tensors(case, seed)
        p = _scaled_mm64(x, w)
        gate, up = p[:, : case["ffn"]], p[:, case["ffn"] :]
        return gate * torch.sigmoid(gate) * up
    if kind == "linear":
        x, w, bias = _linear_tensors(case, seed)
        return _scaled_mm64(x, w) + bias.double()
    if kind == "ulysses":
        s = _prepare_ulysses(case, seed)
        heads, world = case["heads"], case["world"]
        local = -(-heads // world)
        x = _norm_rope64(s["qkv"].double(), heads, s["rope"])
        full = torch.zeros(x.shape[0], 3, world * local, 128, dtype=torch.float64, device=x.device)
        full[:, :, :heads] = x
        full = full.view(x.shape[0], 3, world, local, 128)
        return full.permute(2, 0, 1, 3, 4) if case["token_major"] else full.permute(2, 1, 0, 3, 4)
    s = _prepare_rows(case, seed)
    x = s["x"].double()
    if case["op"] == "swiglu":
        gate, up = x[:, : case["cols"]], x[:, case["cols"] :]
        return gate * torch.sigmoid(gate) * up
    if case["op"] == "norm":
        return _norm64(x, s["w"])
    t = [p[s["index"]].double() for p in s["tables"]]
    if case["op"] == "norm_modulate":
        return _norm64(x, s["w"]) * (1.0 + t[1]) + t[0]
    if case["op"] == "gate":
        return x + t[5] * s["branch"].double()
    hidden = x + t[2] * s["branch"].double()
    return hidden, _norm64(hidden, s["w"]) * (1.0 + t[4]) + t[3]
