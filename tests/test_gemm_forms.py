"""Every form of the INT8 GEMM's last round (whole tiles, the k split, each of the
smaller tiles; behind whole rounds and alone), plain and with SwiGLU: the shapes
take the form they are named for (asked of the dispatch rule, on the CPU), and on
the GPU their results equal an exact float64 product and the stated epilogue bit
for bit."""

from __future__ import annotations

import pytest
import torch

from taomate_hd_amd import _native

CUS = 256
WS = 1 << 30  # a workspace of any size that the split asks for
W, S, T64, T64X128, T128, T192, T256 = range(7)
# form, m, n, k
SHAPES = [
    (W, 1900, 8192, 256), (W, 3928, 8192, 256),
    (S, 256, 2048, 32768), (S, 1314, 14080, 6144),
    (T64, 60, 14336, 1152), (T64, 1283, 11008, 384),
    (T64X128, 127, 14336, 640), (T64X128, 1293, 11776, 384),
    (T128, 68, 28672, 5376), (T128, 1028, 14848, 384),
    (T192, 331, 14336, 1024),
    (T256, 198, 28672, 5376), (T256, 1298, 15360, 256),
]
IDS = [f"{form}-{m}x{n}x{k}" for form, m, n, k in SHAPES]


def _behind_whole_rounds(m, n):
    return -(-m // 256) * -(-n // 256) > CUS


def test_form_numbers():
    assert (W, S, T64, T64X128, T128, T192, T256) == (
        _native.GEMM_WHOLE, _native.GEMM_SPLIT_K, _native.GEMM_64X64, _native.GEMM_64X128, _native.GEMM_128X128,
        _native.GEMM_192X128, _native.GEMM_256X128)


@pytest.mark.parametrize("form,m,n,k", SHAPES, ids=IDS)
def test_shapes_take_their_form(form, m, n, k):
    last_round_form = _native.load().tmhd_gemm_last_round_form
    assert last_round_form(m, n, k, WS, CUS) == form
    assert last_round_form(m, n - 3, k, WS, CUS) == form  # the plain GEMM is compared with ragged columns
    if form == S:
        assert last_round_form(m, n, k, 0, CUS) != S


def test_every_form_is_reached():
    got = {(form, _behind_whole_rounds(m, n)) for form, m, n, _ in SHAPES}
    both = {(form, part) for form in (W, S, T64, T64X128, T128, T256) for part in (False, True)}
    assert got == both | {(T192, False)}  # 192 rows do not divide a 256 x 256 tile


# 120 to 224 tiles of few k blocks: smaller tiles take two or more rounds of first loads and
# epilogues there, and 1.13 to 1.30 times as long as the 256 x 256 tiles
@pytest.mark.parametrize("m,n,k", [(331, 28672, 640), (331, 28672, 1280), (700, 13824, 640), (700, 13824, 1280),
                                   (1024, 10752, 640), (1024, 28672, 640), (1500, 28672, 640), (2048, 5120, 640),
                                   (2048, 5376, 640), (2048, 13824, 640), (3084, 13824, 640), (3084, 28672, 640),
                                   (4836, 5376, 640)])
def test_short_k_keeps_whole_tiles(m, n, k):
    assert _native.load().tmhd_gemm_last_round_form(m, n, k, WS, CUS) == W


@pytest.mark.parametrize("m,n,k", [(0, 256, 128), (16, 0, 128), (16, 256, 64), (16, 256, 192)])
def test_no_rounds(m, n, k):
    assert _native.load().tmhd_gemm_last_round_form(m, n, k, WS, CUS) == -1


def _operands(dev, m, n, k):
    g = torch.Generator(device=dev).manual_seed(m + n + k)
    a = torch.randint(-128, 128, (m, k), generator=g, device=dev, dtype=torch.int8)
    w = torch.randint(-127, 128, (n, k), generator=g, device=dev, dtype=torch.int8)
    sa = torch.rand(m, 1, generator=g, device=dev) * 0.005 + 1e-4
    sb = torch.rand(1, n, generator=g, device=dev) * 0.01 + 1e-4
    bias = (torch.randn(n, generator=g, device=dev) * 0.02).to(torch.bfloat16)
    return a, w, sa, sb, bias, a.double() @ w.double().t().contiguous()  # exact: |sum| < 2^53


def _here(dev, form, m, n, k):
    """Skips unless the shape takes its form on this device with the workspace that the calls below allocate."""
    lib = _native.load()
    if torch.cuda.get_device_properties(dev).multi_processor_count != CUS:
        pytest.skip(f"the shapes are chosen for {CUS} CUs")
    assert lib.tmhd_gemm_last_round_form(m, n, k, lib.tmhd_gemm_split_workspace_bytes(m, n, k), 0) == form


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [s[1:] for s in SHAPES] + [(12252, 13824, 5120), (331, 13824, 5120), (16, 256, 192)])
def test_workspace_is_asked_for_only_where_the_split_runs(dev, m, n, k):
    lib = _native.load()
    need = lib.tmhd_gemm_split_workspace_bytes(m, n, k)
    assert (need > 0) == (lib.tmhd_gemm_last_round_form(m, n, k, WS, 0) == S)
    if need:
        assert lib.tmhd_gemm_last_round_form(m, n, k, need, 0) == S
        assert lib.tmhd_gemm_last_round_form(m, n, k, need - 1, 0) != S


@pytest.mark.gpu
@pytest.mark.parametrize("form,m,n,k", SHAPES, ids=IDS)
def test_plain(dev, form, m, n, k):
    from taomate_hd_amd import quant

    n -= 3
    _here(dev, form, m, n, k)
    a, w, sa, sb, bias, exact = _operands(dev, m, n, k)
    assert torch.equal(quant.int8_mm_i32(a, w.t()).long(), exact.long())
    for b in (None, bias):
        want = exact.float() * sb * sa  # the epilogue in fp32, in its order
        if b is not None:
            want = want + b.float()
        out = quant.cutlass_scaled_mm(a, w.t(), sa, sb, torch.bfloat16, b)
        assert torch.equal(out.view(torch.int16), want.to(torch.bfloat16).view(torch.int16))


@pytest.mark.gpu
@pytest.mark.parametrize("form,m,n,k", SHAPES, ids=IDS)
def test_swiglu(dev, form, m, n, k):
    from taomate_hd_amd import fused_swiglu, interleave_swiglu_rows, quant

    _here(dev, form, m, n, k)
    a, w, sa, sb, bias, exact = _operands(dev, m, n, k)
    for b in (None, bias):
        proj = exact.float() * sb * sa
        if b is not None:
            proj = proj + b.float()
        want = fused_swiglu(proj.to(torch.bfloat16))
        got = quant.cutlass_scaled_mm_swiglu(a, interleave_swiglu_rows(w).t(), sa, interleave_swiglu_rows(sb.t()).t(),
                                             None if b is None else interleave_swiglu_rows(b))
        assert torch.equal(got.view(torch.int16), want.view(torch.int16))
