"""The GEMM tiles smaller than 256 x 256 (few rows, few columns, partial last
rounds) and their SwiGLU form: accumulators and bf16 outputs bit for bit
against an exact float64 product on the GPU and the stated epilogue, at the
edges of the tiles, of k (one block, fewer blocks than the ring) and of the
choice between the forms."""

from __future__ import annotations

import pytest

pytestmark = pytest.mark.gpu


def _operands(torch, dev, m, n, k, seed):
    g = torch.Generator(device=dev).manual_seed(seed)
    a = torch.randint(-128, 128, (m, k), generator=g, device=dev, dtype=torch.int8)
    w = torch.randint(-127, 128, (n, k), generator=g, device=dev, dtype=torch.int8)
    sa = torch.rand(m, 1, generator=g, device=dev) * 0.05 + 1e-3
    sb = torch.rand(1, n, generator=g, device=dev) * 0.01 + 1e-4
    bias = (torch.randn(n, generator=g, device=dev) * 0.02).to(torch.bfloat16)
    exact = a.double() @ w.double().t().contiguous()  # exact: |sum| < 2^53
    return a, w, sa, sb, bias, exact


SHAPES = [
    # m, n, k: 64 x 64 tiles down to one row and one k block
    (1, 64, 128), (1, 5376, 5376), (16, 1001, 256), (63, 640, 384), (65, 130, 1152), (64, 13824, 640),
    # 64 x 128, 128 x 128 and 192 x 128 tiles, ragged rows and columns
    (129, 5376, 1280), (200, 10752, 2688), (331, 5373, 5376), (331, 10752, 896), (333, 13824, 5120), (512, 10750, 5376),
    # 256 x 128 tiles, and parts of 256 x 256 ones in a last round behind whole rounds
    (700, 10752, 5376), (513, 13824, 5120), (2048, 10752, 512), (4100, 4352, 256), (4836, 10752, 384),
    # long k: few tiles split along k
    (256, 2048, 32768),
]


@pytest.mark.parametrize("m,n,k", SHAPES)
def test_tiles_bit_exact(torch_mod, dev, m, n, k):
    torch = torch_mod
    from taomate_hd_amd import quant

    a, w, sa, sb, bias, exact = _operands(torch, dev, m, n, k, m + n + k)
    acc = quant.int8_mm_i32(a, w.t())
    assert torch.equal(acc.long(), exact.long())
    for b in (None, bias):
        out = quant.cutlass_scaled_mm(a, w.t(), sa, sb, torch.bfloat16, b)
        want = exact.float() * sb * sa  # the epilogue in fp32, in its order
        if b is not None:
            want = want + b.float()
        assert torch.equal(out.view(torch.int16), want.to(torch.bfloat16).view(torch.int16))
    # output rows that 8-byte stores do not fit
    wide = torch.full((m, n + 3), 7.0, dtype=torch.bfloat16, device=dev)
    quant.cutlass_scaled_mm_out(wide[:, 1 : n + 1], a, w.t(), sa, sb, bias)
    assert torch.equal(wide[:, 1 : n + 1].contiguous().view(torch.int16), out.view(torch.int16))
    assert bool((wide[:, 0] == 7.0).all()) and bool((wide[:, n + 1 :] == 7.0).all())


@pytest.mark.parametrize("m,f,k", [(1, 128, 128), (60, 7168, 5376), (127, 7168, 640), (130, 14336, 5376), (257, 7168, 384),
                                   (331, 7168, 5376), (640, 7168, 1024), (1500, 14336, 256),
                                   (256, 1024, 32768)])
def test_swiglu_tiles_match_two_steps(torch_mod, dev, m, f, k):
    torch = torch_mod
    from taomate_hd_amd import fused_swiglu, interleave_swiglu_rows, quant

    a, w, sa, sb, bias, exact = _operands(torch, dev, m, 2 * f, k, m + f + k)
    sa = sa * 0.1  # projections of order 1 to 100
    for b in (None, bias):
        proj = exact.float() * sb * sa
        if b is not None:
            proj = proj + b.float()
        want = fused_swiglu(proj.to(torch.bfloat16))
        ib = None if b is None else interleave_swiglu_rows(b)
        got = quant.cutlass_scaled_mm_swiglu(a, interleave_swiglu_rows(w).t(), sa, interleave_swiglu_rows(sb.t()).t(), ib)
        assert torch.equal(got.view(torch.int16), want.view(torch.int16))
