"""The operand buffers that the smooth-K quantization asks for, checked on the host."""

import pytest

from taomate_hd_amd import _native


@pytest.mark.parametrize("missing,message", [(None, "segment 0 keys"), ("mean_workspace", "segment 0 keys"),
                                             ("k_mean", "null output"), ("q_i8", "null output"), ("q_scale", "null output")])
def test_mean_workspace_is_not_needed(missing, message):
    args, quant = _native.AttnArgs(), _native.QKQuant()
    args.heads, args.head_dim, args.lq, args.n_segments = 1, 128, 0, 1  # its segment has no tokens: refused last
    quant.k_mean = quant.mean_workspace = quant.q_i8 = quant.q_scale = 1 << 20
    if missing:
        setattr(quant, missing, None)
    with pytest.raises(ValueError, match=message):
        _native.check(_native.load().tmhd_qk_smooth_quant(args, quant, None), "quant")
