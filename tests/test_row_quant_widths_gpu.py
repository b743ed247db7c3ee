"""Row quantization at the edges of its forms: one wave or four per row, 1 to 8
chunks of 8 columns a lane or the streamed row, ragged last chunks, and rows
whose largest value lies in each wave's part. Bytes and scales as the oracle's."""

import numpy as np
import pytest

from oracle import bf16
from oracle import quant as oq
from tests.helpers import randn_bf16, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize(
    "rows,cols",
    [(rows, cols) for rows in (1, 5) for cols in (8, 512, 520, 1024, 1032, 2048, 2056, 2560, 2568, 3072, 3080, 4096,
                                                  4104, 6144, 6152, 8192, 8200, 16384, 16392)]
    # four waves from 4,097 rows on
    + [(rows, cols) for rows in (4096, 4097) for cols in (3080, 4096)],
)
def test_row_quant_at_form_edges(torch_mod, dev, rows, cols):
    from taomate_hd_amd import quant

    x = randn_bf16((rows, cols), cols)
    for r in range(rows):
        x[r, (r * cols // rows + cols // (2 * rows)) % cols] = 37.0  # the row's maximum
    x[0, -1] = -41.0
    x = bf16.round_f32(x)
    q, s, _ = quant.scaled_int8_quant(to_dev(x, dev))
    wq, ws = oq.token_quant(x)
    assert np.array_equal(q.cpu().numpy(), wq)
    assert np.array_equal(s.cpu().numpy().reshape(-1), ws)
