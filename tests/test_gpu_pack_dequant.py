"""The packer and the dequantizer at the sizes and values where their kernels
can go wrong: bit for bit against the CPU oracle."""
import numpy as np
import pytest
import torch

import oracle as O
import q4rdna
from q4rdna import api
from test_gpu_parity import dev_f32, dev_u8, random_tiles

pytestmark = pytest.mark.gpu


# Runs of four tiles: whole, short (1..3 tiles), several per row tile.
@pytest.mark.parametrize("rows,cols", [(32, 64), (64, 128), (96, 192), (32, 256), (160, 320), (64, 27 * 64)])
@pytest.mark.parametrize("shift", [0, 1, 3])
def test_dequant_short_runs_and_unaligned_outputs(cuda, rows, cols, shift):
    """out is any 4-byte aligned buffer; nothing outside it is written."""
    tiles = random_tiles(rows, cols, rows + cols, subnormal=True)
    buf = torch.full((rows * cols + 8,), 7.0, device="cuda")
    out = buf[shift:shift + rows * cols]
    api.dequantize(api.QWeight.from_tiles(dev_u8(tiles), rows, cols), out)
    want = O.dequant(tiles, rows, cols).reshape(-1)
    assert np.array_equal(out.cpu().numpy().view(np.uint32), want.view(np.uint32))
    rest = torch.cat([buf[:shift], buf[shift + rows * cols:]])
    assert (rest == 7.0).all()
