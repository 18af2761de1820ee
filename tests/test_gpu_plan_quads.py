"""Single-vector plans where the waves' shares of an item are uneven: rows of
1 to 195 groups, so that passes end inside a quad of four groups, a second
pass starts at any of the four waves, and items follow each other with and
without a full first quad.  Against both parity bars."""
import numpy as np
import pytest
import torch

import oracle as O
from conftest import assert_gemv_parity
from q4rdna import api
from test_gpu_parity import dev_f32, dev_u8, random_tiles

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("groups", [[1, 2, 3, 4], [5, 7, 8, 9, 11], [13, 15, 16, 17, 24], [41, 63, 64, 65, 193, 195]])
@pytest.mark.parametrize("kind", ["plain", "add", "glu"])
@pytest.mark.parametrize("repeat", [0, 60])
def test_plan_uneven_groups(cuda, groups, kind, repeat):
    items, want = [], []
    for i, g in enumerate(groups):
        rows, cols = (32, 96, 160, 192, 320)[i % 5], 64 * g
        tiles, x = random_tiles(rows, cols, 100 * g + i), O.gaussian_x(cols, 7 * g)
        gate_t = random_tiles(rows, cols, 100 * g + 50) if kind == "glu" else None
        add = O.gaussian_x(rows, 9 * g) if kind == "add" else None
        y = torch.full((rows,), float("nan"), device="cuda")
        items.append((api.QWeight.from_tiles(dev_u8(tiles), rows, cols), dev_f32(x), y,
                      None if gate_t is None else api.QWeight.from_tiles(dev_u8(gate_t), rows, cols),
                      None if add is None else dev_f32(add)))
        want.append((tiles, rows, cols, x, gate_t, add))
    copies = []
    for _ in range(repeat):
        for w, x, y, gate, add in items:
            copies.append((w, x, torch.full_like(y, float("nan")), gate, add))
    plan = api.Plan(items + copies)
    assert plan.launch()
    torch.cuda.synchronize()
    for (_, _, y, _, _), (tiles, rows, cols, x, gate_t, add) in zip(items, want):
        assert_gemv_parity(y.cpu().numpy(), tiles, rows, cols, x, gate_tiles=gate_t, add=add, label=(kind, cols))
    for i, c in enumerate(copies):
        assert torch.equal(c[2], items[i % len(items)][2]), i
    plan.close()
    # Alone, a GEMV runs the smaller items: the same bits.
    w, x, y, gate, add = items[-1]
    alone = torch.full_like(y, float("nan"))
    plan = api.Plan([(w, x, alone, gate, add)])
    assert plan.launch()
    torch.cuda.synchronize()
    assert torch.equal(alone, y)
    plan.close()
