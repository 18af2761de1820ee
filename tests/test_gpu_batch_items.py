"""Batched plans at the sizes where their items change: plans of little work
(rows cut into K chunks, streams and chunks meeting in memory), of more
(whole rows), and of many items per workgroup, at one and two vector
quads.  Every vector against both parity bars."""
import numpy as np
import pytest
import torch

import oracle as O
from conftest import assert_gemv_parity
from q4rdna import api
from test_gpu_parity import dev_f32, dev_u8, random_tiles

pytestmark = pytest.mark.gpu

# rows, cols, kind: uneven groups, rows ending inside a 256-row block, rows longer than a chunk
SHAPES = [(288, 64 * 41, "plain"), (512, 4096, "glu"), (96, 64 * 7, "add"), (256, 64 * 195, "add"), (32, 64, "plain"),
          (320, 64 * 33, "glu")]


@pytest.mark.parametrize("n", [2, 4, 5, 8])
@pytest.mark.parametrize("repeat", [1, 40])
def test_batched_items(cuda, n, repeat):
    items, want = [], []
    for i, (rows, cols, kind) in enumerate(SHAPES):
        t = random_tiles(rows, cols, 3000 + i)
        gt = random_tiles(rows, cols, 3100 + i) if kind == "glu" else None
        xs = np.stack([O.gaussian_x(cols, 3200 + 10 * i + v) for v in range(n)])
        add = np.stack([O.gaussian_x(rows, 3300 + 10 * i + v) for v in range(n)]) if kind == "add" else None
        args = (api.QWeight.from_tiles(dev_u8(t), rows, cols), dev_f32(xs),
                None if gt is None else api.QWeight.from_tiles(dev_u8(gt), rows, cols),
                None if add is None else dev_f32(add))
        ys = [torch.full((n, rows), float("nan"), device="cuda") for _ in range(repeat)]
        items += [(args[0], args[1], y, args[2], args[3]) for y in ys]
        want.append((t, rows, cols, xs, gt, add, ys))
    plan = api.Plan(items, batch=n)
    for _ in range(2):  # the second launch finds the counters as the first left them
        for it in items:
            it[2].fill_(float("nan"))
        assert plan.launch()
        torch.cuda.synchronize()
        for t, rows, cols, xs, gt, add, ys in want:
            yh = ys[0].cpu().numpy()
            for v in range(n):
                assert_gemv_parity(yh[v], t, rows, cols, xs[v], gate_tiles=gt, add=None if add is None else add[v],
                                   label=(rows, cols, n, v))
            for y in ys[1:]:
                assert torch.equal(y, ys[0]), (rows, cols, n)
    plan.close()


def test_batched_queue(cuda):
    """Ten items of 16 steps per workgroup, over several launches."""
    rows, cols, n = 256, 4096, 3
    t = random_tiles(rows, cols, 3400)
    w = api.QWeight.from_tiles(dev_u8(t), rows, cols)
    xs = np.stack([O.gaussian_x(cols, 3500 + v) for v in range(n)])
    xd = dev_f32(xs)
    count = 512 * 10  # 16 steps each
    out = torch.empty((count, n, rows), device="cuda")
    plan = api.Plan([(w, xd, out[i]) for i in range(count)], batch=n)
    for _ in range(3):
        out.fill_(float("nan"))
        assert plan.launch()
        torch.cuda.synchronize()
        yh = out[0].cpu().numpy()
        for v in range(n):
            assert_gemv_parity(yh[v], t, rows, cols, xs[v], label=("queue", v))
        assert (out == out[0]).all()
    plan.close()
