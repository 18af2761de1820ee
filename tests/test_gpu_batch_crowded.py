"""q4rdna_mul_mat_batch on either side of the lines where its codes enter the
sums in another form (more than one workgroup per CU with a gate, more than two
without and five or six vectors): every vector equals q4rdna_mul_mat_ex of it at the same split bit for bit."""
import pytest
import torch

import oracle as O
from q4rdna import api
from test_gpu_parity import dev_f32, dev_u8, random_tiles

pytestmark = pytest.mark.gpu


# 256 workgroups are one per CU; single launches run eight waves up to 1024.
@pytest.mark.parametrize("rows", [32 * 128, 32 * 129, 32 * 256, 32 * 257, 32 * 512])
@pytest.mark.parametrize("n", [2, 4, 5, 6, 7, 8])
@pytest.mark.parametrize("kind", ["plain", "add", "glu"])
def test_batch_equals_single(cuda, rows, n, kind):
    cols, split = 64 * 19, 2
    w = api.QWeight.from_tiles(dev_u8(random_tiles(rows, cols, rows + n, subnormal=True)), rows, cols)
    gate = api.QWeight.from_tiles(dev_u8(random_tiles(rows, cols, rows + 9)), rows, cols) if kind == "glu" else None
    xs = torch.stack([dev_f32(O.gaussian_x(cols, 20 + v)) for v in range(n)])
    add = torch.stack([dev_f32(O.gaussian_x(rows, 40 + v)) for v in range(n)]) if kind == "add" else None
    y = torch.full((n, rows), float("nan"), device="cuda")
    assert api.mul_mat_batch(w, xs, y, gate=gate, add=add, split_k=split)
    for v in range(n):
        one = torch.full((rows,), float("nan"), device="cuda")
        assert api.mul_mat_ex(w, xs[v], one, gate=gate, add=None if add is None else add[v], split_k=split)
        assert torch.equal(y[v], one), v
