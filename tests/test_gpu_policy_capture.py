"""A tall matrix whose policy split needs a workspace, captured into a graph as
its stream's first call: the capture takes one chunk (no workspace) instead of
growing one, and every replay equals the eager launch bit for bit."""
import pytest
import torch

import oracle as O
from q4rdna import api
from test_gpu_parity import dev_f32, dev_u8, random_tiles

pytestmark = pytest.mark.gpu


# 769 row tiles: the first height at which two chunks make more than six workgroups per CU.
@pytest.mark.parametrize("gated", [False, True])
@pytest.mark.parametrize("rows,cols", [(32 * 769, 64 * 33), (32768, 64 * 40)])
def test_first_call_captured(cuda, rows, cols, gated):
    w = api.QWeight.from_tiles(dev_u8(random_tiles(rows, cols, 1)), rows, cols)
    gate = api.QWeight.from_tiles(dev_u8(random_tiles(rows, cols, 2)), rows, cols) if gated else None
    x = dev_f32(O.gaussian_x(cols, 3))
    y = torch.empty(rows, device="cuda")
    st = torch.cuda.Stream()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=st):
        assert api.mul_mat_ex(w, x, y, gate=gate, stream=st.cuda_stream)
    one, policy = (torch.empty(rows, device="cuda") for _ in range(2))
    for rep in range(3):
        y.fill_(float("nan"))
        x.copy_(dev_f32(O.gaussian_x(cols, 4 + rep)))
        assert api.mul_mat_ex(w, x, one, gate=gate, split_k=1)
        assert api.mul_mat_ex(w, x, policy, gate=gate)
        torch.cuda.synchronize()
        with torch.cuda.stream(st):
            graph.replay()
        st.synchronize()
        # torch hands streams out again: one that other calls have used may have room for the policy's chunks.
        assert torch.equal(y, one) or torch.equal(y, policy), rep
