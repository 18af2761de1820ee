"""Tall matrices and groups whose policy split needs a workspace, captured into
a graph as their stream's first call: the capture takes the several-vector
rule's one chunk (no workspace) instead of growing one, and every replay equals
that split's eager launch bit for bit.  On a stream that has room the capture
takes the policy's split.  And calls on a stream that is not captured, whose
workspaces are made while another stream is."""
import ctypes

import pytest
import torch

import oracle as O
from q4rdna import api
from test_gpu_parity import dev_f32, dev_u8, random_tiles

pytestmark = pytest.mark.gpu


def fresh_stream():
    """A stream the library has not seen (torch hands its pooled streams out
    again); never destroyed, so that its handle stays its own."""
    handle = ctypes.c_void_p()
    assert ctypes.CDLL("libamdhip64.so").hipStreamCreateWithFlags(ctypes.byref(handle), 1) == 0
    return torch.cuda.ExternalStream(handle.value)


def check_captured(call, ys, x, warm):
    """call(split_k) on the current stream, captured with the policy's split
    and replayed, against the eager call at split 1 (cold) or the policy's."""
    st = fresh_stream()
    if warm:
        with torch.cuda.stream(st):
            call(0)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=st):
        call(0)
    for rep in range(3):
        x.copy_(dev_f32(O.gaussian_x(x.numel(), 4 + rep)))
        call(0 if warm else 1)
        want = [y.clone() for y in ys]
        call(1 if warm else 0)
        assert not all(torch.equal(y, w) for y, w in zip(ys, want)), "the two splits' sums do not differ"
        for y in ys:
            y.fill_(float("nan"))
        torch.cuda.synchronize()
        with torch.cuda.stream(st):
            graph.replay()
        st.synchronize()
        for y, w in zip(ys, want):
            assert torch.equal(y, w), rep


# 769 row tiles: the first height at which two chunks make more than six workgroups per CU.
@pytest.mark.parametrize("warm", [False, True])
@pytest.mark.parametrize("gated", [False, True])
@pytest.mark.parametrize("rows,cols", [(32 * 769, 64 * 33), (32768, 64 * 40)])
def test_first_call_captured(cuda, rows, cols, gated, warm):
    w = api.QWeight.from_tiles(dev_u8(random_tiles(rows, cols, 1)), rows, cols)
    gate = api.QWeight.from_tiles(dev_u8(random_tiles(rows, cols, 2)), rows, cols) if gated else None
    x = dev_f32(O.gaussian_x(cols, 3))
    y = torch.empty(rows, device="cuda")
    check_captured(lambda split: api.mul_mat_ex(w, x, y, gate=gate, split_k=split), [y], x, warm)


@pytest.mark.parametrize("warm", [False, True])
@pytest.mark.parametrize("gated", [False, True])
@pytest.mark.parametrize("heights,cols", [((32 * 385, 32 * 384), 64 * 33), ((16384, 8192, 8192), 64 * 48)])
def test_first_group_captured(cuda, heights, cols, gated, warm):
    items = []
    for i, rows in enumerate(heights):
        w, g = (api.QWeight.from_tiles(dev_u8(random_tiles(rows, cols, 2 * i + j)), rows, cols) for j in range(2))
        items.append((w, torch.empty(rows, device="cuda"), g if gated else None))
    x = dev_f32(O.gaussian_x(cols, 3))
    check_captured(lambda split: api.mul_mat_group(items, x, split_k=split), [it[1] for it in items], x, warm)


def test_workspace_made_while_another_stream_is_captured(cuda):
    """The first tall call of a stream runs while another stream is captured
    (in the default mode), and the capture goes on; so it does after a call on
    the captured stream that is refused for want of room."""
    rows, cols = 32768, 64 * 33
    w = api.QWeight.from_tiles(dev_u8(random_tiles(rows, cols, 1)), rows, cols)
    x = dev_f32(O.gaussian_x(cols, 3))
    y, want, count = (torch.full((rows,), float("nan"), device="cuda") for _ in range(3))
    assert api.mul_mat_ex(w, x, want)
    count.zero_()
    captured, other = fresh_stream(), fresh_stream()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=captured):
        count.add_(1)
        assert api.mul_mat_ex(w, x, y, stream=other.cuda_stream)
        with pytest.raises(RuntimeError, match="cannot grow"):
            api.mul_mat_ex(w, x, y, split_k=2)
        count.add_(1)
    other.synchronize()
    assert torch.equal(y, want)
    for rep in range(3):
        with torch.cuda.stream(captured):
            graph.replay()
        captured.synchronize()
        assert (count == 2 * rep + 2).all()
