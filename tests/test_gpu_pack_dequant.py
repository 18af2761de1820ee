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


def special_groups() -> np.ndarray:
    """64-column groups on and beside what the quick evaluation of a scale
    may take: exact ties v = (n + 1/2) s and their fp32 neighbours, bf16 and
    fp16 values, tiny and huge ranges (fp16-subnormal, zero and infinite
    scales, values 2^31 scales and more), infinities and NaNs."""
    rng = np.random.default_rng(7)
    rows = []
    for i in range(96):  # a maximum of 7 s (or -8 s) makes s the first scale tried
        s = np.float32(np.float16(rng.uniform(1e-3, 2.0) * 2.0 ** rng.integers(-6, 6)))
        v = (rng.integers(-8, 8, 64) + 0.5).clip(-7.5, 6.5).astype(np.float32) * s
        v[0] = 7 * s if i & 1 else -8 * s
        step = rng.integers(-1, 2, 64)
        v = np.where(step > 0, np.nextafter(v, np.float32(np.inf)), np.where(step < 0, np.nextafter(v, np.float32(-np.inf)), v))
        v[0] = 7 * s if i & 1 else -8 * s
        rows.append(v)
    base = rng.standard_normal((32, 64)).astype(np.float32)
    rows += list((base.view(np.uint32) & 0xFFFF0000).view(np.float32))
    rows += list(base.astype(np.float16).astype(np.float32))
    for scale in (1e-42, 1e-30, 1e-9, 1e-7, 4e-7, 2e-6, 1e-5, 3e5, 5e5, 6e5, 1e9, 1e30, 3e38):
        with np.errstate(over="ignore"):
            rows += list((base[:2] / 4 * np.float32(scale)).astype(np.float32))
    for bad in (np.inf, -np.inf, np.nan, 3.4e38, 1e-45, 0.0):
        for at in (0, 63):
            v = base[3].copy()
            v[at] = bad
            rows.append(v)
    rows += [np.zeros(64, np.float32), np.full(64, -0.0, np.float32), np.full(64, np.nan, np.float32)]
    one = np.zeros(64, np.float32)
    one[5] = -1e-40
    rows.append(one)
    while len(rows) % 32:
        rows.append(base[len(rows) % 32] * np.float32(len(rows)))
    return np.stack(rows).astype(np.float32)


def test_pack_special_groups_match_the_oracle(cuda):
    groups = special_groups()
    # Each special group beside an ordinary one, so that lanes of one wave take both ways.
    other = O.gaussian_weights(groups.shape[0], 64, 9)
    w = np.concatenate([groups, other], axis=1)
    assert np.array_equal(api.pack(dev_f32(w)).cpu().numpy(), O.pack(w, q4rdna.ALGO_SIDECAR))


@pytest.mark.parametrize("rows,cols", [(32, 64), (64, 192), (480, 4096)])
def test_pack_many_refits_match_the_oracle(cuda, rows, cols):
    """bf16 and uniform weights with outliers: many starts, repeated scales
    and starts cut off at 12 evaluations."""
    rng = np.random.default_rng(rows)
    w = rng.uniform(-1, 1, (rows, cols)).astype(np.float32) * np.float32(0.02)
    w[: rows // 2] = rng.standard_normal((rows // 2, cols)).astype(np.float32)
    w.reshape(-1, 64)[::13, :5] *= 20
    w.reshape(-1, 64)[::3] = (w.reshape(-1, 64)[::3].view(np.uint32) & 0xFFFF0000).view(np.float32)
    assert np.array_equal(api.pack(dev_f32(w)).cpu().numpy(), O.pack(w, q4rdna.ALGO_SIDECAR))
