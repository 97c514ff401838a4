"""GEMV over block shapes at the edges of its block kernels, against numpy.

Operands are small integers times powers of two, so every order of summation
gives the same float32 and float64 sums and y must equal A @ x exactly.
Shapes sit around the 16-element groups of byte-shuffled blocks, the
32-element quads of bit-shuffled ones, and blocks narrower than a group;
matrices of few blocks share a block's rows among workgroups, one of more
than 1024 blocks does not.
"""
import numpy as np
import pytest

import pyiarray as ia

pytestmark = pytest.mark.gpu

# shape, chunks, blocks
SHAPES = [
    ((40, 37), (20, 30), (20, 15)), ((40, 37), (20, 32), (10, 16)), ((33, 51), (33, 34), (11, 17)),
    ((3, 64), (3, 64), (3, 31)), ((129, 200), (65, 100), (65, 33)), ((300, 1025), (150, 1024), (75, 1024)),
    ((1, 500), (1, 250), (1, 125)), ((701, 66), (701, 66), (700, 5)), ((530, 530), (265, 265), (15, 16)),
]


@pytest.mark.parametrize("filters", [ia.COMP_SHUFFLE, ia.COMP_BITSHUFFLE], ids=["bytes", "bits"])
@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("case", SHAPES, ids=[f"{s[0]}x{s[1]}-{b[0]}x{b[1]}" for s, _, b in SHAPES])
def test_gemv_block_shapes_exact(case, dt, filters):
    shape, chunks, blocks = case
    print(f"case: gemv {shape} blocks {blocks} {np.dtype(dt).name} filters {filters}", flush=True)
    rng = np.random.default_rng(shape[0] * 1009 + shape[1])
    A = (rng.integers(-9, 10, shape) * 0.25).astype(dt)
    A[: shape[0] // 3] *= 2.0 ** 20  # several exponents, and constant planes in some blocks only
    A[-1] = 0
    x = rng.integers(-4, 5, shape[1]).astype(dt)
    ctx = ia.Context(clevel=5, filters=filters)
    cA = ia.Container.from_numpy(ctx, A, chunks, blocks)
    cx = ia.Container.from_numpy(ctx, x, (chunks[1],), (blocks[1],))
    y = ia.matmul(cA, cx, (chunks[0],), (blocks[0],)).to_numpy()
    assert np.array_equal(y, (A.astype(np.float64) @ x.astype(np.float64)).astype(dt))
