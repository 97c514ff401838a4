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


# unfiltered blocks read eight elements at once, in one stream and in one a byte (whose ends fall inside groups of
# eight, or do not), and few blocks of just under, at and over two workgroups' work
@pytest.mark.parametrize("split", [ia.ALWAYS_SPLIT, ia.NEVER_SPLIT], ids=["split", "one"])
@pytest.mark.parametrize("filters", [ia.COMP_SHUFFLE, ia.COMP_BITSHUFFLE, 0], ids=["bytes", "bits", "none"])
@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("shape,block", [((40, 37), (20, 15)), ((64, 64), (32, 32)), ((126, 130), (63, 65)),
                                         ((128, 128), (64, 64)), ((91, 90), (91, 90)), ((90, 92), (90, 91)),
                                         ((270, 9), (135, 9)), ((200, 7), (100, 7))])
def test_gemv_unfiltered_and_shared_blocks(shape, block, dt, filters, split):
    print(f"case: gemv {shape} blocks {block} {np.dtype(dt).name} filters {filters} split {split}", flush=True)
    rng = np.random.default_rng(shape[0] * 1009 + block[1])
    A = (rng.integers(-9, 10, shape) * 0.25).astype(dt)
    A[: shape[0] // 3] *= 2.0 ** 20
    A[-1] = 0
    x = rng.integers(-4, 5, shape[1]).astype(dt)
    ctx = ia.Context(clevel=5, filters=filters, splitmode=split)
    cA = ia.Container.from_numpy(ctx, A, shape, block)
    cx = ia.Container.from_numpy(ctx, x, (shape[1],), (block[1],))
    y = ia.matmul(cA, cx, (shape[0],), (block[0],)).to_numpy()
    assert np.array_equal(y, (A.astype(np.float64) @ x.astype(np.float64)).astype(dt))
