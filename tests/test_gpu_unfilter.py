"""Un-filter pass at the edges of its pieces: to_numpy of a container and of
its transposed view must give the input back, bit for bit.

Blocks sit around the 4-element groups of byte planes, the 32-element groups of
bit planes and the staged pieces of 16128 bytes (whole rows, and rows longer
than a piece); few blocks are shared among workgroups, more than 4096 are not.
"""
import numpy as np
import pytest

import pyiarray as ia

pytestmark = pytest.mark.gpu

# shape, chunks, blocks
SHAPES = [
    ((37, 41), (20, 30), (7, 9)), ((64, 96), (64, 96), (32, 32)), ((5, 9000), (5, 9000), (5, 4100)),
    ((3, 2100), (3, 2100), (3, 2017)), ((2100, 3), (2100, 3), (2017, 3)), ((130, 127), (65, 64), (33, 31)),
    ((1, 77), (1, 77), (1, 33)), ((300, 310), (150, 155), (150, 155)), ((528, 520), (264, 260), (8, 8)),
]


@pytest.mark.parametrize("filters", [ia.COMP_SHUFFLE, ia.COMP_BITSHUFFLE, 0], ids=["bytes", "bits", "none"])
@pytest.mark.parametrize("dt", [np.float32, np.float64, np.int16])
@pytest.mark.parametrize("case", SHAPES, ids=[f"{s[0]}x{s[1]}-{b[0]}x{b[1]}" for s, _, b in SHAPES])
def test_unfilter_shapes(case, dt, filters):
    shape, chunks, blocks = case
    print(f"case: unfilter {shape} blocks {blocks} {np.dtype(dt).name} filters {filters}", flush=True)
    rng = np.random.default_rng(shape[0] * 1009 + shape[1])
    a = (rng.standard_normal(shape) * 1000).astype(dt)
    a[: shape[0] // 2, : shape[1] // 2] = 7  # constant planes in some blocks
    ctx = ia.Context(clevel=5, filters=filters)
    c = ia.Container.from_numpy(ctx, a, chunks, blocks)
    assert c.to_numpy().tobytes() == a.tobytes()
    assert c.transpose().to_numpy().tobytes() == np.ascontiguousarray(a.T).tobytes()
