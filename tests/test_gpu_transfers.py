"""Containers to the device and arrays back, at the sizes where the transfers
change: one pinned stage or several (16 MiB pieces, 512 KiB copies), small
results in one copy, large ones piece by piece; and device blocks handed from
freed containers to new ones.
"""
import numpy as np
import pytest

import pyiarray as ia

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 255, 256, 257, 1023, 1024, 2047, 2048, 2049, 4100, 8192, 8193, 12300])
def test_roundtrip_sizes(rows):
    """Random bytes stored raw: `rows` rows of 2 KiB in chunks of 512 KiB."""
    rng = np.random.default_rng(rows)
    a = rng.integers(-2 ** 62, 2 ** 62, (rows, 256))
    ctx = ia.Context(clevel=1, filters=0)
    c = ia.Container.from_numpy(ctx, a, (min(rows, 256), 256), (min(rows, 64), 256))
    assert np.array_equal(c.to_numpy(), a)


@pytest.mark.parametrize("n", [1, 3, 4, 5, 1023, 1024, 1025, 4095, 4097, 65_536, 524_287, 524_288, 524_289])
def test_small_results_to_host(n):
    """float32 results of up to 2 MiB leave in one launch, 16 bytes a thread and
    the last ones alone; larger ones through the pinned stages.  A smaller result
    after a larger one shows none of its bytes."""
    rng = np.random.default_rng(n)
    ctx = ia.Context(clevel=5, filters=ia.COMP_SHUFFLE)
    big = rng.integers(-9, 9, (1, 300_001)).astype(np.float32)
    assert np.array_equal(ia.Container.from_numpy(ctx, big, (1, 300_001), (1, 4096)).to_numpy(), big)
    a = rng.integers(-9, 9, (1, n)).astype(np.float32)
    c = ia.Container.from_numpy(ctx, a, (1, n), (1, min(n, 4096)))
    assert np.array_equal(c.to_numpy(), a)


def test_blocks_reused_by_other_containers():
    """Containers freed and made in turn, each decoded while others live: a
    reused device block never shows another container's data."""
    rng = np.random.default_rng(5)
    ctx = ia.Context(clevel=5, filters=ia.COMP_SHUFFLE)
    live = []
    for i in range(60):
        n = int(rng.choice([40, 41, 100, 333, 700]))
        a = rng.integers(-50, 50, (n, n)).astype(np.float64)
        c = ia.Container.from_numpy(ctx, a, (n, n), (min(n, 64), min(n, 64)))
        live.append((a, c))
        if len(live) > 4:
            live.pop(int(rng.integers(0, len(live))))
        for a, c in live:
            assert np.array_equal(c.to_numpy(), a)
        a, c = live[int(rng.integers(0, len(live)))]
        p = ia.matmul(c, c, a.shape, (min(a.shape[0], 64),) * 2)
        assert np.array_equal(p.to_numpy(), a @ a)


@pytest.mark.parametrize("rows", [32_767, 32_768, 32_769, 49_160, 70_001])
def test_results_through_the_ring(rows):
    """Results of just under, at and over the 64 MiB of the ring of pinned pieces, and some halves more."""
    rng = np.random.default_rng(rows)
    a = rng.integers(-2 ** 62, 2 ** 62, (rows, 256))
    ctx = ia.Context(clevel=0, filters=0)
    c = ia.Container.from_numpy(ctx, a, (min(rows, 4096), 256), (64, 256))
    for _ in range(2):
        assert np.array_equal(c.to_numpy(), a)
