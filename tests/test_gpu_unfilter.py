"""Un-filter pass at the edges of its pieces: to_numpy of a container and of
its transposed view must give the input back, bit for bit.

Blocks sit around the 4-element groups of byte planes, the 32-element groups of
bit planes and the staged pieces of 16128 bytes (whole rows, and rows longer
than a piece); few blocks are shared among workgroups, more than 4096 are not.
"""
import ctypes

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



# unfiltered and bit-shuffled blocks in a stream a byte of the elements: whole groups of eight and not, groups of four
# elements across a stream's end, streams and blocks of one byte throughout, blocks of fewer than four elements
@pytest.mark.parametrize("split", [ia.ALWAYS_SPLIT, ia.NEVER_SPLIT], ids=["split", "one"])
@pytest.mark.parametrize("filters", [ia.COMP_SHUFFLE, ia.COMP_BITSHUFFLE, 0], ids=["bytes", "bits", "none"])
@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("shape,block", [((96, 64), (32, 32)), ((70, 66), (35, 22)), ((60, 63), (20, 21)),
                                         ((5, 9000), (5, 4104)), ((2017, 8), (2017, 8)), ((24, 26), (1, 2)),
                                         ((33, 40), (3, 1)), ((520, 528), (8, 8))])
def test_unfilter_split_streams(shape, block, dt, filters, split):
    print(f"case: unfilter {shape} blocks {block} {np.dtype(dt).name} filters {filters} split {split}", flush=True)
    rng = np.random.default_rng(shape[0] + block[0])
    a = rng.standard_normal(shape).astype(dt)
    a[: shape[0] // 3] = np.round(a[: shape[0] // 3])
    a[shape[0] // 2:, : shape[1] // 2] = np.frombuffer(b"\x2a" * 8, dt)[0]
    a[-1:] = 0
    ctx = ia.Context(clevel=5, filters=filters, splitmode=split)
    c = ia.Container.from_numpy(ctx, a, shape, block)
    assert c.to_numpy().tobytes() == a.tobytes()
    assert c.transpose().to_numpy().tobytes() == np.ascontiguousarray(a.T).tobytes()


class _Job(ctypes.Structure):
    """iamx_block_job_t"""
    _fields_ = [("src", ctypes.c_uint64 * 8), ("kind", ctypes.c_uint8 * 8), ("fill", ctypes.c_uint8 * 8),
                ("neblock", ctypes.c_int32), ("nstreams", ctypes.c_int16), ("typesize", ctypes.c_int16),
                ("filter", ctypes.c_int32), ("bsize", ctypes.c_int32), ("rows", ctypes.c_int32),
                ("cols", ctypes.c_int32), ("vrows", ctypes.c_int32), ("vcols", ctypes.c_int32),
                ("dst_off", ctypes.c_int64), ("dst_ld", ctypes.c_int64)]


@pytest.mark.parametrize("transposed", [False, True])
@pytest.mark.parametrize("streams", ["one", "planes"])
@pytest.mark.parametrize("filt", [0, 1], ids=["none", "bytes"])
@pytest.mark.parametrize("dt", [np.uint16, np.float32, np.float64])
@pytest.mark.parametrize("vrows,vcols", [(3, 5), (5, 5), (9, 5), (4, 7)])
def test_tile_larger_than_its_block(dt, filt, streams, transposed, vrows, vcols):
    """A caller's job whose valid extent names more elements than the block of
    17 holds, or (shuffled) more columns than its rows have: the block's own
    elements are written, nothing else of dst is."""
    if vcols > 5 and not filt:
        vcols = 5
    n, cols, ld = 17, 5, 12
    print(f"case: tile {vrows}x{vcols} of a block of {n}, {np.dtype(dt).name} filter {filt} {streams} {transposed}",
          flush=True)
    a = np.random.default_rng(3).integers(1, 2 ** 15, n).astype(dt)
    ts = a.itemsize
    raw = a.view(np.uint8).reshape(n, ts)
    raw = np.ascontiguousarray(raw.T if filt else raw).ravel()
    h = ctypes.CDLL(ia.HIP_LIB_PATH)
    h.iamx_malloc.restype = ctypes.c_void_p
    h.iamx_malloc.argtypes = [ctypes.c_size_t]
    h.iamx_free.argtypes = [ctypes.c_void_p]
    for f in ("iamx_h2d", "iamx_d2h"):
        getattr(h, f).argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t]
    h.iamx_decode.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.c_void_p, ctypes.c_int, ctypes.c_void_p,
                              ctypes.c_void_p]
    assert h.iamx_init() == 0
    want = np.full((16, ld), 3, dt)
    for e in range(n):
        r, c = divmod(e, cols)
        if r < vrows and c < vcols:
            want[(c, r) if transposed else (r, c)] = a[e]
    got = np.full_like(want, 3)
    d = h.iamx_malloc(4096)
    try:
        job = _Job(neblock=n * ts if streams == "one" else n, nstreams=1 if streams == "one" else ts, typesize=ts,
                   filter=filt | (0x100 if transposed else 0), bsize=n * ts, rows=4, cols=cols, vrows=vrows,
                   vcols=vcols, dst_off=0, dst_ld=ld)
        for s in range(job.nstreams):
            job.src[s], job.kind[s] = d + 1024 + s * n, 1  # raw bytes, read in place
        assert h.iamx_h2d(d, ctypes.byref(job), ctypes.sizeof(job)) == 0
        assert h.iamx_h2d(d + 1024, raw.ctypes.data, raw.nbytes) == 0
        assert h.iamx_h2d(d + 2048, got.ctypes.data, got.nbytes) == 0
        assert h.iamx_decode(None, 0, d, 1, None, d + 2048) == 0
        assert h.iamx_d2h(got.ctypes.data, d + 2048, got.nbytes) == 0
    finally:
        h.iamx_free(d)
    assert np.array_equal(got, want)
