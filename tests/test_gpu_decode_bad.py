"""Malformed LZ4 streams among good ones, in every form of the decoder: 8
wavefronts a stream up to 4 streams a CU, 4 up to 12, and 1 above, where a
stream that begins with a literal run of 8 KB or more has a body of its own.

The kernel must flag each in the status word, decode every other stream, and
write nothing outside the bad stream's slot.
"""
import ctypes
import struct

import numpy as np
import pytest

import pyiarray as ia
from test_gpu_decode import _craft_lz4

GUARD = 64


class Job(ctypes.Structure):
    """iamx_lz4_job_t"""
    _fields_ = [("src", ctypes.c_uint64), ("dst_off", ctypes.c_int64), ("csize", ctypes.c_int32),
                ("nbytes", ctypes.c_int32), ("codec", ctypes.c_int32), ("reserved", ctypes.c_int32)]


def _sequences(s):
    """(token, offset field, next) positions of every sequence with a match."""
    out, p = [], 0
    while True:
        t, n = p, s[p] >> 4
        p += 1
        if n == 15:
            while True:
                n += s[p]
                p += 1
                if s[p - 1] != 255:
                    break
        p += n
        if p >= len(s):
            return out
        o = p
        p += 2
        if s[t] & 15 == 15:
            while s[p] == 255:
                p += 1
            p += 1
        out.append((t, o, p))


def _stream(first, n, seed):
    """A stream of n bytes that begins with `first` literals (or none), then short and longer sequences."""
    at = [0]

    def pick(r):
        at[0] += 1
        if at[0] == 1 and first:
            return first, int(r.integers(1, first)), 20
        if at[0] % 97 == 0:
            return int(r.integers(0, 400)), int(r.integers(1, 3000)), int(r.integers(274, 900))
        return int(r.integers(0, 12)), int(r.integers(1, 6000)), int(r.integers(4, 60))

    return _craft_lz4(np.random.default_rng(seed), n, pick)


def _spoil(kind, s, n):
    """The stream and decoded length of a malformed variant, spoilt three quarters of the way in."""
    s = bytearray(s)
    q = _sequences(s)
    t, o, nxt = q[3 * len(q) // 4]
    if kind == "cut in a match":
        return bytes(s[:o + 1]), n
    if kind == "cut in literals":
        t = next(x for x in q[len(q) // 2:] if x[1] - x[0] > 4)
        return bytes(s[:t[0] + 3]), n
    if kind == "tail":
        return bytes(s[:-7]), n
    if kind == "zero offset":
        s[o:o + 2] = b"\0\0"
        return bytes(s), n
    if kind == "offset before the output":
        t, o, nxt = q[1]
        s[o:o + 2] = b"\xff\xff"
        return bytes(s), n
    if kind == "more output":
        return bytes(s), n - 300
    if kind == "less output":
        return bytes(s), n + 40
    assert kind == "length without end"
    s[t] |= 0xf0
    return bytes(s[:t + 1]) + b"\xff" * 300, n


KINDS = ["cut in a match", "cut in literals", "tail", "zero offset", "offset before the output", "more output",
         "less output", "length without end"]


@pytest.mark.parametrize("first", [0, 9_000])
@pytest.mark.parametrize("kind", KINDS)
def test_oracle_refuses_the_spoilt_streams(orc, kind, first):
    s, raw = _stream(first, first + 9_000, 5)
    assert orc.lz4_decode(s, len(raw)) == raw
    bad, n = _spoil(kind, s, len(raw))
    try:
        assert len(orc.lz4_decode(bad, n)) != n
    except ValueError:
        pass


@pytest.mark.gpu
@pytest.mark.parametrize("per_cu", [0, 8, 13], ids=["8-wavefronts", "4-wavefronts", "1-wavefront"])
@pytest.mark.parametrize("first", [0, 9_000])
@pytest.mark.parametrize("kind", KINDS)
def test_bad_stream_among_good_ones(kind, first, per_cu):
    name, cus, arch = ia.device_info()
    copies = max(5, per_cu * cus)
    print(f"case: {kind}, {first} literals first, {copies} streams on {cus} CUs", flush=True)
    h = ctypes.CDLL(ia.HIP_LIB_PATH)
    h.iamx_malloc.restype = ctypes.c_void_p
    h.iamx_malloc.argtypes = [ctypes.c_size_t]
    h.iamx_free.argtypes = [ctypes.c_void_p]
    for f in ("iamx_h2d", "iamx_d2h"):
        getattr(h, f).argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t]
    h.iamx_decode.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.c_void_p, ctypes.c_int, ctypes.c_void_p,
                              ctypes.c_void_p]
    assert h.iamx_init() == 0
    s, raw = _stream(first, first + 9_000, 5)
    bad, nbad = _spoil(kind, s, len(raw))
    where = copies // 2
    slot = (max(len(raw), nbad) + 15) // 16 * 16 + GUARD
    arena = np.zeros((len(s) + 63) // 16 * 16 + len(bad) + 64, np.uint8)
    at_bad = (len(s) + 63) // 16 * 16 + 1
    arena[:len(s)] = np.frombuffer(s, np.uint8)
    arena[at_bad:at_bad + len(bad)] = np.frombuffer(bad, np.uint8)
    d_arena, d_jobs = h.iamx_malloc(arena.nbytes), h.iamx_malloc(copies * ctypes.sizeof(Job))
    d_scratch = h.iamx_malloc(copies * slot)
    try:
        assert d_arena and d_jobs and d_scratch
        jobs = (Job * copies)()
        for i in range(copies):
            b = i == where
            jobs[i] = Job(d_arena + (at_bad if b else 0), i * slot, len(bad if b else s), nbad if b else len(raw), 0, 0)
        out = np.full(copies * slot, 0xa5, np.uint8)
        assert h.iamx_h2d(d_arena, arena.ctypes.data, arena.nbytes) == 0
        assert h.iamx_h2d(d_jobs, ctypes.byref(jobs), ctypes.sizeof(jobs)) == 0
        assert h.iamx_h2d(d_scratch, out.ctypes.data, out.nbytes) == 0
        assert h.iamx_decode(d_jobs, copies, None, 0, d_scratch, None) == 0
        status = h.iamx_decode_status()
        assert h.iamx_d2h(out.ctypes.data, d_scratch, out.nbytes) == 0
    finally:
        for d in (d_arena, d_jobs, d_scratch):
            h.iamx_free(d)
    assert status & 0xfe, status
    assert not status & ~0xfe, status
    out = out.reshape(copies, slot)
    good = np.delete(out, where, 0)
    assert np.array_equal(good[:, :len(raw)], np.broadcast_to(np.frombuffer(raw, np.uint8), (copies - 1, len(raw))))
    assert (good[:, (len(raw) + 15) // 16 * 16:] == 0xa5).all()
    assert (out[where, (nbad + 15) // 16 * 16:] == 0xa5).all()
