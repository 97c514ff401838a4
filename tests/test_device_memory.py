"""Device and pinned memory at their limits, against a stand-in for the HIP
runtime (fake_device.c): a device of a set size in host memory, so that these
run, and run out of memory, without a GPU.  Each test is a process of its own,
with the stand-in's symbols before the runtime's.
"""
import os
import subprocess
import sys
import textwrap

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def fake_device(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("fake") / "libfake_device.so")
    subprocess.check_call(["gcc", "-O2", "-fPIC", "-shared", "-w", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                           "-o", so, os.path.join(HERE, "fake_device.c")])
    head = textwrap.dedent(f"""
        import ctypes, sys
        sys.path.insert(0, {HERE!r})
        sys.path.insert(0, {os.path.join(os.path.dirname(HERE), "iron-array_amd")!r})
        fake = ctypes.CDLL({so!r}, mode=ctypes.RTLD_GLOBAL)
        fake.fake_limits.argtypes = [ctypes.c_size_t, ctypes.c_size_t]
        fake.fake_device_used.restype = fake.fake_pinned_peak.restype = ctypes.c_size_t
        import numpy as np
        import pyiarray as ia
        ia.lib()
        h = ctypes.CDLL(ia.HIP_LIB_PATH)
        h.iamx_malloc.restype = h.iamx_workspace.restype = ctypes.c_void_p
        h.iamx_malloc.argtypes = [ctypes.c_size_t]
        h.iamx_free.argtypes = [ctypes.c_void_p]
        h.iamx_workspace.argtypes = [ctypes.c_int, ctypes.c_size_t]
        h.iamx_mem_info.argtypes = [ctypes.POINTER(ctypes.c_size_t)] * 2
        MB = 1 << 20
    """)

    def run(code):
        r = subprocess.run([sys.executable, "-c", head + textwrap.dedent(code)], capture_output=True, text=True,
                           timeout=100)
        assert r.returncode == 0, r.stdout + r.stderr

    return run


KEEP_BLOCKS = """
    fake.fake_limits(1024 * MB, 1024 * MB)
    assert h.iamx_init() == 0
    def free_bytes():
        f, t = ctypes.c_size_t(), ctypes.c_size_t()
        assert h.iamx_mem_info(ctypes.byref(f), ctypes.byref(t)) == 0
        return f.value
    before = free_bytes()
    blocks = [h.iamx_malloc(60 * MB) for _ in range(4)]
    assert all(blocks)
    for b in blocks:
        h.iamx_free(b)
    assert fake.fake_device_used() >= 240 * MB  # kept for later calls
"""


def test_kept_blocks_count_as_free_memory(fake_device):
    fake_device(KEEP_BLOCKS + """
    assert free_bytes() == before
    """)


@pytest.mark.parametrize("what", ["h.iamx_workspace(3, 420 * MB)", "h.iamx_malloc(480 * MB)"])
def test_kept_blocks_are_given_back_to_an_allocation(fake_device, what):
    """Workspaces are the largest allocations: one that fits without the blocks
    kept is had."""
    fake_device(KEEP_BLOCKS + f"""
    big = h.iamx_malloc(500 * MB)
    assert big
    assert {what}
    assert fake.fake_device_used() <= 1024 * MB
    """)


RESULT = """
    def result(rows):
        a = np.zeros((rows, 65536 // 4), np.float32)
        c = ia.Container.from_numpy(ia.Context(clevel=0, filters=0), a, (min(rows, 64), a.shape[1]), (8, 4096))
        return c.to_numpy().view(np.uint32).ravel()  # the device image: nothing wrote over the numbers it began with
"""


@pytest.mark.parametrize("rows", [32, 33, 1023, 1024, 1025, 1536, 1537, 2048, 4000])
def test_results_of_any_size_pin_a_bounded_ring(fake_device, rows):
    """64 KiB a row: one piece, all slots of the ring, one more, and rings full."""
    fake_device(RESULT + f"""
    fake.fake_limits(4096 * MB, 4096 * MB)
    got = result({rows})
    assert np.array_equal(got, np.arange(got.size, dtype=np.uint32))
    assert fake.fake_pinned_peak() < 120 * MB
    """)


def test_result_without_pinned_memory_for_the_ring(fake_device):
    fake_device(RESULT + """
    fake.fake_limits(4096 * MB, 50 * MB)  # two upload stages of 16 MiB and a little more
    got = result(2048)
    assert np.array_equal(got, np.arange(got.size, dtype=np.uint32))
    """)


@pytest.mark.parametrize("pinned", [1, 10, 20, 1024])
@pytest.mark.parametrize("rows", [1, 40, 512, 700])
def test_uploads_with_and_without_pinned_stages(fake_device, rows, pinned):
    """The blocks of a container stored raw, of 64 KiB to 44 MiB, read back from
    the device addresses that its plan names, with no stage, one of two, and both."""
    fake_device(f"""
    from test_zz_no_alloc import DevicePlan
    class Job(ctypes.Structure):
        _fields_ = [("src", ctypes.c_uint64 * 8), ("rest", ctypes.c_uint8 * 64)]
    fake.fake_limits(4096 * MB, {pinned} * MB)
    rng = np.random.default_rng(1)
    a = rng.integers(0, 2 ** 62, ({rows}, 8192))
    c = ia.Container.from_numpy(ia.Context(clevel=0, filters=0), a, (min({rows}, 16), 8192), (1, 8192))
    p = DevicePlan()
    assert ia.lib().iarray_container_device_plan(c.ptr, ctypes.cast(ctypes.byref(p), ctypes.c_void_p)) == 0
    jobs = (Job * p.n_blocks).from_address(p.blocks)
    assert p.n_blocks == {rows}
    for i in range({rows}):
        got = np.frombuffer((ctypes.c_uint8 * 65536).from_address(jobs[i].src[0]), np.int64)
        assert np.array_equal(got, a[i]), i
    c.to_numpy()  # launches and their error checks, after the allocations that failed
    """)
