"""Performance cases of the compressed matrix product path.

Each case is one thing a program does with this library on one MI355X: a
product of compressed containers read back as an array (the drop-in API of
include/iarray.h through its Python binding), or one stage of it on device
memory (the C layer of include/iamx.h, for another host runtime).  The
operands, contexts, decode plans and device buffers a program keeps between
calls are made by prepare(); run() is one call.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "iron-array_amd"))
import pyiarray as ia  # noqa: E402

PRECISION = {"plain": ia.PLAIN, "split_bf16": ia.SPLIT_BF16, "ozaki_int8": ia.OZAKI_INT8, "ozaki_crt": ia.OZAKI_CRT}
CRT_MODULI = 13  # what the automatic pick settles on for 64-bit operands of six decades


def listed():
    return [
        # the smallest call: a 500 x 500 matrix in four blocks times a vector, bound by latency
        {"name": "gemv_small", "kind": "gemv", "M": 500, "K": 500, "chunk": 250, "block": 250, "uneven": False,
         "dtype": "f32", "filter": "bits", "data": "smooth", "transposed": False},
        # the headline: a 20000 x 20000 float32 matrix (1.6 GB, bitshuffled) times a vector, as in bench.py
        {"name": "gemv_large", "kind": "gemv", "M": 20000, "K": 20000, "chunk": 2000, "block": 250, "uneven": False,
         "dtype": "f32", "filter": "bits", "data": "smooth", "transposed": False},
        # an ordinary float64 matrix under the default byte shuffle, ragged in both dimensions
        {"name": "gemv_ragged_f64", "kind": "gemv", "M": 7001, "K": 5003, "chunk": 1000, "block": 125,
         "uneven": False, "dtype": "f64", "filter": "bytes", "data": "smooth", "transposed": False},
        # the transposed view of a matrix times a vector (the other direction of a solver's iteration)
        {"name": "gemv_transposed", "kind": "gemv", "M": 6007, "K": 4001, "chunk": 500, "block": 125,
         "uneven": False, "dtype": "f64", "filter": "bytes", "data": "uniform", "transposed": True},
        # a small matrix product, compressed result included, read back: launches and host calls
        {"name": "gemm_small", "kind": "gemm", "M": 300, "N": 170, "K": 250, "chunk": 100, "block": 50,
         "uneven": False, "dtype": "f64", "filter": "bytes", "data": "uniform", "precision": "plain"},
        # 2000^3 float64, chunks of 500, blocks of 125: bench.py's gemm2k_f64, read back
        {"name": "gemm_f64", "kind": "gemm", "M": 2000, "N": 2000, "K": 2000, "chunk": 500, "block": 125,
         "uneven": False, "dtype": "f64", "filter": "bytes", "data": "uniform", "precision": "plain"},
        # a ragged float32 product in the split-bfloat16 form, read back
        {"name": "gemm_split", "kind": "gemm", "M": 3001, "N": 2503, "K": 2749, "chunk": 512, "block": 128,
         "uneven": False, "dtype": "f32", "filter": "bytes", "data": "normal", "precision": "split_bf16"},
        # many independent ragged float32 products in one call, each result read back
        {"name": "batch", "kind": "batch", "count": 48, "low": 64, "high": 768, "dtype": "f32"},
        # the block fetch of one operand of an 8192^3 float32 product: 256 MiB decoded into device memory
        {"name": "fetch_f32", "kind": "fetch", "M": 8192, "K": 8192, "chunk": 1024, "block": 256, "uneven": False,
         "dtype": "f32", "filter": "bytes", "data": "normal", "clevel": 3},
        # the block fetch of a ragged bitshuffled float64 matrix
        {"name": "fetch_ragged", "kind": "fetch", "M": 3001, "K": 4507, "chunk": 1000, "block": 125, "uneven": False,
         "dtype": "f64", "filter": "bits", "data": "smooth", "clevel": 5},
        # both operands of a 6000^3 float64 product fetched and multiplied in the CRT form, C left on the device
        {"name": "product_crt", "kind": "product", "M": 6000, "N": 6000, "K": 6000, "chunk": 1500, "block": 250,
         "uneven": False, "dtype": "f64", "filter": "bytes", "data": "wide", "precision": "ozaki_crt"},
        # a serving loop's GEMV on a resident plan, without allocation (iamx_gemv_fused_noalloc)
        {"name": "serve", "kind": "serve", "M": 2500, "K": 2500, "chunk": 1250, "block": 250, "uneven": False,
         "dtype": "f32", "filter": "bits", "data": "smooth"},
    ]


def _size(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["gemv", "gemv", "gemm", "gemm", "fetch", "product", "serve", "batch"])
    if kind == "batch":
        low = rng.randint(16, 96)
        return {"kind": "batch", "count": rng.randint(4, 48), "low": low, "high": rng.randint(low + 32, 768),
                "dtype": rng.choice(["f32", "f64"])}
    block = rng.choice([48, 64, 100, 125, 128, 250, 256, rng.randint(33, 256)])
    case = {"kind": kind, "chunk": block * rng.choice([1, 2, 4, 8]), "block": block, "uneven": rng.random() < 0.25,
            "dtype": rng.choice(["f32", "f64"]), "filter": rng.choice(["bytes", "bits"]),
            "data": rng.choice(["smooth", "uniform", "normal"])}
    if kind == "gemv":
        case.update(M=_size(rng, 200, 12000), K=_size(rng, 200, 12000), transposed=rng.random() < 0.25)
    elif kind == "serve":
        case.update(M=_size(rng, 200, 2500), K=_size(rng, 200, 2500))
    elif kind == "fetch":
        case.update(M=_size(rng, 300, 8192), K=_size(rng, 300, 8192), clevel=rng.choice([1, 3, 5, 9]))
    else:
        high = 3000 if kind == "gemm" else 5000
        case.update(M=_size(rng, 100, high), N=_size(rng, 100, high), K=_size(rng, 100, high),
                    precision=rng.choice(["plain", "split_bf16" if case["dtype"] == "f32" else "ozaki_crt"]))
    return case


# ---- inputs -------------------------------------------------------------------------------------
def _torch_type(case):
    return torch.float32 if case["dtype"] == "f32" else torch.float64


def _matrix(rows, cols, dtype, data, seed):
    """A dense operand on the GPU.  smooth: sin(0.001 i) + cos(0.0007 j) plus
    noise of 1e-3 (bench.py's GEMV); uniform in [-1, 1); normal; wide: a random
    sign times 10^u, u uniform in [-3, 3)."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    if data == "smooth":
        a = torch.randn(rows, cols, device="cuda", generator=gen, dtype=dtype)
        a *= 1e-3
        a += torch.sin(0.001 * torch.arange(rows, device="cuda", dtype=torch.float64)).to(dtype)[:, None]
        a += torch.cos(0.0007 * torch.arange(cols, device="cuda", dtype=torch.float64)).to(dtype)[None, :]
        return a
    if data == "normal":
        return torch.randn(rows, cols, device="cuda", generator=gen, dtype=dtype)
    u = torch.rand(rows, cols, device="cuda", generator=gen, dtype=dtype)
    if data == "uniform":
        return 2 * u - 1
    sign = torch.rand(rows, cols, device="cuda", generator=gen) < 0.5
    mag = torch.pow(10.0, 6 * u - 3)
    return torch.where(sign, -mag, mag)


def _vector(n, dtype, seed):
    return _matrix(1, n, dtype, "uniform", seed)[0]


def _tile(dim, case):
    """Chunk and block length along an axis of `dim` elements; uneven chunks
    are not a multiple of the block."""
    chunk = case["chunk"] - (case["block"] // 3 if case["uneven"] else 0)
    chunk = min(dim, max(1, chunk))
    return chunk, min(chunk, case["block"])


def _container(ctx, dense, case):
    tiles = [_tile(d, case) for d in dense.shape]
    return ia.Container.from_numpy(ctx, dense.cpu().numpy(), [t[0] for t in tiles], [t[1] for t in tiles])


def _context(case):
    filters = ia.COMP_SHUFFLE if case.get("filter", "bytes") == "bytes" else ia.COMP_BITSHUFFLE
    return ia.Context(clevel=case.get("clevel", 5), filters=filters)


def _gemm_operands(case, seed):
    dt = _torch_type(case)
    return (_matrix(case["M"], case["K"], dt, case["data"], 4 * seed + 1),
            _matrix(case["K"], case["N"], dt, case["data"], 4 * seed + 2))


def _gemv_operands(case, seed):
    """The stored matrix (the transpose of the one multiplied when the case is transposed) and x."""
    dt = _torch_type(case)
    rows, cols = (case["K"], case["M"]) if case.get("transposed") else (case["M"], case["K"])
    return _matrix(rows, cols, dt, case["data"], 4 * seed + 1), _vector(case["K"], dt, 4 * seed + 2)


def _batch_dims(case):
    rng = np.random.default_rng(case["count"] * 100003 + case["low"] * 1009 + case["high"])
    return [tuple(int(v) for v in row) for row in rng.integers(case["low"], case["high"] + 1, (case["count"], 3))]


def _batch_operands(case, seed):
    dt = _torch_type(case)
    for i, (m, n, k) in enumerate(_batch_dims(case)):
        yield (_matrix(m, k, dt, "uniform", (seed << 8) + 2 * i), _matrix(k, n, dt, "uniform", (seed << 8) + 2 * i + 1))


class _DevicePlan(ctypes.Structure):
    """iarray_device_plan_t of include/iarray_amd.h"""
    _fields_ = [("lz4", ctypes.c_void_p), ("n_lz4", ctypes.c_int), ("blocks", ctypes.c_void_p),
                ("blk_rc", ctypes.c_void_p), ("n_blocks", ctypes.c_int), ("nbcols", ctypes.c_int),
                ("scratch_bytes", ctypes.c_int64), ("blockshape", ctypes.c_int64 * 2)]


_hip = None


def _device_layer():
    """libiamx.so, the C ABI of include/iamx.h"""
    global _hip
    if _hip is None:
        ia.lib()
        h = ctypes.CDLL(ia.HIP_LIB_PATH)
        ptr, num, i64 = ctypes.c_void_p, ctypes.c_int, ctypes.c_int64
        h.iamx_last_error.restype = ctypes.c_char_p
        h.iamx_decode.argtypes = [ptr, num, ptr, num, ptr, ptr]
        h.iamx_gemm.argtypes = [num, num, num, i64, i64, i64, ptr, i64, ptr, i64, ptr, i64]
        h.iamx_gemv_fused_noalloc.argtypes = [num, ptr, num, ptr, ptr, num, num, num, num, ptr, i64, ptr, i64, i64]
        assert h.iamx_init() == 0, h.iamx_last_error()
        _hip = h
    return _hip


def _plan(container):
    plan = _DevicePlan()
    rc = ia.lib().iarray_container_device_plan(container.ptr, ctypes.cast(ctypes.byref(plan), ctypes.c_void_p))
    assert rc == 0, ia.lib().iarray_err_strerror(rc)
    return plan


def _resident(ctx, dense, case):
    """A container with its decode plan, and the device buffers its fetch fills."""
    c = _container(ctx, dense, case)
    plan = _plan(c)
    return {"container": c, "plan": plan, "dense": torch.empty_like(dense),
            "scratch": torch.empty(plan.scratch_bytes + 16, dtype=torch.uint8, device="cuda")}


def _fetch(op):
    h, p = _device_layer(), op["plan"]
    rc = h.iamx_decode(p.lz4, p.n_lz4, p.blocks, p.n_blocks, op["scratch"].data_ptr(), op["dense"].data_ptr())
    assert rc == 0, h.iamx_last_error()
    return op["dense"]


def prepare(case, seed):
    kind = case["kind"]
    ctx = _context(case)
    state = {"case": case, "ctx": ctx}
    if kind == "gemv":
        a, x = _gemv_operands(case, seed)
        state["a"] = _container(ctx, a, case)
        if case["transposed"]:
            state["a"] = state["a"].transpose()
        state["x"] = _container(ctx, x, case)
        state["out"] = [[t] for t in _tile(case["M"], case)]
    elif kind == "gemm":
        a, b = _gemm_operands(case, seed)
        state["a"], state["b"] = _container(ctx, a, case), _container(ctx, b, case)
        state["out"] = list(zip(_tile(case["M"], case), _tile(case["N"], case)))
    elif kind == "batch":
        tile = {"chunk": 512, "block": 128, "uneven": False}
        state["pairs"] = [(_container(ctx, a, tile), _container(ctx, b, tile)) for a, b in _batch_operands(case, seed)]
        state["chunks"] = [(min(m, 512), min(n, 512)) for m, n, _ in _batch_dims(case)]
        state["blocks"] = [(min(m, 128), min(n, 128)) for m, n, _ in _batch_dims(case)]
    elif kind == "fetch":
        state["a"] = _resident(ctx, _matrix(case["M"], case["K"], _torch_type(case), case["data"], 4 * seed + 1), case)
    elif kind == "product":
        a, b = _gemm_operands(case, seed)
        state["a"], state["b"] = _resident(ctx, a, case), _resident(ctx, b, case)
        state["c"] = torch.empty(case["M"], case["N"], dtype=a.dtype, device="cuda")
    else:  # serve
        a, x = _gemv_operands(case, seed)
        state["a"] = _container(ctx, a, case)
        state["plan"], state["x"], state["y"] = _plan(state["a"]), x, torch.empty(case["M"], dtype=x.dtype, device="cuda")
    torch.cuda.synchronize()  # the device layer runs on a stream of its own
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "gemv":
        return ia.matmul(state["a"], state["x"], *state["out"]).to_numpy()
    if kind == "gemm":
        return ia.matmul(state["a"], state["b"], *state["out"], precision=PRECISION[case["precision"]]).to_numpy()
    if kind == "batch":
        return [c.to_numpy() for c in ia.matmul_batch(state["pairs"], state["chunks"], state["blocks"])]
    if kind == "fetch":
        return _fetch(state["a"])
    h = _device_layer()
    dt = 1 if case["dtype"] == "f32" else 0
    if kind == "product":
        a, b, c = _fetch(state["a"]), _fetch(state["b"]), state["c"]
        moduli = CRT_MODULI if case["precision"] == "ozaki_crt" else 0
        rc = h.iamx_gemm(dt, PRECISION[case["precision"]], moduli, case["M"], case["N"], case["K"], a.data_ptr(),
                         case["K"], b.data_ptr(), case["N"], c.data_ptr(), case["N"])
        assert rc == 0, h.iamx_last_error()
        return c
    p, x, y = state["plan"], state["x"], state["y"]
    rc = h.iamx_gemv_fused_noalloc(dt, p.lz4, p.n_lz4, p.blocks, p.blk_rc, p.n_blocks, p.nbcols, p.blockshape[0],
                                   p.blockshape[1], x.data_ptr(), case["K"], y.data_ptr(), case["M"],
                                   p.scratch_bytes)
    assert rc == 0, h.iamx_last_error()
    return y


# ---- what a pass cannot do without ----------------------------------------------------------------
def _ratio(case):
    """Compressed over raw bytes of the operands, as measured on each kind of data."""
    if case.get("data") == "smooth":
        if case["dtype"] == "f64":
            return 0.75
        return 0.615 if case["filter"] == "bits" else 0.65
    return 0.95


def work(case):
    size = 4 if case["dtype"] == "f32" else 8
    ratio, kind = _ratio(case), case["kind"]
    if kind == "batch":
        dims = _batch_dims(case)
        return {"bytes": float(sum(size * (ratio * (m * k + k * n) + m * n) for m, n, k in dims)),
                "flops": float(sum(2 * m * n * k for m, n, k in dims))}
    m, k = case["M"], case["K"]
    if kind in ("gemv", "serve"):
        return {"bytes": size * (ratio * m * k + k + m), "flops": 2.0 * m * k}
    if kind == "fetch":
        return {"bytes": size * (ratio + 1) * m * k, "flops": 0.0}
    n = case["N"]
    products = {"plain": 1, "split_bf16": 3, "ozaki_crt": CRT_MODULI}[case["precision"]]
    return {"bytes": size * (ratio * (m * k + k * n) + m * n), "flops": 2.0 * products * m * n * k}


# ---- the same in 64 bits ----------------------------------------------------------------------------
def exact(case, seed):
    kind = case["kind"]
    if kind in ("gemv", "serve"):
        a, x = _gemv_operands(case, seed)
        a = a.double()
        return ((a.t() if case.get("transposed") else a) @ x.double()).cpu().numpy()
    if kind == "batch":
        return [(a.double() @ b.double()).cpu().numpy() for a, b in _batch_operands(case, seed)]
    if kind == "fetch":
        return _matrix(case["M"], case["K"], _torch_type(case), case["data"], 4 * seed + 1).double()
    a, b = _gemm_operands(case, seed)
    c = a.double() @ b.double()
    return c if kind == "product" else c.cpu().numpy()
