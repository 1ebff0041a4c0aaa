"""Helpers of the GPU parity tests: device buffers (torch as plumbing), host
copies of raw device pointers, synthetic data."""
import ctypes

import numpy as np
import torch

import s2pamd

DEV = "cuda:0"
_hip = None
# Every device buffer made by to_dev()/empty() stays referenced until the test
# ends (conftest clears it after a device synchronisation): pointers handed to
# the C ABI must never outlive their torch tensor, whose block the caching
# allocator would otherwise hand to the next allocation.
LIVE = []
# (what, largest per-row gpu-oracle L2 distance, exception rows used, rows) of
# every logits check, summarised at the end of the pytest run (conftest)
LOGITS_RECORD = []


def hip():
    global _hip
    if _hip is None:
        _hip = ctypes.CDLL("libamdhip64.so")
        _hip.hipMemcpy.restype = ctypes.c_int
        _hip.hipMemcpy.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t, ctypes.c_int]
        _hip.hipDeviceSynchronize.restype = ctypes.c_int
    return _hip


def sync():
    torch.cuda.synchronize()


def d2h(ptr, nbytes, dtype):
    """Copy nbytes from a raw device pointer into a new numpy array."""
    sync()
    out = np.empty(nbytes // np.dtype(dtype).itemsize, dtype)
    rc = hip().hipMemcpy(out.ctypes.data, ptr, nbytes, 2)
    assert rc == 0, f"hipMemcpy D2H failed: {rc}"
    return out


def h2d_raw(host, dev_ptr):
    """Copy a numpy array into raw device memory."""
    host = np.ascontiguousarray(host)
    rc = hip().hipMemcpy(dev_ptr, host.ctypes.data, host.nbytes, 1)
    assert rc == 0, f"hipMemcpy H2D failed: {rc}"
    sync()


def to_dev(a):
    """numpy -> device tensor (uint16 travels as int16 bits)."""
    a = np.ascontiguousarray(a)
    if a.dtype == np.uint16:
        t = torch.from_numpy(a.view(np.int16)).to(DEV)
    elif a.dtype == np.uint64:
        t = torch.from_numpy(a.view(np.int64)).to(DEV)
    else:
        t = torch.from_numpy(a).to(DEV)
    LIVE.append(t)
    return t


def to_host(t, dtype=None):
    sync()
    a = t.detach().cpu().numpy()
    if dtype is not None:
        a = a.view(dtype)
    return a


def empty(shape, dtype=torch.int16):
    t = torch.empty(shape, dtype=dtype, device=DEV)
    LIVE.append(t)
    return t


def P(t):
    return s2pamd.dptr(t)


def S():
    return s2pamd.stream_ptr()


def bf16_bits(a):
    return torch.from_numpy(np.ascontiguousarray(a, np.float32)).to(torch.bfloat16).view(
        torch.int16).numpy().view(np.uint16)


def bf16_vals(bits):
    return (np.ascontiguousarray(bits, np.uint16).astype(np.uint32) << 16).view(np.float32)


class GemvArgs(ctypes.Structure):
    """The launch descriptor of csrc/gemv_internal.h (zero: plain, STORE, AUTO)."""
    _fields_ = [("w", ctypes.c_void_p), ("s", ctypes.c_void_p), ("x", ctypes.c_void_p),
                ("ldx", ctypes.c_int), ("y", ctypes.c_void_p), ("ldy", ctypes.c_int),
                ("M", ctypes.c_int), ("N", ctypes.c_int), ("K", ctypes.c_int),
                ("wfmt", ctypes.c_int), ("gps", ctypes.c_int), ("splits", ctypes.c_int),
                ("win", ctypes.c_int), ("nrb", ctypes.c_int), ("ks", ctypes.c_int),
                ("rt", ctypes.c_int), ("xmode", ctypes.c_int), ("norm_w", ctypes.c_void_p),
                ("norm_eps", ctypes.c_float), ("ssq_in", ctypes.c_void_p),
                ("ssq_in_blocks", ctypes.c_int), ("epi", ctypes.c_int),
                ("ssq_out", ctypes.c_void_p), ("part", ctypes.c_void_p),
                ("part_cap", ctypes.c_int64), ("counters", ctypes.c_void_p),
                ("engine", ctypes.c_int), ("inv_in", ctypes.c_void_p),
                ("inv_out", ctypes.c_void_p), ("inv_eps", ctypes.c_float),
                ("deferred", ctypes.c_void_p)]


GEMV_AUTO, GEMV_STAGED = 0, 1
GEMV_STORE, GEMV_RESID, GEMV_SWIGLU = 0, 1, 2
GEMV_FMT = {"int4": 0, "int8": 1, "bf16": 2}
SSQ_ROWS = 128  # rows a block of sums of squares has room for


def gemv_launch(lib, fmt, w, s, x, y, M, N, K, ldy=None, engine=GEMV_AUTO, epi=GEMV_STORE,
                norm_w=None, ssq_in=None, ssq_out=None, eps=1e-6):
    """s2p_gemv_launch on the library's scratch; w, s, x, y, ..: device
    addresses; norm_w: with an input RMSNorm over rows of K"""
    for f, r in (("part", ctypes.c_void_p), ("part_cap", ctypes.c_int64),
                 ("counters", ctypes.c_void_p)):
        getattr(lib, "s2p_gemm_ctx_" + f).restype = r
    a = GemvArgs(w=w, s=s, x=x, ldx=K, y=y, ldy=N if ldy is None else ldy, M=M, N=N, K=K,
                 wfmt=GEMV_FMT[fmt], epi=epi, engine=engine, ssq_out=ssq_out,
                 part=lib.s2p_gemm_ctx_part(), part_cap=lib.s2p_gemm_ctx_part_cap(),
                 counters=lib.s2p_gemm_ctx_counters())
    if norm_w is not None:
        a.xmode, a.norm_w, a.norm_eps, a.ssq_in, a.ssq_in_blocks = 1, norm_w, eps, ssq_in, K // 16
    fn = lib.s2p_gemv_launch
    fn.restype, fn.argtypes = ctypes.c_int, [ctypes.c_void_p, ctypes.c_void_p]
    s2pamd.hip_check(fn(ctypes.byref(a), S()), "gemv launch")


def assert_close_rel(got, want, rel=1e-2, floor_frac=1e-2, what=""):
    """|got - want| <= rel * |want| + floor_frac * rms(want), elementwise."""
    got = np.asarray(got, np.float64)
    want = np.asarray(want, np.float64)
    rms = float(np.sqrt(np.mean(want ** 2))) if want.size else 0.0
    err = np.abs(got - want)
    bound = rel * np.abs(want) + floor_frac * rms
    bad = err > bound
    assert not bad.any(), (
        f"{what}: {int(bad.sum())}/{bad.size} beyond tolerance; max err {err.max():.4g} "
        f"(rms {rms:.4g}); worst at {np.unravel_index(np.argmax(err - bound), err.shape)}")


def assert_close_norm(got, want, rel=1e-2, what="", max_factor=2.0):
    """Per row: ||got - want||_2 <= rel ||want||_2 (the relative error of the
    row vector) and, as a guard against a few wild elements,
    max|got - want| <= max_factor * rel * max|want|; rel may be a per-row
    array."""
    got = np.asarray(got, np.float64)
    want = np.asarray(want, np.float64)
    d = got - want
    l2 = np.linalg.norm(d, axis=-1) / np.maximum(np.linalg.norm(want, axis=-1), 1e-30)
    mx = np.abs(d).max(axis=-1) / np.maximum(np.abs(want).max(axis=-1), 1e-30)
    rel = np.broadcast_to(np.asarray(rel, np.float64), l2.shape)
    assert (l2 <= rel).all() and (mx <= max_factor * rel).all(), (
        f"{what}: worst row L2 rel {l2.max():.3g} (row {int(l2.argmax())}), "
        f"worst row max-norm rel {mx.max():.3g} (row {int(mx.argmax())}), "
        f"tolerance {rel.min():.3g}..{rel.max():.3g}; failing rows "
        f"{[(int(i), round(float(l2[i]), 4), round(float(mx[i]), 4), round(float(rel[i]), 4)) for i in np.nonzero((l2 > rel) | (mx > max_factor * rel))[0]]}")
