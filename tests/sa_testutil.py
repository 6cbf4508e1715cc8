"""Helpers shared by the tests: the launch plan the library will choose.

Several tests exercise one kernel path (shared-row tiles, no split; one form of
the fused_moe tiles) and pick their shapes for it. They assert the plan first,
through the g++ build of the host-side planners (``libsa_host_test.so``, the
same ``sa_plan.h`` and ``fm_plan.h`` the HIP libraries compile); sparse_attn's
depends on the device's compute-unit count.
"""
import ctypes
import os

import torch

import sa_capi

_LIB = os.path.join(os.path.dirname(sa_capi.LIB_PATH), "libsa_host_test.so")
_host = None
_KEYS = ["nsplit", "split_len", "tiles", "tiles_per_b", "ntiles", "tile_cap", "ws",
         "meta_off", "order_off", "rows_off", "cnts_off", "part_off"]


def device_cus() -> int:
    return torch.cuda.get_device_properties(torch.cuda.current_device()).multi_processor_count


def host_lib():
    global _host
    if _host is None:
        _host = ctypes.CDLL(_LIB)
        _host.sa_host_plan_full.argtypes = [ctypes.POINTER(sa_capi.SaArgs), ctypes.c_int,
                                            ctypes.POINTER(ctypes.c_int64)]
        _host.fm_host_plan.argtypes = [ctypes.POINTER(sa_capi.FmArgs),
                                       ctypes.POINTER(ctypes.c_int64)]
    return _host


def moe_plan(M, K, N, E, topk, flags=0) -> dict:
    """The kernel and tiles fused_moe runs for this shape: gemm (fm_gemm_kernel),
    tile_rows, narrow_rows (tiles of at most this many pairs are narrow), pb."""
    a = sa_capi.FmArgs()
    a.hidden = a.w1 = a.w2 = a.score = a.out = 0x10000  # only their alignment is read
    a.M, a.K, a.N, a.E, a.topk, a.flags = M, K, N, E, topk, flags
    a.s_hidden, a.s_score, a.s_out = K, E, K
    out = (ctypes.c_int64 * 4)()
    rc = host_lib().fm_host_plan(ctypes.byref(a), out)
    assert rc == sa_capi.FM_OK, f"moe plan: code {rc}"
    return dict(zip(("gemm", "tile_rows", "narrow_rows", "pb"), out))


def plan_of(q, kv, idx, flags=0) -> dict:
    """The plan sa_forward makes for these tensors on the current device."""
    o = q  # only its strides and pointer alignment are read
    a = sa_capi.make_args(q, kv, q.new_zeros(16, dtype=torch.float32), idx, o, 1.0, flags)
    out = (ctypes.c_int64 * len(_KEYS))()
    rc = host_lib().sa_host_plan_full(ctypes.byref(a), device_cus(), out)
    assert rc == sa_capi.SA_OK, f"plan: code {rc}"
    return dict(zip(_KEYS, list(out)))


def expect_plan(q, kv, idx, flags=0, tiles=None, nsplit=None) -> dict:
    """Assert the plan these tests rely on (shared-row tiles, no split, ...)."""
    p = plan_of(q, kv, idx, flags)
    if tiles is not None:
        assert bool(p["tiles"]) == tiles, f"plan has tiles={bool(p['tiles'])} on " \
                                          f"{device_cus()} CUs; the test needs {tiles}"
    if nsplit is not None:
        assert p["nsplit"] == nsplit, f"plan splits {p['nsplit']} ways on {device_cus()} CUs"
    return p
