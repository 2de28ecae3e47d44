"""mambo_gemm_plan for the tests: which kernel takes a call."""

from __future__ import annotations

import ctypes


def raw_plan(m, ns, blocks, ldxv=None, ldxs=None, config=None):
    """(status, GemmConfig) of a call of `ns` rows per projection and rows of K = 256 * blocks."""
    from mambo_amd import _native
    projections = (_native.Projection * len(ns))(*(_native.Projection(0, n, 0, n) for n in ns))
    cfg = None if config is None else ctypes.byref(_native.GemmConfig.from_dict(config))
    out = _native.GemmConfig()
    rc = _native.lib().mambo_gemm_plan(m, projections, len(ns), blocks, 256 * blocks if ldxv is None else ldxv,
                                       8 * blocks if ldxs is None else ldxs, cfg, ctypes.byref(out))
    return rc, out


def plan(m, ns, blocks, **kwargs) -> dict:
    from mambo_amd import _native
    rc, out = raw_plan(m, ns, blocks, **kwargs)
    _native.check(rc)
    return out.as_dict()


def wide_shape(p) -> tuple:
    """(32-token sub-tiles, waves of a K group, K groups, K slices) of a plan of the 32 x 32 MFMA
    kernel; None of another kernel's."""
    from mambo_amd import _native
    if p["kernel"] != _native.GEMM_WIDE:
        return None
    return p["tile_m"] // 32, p["tile_n"] // 32, p["waves"] // (p["tile_n"] // 32), p["split_k"]
