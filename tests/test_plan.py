"""mambo_gemm_plan (no GPU): what a projection call launches, and what it refuses."""

from __future__ import annotations

import ctypes

import pytest

from plan import plan, raw_plan


def test_plan_reports_the_kernel_of_a_call():
    from mambo_amd import _native
    # a named configuration comes back as it runs, its zero fields filled, its K slices counted
    named = {"kernel": _native.GEMM_TILED, "waves": 8, "tile_m": 64, "tile_n": 128, "split_k": 5}
    assert plan(512, [4096], 16, config=named) == {**named, "split_k": 4}
    assert plan(1, [4096], 16)["kernel"] == _native.GEMM_STREAM
    # the library's choice from 33 tokens: 128 x 256 tiles, and none of a family's configurations
    wide = plan(2048, [28672], 16)
    assert wide == {"kernel": _native.GEMM_WIDE, "waves": 8, "split_k": 1, "tile_m": 128, "tile_n": 256}
    default = _native.GemmConfig()
    assert _native.lib().mambo_gemm_default_config(2048, 28672, 16, ctypes.byref(default)) == 0
    assert default.kernel != _native.GEMM_WIDE
    assert plan(2048, [28672], 16, config=default.as_dict()) == default.as_dict()
    # few workgroups: small tiles of the tiled kernel, no K split
    small = plan(128, [1024], 16)
    assert (small["kernel"], small["split_k"]) == (_native.GEMM_TILED, 1) and small["tile_m"] <= 32
    # by the N of each projection, not by their sum alone
    assert plan(128, [16384], 16)["tile_m"] == 64 and plan(128, [16192, 64, 64, 64], 16)["tile_m"] == 128


def test_plan_refuses_what_the_call_refuses():
    from mambo_amd import _native
    lib, err = _native.lib(), _native.MAMBO_ERR_VALUE
    out = _native.GemmConfig()
    one = (_native.Projection * 1)(_native.Projection(0, 64, 0, 64))
    assert lib.mambo_gemm_plan(1, None, 1, 4, 1024, 32, None, ctypes.byref(out)) == err
    assert lib.mambo_gemm_plan(1, one, 1, 4, 1024, 32, None, None) == err
    for m, ns, blocks, kwargs, text in (
            (0, [64], 4, {}, "positive"), (1, [0], 4, {}, "n must be positive"), (1, [64] * 5, 4, {}, "count"),
            (64, [64], 4, {"ldxv": 1008}, "cover the row"), (64, [64], 4, {"ldxs": 24}, "cover the row"),
            (64, [64], 4, {"ldxv": 1 << 27}, "stride too large"),
            (64, [64], 4, {"config": {"kernel": _native.GEMM_WIDE}}, "unsupported kernel family"),
            (64, [64], 4, {"config": {"kernel": _native.GEMM_TILED, "waves": 3}}, "waves")):
        rc, _ = raw_plan(m, ns, blocks, **kwargs)
        assert rc == err and text in lib.mambo_last_error().decode(), (m, ns, kwargs, lib.mambo_last_error())
    with pytest.raises(ValueError, match="positive"):
        plan(0, [64], 4)


def test_plan_strides_within_32_bit_offsets():
    """The copies of a token tile address its rows with 32-bit offsets, values and scales alike. A call
    whose row strides do not fit a kernel's tile goes to one whose tile they fit, and is
    refused where the named default's tile is too tall for them."""
    from mambo_amd import _native
    top = (1 << 27) - 16  # strides end below 2^27
    for name, unit in (("ldxv", 16), ("ldxs", 8)):
        for m, ns, blocks in ((2048, [28672], 16), (128, [8192], 112), (48, [28672], 16), (300, [4096], 112)):
            assert plan(m, ns, blocks)["kernel"] == _native.GEMM_WIDE
            default = _native.GemmConfig()
            _native.check(_native.lib().mambo_gemm_default_config(m, sum(ns), blocks, ctypes.byref(default)))
            for ld in sorted({unit * (x // unit) + d * unit for s in range(20, 27) for d in (-1, 0, 1)
                              for x in (1 << s, (1 << s) * 33 // 32)} | {top}):
                rc, p = raw_plan(m, ns, blocks, **{name: ld})
                fits = default.kernel != _native.GEMM_TILED or default.tile_m * ld < 1 << 32
                assert (rc == 0) == fits, (m, name, ld)
                if rc == 0 and p.kernel in (_native.GEMM_WIDE, _native.GEMM_TILED):
                    assert (p.tile_m - 1) * ld + 256 * blocks < 1 << 32, (m, name, ld, p.as_dict())


def test_plan_where_the_named_default_is_the_faster():
    """Launches that the small tiles and the 32 x 32 kernel leave to the named default, and the other
    side of each line."""
    from mambo_amd import _native
    dense, tiled, wide = _native.GEMM_DENSE, _native.GEMM_TILED, _native.GEMM_WIDE
    # up to 10 tokens, 64-row tiles of one workgroup per CU, or of two on a long K
    assert [plan(m, [15692], 64)["kernel"] for m in (5, 10, 11)] == [dense, dense, tiled]
    assert [plan(m, [28569], 64)["kernel"] for m in (5, 10, 11)] == [dense, dense, tiled]
    assert plan(5, [28672], 32)["kernel"] == tiled  # two on a shorter K
    assert plan(8, [14336], 32)["tile_n"] == 32 and plan(8, [14336], 32)["kernel"] == tiled
    # four K blocks where 64-token tiles are one round of two workgroups per CU
    assert plan(400, [8192], 4) == {"kernel": tiled, "waves": 8, "split_k": 1, "tile_m": 64, "tile_n": 128}
    assert plan(400, [10240], 4)["kernel"] == wide and plan(400, [8192], 5)["kernel"] == wide
    # eight waves of 32 rows from nine K blocks, and on fewer where four would just pass a workgroup per CU
    assert plan(959, [7383], 5)["tile_n"] == 128 and plan(960, [28672], 9)["tile_n"] == 256
    assert plan(384, [13208], 6)["tile_n"] == 256
