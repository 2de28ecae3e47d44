"""The 32 x 32 MFMA kernel (gemm_wide_kernel), which takes calls of 33 tokens and more that
leave the configuration to the library, and the small tiles of the tiled kernel, which take those of few
workgroups: each shape of either at ragged token and row counts, odd and even K blocks, with and
without a K split, grouped, strided, and with the scales and block scales that a wrong lane or a wrong
block would show. Which kernel and shape a case runs is part of the case (mambo_gemm_plan).

Tolerance: the products of 8-bit floats are exact in f32 and every kernel here sums them in
f32 inside the MFMA; two orders of those sums differ by 2.6e-5 rel-L2 from the oracle's float64
product at K = 512 to 28672. 1e-4 is four times that; a wrong group, scale or sign is > 1e-2."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from conftest import make_synthetic_iq3_s, rel_l2
from oracle import oracle
from plan import plan, wide_shape
from test_gpu_configs import columns, oracle_rows, sample_rows
from test_gpu_matmul import _synth_act, _synth_weight, step

pytestmark = pytest.mark.gpu


def project(gpu, xv, xs, raws, config=None, pad=0):
    """Outputs of one call, in buffers with `pad` guard columns and one guard row that the
    kernel must leave alone."""
    from mambo_amd.kernels.iq3_s_fp8 import launch_iq3_s_fp8_matmul_grouped
    from mambo_amd.utils.iq3_s_weight import prepare_iq3_s_fields
    weights = [prepare_iq3_s_fields(torch.from_numpy(r).to(gpu), fields=False) for r in raws]
    m = xv.shape[0]
    bufs = [torch.full((m + 1, r.shape[0] + pad), 12345.0, device=gpu) for r in raws]
    outs = [b[:m, :r.shape[0]] for b, r in zip(bufs, raws)]
    launch_iq3_s_fp8_matmul_grouped(torch.from_numpy(xv).to(gpu), torch.from_numpy(xs).to(gpu), weights,
                                    config=config or {"kernel": 0}, outs=outs)
    torch.cuda.synchronize()
    for b, r in zip(bufs, raws):
        assert bool((b[m:] == 12345.0).all()) and bool((b[:, r.shape[0]:] == 12345.0).all())
    return [o.cpu().numpy() for o in outs]


# tokens, rows of each projection, K blocks, shape: 32-token sub-tiles, waves of a K group, K groups and K
# slices. Each of the six shapes of the kernel unsplit and, where a split takes it, split: K groups
# that a slice leaves one to three blocks short (9 blocks for two groups, 7, 10, 15, 18 and 33 for four),
# slices of one and of several blocks with a short last one, last 16-row tile alone in its pair, tokens
# one past and one short of a tile, one to all of a tile's rows padded
SHAPES = [(1000, [4090], 4, (4, 4, 2, 1)), (1025, [3000, 1100], 5, (2, 4, 1, 1)), (961, [8190], 5, (4, 4, 1, 1)),
          (1024, [8000, 190], 4, (4, 4, 1, 1)), (450, [8208], 4, (4, 8, 1, 1)), (2048, [16000], 4, (4, 4, 1, 1)),
          (48, [57344], 4, (2, 4, 1, 1)), (338, [11079], 9, (4, 8, 1, 1)), (1000, [8190], 10, (4, 8, 1, 1)),
          (129, [8192], 13, (2, 4, 2, 1)), (76, [10895, 18], 9, (2, 4, 2, 1)), (146, [11106], 9, (4, 4, 2, 1)),
          (35, [8882], 7, (2, 2, 4, 1)), (718, [2], 10, (2, 2, 4, 1)), (128, [4100, 4000], 23, (2, 2, 4, 1)),
          (96, [8100], 33, (2, 2, 4, 1)), (128, [6000, 130], 18, (2, 2, 4, 1)), (97, [8192], 15, (2, 2, 4, 1)),
          (65, [1000], 64, (2, 2, 4, 8)), (875, [3], 17, (2, 2, 4, 6)), (470, [21, 251], 26, (2, 4, 1, 9)),
          (64, [4384], 61, (2, 4, 2, 6)), (912, [1, 104], 41, (2, 4, 2, 7)), (206, [10810], 63, (4, 4, 1, 3)),
          (69, [6290, 159], 33, (4, 4, 2, 4)), (1134, [326, 170], 49, (4, 4, 2, 4)), (263, [6375, 137], 46, (4, 8, 1, 3))]


@pytest.mark.parametrize("m,ns,blocks,shape", SHAPES)
def test_wide_shapes(gpu, m, ns, blocks, shape):
    assert wide_shape(plan(m, ns, blocks)) == shape
    k = 256 * blocks
    raws = [make_synthetic_iq3_s(n, k, seed=7 * m + i) for i, n in enumerate(ns)]
    x = np.random.default_rng(m).standard_normal((m, k)).astype(np.float32)
    xv, xs = oracle.quantize_mxfp8(x)
    step(f"wide M={m} N={ns} K={k}")
    for o, raw in zip(project(gpu, xv, xs, raws, pad=5), raws):
        rows = np.unique(np.r_[np.arange(min(48, raw.shape[0])), np.arange(max(0, raw.shape[0] - 40), raw.shape[0]),
                               np.random.default_rng(1).choice(raw.shape[0], 40)])
        assert np.isfinite(o).all()
        assert rel_l2(o[:, rows], oracle.iq3s_fp8_matmul(xv, xs, raw[rows], threads=oracle.default_threads())) < 1e-4


# each shape with its K groups a block or more short, and split
SPECIAL = [(1000, 4090, 4, (4, 4, 2, 1)), (146, 11106, 9, (4, 4, 2, 1)), (76, 10913, 9, (2, 4, 2, 1)),
           (97, 8192, 15, (2, 2, 4, 1)), (718, 20, 10, (2, 2, 4, 1)), (961, 8190, 5, (4, 4, 1, 1)),
           (338, 11079, 9, (4, 8, 1, 1)), (1025, 4100, 5, (2, 4, 1, 1)), (875, 30, 17, (2, 2, 4, 6)),
           (64, 4384, 61, (2, 4, 2, 6))]


@pytest.mark.parametrize("m,n,blocks,shape", SPECIAL)
def test_wide_scales_and_special_values(gpu, m, n, blocks, shape):
    """Activation scales spread over 80 binades, zero and negative block scales, NaN activation
    scales and block scales, in the last block too, which a short K group takes again: the same values, and NaN in
    the same places, as an explicit configuration of the tiled kernel."""
    assert wide_shape(plan(m, [n], blocks)) == shape
    k = 256 * blocks
    rng = np.random.default_rng(n)
    raw = make_synthetic_iq3_s(n, k, seed=n)
    d = raw[..., :2].view(np.float16)
    d[3::7, blocks // 2] = 0.0
    d[5::11] = -d[5::11]
    d[1::13, blocks - 1] = 0.0
    d[8, blocks - 1] = np.nan
    xv, _ = oracle.quantize_mxfp8(rng.standard_normal((m, k)).astype(np.float32))
    xs = rng.integers(87, 168, size=(m, k // 32)).astype(np.uint8)
    xs[m - 1, 5] = 255
    xs[m - 3, k // 32 - 1] = 255
    step(f"wide scales M={m} N={n} K={k}")
    got, = project(gpu, xv, xs, [raw])
    want, = project(gpu, xv, xs, [raw], config={"kernel": 2, "tile_m": 64, "tile_n": 128, "waves": 8, "split_k": 1})
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.isnan(want[m - 1]).all() and np.isnan(want[m - 3]).all() and np.isnan(want[:, 8]).all()
    rest = np.delete(np.delete(want, [m - 1, m - 3], 0), 8, 1)
    assert np.isfinite(rest).all()
    ok = np.isfinite(want)
    for i in range(0, m, 37):  # per token: their scales differ by 80 binades
        j = ok[i]
        if j.any():
            assert rel_l2(got[i, j], want[i, j]) < 1e-4


# tokens, rows of each projection, K blocks, tokens and rows of the small tile: each tile (16 and 32
# tokens, 16, 32 and 64 rows), first and last tokens and rows of a tile, blocks that divide among eight waves'
# K groups or leave some without, the first and last token counts of the rule
SMALL = [(33, [1], 4, (16, 32)), (64, [16, 17], 5, (16, 16)), (65, [100, 33, 1], 8, (16, 16)),
         (48, [4090], 16, (32, 32)), (96, [1000], 9, (16, 32)), (129, [2050], 7, (32, 32)),
         (256, [700, 64], 13, (32, 32)), (48, [8190], 23, (32, 64)), (128, [4100], 4, (32, 64)),
         (34, [3000], 112, (32, 32)), (5, [640], 13, (16, 16)), (16, [1, 300], 3, (16, 32)), (17, [250], 2, (16, 64)),
         (12, [2300], 47, (16, 16)), (400, [330], 7, (32, 32)), (400, [330], 2, (16, 64)), (400, [1000], 3, (32, 64)),
         (257, [100], 9, (16, 16)), (320, [33], 10, (16, 16)), (256, [16, 17, 48], 11, (16, 16)),
         (300, [130], 16, (16, 16)), (385, [64, 1], 33, (16, 16)), (33, [6204], 11, (32, 32)),
         (63, [12288 + 16], 4, (32, 64)), (40, [10200], 5, (32, 64)), (81, [700], 5, (32, 16)), (284, [247], 8, (32, 16)),
         (11, [15692], 8, (16, 64))]


@pytest.mark.parametrize("m,ns,blocks,tile", SMALL)
def test_launches_of_few_workgroups(gpu, m, ns, blocks, tile):
    """Against the oracle, and the same bits again (no K split takes these calls)."""
    p = plan(m, ns, blocks)
    assert p == {"kernel": 2, "waves": 8, "split_k": 1, "tile_m": tile[0], "tile_n": tile[1]}
    k = 256 * blocks
    raws = [make_synthetic_iq3_s(n, k, seed=11 * m + i) for i, n in enumerate(ns)]
    x = np.random.default_rng(m).standard_normal((m, k)).astype(np.float32)
    xv, xs = oracle.quantize_mxfp8(x)
    step(f"few workgroups M={m} N={ns} K={k}")
    first = project(gpu, xv, xs, raws, pad=3)
    for o, raw in zip(first, raws):
        rows = np.unique(np.r_[np.arange(min(40, raw.shape[0])), np.arange(max(0, raw.shape[0] - 40), raw.shape[0])])
        assert np.isfinite(o).all()
        assert rel_l2(o[:, rows], oracle.iq3s_fp8_matmul(xv, xs, raw[rows], threads=oracle.default_threads())) < 1e-4
    for o, again in zip(first, project(gpu, xv, xs, raws)):
        assert np.array_equal(o, again)


# each shape, with K groups one to three blocks short, and split
INFINITE = [(128, 6000, 17, (2, 2, 4, 1)), (97, 8192, 15, (2, 2, 4, 1)), (718, 20, 10, (2, 2, 4, 1)),
            (76, 10913, 9, (2, 4, 2, 1)), (146, 11106, 9, (4, 4, 2, 1)), (1000, 4090, 4, (4, 4, 2, 1)),
            (961, 8190, 5, (4, 4, 1, 1)), (338, 11079, 9, (4, 8, 1, 1)), (1025, 4100, 5, (2, 4, 1, 1)),
            (875, 30, 17, (2, 2, 4, 6)), (64, 4384, 61, (2, 4, 2, 6))]


@pytest.mark.parametrize("m,n,blocks,shape", INFINITE)
def test_wide_infinite_sums(gpu, m, n, blocks, shape):
    """A token all of whose products overflow f32 with one sign (weights of one four-bit term, no signs):
    each block's sum is infinite, so a row of positive block scales gives +inf, one of negative ones -inf, one
    with both or with a zero among them NaN - element by element, with no NaN from a K group's missing
    last block - and the other tokens stay finite."""
    assert wide_shape(plan(m, [n], blocks)) == shape
    k = 256 * blocks
    raw = make_synthetic_iq3_s(n, k, seed=n)
    raw[..., 74:] = 0  # signs and scale nibbles
    d = raw[..., :2].view(np.float16)
    d[1::4] = -d[1::4]
    d[2::5, blocks - 1] = -d[2::5, blocks - 1]
    d[3::6, 0] = 0.0
    xv = np.full((m, k), 0x38, dtype=np.uint8)  # 1.0
    xs = np.full((m, k // 32), 127, dtype=np.uint8)
    xv[7], xs[7] = 0x7E, 254  # 448 * 2^127
    step(f"wide infinities M={m} N={n} K={k}")
    got, = project(gpu, xv, xs, [raw])
    dd = d.reshape(n, blocks).astype(np.float64)
    want = np.where((dd > 0).all(1), np.inf, np.where((dd < 0).all(1), -np.inf, np.nan))
    assert {np.inf, -np.inf} <= set(want) and np.isnan(want).any()
    np.testing.assert_array_equal(got[7], want)
    assert np.isfinite(np.delete(got, 7, 0)).all()


@pytest.mark.parametrize("m,n,second,blocks,shape", [
    (961, 8190, 900, 5, (4, 4, 1, 1)), (1025, 4100, 300, 5, (2, 4, 1, 1)), (718, 30, 16, 10, (2, 2, 4, 1)),
    (76, 10900, 13, 9, (2, 4, 2, 1)), (146, 11000, 106, 9, (4, 4, 2, 1)), (338, 11079, 100, 9, (4, 8, 1, 1))])
def test_wide_same_bits_without_a_split_and_under_capture(gpu, m, n, second, blocks, shape):
    """No K split: repeated calls, a grouped call of the same shape of workgroup and replays of a
    captured call give the same bits."""
    from mambo_amd.kernels.iq3_s_fp8 import launch_iq3_s_fp8_matmul
    from mambo_amd.utils.iq3_s_weight import prepare_iq3_s_fields
    assert wide_shape(plan(m, [n], blocks)) == wide_shape(plan(m, [n, second], blocks)) == shape
    k = 256 * blocks
    raw = make_synthetic_iq3_s(n, k, seed=2)
    x = np.random.default_rng(3).standard_normal((m, k)).astype(np.float32)
    xv, xs = oracle.quantize_mxfp8(x)
    step(f"wide, same bits M={m} N={n} K={k}")
    first, = project(gpu, xv, xs, [raw])
    again = project(gpu, xv, xs, [raw, raw[:second].copy()])
    assert np.array_equal(first, again[0]) and np.array_equal(first[:, :second], again[1])
    w = prepare_iq3_s_fields(torch.from_numpy(raw).to(gpu), fields=False)
    for out in replays(gpu, lambda a, s, out: launch_iq3_s_fp8_matmul(a, s, w, config={"kernel": 0}, out=out),
                       xv, xs, n):
        assert np.array_equal(out, first)


def replays(gpu, call, xv, xs, n):
    """The output of each of three replays of a captured call, written to between them."""
    a, s = torch.from_numpy(xv).to(gpu), torch.from_numpy(xs).to(gpu)
    out = torch.empty((xv.shape[0], n), device=gpu)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(side), torch.cuda.graph(graph, stream=side):
        call(a, s, out)
    torch.cuda.current_stream().wait_stream(side)
    for _ in range(3):
        out.fill_(-1.0)
        graph.replay()
        torch.cuda.synchronize()
        yield out.cpu().numpy()


@pytest.mark.parametrize("m,n,blocks,shape", [(65, 1000, 64, (2, 2, 4, 8)), (64, 4384, 61, (2, 4, 2, 6)),
                                              (470, 272, 26, (2, 4, 1, 9))])
def test_wide_split_under_capture(gpu, m, n, blocks, shape):
    """A captured K split clears its outputs in every replay: each within two orders of f32
    atomics (a few ulp of the largest partial sum, 1e-6 of the result's norm) of the eager call."""
    from mambo_amd.kernels.iq3_s_fp8 import launch_iq3_s_fp8_matmul
    from mambo_amd.utils.iq3_s_weight import prepare_iq3_s_fields
    assert wide_shape(plan(m, [n], blocks)) == shape
    k = 256 * blocks
    raw = make_synthetic_iq3_s(n, k, seed=6)
    xv, xs = oracle.quantize_mxfp8(np.random.default_rng(6).standard_normal((m, k)).astype(np.float32))
    step(f"wide split, captured M={m} N={n} K={k}")
    eager, = project(gpu, xv, xs, [raw])
    w = prepare_iq3_s_fields(torch.from_numpy(raw).to(gpu), fields=False)
    for out in replays(gpu, lambda a, s, out: launch_iq3_s_fp8_matmul(a, s, w, config={"kernel": 0}, out=out),
                       xv, xs, n):
        assert rel_l2(out, eager) < 1e-6


# the default path at the sweep's launches (70B q/k/v and o, 8B q/k/v, o, gate/up and down) at both
# ends of the token buckets from 64 to 512
@pytest.mark.parametrize("n,k,bucket", [(10240, 8192, 64), (10240, 8192, 128), (10240, 8192, 256), (28672, 4096, 64),
                                        (28672, 4096, 128), (4096, 14336, 256), (4096, 4096, 128), (4096, 4096, 256),
                                        (6144, 4096, 64), (6144, 4096, 128), (6144, 4096, 256), (6144, 4096, 512),
                                        (8192, 8192, 64), (8192, 8192, 128)])
def test_default_path_at_the_sweep_launches(gpu, n, k, bucket):
    from mambo_amd.kernels.iq3_s_fp8 import launch_iq3_s_fp8_matmul
    from mambo_amd.kernels.quantize_fp8 import launch_quantize_fp8
    seed = 700 + (n // 16 + k // 256 + bucket) % 200
    step(f"synth weight {n}x{k}")
    fields = _synth_weight(gpu, n, k, seed=seed)
    rows = sample_rows(n, 24, seed)
    for m in (bucket, bucket // 2 + 1):
        xq, xs = launch_quantize_fp8(_synth_act(gpu, m, k, seed=seed + m))
        step(f"default path M={m} {n}x{k}: {plan(m, [n], k // 256)}")
        out = launch_iq3_s_fp8_matmul(xq, xs, fields)
        torch.cuda.synchronize()
        assert rel_l2(columns(out, rows), oracle_rows(xq, xs, seed, k, rows)) < 1e-4
        assert bool(torch.isfinite(out).all())


def test_scale_rows_beyond_32_bit_offsets(gpu):
    """Rows of scales so far apart that 63 of them pass 4 GiB: not for tiles with 32-bit offsets."""
    from mambo_amd.kernels.iq3_s_fp8 import launch_iq3_s_fp8_matmul
    from mambo_amd.utils.iq3_s_weight import prepare_iq3_s_fields
    m, n, blocks, ld = 63, 12304, 4, (1 << 32) // 62 // 8 * 8 + 8
    k = 256 * blocks
    raw = make_synthetic_iq3_s(n, k, seed=5)
    xv, xs = oracle.quantize_mxfp8(np.random.default_rng(5).standard_normal((m, k)).astype(np.float32))
    w = prepare_iq3_s_fields(torch.from_numpy(raw).to(gpu), fields=False)
    far = torch.empty(m * ld, dtype=torch.uint8, device=gpu).as_strided((m, k // 32), (ld, 1))
    far.copy_(torch.from_numpy(xs).to(gpu))
    step(f"scale rows {ld} bytes apart")
    out = launch_iq3_s_fp8_matmul(torch.from_numpy(xv).to(gpu), far, w, config={"kernel": 0}).cpu().numpy()
    rows = np.random.default_rng(1).choice(n, 64, replace=False)
    assert rel_l2(out[:, rows], oracle.iq3s_fp8_matmul(xv, xs, raw[rows], threads=oracle.default_threads())) < 1e-4
