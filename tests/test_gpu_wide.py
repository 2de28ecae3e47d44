"""The 32 x 32 MFMA kernel (gemm_wide_kernel), which takes calls of 33 tokens and more that
leave the configuration to the library: each of its shapes at ragged token and row counts, odd
and even K blocks, with and without a K split, grouped, strided, and with the scales and block
scales that a wrong lane or a wrong block would show.

Tolerance: the products of 8-bit floats are exact in f32 and every kernel here sums them in
f32 inside the MFMA; two orders of those sums differ by 2.6e-5 rel-L2 from the oracle's float64
product at K = 512 to 28672. 1e-4 is four times that; a wrong group, scale or sign is > 1e-2."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from conftest import make_synthetic_iq3_s, rel_l2
from oracle import oracle
from test_gpu_matmul import step

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


# tokens, rows of each projection, K blocks: 64-token tiles of one and two K groups (odd and even
# blocks, the second group's last one missing) without and with a K split (9 and 16 blocks: unsplit
# and split other plans; slices of one and of several blocks), 128-token tiles of two K groups and of
# eight waves, the shapes taken over from the dense kernel; last 16-row tile alone in its pair, tokens
# one past and one short of a tile, one to all of a tile's rows padded
SHAPES = [(257, [100], 9), (320, [33], 10), (256, [16, 17, 48], 11), (300, [130], 16), (385, [64, 1], 33),
          (1000, [4090], 4), (1025, [3000, 1100], 5), (961, [8190], 5), (1024, [8000, 190], 4),
          (33, [6204], 11), (63, [12288 + 16], 4), (40, [10200], 5), (128, [4100, 4000], 23), (129, [8192], 13),
          (65, [1000], 64), (2048, [16000], 4), (48, [57344], 4),
          # four K groups of 64 x 64 tiles: blocks that leave one to three groups short
          (96, [8100], 33), (128, [6000, 130], 18), (97, [8192], 15)]


@pytest.mark.parametrize("m,ns,blocks", SHAPES)
def test_wide_shapes(gpu, m, ns, blocks):
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


@pytest.mark.parametrize("m,n,blocks", [(257, 100, 9), (300, 130, 16), (1000, 4090, 4)])
def test_wide_scales_and_special_values(gpu, m, n, blocks):
    """Activation scales spread over 80 binades, zero and negative block scales, a NaN activation
    scale and a NaN block scale: the same values, and NaN in the same places, as an explicit
    configuration of the tiled kernel."""
    k = 256 * blocks
    rng = np.random.default_rng(n)
    raw = make_synthetic_iq3_s(n, k, seed=n)
    d = raw[..., :2].view(np.float16)
    d[3::7, blocks // 2] = 0.0
    d[5::11] = -d[5::11]
    d[8, blocks - 1] = np.nan
    xv, _ = oracle.quantize_mxfp8(rng.standard_normal((m, k)).astype(np.float32))
    xs = rng.integers(87, 168, size=(m, k // 32)).astype(np.uint8)
    xs[m - 1, 5] = 255
    step(f"wide scales M={m} N={n} K={k}")
    got, = project(gpu, xv, xs, [raw])
    want, = project(gpu, xv, xs, [raw], config={"kernel": 2, "tile_m": 64, "tile_n": 128, "waves": 8, "split_k": 1})
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.isnan(want[m - 1]).all() and np.isnan(want[:, 8]).all() and np.isfinite(want).any()
    ok = np.isfinite(want)
    for i in range(0, m, 37):  # per token: their scales differ by 80 binades
        j = ok[i]
        if j.any():
            assert rel_l2(got[i, j], want[i, j]) < 1e-4


# tokens, rows of each projection, K blocks for the small tiles that take launches of few
# workgroups: each tile (16 and 32 tokens, 16, 32 and 64 rows), first and last tokens and rows of a tile, blocks
# that divide among eight waves' K groups or leave some without, the last token count of the rule
SMALL = [(33, [1], 4), (64, [16, 17], 5), (65, [100, 33, 1], 8), (48, [4090], 16), (96, [1000], 9), (129, [2050], 7),
         (256, [700, 64], 13), (48, [8190], 23), (128, [4100], 4), (34, [3000], 112), (5, [640], 13), (16, [1, 300], 3),
         (17, [250], 2), (12, [2300], 47), (400, [330], 7), (400, [3170], 2)]


@pytest.mark.parametrize("m,ns,blocks", SMALL)
def test_launches_of_few_workgroups(gpu, m, ns, blocks):
    """Against the oracle, and the same bits again (no K split takes these calls)."""
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


@pytest.mark.parametrize("m,n,blocks", [(128, 6000, 17), (300, 130, 9)])
def test_wide_infinite_sums(gpu, m, n, blocks):
    """A token whose sums overflow f32: infinities (no NaN from a K group's missing last block),
    as the tiled kernel gives them, and finite values elsewhere."""
    k = 256 * blocks
    raw = make_synthetic_iq3_s(n, k, seed=n)
    xv = np.full((m, k), 0x38, dtype=np.uint8)  # 1.0
    xs = np.full((m, k // 32), 127, dtype=np.uint8)
    xv[7], xs[7] = 0x7E, 254  # 448 * 2^127
    step(f"wide infinities M={m} N={n} K={k}")
    got, = project(gpu, xv, xs, [raw])
    want, = project(gpu, xv, xs, [raw], config={"kernel": 2, "tile_m": 64, "tile_n": 128, "waves": 8, "split_k": 1})
    assert np.isfinite(np.delete(got, 7, 0)).all() and not np.isfinite(want[7]).any()
    assert np.array_equal(np.isinf(got[7]).any(), np.isinf(want[7]).any())
    last = blocks - 1
    assert last % 2 == 0  # both counts leave a group's last block out


def test_wide_same_bits_without_a_split_and_under_capture(gpu):
    """No K split: repeated calls, a grouped call of the same shape of workgroup and replays of a
    captured call give the same bits."""
    from mambo_amd.kernels.iq3_s_fp8 import launch_iq3_s_fp8_matmul
    from mambo_amd.utils.iq3_s_weight import prepare_iq3_s_fields
    m, n, k = 1000, 2000, 1024
    raw = make_synthetic_iq3_s(n, k, seed=2)
    x = np.random.default_rng(3).standard_normal((m, k)).astype(np.float32)
    xv, xs = oracle.quantize_mxfp8(x)
    step("wide, same bits")
    first, = project(gpu, xv, xs, [raw])
    again = project(gpu, xv, xs, [raw, raw[:900].copy()])
    assert np.array_equal(first, again[0]) and np.array_equal(first[:, :900], again[1])
    w = prepare_iq3_s_fields(torch.from_numpy(raw).to(gpu), fields=False)
    a, s = torch.from_numpy(xv).to(gpu), torch.from_numpy(xs).to(gpu)
    out = torch.empty((m, n), device=gpu)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(side), torch.cuda.graph(graph, stream=side):
        launch_iq3_s_fp8_matmul(a, s, w, config={"kernel": 0}, out=out)
    torch.cuda.current_stream().wait_stream(side)
    for _ in range(3):
        out.fill_(-1.0)
        graph.replay()
        torch.cuda.synchronize()
        assert np.array_equal(out.cpu().numpy(), first)


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
