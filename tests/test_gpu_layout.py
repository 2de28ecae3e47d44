"""Weight preparation and decoding at the edges of their workgroups (64 rows x 4 blocks or a tile;
32 rows x 4 blocks or 16 x 1), from every form of source: whole fields against numpy, bit for bit,
and the tile layout against the one that the byte path builds."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from conftest import make_synthetic_iq3_s
from oracle import oracle
from test_gpu_matmul import step

pytestmark = pytest.mark.gpu


def reference_fields(raw):
    """numpy form of the five fields of u8 [N, B, 110]."""
    x = np.ascontiguousarray(raw.transpose(1, 0, 2))

    def field(a, b, dtype):
        return np.ascontiguousarray(x[:, :, a:b]).view(dtype)

    return {"d": field(0, 2, np.float16)[..., 0], "qs": field(2, 66, np.uint32), "qh": field(66, 74, np.uint16),
            "signs": field(74, 106, np.int32), "scales": field(106, 110, np.uint32)[..., 0]}


def sources(raw, gpu):
    """The same blocks as tensors of other bases and strides: the first six hold contiguous blocks,
    the last two do not (read in bytes)."""
    n, blocks, size = raw.shape
    x = torch.from_numpy(raw).to(gpu)
    yield "aligned", x
    for off in (1, 2, 3):
        flat = torch.empty(raw.size + off, dtype=torch.uint8, device=gpu)
        v = flat[off:].view(raw.shape)
        v.copy_(x)
        yield f"base + {off}", v
    wide = torch.empty((n, blocks + 1, size), dtype=torch.uint8, device=gpu)[:, 1:]
    wide.copy_(x)
    yield "rows of a wider matrix", wide
    rows = torch.empty((2 * n, blocks, size), dtype=torch.uint8, device=gpu)[::2]
    rows.copy_(x)
    yield "every second row", rows
    apart = torch.empty((n, blocks, 2 * size), dtype=torch.uint8, device=gpu)[..., ::2]
    apart.copy_(x)
    yield "every second byte", apart
    yield "blocks first", x.transpose(0, 1).contiguous().transpose(0, 1)


@pytest.mark.parametrize("n,blocks", [
    (1, 1), (16, 2), (45, 5),  # a tile per workgroup
    # 64 rows x 4 blocks: from 192 workgroups on whose rows hold 600 blocks together
    (1, 768), (65, 383), (192, 254), (12225, 1), (1100, 61), (38337, 1), (13000, 3)])
def test_prepare_forms_agree(gpu, n, blocks):
    from mambo_amd.kernels.iq3_s_fp8 import launch_dequant_iq3_s
    from mambo_amd.utils.iq3_s_weight import IQ3SFields, ensure_packed, prepare_iq3_s_fields
    raw = make_synthetic_iq3_s(n, blocks * 256, seed=n + blocks)
    want = reference_fields(raw)
    step(f"prepare, byte path [{n},{blocks},110]")
    forms = dict(sources(raw, gpu))
    tile = prepare_iq3_s_fields(forms["every second byte"], fields=False).packed
    for name, source in forms.items():
        step(f"prepare {name} [{n},{blocks},110]")
        f = prepare_iq3_s_fields(source, pack=True)
        for field, value in want.items():
            got = getattr(f, field).cpu().contiguous().view(torch.uint8).numpy()
            np.testing.assert_array_equal(got.ravel(), value.view(np.uint8).ravel(), err_msg=f"{name}: {field}")
        assert torch.equal(f.packed, tile), name
        assert torch.equal(prepare_iq3_s_fields(source, fields=False).packed, tile), name
    step(f"pack and dequant [{n},{blocks},110]")
    assert torch.equal(ensure_packed(IQ3SFields(f.d, f.qs, f.qh, f.signs, f.scales)), tile)
    bits, scales = launch_dequant_iq3_s(f)
    torch.cuda.synchronize()
    want_bits, want_scales = oracle.dequant_iq3s_fp8(raw)
    np.testing.assert_array_equal(bits.cpu().numpy(), want_bits)
    np.testing.assert_array_equal(scales.cpu().numpy(), want_scales)


def test_prepare_of_repeated_rows(gpu):
    """A row stride of zero, the smallest there is."""
    from mambo_amd.utils.iq3_s_weight import prepare_iq3_s_fields
    raw = make_synthetic_iq3_s(1, 5 * 256, seed=4)
    x = torch.from_numpy(raw).to(gpu)
    step("prepare expanded rows [7000,5,110]")
    a = prepare_iq3_s_fields(x.expand(7000, -1, -1), pack=True)
    b = prepare_iq3_s_fields(x.expand(7000, -1, -1).contiguous(), pack=True)
    assert torch.equal(a.packed, b.packed) and torch.equal(a.signs, b.signs) and torch.equal(a.d, b.d)


# (16 rows x 1 block up to 32767 blocks, 32 x 4 from there)
@pytest.mark.parametrize("n,blocks", [(1, 1), (31, 3), (33, 4), (64, 5), (100, 9), (32767, 1), (16384, 2), (33, 993),
                                      (8193, 5), (31, 1059)])
def test_dequant_into_scales_of_any_float_alignment(gpu, n, blocks):
    """Edges of the decoder's workgroups, the scales four bytes off a 16-byte boundary, and
    nothing written outside either output."""
    from mambo_amd import _native
    from mambo_amd.utils.iq3_s_weight import prepare_iq3_s_fields
    raw = make_synthetic_iq3_s(n, blocks * 256, seed=3 * n + blocks)
    f = prepare_iq3_s_fields(torch.from_numpy(raw).to(gpu))
    bits = torch.full((n * blocks * 256 + 64,), 0x5A, dtype=torch.uint8, device=gpu)
    scales = torch.full((n * blocks * 8 + 2,), 12345.0, device=gpu)
    step(f"dequant, scales off alignment [{n},{blocks},110]")
    _native.check(_native.lib().mambo_iq3s_dequant(
        f.d.data_ptr(), f.qs.data_ptr(), f.qh.data_ptr(), f.signs.data_ptr(), f.scales.data_ptr(), n, blocks,
        bits[32:].data_ptr(), scales[1:].data_ptr(), _native.stream_handle(None)))
    torch.cuda.synchronize()
    want_bits, want_scales = oracle.dequant_iq3s_fp8(raw)
    np.testing.assert_array_equal(bits[32:-32].cpu().numpy(), want_bits.ravel())
    np.testing.assert_array_equal(scales[1:-1].cpu().numpy(), want_scales.ravel())
    assert bool((bits[:32] == 0x5A).all()) and bool((bits[-32:] == 0x5A).all())
    assert float(scales[0]) == 12345.0 and float(scales[-1]) == 12345.0
