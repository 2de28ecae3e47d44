"""Performance cases of the framework: the work its users have it do, through its public
entry points, with the inputs made from a seed and a plain 64-bit statement of the results.

Kinds of case:

  step      the projections of whole decoder layers of the two models whose shapes the
            framework's sweep names (q/k/v and gate/up in one grouped call, o and down alone),
            optionally one GPU's tensor-parallel shard of them, for ``m`` tokens: bf16 rows
            are quantized and multiplied. A serving program captures such a step once in a
            HIP graph and replays it; so does this case.
  call      one eager call: a projection (or two that share their rows, ``n2`` > 0) of ``m``
            rows of any size, on rows quantized before ("pre"), in a call of their own
            ("separate") or by the projection call itself ("fused").
  quantize  the MXFP8 activation quantizer alone.
  load      a weight brought from its GGUF blocks to everything a launch or the decoder
            needs (the fields and the tile layout).
  dequant   the standalone decoder over a prepared weight.
"""

from __future__ import annotations

import math

import torch

from mambo_amd.kernels.iq3_s_fp8 import (launch_dequant_iq3_s, launch_iq3_s_fp8_matmul,
                                         launch_iq3_s_fp8_matmul_grouped, launch_iq3_s_matmul_quantize)
from mambo_amd.kernels.quantize_fp8 import launch_quantize_fp8
from mambo_amd.utils.iq3_s_weight import prepare_iq3_s_fields
from mambo_amd.utils.sweep import capture, layer_shapes

DTYPES = {"bf16": torch.bfloat16, "f32": torch.float32}

# The 512 four-weight codes of the IQ3_S codebook, three hex digits each: level l of weight j
# in bits 3j..3j+2, magnitude 2l + 1.
GRID = (
    "00000100200500700800900a00c00e01001101501b02002202502702902b03003203903c03f04004104204404804904d"
    "05005305705905d06407107507a08008108508708808b08e09109509809c0a20a50a70a90ab0b80bb0c30c90cd0d00d2"
    "0d90db0de0e40e80ea0f70f90fd10010b10f11111411a12012312913814214415015215615b16116516717617b186189"
    "18b1991aa1b91c01c21c41d01d21d61db1e81ec20020120220420820920b20d20f21021221921c21e22c22e23123a240"
    "24124324624824c25125825b26126826a27827e28028a28d28f29029429a2a02a32ad2b02ba2c12c42c72c82cb2d12d7"
    "2d82dc2e12f22f830330530a30c31931b32232632832c34134834b35135835a3693903943973a43a63c13c33c83ca3d1"
    "3dd3e13f23f840040140340540740840a40c40e41141341741841a42142342542842a43743843b43d44044244844b44f"
    "45245545945c46246948148448749149349849f4a14ab4af4b94bc4c04c24c54c94d24d44d94db4e24e84f6501507510"
    "51351a51d52153a53d54454955255f56056b5785805825875915ad5b15c55c95d65d85e35e860260960b60d60f612619"
    "61b61d62262462762963363964164364564c65165366067067a67e68068a69069a69c6a86c16c86cc6d16d36d76d86e1"
    "6e36e76ed6fb70370970e71271972a73073474174874a75575a76476e77b78e7a17c17c37d07d27dd80080480a810814"
    "81781a82182883884284784984b85285885d86386986d88188388888d89189b8a08af8b28b88c48c98cb8d08d28d98dd"
    "90090291491f92093994594795197298b99c9b09c89cd9d89e39e9a02a08a0ca12a20a24a27a2aa36a3ca41a43a45a4a"
    "a51a5aa7aa80a89a93a98a9eaabac2ac7ac8ad7ae4ae9af5afbb01b04b10b1ab26b4ab56b69b6bba2bc2bc4bd2c09c0b"
    "c0dc19c1bc30c40c50c57c74c8ac9cca2cadcb2cb8cc0ccccd1ce0d15d23d32d40d43d5cd70d85da0dc9dcbe00e04e07"
    "e10e12e1ee20e2ce32e42e49e54e63e65e81e84e88e8ee91e98ea9ec2edaeddeebf01f05f0bf10f28f52f62f82f99fc0"
)


def listed() -> list[dict]:
    return [
        # one token through the smallest projection a layer has (k or v of the 8B model), called
        # the way the reference's caller does: launch latency and host time
        {"name": "call_kv_m1", "kind": "call", "m": 1, "n": 1024, "n2": 0, "k": 4096, "mode": "pre", "dtype": "bf16"},
        # single-stream decoding, both models: weight bandwidth and launches
        {"name": "decode_8b_m1", "kind": "step", "model": "llama8b", "tp": 1, "layers": 4, "m": 1, "mode": "fused"},
        {"name": "decode_70b_m1", "kind": "step", "model": "llama70b", "tp": 1, "layers": 1, "m": 1, "mode": "separate"},
        # batched decoding: a few users, a server's running batch, a large one
        {"name": "batch_70b_m16", "kind": "step", "model": "llama70b", "tp": 1, "layers": 1, "m": 16, "mode": "separate"},
        {"name": "batch_8b_m48", "kind": "step", "model": "llama8b", "tp": 1, "layers": 2, "m": 48, "mode": "separate"},
        {"name": "batch_70b_m128", "kind": "step", "model": "llama70b", "tp": 1, "layers": 1, "m": 128, "mode": "separate"},
        # a prompt chunk of a size that divides nothing, rows that the caller holds in f32
        {"name": "call_ragged", "kind": "call", "m": 203, "n": 5003, "n2": 1201, "k": 2816, "mode": "fused", "dtype": "f32"},
        # prefill: a prompt chunk of the large model, a long prompt of the small one
        {"name": "prefill_70b_m512", "kind": "step", "model": "llama70b", "tp": 1, "layers": 1, "m": 512, "mode": "separate"},
        {"name": "prefill_8b_m8192", "kind": "step", "model": "llama8b", "tp": 1, "layers": 1, "m": 8192, "mode": "separate"},
        # the quantizer's own configuration, 4096 rows of 4096
        {"name": "quantize_4096", "kind": "quantize", "m": 4096, "k": 4096, "dtype": "bf16"},
        # loading a model: the 8B gate and up projections as one weight
        {"name": "load_28672x4096", "kind": "load", "n": 28672, "k": 4096},
        # decoding a weight outside a projection, as a check of a loaded file does
        {"name": "dequant_4096x14336", "kind": "dequant", "n": 4096, "k": 14336},
    ]


# The largest listed case's multiply-adds, which no drawn case exceeds.
MOST_MNK = 8192 * sum(n * k for _, n, k, _ in layer_shapes("llama8b"))
MOST_WEIGHTS = sum(n * k for _, n, k, _ in layer_shapes("llama70b"))


def _log_int(rng, lo: int, hi: int) -> int:
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng) -> dict:
    kind = rng.choice(["step", "step", "step", "step", "call", "call", "call", "quantize", "load", "dequant"])
    while True:
        if kind == "step":
            case = {"kind": kind, "model": rng.choice(["llama8b", "llama70b"]), "tp": rng.choice([1, 1, 2, 4, 8]),
                    "layers": rng.choice([1, 2, 3, 4]), "m": _log_int(rng, 1, 8192),
                    "mode": rng.choice(["separate", "fused"])}
            weights = case["layers"] * sum(n * k for _, n, k, _ in layer_shapes(case["model"], case["tp"]))
        elif kind == "call":
            case = {"kind": kind, "m": _log_int(rng, 1, 8192), "n": _log_int(rng, 128, 57344),
                    "n2": rng.choice([0, 0, _log_int(rng, 128, 28672)]), "k": 256 * _log_int(rng, 2, 112),
                    "mode": rng.choice(["pre", "separate", "fused"]), "dtype": rng.choice(["bf16", "bf16", "f32"])}
            weights = (case["n"] + case["n2"]) * case["k"]
        elif kind == "quantize":
            case = {"kind": kind, "m": _log_int(rng, 1, 8192), "k": 32 * _log_int(rng, 8, 896),
                    "dtype": rng.choice(["bf16", "bf16", "f32"])}
            weights = 0
        else:
            case = {"kind": kind, "n": _log_int(rng, 128, 57344), "k": 256 * _log_int(rng, 2, 112)}
            weights = case["n"] * case["k"]
        if weights * case.get("m", 1) <= MOST_MNK and weights <= (MOST_WEIGHTS if "m" in case else 1 << 28):
            return case


# ------------------------------------------------------------------------------ inputs
def _generator(seed: int) -> torch.Generator:
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed))
    return gen


def _rows(m: int, k: int, dtype: torch.dtype, gen: torch.Generator) -> torch.Tensor:
    """Activations as a transformer has them: N(0, 1) with one value in a thousand 20 times
    as large."""
    x = torch.randn((m, k), generator=gen, device="cuda")
    big = torch.rand((m, k), generator=gen, device="cuda") < 1e-3
    return torch.where(big, 20.0 * x, x).to(dtype)


def _raw(n: int, k: int, gen: torch.Generator) -> torch.Tensor:
    """GGUF blocks uint8 [N, K/256, 110]: uniform codes, signs and scale nibbles, block
    scales in [0.002, 0.04]."""
    raw = torch.randint(0, 256, (n, k // 256, 110), dtype=torch.uint8, generator=gen, device="cuda")
    d = 0.002 + 0.038 * torch.rand((n, k // 256, 1), generator=gen, device="cuda")
    raw[..., :2] = d.to(torch.float16).view(torch.uint8)
    return raw


def _launches(case: dict) -> list[tuple[int, list[int]]]:
    """(K, [N, ...]) of each projection launch of a case, in order."""
    if case["kind"] == "call":
        return [(case["k"], [case["n"]] + ([case["n2"]] if case["n2"] else []))]
    out, slots = [], []
    for layer in range(case["layers"]):
        for _, n, k, slot in layer_shapes(case["model"], case["tp"]):
            if slots and slots[-1] == (layer, slot):
                out[-1][1].append(n)
            else:
                slots.append((layer, slot))
                out.append((k, [n]))
    return out


def _inputs(case: dict, seed: int):
    """Rows and raw weights of each launch, one launch at a time."""
    gen = _generator(seed)
    dtype = DTYPES[case.get("dtype", "bf16")]
    for k, ns in _launches(case):
        yield k, ns, _rows(case["m"], k, dtype, gen), [_raw(n, k, gen) for n in ns]


def _project(launch: dict) -> list[torch.Tensor]:
    weights, outs = launch["weights"], launch["outs"]
    if launch["mode"] == "fused":
        return launch_iq3_s_matmul_quantize(launch["rows"], weights, outs=outs)
    if launch["mode"] == "separate":
        values, scales = launch_quantize_fp8(launch["rows"], out=launch["mx"])
    else:
        values, scales = launch["mx"]
    if len(weights) == 1:
        return [launch_iq3_s_fp8_matmul(values, scales, weights[0], out=None if outs is None else outs[0])]
    return launch_iq3_s_fp8_matmul_grouped(values, scales, weights, outs=outs)


def prepare(case: dict, seed: int) -> dict:
    kind = case["kind"]
    if kind == "quantize":
        return {"kind": kind, "rows": _rows(case["m"], case["k"], DTYPES[case["dtype"]], _generator(seed))}
    if kind == "load":
        return {"kind": kind, "raw": _raw(case["n"], case["k"], _generator(seed))}
    if kind == "dequant":
        return {"kind": kind, "weight": prepare_iq3_s_fields(_raw(case["n"], case["k"], _generator(seed)))}
    launches = []
    for k, ns, rows, raws in _inputs(case, seed):
        launch = {"mode": case["mode"], "rows": rows, "mx": None, "outs": None,
                  "weights": [prepare_iq3_s_fields(raw, fields=False) for raw in raws]}
        if case["mode"] == "pre":
            launch["mx"] = launch_quantize_fp8(rows)
        if kind == "step":  # a captured step keeps its buffers
            if case["mode"] == "separate":
                launch["mx"] = (torch.empty((case["m"], k), dtype=torch.uint8, device="cuda"),
                                torch.empty((case["m"], k // 32), dtype=torch.uint8, device="cuda"))
            launch["outs"] = [torch.empty((case["m"], n), dtype=torch.float32, device="cuda") for n in ns]
        launches.append(launch)
    state = {"kind": kind, "launches": launches}
    if kind == "step":
        def step():
            for launch in launches:
                _project(launch)

        step()
        torch.cuda.synchronize()
        state["graph"] = capture(step)
    return state


def run(state: dict):
    kind = state["kind"]
    if kind == "step":
        state["graph"].replay()
        return [launch["outs"] for launch in state["launches"]]
    if kind == "call":
        return _project(state["launches"][0])
    if kind == "quantize":
        return launch_quantize_fp8(state["rows"])
    if kind == "load":
        w = prepare_iq3_s_fields(state["raw"], pack=True)
        # the tile layout is private to the framework; the fields are not
        return [w.d, w.qs.view(torch.int32), w.qh.view(torch.int16), w.signs, w.scales.view(torch.int32)]
    return launch_dequant_iq3_s(state["weight"])


# ------------------------------------------------------------------- what a pass has to do
def work(case: dict) -> dict:
    kind = case["kind"]
    size = DTYPES[case.get("dtype", "bf16")].itemsize
    if kind == "quantize":
        return {"bytes": case["m"] * case["k"] * (size + 33 / 32), "flops": 0}
    if kind in ("load", "dequant"):
        weights = case["n"] * case["k"]
        if kind == "load":  # blocks in, fields and tiles out
            return {"bytes": 3 * weights * 110 / 256, "flops": 0}
        return {"bytes": weights * (110 / 256 + 1 + 4 / 32), "flops": 0}
    if case["mode"] == "pre":
        size = 33 / 32
    total = {"bytes": 0.0, "flops": 0.0}
    for k, ns in _launches(case):
        total["bytes"] += case["m"] * k * size + sum(n * k * 110 / 256 + 4 * case["m"] * n for n in ns)
        total["flops"] += 2.0 * case["m"] * sum(ns) * k
    return total


def tolerance(case: dict):
    if case["kind"] in ("quantize", "load", "dequant"):
        return "exact"
    # f32 accumulation of products of 8-bit floats: against float64 the stream path is
    # 0.5e-5 to 2.5e-5 off and the MFMA paths 2.3e-5 to 2.6e-5 (measured over the listed and
    # some drawn cases), and two orders of the sums differ by as much
    return {"rel": 1e-4, "max": 1e-3}


# ------------------------------------------------------------- the same in plain 64 bits
def _quantized(x: torch.Tensor) -> torch.Tensor:
    """Rows after MXFP8 quantization, as float64: per 32 values the exponent
    ceil(log2(amax / 448)), E4M3 codes rounded to nearest even."""
    m, k = x.shape
    g = x.double().view(m, k // 32, 32)
    mant, exp = torch.frexp(g.abs().amax(-1, keepdim=True))  # amax = mant * 2^exp, mant in [0.5, 1)
    e = torch.where(mant <= 0.875, exp - 9, exp - 8)
    e = torch.where(mant == 0, torch.zeros_like(e), e).clamp(min=-127)
    scale = torch.exp2(e.double())
    codes = (g / scale).float().to(torch.float8_e4m3fn)
    return (codes.double() * scale).view(m, k)


def _levels() -> torch.Tensor:
    codes = torch.tensor([int("".join(GRID)[i:i + 3], 16) for i in range(0, 1536, 3)], device="cuda")
    return 2.0 * ((codes[:, None] >> torch.tensor([0, 3, 6, 9], device="cuda")) & 7).double() + 1.0


def _scales(raw: torch.Tensor) -> torch.Tensor:
    """Group scales d * (1 + 2 * nibble), float64 [N, K/32]."""
    n = raw.shape[0]
    d = raw[..., :2].contiguous().view(torch.float16).double()
    nib = torch.stack((raw[..., 106:110] & 15, raw[..., 106:110] >> 4), -1).view(n, -1, 8)
    return (d * (1 + 2 * nib.double())).view(n, -1)


def _decoded(raw: torch.Tensor) -> torch.Tensor:
    """The weight's values, float64 [N, K]."""
    n, blocks, _ = raw.shape
    bits = torch.arange(8, device="cuda")
    qh = (raw[..., 66:74, None] >> bits) & 1
    idx = raw[..., 2:66].long() + 256 * qh.reshape(n, blocks, 64).long()
    sign = 1.0 - 2.0 * ((raw[..., 74:106, None] >> bits) & 1).reshape(n, blocks * 256).double()
    w = _levels()[idx].reshape(n, blocks * 256) * sign
    return (w.view(n, -1, 32) * _scales(raw)[..., None]).view(n, -1)


def exact(case: dict, seed: int):
    kind = case["kind"]
    if kind == "dequant":
        return [None, _scales(_raw(case["n"], case["k"], _generator(seed)))]
    if kind in ("quantize", "load"):  # bytes, no computed numbers
        return None
    outs = []
    for _, _, rows, raws in _inputs(case, seed):
        x = _quantized(rows)
        per = []
        for raw in raws:  # 4096 weight rows at a time
            per.append(torch.cat([x @ _decoded(part).t().contiguous() for part in raw.split(4096)], 1))
        outs.append(per)
    return outs if kind == "step" else outs[0]
