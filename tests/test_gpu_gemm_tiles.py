"""Every tile of the weight-streaming GEMM and the four-wave GEMM in one launch,
by the sizes that the library routes there (h3q_scaled_mm_plan, checked before
each call, so that a change of the rules cannot empty the coverage), in each form
they take: both layouts, int8 and e4m3, per-row and per-tensor scales, bias,
binary16 output, the adapter and strided output rows.

int8 against the exact product through the oracle's epilogue bit for bit, on every
output; e4m3 against the instruction model and the adapter against binary64, to
the bounds of test_gpu_gemm and test_gpu_gemm_stream, on rows at both ends and
around every seam of 16 to 256 rows."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from _util import bits16, gemm_plan
from test_gpu_gemm import _assert_fp8_close
from test_gpu_gemm_split import _codes, _exact
from test_gpu_gemm_stream import _operands

pytestmark = pytest.mark.gpu

# A tile each; one row or column block past a whole number of them.
_TILES = {(64, 64): (161, 1032), (64, 128): (129, 5496), (80, 128): (194, 8240), (80, 256): (389, 8240),
          (96, 128): (244, 8240), (96, 256): (644, 7176), (112, 128): (289, 8240), (112, 256): (769, 7176),
          (128, 128): (339, 8240), (128, 256): (899, 7176)}
# More tiles than workgroups with a last round of halves, tall, wide, and the least K.
_FOUR_WAVES = [(5130, 4104, 1024), (8000, 1032, 512), (2056, 5128, 640), (2600, 3336, 256)]

# form: (format, tiled activations, tiled weights, per-tensor scales, binary16, adapter rank)
_FORMS = {"int8": ("int8", True, True, False, False, 0),
          "int8 rows": ("int8", False, False, False, False, 0),
          "e4m3": ("e4m3", True, True, False, False, 0),
          "e4m3 rows per tensor": ("e4m3", False, False, True, False, 0),
          "int8 per tensor": ("int8", False, True, True, False, 0),
          "f16": ("int8", False, False, False, True, 0),
          "int8 adapter": ("int8", True, True, False, False, 72),
          "e4m3 rows adapter": ("e4m3", False, False, False, False, 128)}


def _rows(m: int) -> np.ndarray:
    near = np.arange(0, m, 256)[:, None] + np.array([-1, 0, 1])[None, :]
    seams = np.array([h * i + d for h in (64, 80, 96, 112, 128) for i in range(1, 4) for d in (-1, 0)])
    return np.unique(np.clip(np.concatenate([near.ravel(), seams, [15, 16, m - 17, m - 16, m - 1]]), 0, m - 1))


def _check(ops, oracle, device, m, n, k, form, expect):
    fmt, a_tiled, b_tiled, per_tensor, f16, rank = _FORMS[form]
    ldo = n + 8 if form == "int8 rows" else n
    plan = gemm_plan(m, n, k, a_tiled=a_tiled, b_tiled=b_tiled, rank=rank, f16=f16, ldo=ldo)
    assert plan[:2] == expect, plan
    print(f"{expect} {form} {m}x{n}x{k}", flush=True)
    _, _, qa, sa, qw, sw = _operands(ops, device, m, n, k, fmt, a_tiled, b_tiled)
    if per_tensor:
        sa, sw = sa[:1].clone(), sw[:1].clone()
    gen = torch.Generator().manual_seed(n + rank)
    bias = (torch.randn(n, generator=gen) * 0.01).to(torch.float16 if f16 else torch.bfloat16)
    kw = {}
    if rank:
        t = torch.randn(m, rank, generator=gen).to(torch.bfloat16)
        lb = (torch.randn(n, rank, generator=gen) * 0.05).to(torch.bfloat16)
        kw = dict(lora_t=t.to(device), lora_b=lb.to(device), lora_scale=0.75)
    big = torch.full((m, ldo), float("nan"), device=device, dtype=bias.dtype)
    out = ops.scaled_mm(qa, qw, sa, sw, bias=bias.to(device), out=big[:, :n], out_dtype=bias.dtype, a_tiled=a_tiled,
                        b_tiled=b_tiled, m=m, n=n, **kw)
    torch.cuda.synchronize()
    assert torch.isnan(big[:, n:].float()).all()
    rows = _rows(m) if fmt == "e4m3" or rank else np.arange(m)
    codes_a = _codes(qa, m, k, a_tiled)[torch.from_numpy(rows).to(device)]
    codes_w = _codes(qw, n, k, b_tiled)
    got = out[torch.from_numpy(rows).to(device)].contiguous()
    rsa = sa.cpu().numpy()[:1 if per_tensor else m]
    rsa = rsa if per_tensor else rsa[rows]
    rsw = sw.cpu().numpy()[:1 if per_tensor else n]
    if not rank:
        if fmt == "int8":
            bias_bits = bias.view(torch.int16).numpy().view(np.uint16)
            ref = oracle.epilogue(_exact(codes_a, codes_w), rsa, rsw, bias_bits, out_f16=f16)
            np.testing.assert_array_equal(got.view(torch.int16).cpu().numpy().view(np.uint16), ref)
        else:
            _assert_fp8_close(oracle, bits16(got), codes_a.cpu().numpy(), rsa, codes_w.cpu().numpy(), rsw, bits16(bias))
        return
    scale = rsa.astype(np.float64).reshape(-1, 1) * rsw.astype(np.float64).reshape(1, -1)
    if fmt == "int8":
        y, slack = _exact(codes_a, codes_w).astype(np.float64) * scale, 0.0
    else:
        model, rbound = oracle.gemm_e4m3_mfma(codes_a.cpu().numpy(), codes_w.cpu().numpy())
        y, slack = model * scale, rbound * scale
    t64, b64, bias64 = t.double().numpy()[rows], lb.double().numpy(), bias.double().numpy()
    ref = y + bias64 + 0.75 * (t64 @ b64.T)
    mag = np.abs(y) + np.abs(bias64) + 0.75 * (np.abs(t64) @ np.abs(b64).T)
    got = oracle.bf16_to_f32(bits16(got)).astype(np.float64)
    ulp = 2.0 ** (np.floor(np.log2(np.maximum(np.maximum(np.abs(ref), np.abs(got)), 2.0 ** -126))) - 7)
    # one bf16 rounding; rank + 5 binary32 roundings of terms up to mag
    assert np.all(np.abs(got - ref) <= 0.51 * ulp + slack + (rank + 5) * 2.0 ** -24 * mag)


@pytest.mark.parametrize("form", _FORMS)
@pytest.mark.parametrize("tile", _TILES)
def test_stream_tiles(ops, oracle, device, tile, form):
    """11 k-tiles (12 with a tail where no operand is tiled): more than a ring
    holds, not a multiple of two or four K groups."""
    m, n = _TILES[tile]
    fmt, a_tiled, b_tiled, _, _, _ = _FORMS[form]
    _check(ops, oracle, device, m, n, 1408 if a_tiled or b_tiled else 1424, form, ("stream", tile))


@pytest.mark.parametrize("form", _FORMS)
@pytest.mark.parametrize("m,n,k", _FOUR_WAVES)
def test_four_waves(ops, oracle, device, m, n, k, form):
    """One launch of 256 x 256 tiles, ragged in both directions; 357 of them on 256
    workgroups, and fewer tiles than workgroups."""
    _check(ops, oracle, device, m, n, k, form, ("four waves", (0, 0)))


@pytest.mark.parametrize("form", ["int8 rows", "e4m3 rows per tensor", "f16", "e4m3 rows adapter"])
@pytest.mark.parametrize("m,n,k", [(3500, 4104, 656), (6200, 2056, 1040)])
def test_k_tail_per_tile(ops, oracle, device, m, n, k, form):
    """A K tail at sizes that fill the chip with 256 x 256 tiles: the sixteen-wave kernels."""
    _check(ops, oracle, device, m, n, k, form, ("per tile", (0, 0)))
