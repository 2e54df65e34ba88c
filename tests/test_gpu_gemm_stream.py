"""The weight-streaming GEMM over chip-filling tiles (gemm_stream.hpp; some calls of
up to 128 rows take the few-rows kernels instead), at the sizes where a ring or a
reduction can go wrong: one row past 64, 80, 96, 112 and 128, ragged column counts,
fewer k-tiles than the rings hold, k-tiles that do not divide among the K groups, a K
tail (row-major only), both layouts of both operands, binary16 output and the LoRA
epilogue.  These sizes take the smaller tiles; test_gpu_gemm_tiles runs every tile.
int8 against the oracle bit for bit, e4m3 against the instruction model to the
bound of test_gpu_gemm."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from _util import activations, bits16, weights

pytestmark = pytest.mark.gpu


def _operands(ops, device, m, n, k, fmt, a_tiled, b_tiled):
    f, ar = (ops.FMT_E4M3FN, ops.ROUND_DIV) if fmt == "e4m3" else (ops.FMT_INT8, ops.ROUND_RCP_MUL)
    x = activations(m, k, seed=m + k, outlier_channels=max(1, k // 100), outlier_scale=15.0)
    w = weights(n, k, seed=n + k)
    qw, sw = (ops.quant_rows_tiled if b_tiled else ops.quant_rows)(w.to(device), f, ops.ROUND_DIV)
    qa, sa = (ops.quant_rows_tiled if a_tiled else ops.quant_rows)(x.to(device), f, ar)
    return x, w, qa, sa.reshape(-1), qw, sw.reshape(-1)


# (m, n, k): one row past 64, 80, 96, 112 and 128 rows and exact ones; K of 1, 2, 3, 5
# and 9 k-tiles; n = 8 alone and past a tile.
_CASES = [(33, 8200, 256, True, True), (65, 264, 128, True, True), (128, 520, 384, False, True),
          (129, 264, 256, True, True), (161, 1032, 640, True, True), (300, 8, 1152, False, True),
          (337, 2056, 256, True, True), (449, 4104, 384, False, True), (700, 3592, 640, True, True),
          (897, 5128, 512, True, True), (1025, 5120, 256, False, True),
          (17, 40, 3088, False, False), (66, 264, 2064, False, False), (130, 136, 1040, False, False),
          (259, 1000, 528, False, False), (600, 3080, 144, False, False), (1030, 5128, 272, False, False)]


@pytest.mark.parametrize("m,n,k,a_tiled,b_tiled", _CASES)
@pytest.mark.parametrize("fmt", ["int8", "e4m3"])
def test_stream_gemm(ops, oracle, device, m, n, k, a_tiled, b_tiled, fmt):
    from test_gpu_gemm import _assert_fp8_close

    if a_tiled and m > 128 and k < 256:
        pytest.skip("tiled activations above 128 rows need K >= 256")
    print(f"stream gemm {fmt} {m}x{n}x{k} a_tiled={a_tiled} b_tiled={b_tiled}", flush=True)
    x, w, qa, sa, qw, sw = _operands(ops, device, m, n, k, fmt, a_tiled, b_tiled)
    bvec = (torch.randn(n, generator=torch.Generator().manual_seed(n)) * 0.01).to(torch.bfloat16)
    bias = bvec if m % 2 else None
    big = torch.full((m, n + 8), float("nan"), device=device, dtype=torch.bfloat16)
    out = ops.scaled_mm(qa, qw, sa, sw, bias=None if bias is None else bias.to(device), out=big[:, :n],
                        a_tiled=a_tiled, b_tiled=b_tiled, m=m, n=n)
    torch.cuda.synchronize()
    assert torch.isnan(big[:, n:].float()).all()  # the columns past n are never written
    bb = None if bias is None else bits16(bias)
    rqa, rsa = oracle.quant_rows(bits16(x), fmt, "div" if fmt == "e4m3" else "rcp")
    rqw, rsw = oracle.quant_rows(bits16(w), fmt, "div")
    if fmt == "int8":
        ref = oracle.epilogue(oracle.gemm_i8_i32_fast(rqa, rqw), rsa, rsw, bb)
        np.testing.assert_array_equal(bits16(out.contiguous()), ref)
    else:
        rows = np.unique(np.concatenate([np.arange(0, min(m, 130)), np.arange(max(0, m - 130), m)]))
        _assert_fp8_close(oracle, bits16(out.contiguous()), rqa, rsa, rqw, rsw, bb, rows=rows)


@pytest.mark.parametrize("m,n,k,rank", [(5, 520, 256, 8), (40, 1032, 640, 128), (129, 264, 384, 72),
                                        (500, 3592, 1152, 128), (1040, 5128, 256, 24)])
@pytest.mark.parametrize("fmt", ["int8", "e4m3"])
def test_stream_lora(ops, oracle, device, m, n, k, rank, fmt):
    """The adapter is added before the one rounding: within one bf16 ulp of
    the binary64 sum y + scale * (t . lora_b) of the oracle's y (binary32,
    before its rounding; here reconstructed from the exact accumulators for
    int8) plus the binary32 error of the terms, and the same bits from both
    weight layouts."""
    print(f"stream lora {fmt} {m}x{n}x{k} rank={rank}", flush=True)
    x, w, qa, sa, qw, sw = _operands(ops, device, m, n, k, fmt, False, True)
    gen = torch.Generator().manual_seed(rank)
    t = torch.randn(m, rank, generator=gen).to(torch.bfloat16)
    lb = (torch.randn(n, rank, generator=gen) * 0.05).to(torch.bfloat16)
    kw = dict(lora_t=t.to(device), lora_b=lb.to(device), lora_scale=0.75, m=m, n=n)
    out = ops.scaled_mm(qa, qw, sa, sw, b_tiled=True, **kw)
    _, _, qa2, sa2, qw2, sw2 = _operands(ops, device, m, n, k, fmt, False, False)
    rows = ops.scaled_mm(qa2, qw2, sa2, sw2, **kw)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(bits16(out), bits16(rows))
    rqa, rsa = oracle.quant_rows(bits16(x), fmt, "div" if fmt == "e4m3" else "rcp")
    rqw, rsw = oracle.quant_rows(bits16(w), fmt, "div")
    scale = rsa.astype(np.float64).reshape(-1, 1) * rsw.astype(np.float64).reshape(1, -1)
    if fmt == "int8":
        y, slack = oracle.gemm_i8_i32_fast(rqa, rqw).astype(np.float64) * scale, 0.0
    else:
        model, rbound = oracle.gemm_e4m3_mfma(rqa, rqw)
        y, slack = model.astype(np.float64) * scale, rbound * scale
    t64, b64 = t.double().numpy(), lb.double().numpy()
    ref = y + 0.75 * (t64 @ b64.T)
    mag = np.abs(y) + 0.75 * (np.abs(t64) @ np.abs(b64).T)
    got = oracle.bf16_to_f32(bits16(out)).astype(np.float64)
    ulp = 2.0 ** (np.floor(np.log2(np.maximum(np.maximum(np.abs(ref), np.abs(got)), 2.0 ** -126))) - 7)
    # one bf16 rounding; rank + 4 binary32 roundings of terms up to mag
    assert np.all(np.abs(got - ref) <= 0.51 * ulp + slack + (rank + 4) * 2.0 ** -24 * mag)


@pytest.mark.parametrize("m,n,k", [(70, 264, 2064), (300, 520, 1040), (1100, 2056, 272)])
def test_stream_f16_output(ops, oracle, device, m, n, k):
    print(f"stream f16 {m}x{n}x{k}", flush=True)
    x, w, qa, sa, qw, sw = _operands(ops, device, m, n, k, "int8", False, False)
    bias = (torch.randn(n, generator=torch.Generator().manual_seed(3)) * 0.1).to(torch.float16)
    out = ops.scaled_mm(qa, qw, sa, sw, bias=bias.to(device), out_dtype=torch.float16)
    torch.cuda.synchronize()
    rqa, rsa = oracle.quant_rows(bits16(x), "int8", "rcp")
    rqw, rsw = oracle.quant_rows(bits16(w), "int8", "div")
    acc = oracle.gemm_i8_i32_fast(rqa, rqw).astype(np.float64)
    v = (rsw.astype(np.float64).reshape(1, -1) * acc).astype(np.float32).astype(np.float64)
    exact = rsa.astype(np.float64).reshape(-1, 1) * v + bias.double().numpy()  # one rounding each: s_w * acc, the fma
    ref = exact.astype(np.float32).astype(np.float16)
    np.testing.assert_array_equal(out.cpu().numpy().view(np.uint16), ref.view(np.uint16))


@pytest.mark.parametrize("m,n,k", [(129, 8, 144), (2600, 1040, 272), (4400, 2056, 656), (130, 4104, 4080)])
def test_stream_k_tail_at_any_size(ops, oracle, device, m, n, k):
    """K that is not a multiple of 128 above 128 rows, at sizes on both sides of the
    line to the sixteen-wave kernels."""
    print(f"stream K tail {m}x{n}x{k}", flush=True)
    x, w, qa, sa, qw, sw = _operands(ops, device, m, n, k, "int8", False, False)
    out = ops.scaled_mm(qa, qw, sa, sw)
    torch.cuda.synchronize()
    rqa, rsa = oracle.quant_rows(bits16(x), "int8", "rcp")
    rqw, rsw = oracle.quant_rows(bits16(w), "int8", "div")
    ref = oracle.epilogue(oracle.gemm_i8_i32_fast(rqa, rqw), rsa, rsw, None)
    np.testing.assert_array_equal(bits16(out), ref)


@pytest.mark.parametrize("m,n,k", [(200, 264, 272), (300, 520, 1040)])
def test_bias_at_an_odd_element(ops, oracle, device, m, n, k):
    """A bias that starts at an odd 2-byte element takes the kernel that reads it element by element."""
    print(f"odd bias {m}x{n}x{k}", flush=True)
    x, w, qa, sa, qw, sw = _operands(ops, device, m, n, k, "int8", False, False)
    packed = (torch.randn(n + 1, generator=torch.Generator().manual_seed(5)) * 0.1).to(torch.float16)
    bias = packed.to(device)[1:]
    assert bias.data_ptr() % 4 == 2
    out = ops.scaled_mm(qa, qw, sa, sw, bias=bias, out_dtype=torch.float16)
    torch.cuda.synchronize()
    acc = oracle.gemm_i8_i32_fast(*(oracle.quant_rows(bits16(t), "int8", r)[0] for t, r in ((x, "rcp"), (w, "div"))))
    v = (sw.cpu().numpy().astype(np.float64) * acc.astype(np.float64)).astype(np.float32).astype(np.float64)
    exact = sa.cpu().numpy().astype(np.float64)[:, None] * v + packed[1:].double().numpy()
    ref = exact.astype(np.float32).astype(np.float16)  # one rounding each: s_w * acc, the fma
    np.testing.assert_array_equal(out.cpu().numpy().view(np.uint16), ref.view(np.uint16))


@pytest.mark.parametrize("m,n,k", [(5, 520, 256), (16, 264, 3072), (33, 1032, 640), (128, 264, 2048)])
@pytest.mark.parametrize("fmt", ["int8", "e4m3"])
def test_few_tiled_rows_on_row_major_weights(ops, oracle, device, m, n, k, fmt):
    """Tiled activations beside row-major weights up to 128 rows; refused where no kernel reads them so."""
    test_stream_gemm(ops, oracle, device, m, n, k, True, False, fmt)
    _, _, qa, sa, qw, sw = _operands(ops, device, m, n, k, fmt, True, False)
    with pytest.raises(RuntimeError, match="row-major weights"):
        ops.scaled_mm(qa, qw[:n - 4], sa, sw[:n - 4], a_tiled=True, m=m, n=n - 4)
