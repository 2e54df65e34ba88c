"""A GEMM whose last round of 256 x 256 tiles is mostly empty runs in two
launches, full rounds and the rest over smaller tiles: calls split by columns
and by rows, ragged in both, for each layout, bias, per-tensor and per-row
scales, both output types and the adapter.  int8 against the exact product
(binary64 on the device: below 2^53) through the oracle's epilogue bit for bit,
e4m3 against the instruction model to the bound of test_gpu_gemm on the rows
around the seams."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from _util import bits16
from test_gpu_gemm_stream import _operands

pytestmark = pytest.mark.gpu

# (m, n, k): columns from 3072 and 13056 on, rows from 3840 and 1792 on.
_SPLIT = [(5130, 3336, 1536), (1030, 16904, 2048), (4362, 4104, 1536), (2049, 8712, 1536)]


def _codes(q: torch.Tensor, rows: int, k: int, tiled: bool) -> torch.Tensor:
    """Row-major codes of an operand; tiled: 16-row x 128-byte blocks in fragment order."""
    q = q.view(torch.uint8)
    if not tiled:
        return q[:rows]
    v = q.reshape(-1, k // 128, 2, 4, 16, 16)  # [block, step, half, group, row, byte]
    return v.permute(0, 4, 1, 3, 2, 5).reshape(-1, k)[:rows].contiguous()


def _exact(qa: torch.Tensor, qw: torch.Tensor) -> np.ndarray:
    acc = qa.view(torch.int8).double() @ qw.view(torch.int8).double().t().contiguous()
    return acc.to(torch.int32).cpu().numpy()


@pytest.mark.parametrize("a_tiled,b_tiled", [(True, True), (False, True), (False, False)])
@pytest.mark.parametrize("m,n,k", _SPLIT)
def test_split_int8(ops, oracle, device, m, n, k, a_tiled, b_tiled):
    print(f"split int8 {m}x{n}x{k} a_tiled={a_tiled} b_tiled={b_tiled}", flush=True)
    _, _, qa, sa, qw, sw = _operands(ops, device, m, n, k, "int8", a_tiled, b_tiled)
    bias = (torch.randn(n, generator=torch.Generator().manual_seed(n)) * 0.01).to(torch.bfloat16)
    big = torch.full((m, n + 8), float("nan"), device=device, dtype=torch.bfloat16)
    out = ops.scaled_mm(qa, qw, sa, sw, bias=bias.to(device), out=big[:, :n], a_tiled=a_tiled, b_tiled=b_tiled,
                        m=m, n=n)
    torch.cuda.synchronize()
    assert torch.isnan(big[:, n:].float()).all()
    acc = _exact(_codes(qa, m, k, a_tiled), _codes(qw, n, k, b_tiled))
    ref = oracle.epilogue(acc, sa.cpu().numpy()[:m], sw.cpu().numpy()[:n], bits16(bias))
    np.testing.assert_array_equal(bits16(out.contiguous()), ref)


@pytest.mark.parametrize("m,n,k", _SPLIT)
def test_split_e4m3(ops, oracle, device, m, n, k):
    from test_gpu_gemm import _assert_fp8_close

    print(f"split e4m3 {m}x{n}x{k}", flush=True)
    _, _, qa, sa, qw, sw = _operands(ops, device, m, n, k, "e4m3", True, True)
    out = ops.scaled_mm(qa, qw, sa, sw, a_tiled=True, b_tiled=True, m=m, n=n)
    torch.cuda.synchronize()
    rqa = _codes(qa, m, k, True).cpu().numpy()
    rqw = _codes(qw, n, k, True).cpu().numpy()
    rows = np.unique(np.clip(np.array([0, 1791, 1792, 3839, 3840, m - 1]), 0, m - 1))
    _assert_fp8_close(oracle, bits16(out), rqa, sa.cpu().numpy()[:m], rqw, sw.cpu().numpy()[:n], None, rows=rows)


@pytest.mark.parametrize("m,n,k", [_SPLIT[0], _SPLIT[2]])
def test_split_f16_per_tensor(ops, device, m, n, k):
    print(f"split f16 {m}x{n}x{k}", flush=True)
    _, _, qa, sa, qw, sw = _operands(ops, device, m, n, k, "int8", False, False)
    bias = (torch.randn(n, generator=torch.Generator().manual_seed(3)) * 0.1).to(torch.float16)
    out = ops.scaled_mm(qa, qw, sa[:1], sw[:1], bias=bias.to(device), out_dtype=torch.float16)
    torch.cuda.synchronize()
    v = (sw[0].item() * _exact(qa, qw).astype(np.float64)).astype(np.float32).astype(np.float64)
    exact = sa[0].item() * v + bias.double().numpy()  # one rounding each: s_w * acc, the fma
    ref = exact.astype(np.float32).astype(np.float16)
    np.testing.assert_array_equal(out.cpu().numpy().view(np.uint16), ref.view(np.uint16))


@pytest.mark.parametrize("m,n,k", [_SPLIT[0], _SPLIT[2]])
def test_split_lora(ops, oracle, device, m, n, k):
    """The bound of test_gpu_gemm_stream's adapter test, whole output."""
    print(f"split lora {m}x{n}x{k}", flush=True)
    rank = 72
    _, _, qa, sa, qw, sw = _operands(ops, device, m, n, k, "int8", False, True)
    gen = torch.Generator().manual_seed(rank)
    t = torch.randn(m, rank, generator=gen).to(torch.bfloat16)
    lb = (torch.randn(n, rank, generator=gen) * 0.05).to(torch.bfloat16)
    out = ops.scaled_mm(qa, qw, sa, sw, b_tiled=True, lora_t=t.to(device), lora_b=lb.to(device), lora_scale=0.75,
                        m=m, n=n)
    torch.cuda.synchronize()
    scale = sa.cpu().numpy()[:m].astype(np.float64).reshape(-1, 1) * sw.cpu().numpy()[:n].astype(np.float64)
    y = _exact(_codes(qa, m, k, False), _codes(qw, n, k, True)).astype(np.float64) * scale
    t64, b64 = t.double().numpy(), lb.double().numpy()
    ref = y + 0.75 * (t64 @ b64.T)
    mag = np.abs(y) + 0.75 * (np.abs(t64) @ np.abs(b64).T)
    got = oracle.bf16_to_f32(bits16(out)).astype(np.float64)
    ulp = 2.0 ** (np.floor(np.log2(np.maximum(np.maximum(np.abs(ref), np.abs(got)), 2.0 ** -126))) - 7)
    assert np.all(np.abs(got - ref) <= 0.51 * ulp + (rank + 4) * 2.0 ** -24 * mag)
