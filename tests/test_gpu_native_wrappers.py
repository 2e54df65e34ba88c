"""The native tensor wrappers (csrc/torch_ops.cpp) against the Python bodies of
ops.py that they stand in for: every call of the table below is made twice, once
as it is and once with the native wrapper declining, and must give the same
bits (or the same exception) over the argument forms the functions accept."""

from __future__ import annotations

import re
import shutil
import subprocess
import sys

import pytest
import torch

from _util import activations, weights
from conftest import ROOT

pytestmark = pytest.mark.gpu


def _flat(v):
    if v is None:
        return []
    if isinstance(v, torch.Tensor):
        return [v.reshape(-1).view(torch.uint8).cpu()]
    return [t for item in v for t in _flat(item)]


def _both(ops, monkeypatch, call):
    """(result, error) of the call through the native wrapper and without it."""
    got = []
    native = ops._native_call
    taken = []
    for enabled in (True, False):
        def hook(name, first, *args, enabled=enabled):
            out = native(name, first, *args) if enabled else None
            taken.append(out is not None)
            return out

        monkeypatch.setattr(ops, "_native_call", hook)
        try:
            got.append((call(), None))
        except Exception as exc:  # noqa: BLE001 - compared below
            got.append((None, (type(exc), str(exc))))
        torch.cuda.synchronize()
    monkeypatch.setattr(ops, "_native_call", native)
    return got[0], got[1], taken[0] if taken else False


def _calls(ops, device):
    x = activations(37, 512, seed=3, outlier_channels=5).to(device)
    w = weights(264, 512, seed=4).to(device)
    wide = activations(37, 1024, seed=5).to(device)
    e4, i8 = ops.FMT_E4M3FN, ops.FMT_INT8
    qa, sa = ops.quant_rows(x, e4)
    qw, sw = ops.quant_rows(w, e4)
    qt, _ = ops.quant_rows_tiled(w, e4)
    at, _ = ops.quant_rows_tiled(x, e4)
    bias = torch.randn(264, device=device).to(torch.bfloat16)
    t = torch.randn(37, 16, device=device).to(torch.bfloat16)
    lb = torch.randn(264, 16, device=device).to(torch.bfloat16)
    table = torch.randn(3, 512, device=device).to(torch.bfloat16)
    idx = torch.arange(37, device=device) % 3
    g = torch.ones(512, device=device, dtype=torch.bfloat16)
    one = torch.full((1,), 0.01, device=device)
    branch = activations(37, 512, seed=6).to(device)
    q4 = torch.randn(2, 9, 5, 64, device=device).to(torch.bfloat16)
    new = lambda *s, d=torch.bfloat16: torch.zeros(s, device=device, dtype=d)  # noqa: E731
    return {
        "rows": lambda: ops.quant_rows(x, e4),
        "rows int8 rcp, strided": lambda: ops.quant_rows(wide[:, :512], i8, ops.ROUND_RCP_MUL),
        "rows given": lambda: ops.quant_rows(x, i8, codes=new(37, 512, d=torch.int8), scales=new(37, 1, d=torch.float32)),
        "rows one": lambda: ops.quant_rows(x[:1], e4),
        "rows empty": lambda: ops.quant_rows(x[:0], e4),
        "rows transposed": lambda: ops.quant_rows(x.t(), e4),
        "rows fp16": lambda: ops.quant_rows(x.half(), e4),
        "rows bad scales": lambda: ops.quant_rows(x, e4, scales=new(36, d=torch.float32)),
        "rows e4m3 rcp": lambda: ops.quant_rows(x, e4, ops.ROUND_RCP_MUL),
        "tiled given": lambda: ops.quant_rows_tiled(x, e4, codes=new(64, 512, d=torch.float8_e4m3fn), row0=16),
        "tiled too small": lambda: ops.quant_rows_tiled(x, e4, codes=new(32, 512, d=torch.float8_e4m3fn)),
        "tiled K": lambda: ops.quant_rows_tiled(wide[:, :500], e4),
        "mm": lambda: ops.scaled_mm(qa, qw, sa, sw),
        "mm bias": lambda: ops.scaled_mm(qa, qw, sa.reshape(-1), sw.reshape(-1), bias=bias),
        "mm tiled": lambda: ops.scaled_mm(at, qt, sa, sw, bias=bias, a_tiled=True, b_tiled=True, m=37, n=264),
        "mm lora": lambda: ops.scaled_mm(qa, qw, sa, sw, lora_t=t, lora_b=lb, lora_scale=0.5),
        "mm f16": lambda: ops.scaled_mm(qa, qw, sa, sw, bias=bias.half(), out_dtype=torch.float16),
        "mm per tensor": lambda: ops.scaled_mm(qa, qw, one, one),
        "mm out": lambda: ops.scaled_mm(qa, qw, sa, sw, out=new(37, 300)[:, :264]),
        "mm sub rows": lambda: ops.scaled_mm(qa[:5], qw[:40], sa[:5], sw[:40]),
        "mm no rows": lambda: ops.scaled_mm(qa[:0], qw, sa[:0], sw),
        "mm types": lambda: ops.scaled_mm(qa, qw.view(torch.int8), sa, sw),
        "mm scales": lambda: ops.scaled_mm(qa, qw, sa[:7], sw),
        "mm scale type": lambda: ops.scaled_mm(qa, qw, sa.double(), sw),
        "mm half lora": lambda: ops.scaled_mm(qa, qw, sa, sw, lora_t=t),
        "mm rank": lambda: ops.scaled_mm(qa, qw, sa, sw, lora_t=t[:, :4].contiguous(), lora_b=lb[:, :4].contiguous()),
        "mm out type": lambda: ops.scaled_mm(qa, qw, sa, sw, out_dtype=torch.float32),
        "mm device": lambda: ops.scaled_mm(qa, qw.cpu(), sa, sw),
        "down": lambda: ops.lora_down(x, w[:16]),
        "down strided": lambda: ops.lora_down(wide[:, 8:520], w[:24]),
        "down inner": lambda: ops.lora_down(wide, w[:16]),
        "norm": lambda: ops.norm_modulate_quant(x, g, table, table, idx, 1e-6, fmt=i8, rounding=ops.ROUND_RCP_MUL),
        "norm out": lambda: ops.norm_modulate_quant(x, g, table, table, idx, 1e-6, out=True),
        "norm both": lambda: ops.norm_modulate_quant(x, g, table, table, idx, 1e-6, fmt=e4, out=True),
        "norm gate": lambda: ops.norm_modulate_quant(x, g, table, table, idx, 1e-6, fmt=e4,
                                                     residual_gate=(branch, table, new(37, 512))),
        "norm neither": lambda: ops.norm_modulate_quant(x, g, table, table, idx, 1e-6),
        "norm index type": lambda: ops.norm_modulate_quant(x, g, table, table, idx.int(), 1e-6, fmt=e4),
        "norm table": lambda: ops.norm_modulate_quant(x, g, table[:, :256], table, idx, 1e-6, fmt=e4),
        "swiglu": lambda: ops.swiglu_quant(wide, fmt=i8, rounding=ops.ROUND_RCP_MUL),
        "swiglu out": lambda: ops.swiglu_quant(wide, out=True),
        "swiglu neither": lambda: ops.swiglu_quant(wide),
        "swiglu width": lambda: ops.swiglu_quant(wide[:, :1020], fmt=e4),
        "heads": lambda: ops.quant_per_head_e4m3(q4),
        "heads strided": lambda: ops.quant_per_head_e4m3(q4[:, :, :3]),
        "heads shape": lambda: ops.quant_per_head_e4m3(q4[0]),
        "tensor": lambda: ops.quant_tensor_e4m3(x),
        "tensor eager": lambda: ops.quant_tensor_e4m3(x, eager=True),
        "tensor static": lambda: ops.quant_tensor_e4m3(x, one.reshape(())),
        "tensor f16 3-d": lambda: ops.quant_tensor_e4m3(x.half().reshape(1, 37, 512), eager=True),
        "tensor f32 strided": lambda: ops.quant_tensor_e4m3(wide.float()[:, :512]),
        "tensor scale type": lambda: ops.quant_tensor_e4m3(x, one.double()),
    }


DECLINED = {"rows empty", "rows transposed", "rows fp16", "rows bad scales", "rows e4m3 rcp", "tiled too small", "tiled K",
            "mm no rows", "mm types", "mm scales", "mm scale type", "mm half lora", "mm rank", "mm out type",
            "mm device", "down inner", "norm neither", "norm index type", "norm table", "swiglu neither",
            "swiglu width", "heads strided", "heads shape", "tensor f32 strided", "tensor scale type"}


def test_native_wrappers_equal_the_python_ones(ops, device, monkeypatch):
    for name, call in _calls(ops, device).items():
        print(name, flush=True)
        (a, ea), (b, eb), taken = _both(ops, monkeypatch, call)
        assert ea == eb, (name, ea, eb)
        assert taken == (name not in DECLINED), name
        fa, fb = _flat(a), _flat(b)
        assert len(fa) == len(fb) and all(torch.equal(p, q) for p, q in zip(fa, fb)), name


def test_native_wrappers_refuse_what_the_python_ones_refuse(ops, device, monkeypatch):
    """Row counts and formats below zero, and a residual gate without its
    tensors, are no way to say "not given", and an output that does not hold the
    result is refused before the launch: the same error as without the native
    wrapper."""
    x = activations(37, 512, seed=3).to(device)
    q, s = ops.quant_rows(x, ops.FMT_INT8)
    one = torch.ones(1, device=device)
    table = torch.zeros(1, 512, device=device, dtype=torch.bfloat16)
    idx = torch.zeros(37, device=device, dtype=torch.int64)
    g = torch.ones(512, device=device, dtype=torch.bfloat16)
    norm = lambda **kw: ops.norm_modulate_quant(x, g, table, table, idx, 1e-6, out=True, **kw)  # noqa: E731
    calls = {
        "m": lambda: ops.scaled_mm(q, q, one, s, m=-1),
        "m below": lambda: ops.scaled_mm(q, q, one, s, m=-3),
        "n": lambda: ops.scaled_mm(q, q, s, one, n=-1),
        "both scales": lambda: ops.scaled_mm(q, q, s, s, m=-1, n=-1),
        "norm format": lambda: norm(fmt=-1),
        "norm gate of nothing": lambda: norm(residual_gate=(None, None, None)),
        "norm gate without a branch": lambda: norm(residual_gate=(None, table, torch.empty_like(x))),
        "norm gate without a table": lambda: norm(residual_gate=(x, None, torch.empty_like(x))),
        "swiglu format": lambda: ops.swiglu_quant(x, fmt=-1, out=True),
        "down rows": lambda: ops.lora_down(x, x[:16], out=torch.empty(36, 16, device=device, dtype=torch.bfloat16)),
        "down rank": lambda: ops.lora_down(x, x[:16], out=torch.empty(37, 8, device=device, dtype=torch.bfloat16)),
    }
    for name, call in calls.items():
        print(name, flush=True)
        (_, ea), (_, eb), taken = _both(ops, monkeypatch, call)
        assert eb is not None and ea == eb and not taken, (name, ea, eb)


# A kernel library whose h3q_quant_rows returns once another Python thread has
# run since it was entered (0), or after five seconds without (1).
_STUB = """
#include <time.h>
volatile int entered, released;
{others}
int h3q_quant_rows() {{
    entered = 1;
    for (int i = 0; i < 5000 && !released; ++i) nanosleep(&(struct timespec){{0, 1000000}}, 0);
    return !released;
}}
"""
_CHILD = """
import ctypes, importlib.util, sys, threading, torch
folder = sys.argv[1]
stub = ctypes.CDLL(folder + "/libtaomate_h3_amd.so")
spec = importlib.util.spec_from_file_location("_h3q_torch", folder + "/_h3q_torch.so")
native = importlib.util.module_from_spec(spec)
spec.loader.exec_module(native)
x = torch.zeros(2, 16, device="cuda:0", dtype=torch.bfloat16)
codes, scales = x.to(torch.int8), torch.zeros(2, 1, device="cuda:0")
entered, released = (ctypes.c_int.in_dll(stub, name) for name in ("entered", "released"))

def other():
    while not entered.value:
        pass
    released.value = 1

thread = threading.Thread(target=other, daemon=True)
thread.start()
result = native.quant_rows(x, 1, 1, codes, scales, 0)
print("other thread ran" if result is not None else "other thread held up", flush=True)
released.value = entered.value = 1
thread.join(10)
"""


def test_native_wrappers_release_the_interpreter_lock(device, tmp_path):
    """While a wrapper is inside the kernel library another Python thread runs:
    with a stand-in library (a process of its own, nothing launched) whose entry
    point waits for one, as a full launch queue waits for the GPU."""
    from taomate_h3_amd import _lib, _native

    names = set(re.findall(r"\b(h3q_\w+)\s*\(", (ROOT / "include" / "taomate_h3_amd.h").read_text()))
    others = "\n".join(f"int {name}() {{ return 1; }}" for name in sorted(names - {"h3q_quant_rows"}))
    (tmp_path / "stub.c").write_text(_STUB.format(others=others))
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", str(tmp_path / _lib.LIB_PATH.name), str(tmp_path / "stub.c")],
                   check=True)
    shutil.copy(_native.PATH, tmp_path)
    (tmp_path / "child.py").write_text(_CHILD)
    res = subprocess.run([sys.executable, str(tmp_path / "child.py"), str(tmp_path)], capture_output=True, text=True,
                         timeout=100)
    assert res.stdout.strip() == "other thread ran", (res.stdout, res.stderr[-2000:])
