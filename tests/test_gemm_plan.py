"""Which kernels a scaled GEMM call takes (h3q_scaled_mm_plan, on the host): the
sizes on both sides of every line of the rules, so that a change of a rule shows
here and not only in a measurement."""

from __future__ import annotations

import random

import pytest

from _util import gemm_plan

FEW, STREAM = "few rows", "stream"


@pytest.mark.parametrize("m,n,k,kernel", [
    # 65 .. 128 rows: up to 8192 columns the few-rows kernel until K is long
    (128, 5120, 5120, FEW), (65, 5120, 5120, FEW), (128, 2048, 2048, FEW), (96, 8192, 10240, FEW),
    (128, 5120, 12288, STREAM), (128, 5120, 13824, STREAM), (65, 8200, 256, STREAM), (77, 10752, 5376, STREAM),
    # 33 .. 64 rows: streaming tiles for wide weights with K from 5120
    (40, 10752, 5376, STREAM), (64, 10248, 5120, STREAM), (64, 10240, 5120, FEW), (40, 16384, 4096, FEW),
    (40, 8208, 5120, FEW), (64, 5120, 13824, FEW),
    (32, 16384, 13824, FEW), (1, 10752, 5376, FEW)])
def test_few_rows_tiled_weights(m, n, k, kernel):
    assert gemm_plan(m, n, k, a_tiled=True, b_tiled=True)[0] == kernel
    assert gemm_plan(m, n, k, b_tiled=True)[0] == kernel


@pytest.mark.parametrize("m,n,k,kernel", [
    (16, 10752, 13824, FEW), (17, 10752, 3072, STREAM), (17, 10752, 2944, FEW),
    (17, 5120, 5120, STREAM), (17, 5120, 4992, FEW), (24, 8192, 5120, FEW), (24, 8192, 7168, STREAM),
    (24, 5120, 13840, FEW), (25, 5120, 3072, STREAM), (32, 5120, 3088, FEW), (32, 5120, 4112, STREAM),
    (32, 4096, 13824, FEW), (48, 1024, 3072, FEW), (56, 4096, 13824, FEW), (57, 4096, 5120, STREAM),
    (33, 4104, 3072, STREAM), (33, 4104, 2944, FEW),
    (65, 1024, 2048, STREAM), (65, 1024, 1920, FEW), (65, 1024, 2064, FEW), (65, 2048, 3088, FEW),
    (65, 2048, 4112, STREAM), (81, 2048, 3088, STREAM), (128, 2048, 2064, FEW), (65, 5120, 2064, STREAM),
    (128, 5120, 1920, FEW)])
def test_few_rows_row_major_weights(m, n, k, kernel):
    assert gemm_plan(m, n, k)[0] == kernel


@pytest.mark.parametrize("m,n,k", [(1, 8, 128), (32, 1024, 3072), (128, 2048, 2048), (16, 5120, 5120)])
def test_few_rows_of_tiled_activations_on_row_major_weights(m, n, k):
    """The few-rows kernel of row-major weights reads row-major activations only."""
    assert gemm_plan(m, n, k, a_tiled=True)[0] == STREAM
    assert gemm_plan(m, n + 4, k, a_tiled=True)[0] == "per tile"  # h3q_scaled_mm refuses it


def test_few_rows_with_an_adapter():
    """The few-rows kernels take no adapter: streaming tiles where their form allows, else per tile."""
    assert gemm_plan(16, 5120, 5120, b_tiled=True, rank=64)[0] == STREAM
    assert gemm_plan(128, 2048, 2048, rank=8)[0] == STREAM
    assert gemm_plan(16, 5116, 5120, b_tiled=True, rank=64)[0] == "per tile"


@pytest.mark.parametrize("m,n,k,split", [(5130, 3336, 1536, 3072), (1030, 16904, 2048, 13056),
                                         (4362, 4104, 1536, -3840), (2049, 8712, 1536, -1792),
                                         (4608, 4096, 1024, -4096), (5130, 4104, 1024, 0), (8192, 15360, 5120, 0)])
def test_calls_in_two_launches(m, n, k, split):
    """First columns, or (negative) first rows, of the four-wave part; 0: one launch."""
    plan = gemm_plan(m, n, k, a_tiled=True, b_tiled=True)
    assert plan[0] == ("split" if split else "four waves") and plan[2] == split


@pytest.mark.parametrize("m,n,k,f16,rank,kernel", [
    (600, 3520, 1040, True, 0, STREAM), (2600, 256, 4112, False, 0, STREAM), (4400, 4096, 2064, False, 64, STREAM),
    (3500, 3520, 4112, True, 0, "per tile"), (3500, 3520, 4112, False, 64, "per tile"),
    (16384, 4096, 624, False, 0, "per tile"), (9000, 3520, 2064, False, 0, "per tile"),
    (12800, 2304, 1040, True, 0, "per tile"), (129, 8, 144, False, 0, STREAM)])
def test_k_tails_above_128_rows(m, n, k, f16, rank, kernel):
    """Row-major calls with a K that is not a multiple of 128: streaming tiles while
    the 256 x 256 tiles of the sixteen-wave kernels leave most of the chip idle."""
    assert gemm_plan(m, n, k, f16=f16, rank=rank)[0] == kernel


def test_the_layouts_do_not_decide_above_128_rows():
    """Nor at any row count with an adapter: such a call gives the same bits in every layout."""
    rng = random.Random(7)
    for _ in range(2000):
        m = round(129 * (20000 / 129) ** rng.random())
        n, k = 8 * rng.randint(1, 2000), 128 * rng.randint(2, 110)
        rank = rng.choice((0, 0, 64))
        plans = {gemm_plan(m, n, k, a_tiled=a, b_tiled=b, rank=rank)
                 for a in (False, True) for b in (False, True)}
        assert len(plans) == 1, (m, n, k, rank, plans)
        few = 1 + m % 128
        assert gemm_plan(few, n, k, rank=64) == gemm_plan(few, n, k, b_tiled=True, rank=64)
