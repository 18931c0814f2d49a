"""CPU checks of two arithmetic shortcuts of the plan-based rotate+quantize kernel, on models of
them in C (oracle/kernel_arith_check.c) against the plain IEEE operations: the four-instruction
division, over billions of operand pairs of the admitted ranges, and the folding of the
1/sqrt(block) factor into the bucketize thresholds, around every boundary of the codebooks."""

from __future__ import annotations

import ctypes
from pathlib import Path

import numpy as np
import pytest

ROOT = Path(__file__).resolve().parent.parent


@pytest.fixture(scope="module")
def checks():
    so = ROOT / "oracle" / "liboq_kernel_checks.so"
    if not so.exists():
        from oracle.build import build_oracle

        build_oracle()
    lib = ctypes.CDLL(str(so))
    f32p = ctypes.POINTER(ctypes.c_float)
    lib.oqk_division_mismatches.restype = ctypes.c_int64
    lib.oqk_division_mismatches.argtypes = [ctypes.c_int64, ctypes.c_uint64, ctypes.c_int, f32p, f32p]
    u32p = ctypes.POINTER(ctypes.c_uint32)
    lib.oqk_short_quotient_sample.restype = ctypes.c_int64
    lib.oqk_short_quotient_sample.argtypes = [ctypes.c_int64, ctypes.c_uint64, ctypes.c_int, f32p, f32p, u32p, ctypes.c_int64]
    lib.oqk_short_quotient_mismatches.restype = ctypes.c_int64
    lib.oqk_short_quotient_mismatches.argtypes = [ctypes.c_int, u32p, ctypes.c_int64]
    lib.oqk_fold_threshold.restype = ctypes.c_float
    lib.oqk_fold_threshold.argtypes = [ctypes.c_float, ctypes.c_float]
    lib.oqk_fold_mismatches.restype = ctypes.c_int64
    lib.oqk_fold_mismatches.argtypes = [ctypes.c_float, ctypes.c_float, ctypes.c_int]
    return lib


@pytest.mark.parametrize("mode", [0, 1, 2])
def test_four_instruction_division_is_the_ieee_quotient(checks, mode):
    x, d = ctypes.c_float(), ctypes.c_float()
    bad = checks.oqk_division_mismatches(1_000_000_000, 11 + mode, mode, ctypes.byref(x), ctypes.byref(d))
    assert bad == 0, f"{bad} quotients differ, first x={x.value!r} d={d.value!r}"


def test_the_division_check_catches_an_inexact_sequence(checks):
    x, d = ctypes.c_float(), ctypes.c_float()
    assert checks.oqk_division_mismatches(200_000_000, 5, 16, ctypes.byref(x), ctypes.byref(d)) > 0


SHORT_QUOTIENT_FAILS = {8: [0x50ab43, 0x792863],
                        11: [0x50ab43, 0x5562af, 0x56edff, 0x59c6cb, 0x5eca3f, 0x6828eb, 0x722cf3, 0x742bcb, 0x74458f, 0x7453bb, 0x792863, 0x7f3c33]}


@pytest.mark.parametrize("xbits", [8, 11])
def test_quotients_of_16_bit_inputs_without_the_correction(checks, xbits):
    """All significands: the denominators with a wrong quotient are those whose rows the kernel sends to the IEEE division.
    And a sample over the admitted exponents, where products may be subnormal."""
    found = (ctypes.c_uint32 * 64)()
    count = checks.oqk_short_quotient_mismatches(xbits, found, 64)
    assert list(found[:min(count, 64)]) == SHORT_QUOTIENT_FAILS[xbits]
    source = (ROOT / "orbitquant_amd/csrc/rotate_quantize_fast.h").read_text()
    assert all(f"0x{m:06x}u" in source for m in SHORT_QUOTIENT_FAILS[xbits])
    x, d = ctypes.c_float(), ctypes.c_float()
    skip = (ctypes.c_uint32 * count)(*SHORT_QUOTIENT_FAILS[xbits])
    bad = checks.oqk_short_quotient_sample(300_000_000, 77, int(xbits == 11), ctypes.byref(x), ctypes.byref(d), skip, count)
    assert bad == 0, f"{bad} quotients differ, first x={x.value!r} d={d.value!r}"


@pytest.mark.parametrize("block", [8, 64, 128, 512, 2048, 4096])
def test_folded_thresholds_decide_like_multiply_then_compare(checks, block):
    from oracle import oracle_np

    c = np.float32(1.0 / np.sqrt(block))
    for bits in (2, 3, 4, 6):
        _, bounds = oracle_np.lloyd_max_tables(max(block, 64), bits)
        for b in bounds:
            assert checks.oqk_fold_mismatches(float(b), float(c), 4096) == 0
    # boundaries no codebook has: zero, denormals, huge, infinities
    for b in (0.0, -0.0, 1e-45, -1e-45, 1e-38, 3e38, -3e38, float("inf"), float("-inf")):
        assert checks.oqk_fold_mismatches(b, float(c), 4096) == 0
    t = checks.oqk_fold_threshold(float("nan"), float(c))
    assert t != t


def test_parts_of_k_leave_no_larger_error_than_wavefronts_that_share_it():
    """The 128 x 192 tile keeps the sums of parts of K apart, whole rounds of three K-steps and no longer than a quarter, where it takes the
    place of four wavefronts with a quarter each.  Rounding errors as independent, of a sum's size, which grows with the root of its
    length: one for each of a step's four products, and one for each part added to the others.  Four to eight parts."""
    def variance(parts):
        return 2 * sum(p * p for p in parts) + sum(sum(parts[:i]) for i in range(2, len(parts) + 1))

    for steps in range(12, 1000):
        part = steps // 12 * 3
        parts = [min(part, steps - at) for at in range(0, steps, part)]
        quarters = [steps * (w + 1) // 4 - steps * w // 4 for w in range(4)]
        assert sum(parts) == sum(quarters) == steps and 4 <= len(parts) <= 8
        assert variance(parts) <= variance(quarters), steps
