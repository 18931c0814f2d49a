"""Which kernel a problem takes, read off the workspace sizes the library asks for (no GPU): the rules weigh a kernel
against the launch it takes the place of, and must not send a call to the slower one.  The times named are single
calls on an MI355X, the one side then the other."""

from __future__ import annotations

import pytest

from orbitquant_amd import _lib


@pytest.fixture(scope="module")
def lib():
    return _lib.load()


def operand_order(rows, k, value_bytes=2):
    return -(-rows // 32) * -(-k * value_bytes // 128) * 4096


@pytest.mark.parametrize("m,n,k,wbits,abits", [
    (4608, 12288, 3072, 3, 3),     # 333 -> 300 us
    (4608, 3072, 12288, 3, 3),     # 319 -> 305 us
    (8192, 13824, 5120, 3, 4),     # 1016 -> 884 us
    (32760, 13824, 5120, 4, 6),    # 4368 -> 3419 us
    (2048, 4096, 4096, 6, 6)])     # 123 -> 75 us
def test_large_problems_are_decoded_first(lib, m, n, k, wbits, abits):
    fmt = _lib.OQ_CODES_U8 if abits > 4 else _lib.OQ_CODES_NIBBLE
    assert lib.oq_packed_linear_workspace_bytes(m, n, k, wbits, fmt, abits) == operand_order(m, k) + operand_order(n, k)


@pytest.mark.parametrize("m,n,k,wbits,abits", [
    (2057, 9824, 13056, 3, 4),     # 521 us packed, 592 decoded first
    (1514, 13008, 12736, 2, 4),    # 451, 581
    (974, 6640, 15424, 3, 3),      # 230, 291
    (6144, 4096, 16384, 3, 4),     # 711, 998
    (4971, 3704, 1088, 2, 4),      # 54, 77
    (2048, 3072, 12288, 3, 4),     # 155, 175
    (4608, 3072, 3072, 3, 3),      # 85, 86
    (1024, 14336, 4096, 4, 4)])    # 95, 114
def test_the_packed_kernel_keeps_what_it_is_faster_on(lib, m, n, k, wbits, abits):
    assert lib.oq_packed_linear_workspace_bytes(m, n, k, wbits, _lib.OQ_CODES_NIBBLE, abits) == 0
