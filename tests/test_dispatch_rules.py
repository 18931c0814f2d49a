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
    (1024, 14336, 4096, 4, 4),     # 95, 114
    # its wavefronts share K, and leave a third of the error
    (2048, 4096, 14336, 3, 4), (2048, 9216, 3072, 3, 4), (4608, 4096, 8192, 2, 4), (1341, 5248, 9216, 2, 4)])
def test_the_packed_kernel_keeps_what_it_is_faster_on(lib, m, n, k, wbits, abits):
    assert lib.oq_packed_linear_workspace_bytes(m, n, k, wbits, _lib.OQ_CODES_NIBBLE, abits) == 0


@pytest.mark.parametrize("m,n,k", [(4608, 36864, 4096), (1024, 14336, 4096), (2048, 4096, 4096), (4608, 3072, 12288)])
def test_int8_tables_are_multiplied_as_integers_on_large_problems(lib, m, n, k):
    assert lib.oq_packed_linear_int8_workspace_bytes(m, n, k) == operand_order(m, k, 1) + operand_order(n, k, 1)


@pytest.mark.parametrize("m,n,k", [
    (74, 784, 8000),               # K shared between workgroups 18 us, as integers 45
    (128, 2048, 8128),             # 20, 53
    (200, 1024, 4160),             # 17, 29
    (300, 2048, 7488),             # 25, 50
    (2237, 376, 15232),            # 39, 84
    (1587, 10568, 512),            # one launch 30, as integers 43
    (2048, 4608, 1152),            # 34, 46
    (64, 36864, 4096), (4608, 36864, 131072), (4608, 36868, 4096), (4608, 36864, 4064), (0, 36864, 4096)])   # not taken at all
def test_int8_tables_stay_with_the_launch_that_is_faster(lib, m, n, k):
    assert lib.oq_packed_linear_int8_workspace_bytes(m, n, k) == 0


@pytest.mark.parametrize("m,n,k,wbits", [(4608, 14336, 4096, 3), (4608, 14336, 4096, 4), (2048, 4096, 4096, 6), (8, 512, 7488, 6)])
def test_values_decode_the_weights_where_that_is_faster(lib, m, n, k, wbits):
    # bf16: 559 -> 419, 510 -> 414, 136 -> 75, 115 -> 74 us
    assert lib.oq_matmul_packed_weight_workspace_bytes(m, n, k, wbits, _lib.OQ_BF16) == operand_order(m, k) + operand_order(n, k)


@pytest.mark.parametrize("m,n,k,wbits", [
    (2, 512, 7488, 3), (64, 512, 7488, 3), (4608, 512, 7488, 3),        # 53, 59, 88 us packed; 74, 75, 93 decoded first
    (2, 952, 15552, 2), (2701, 696, 8000, 2), (1445, 1000, 16320, 2),   # 107, 80, 143; 147, 93, 166
    (3416, 2352, 3072, 2)])                                             # the packed launch shares K between wavefronts
def test_values_leave_the_weights_packed_elsewhere(lib, m, n, k, wbits):
    assert lib.oq_matmul_packed_weight_workspace_bytes(m, n, k, wbits, _lib.OQ_BF16) == operand_order(m, k)


def test_the_least_workspace_holds_partial_tiles_only(lib):
    sizes = lambda *shape: (lib.oq_packed_linear_workspace_bytes(*shape), lib.oq_packed_linear_least_workspace_bytes(*shape))
    nibble, u8 = _lib.OQ_CODES_NIBBLE, _lib.OQ_CODES_U8
    full, least = sizes(4608, 12288, 3072, 3, nibble, 3)
    assert full > 0 and least == 0
    full, least = sizes(32760, 13824, 5120, 4, u8, 6)
    assert full > 0 and least == 0
    full, least = sizes(128, 4096, 14336, 4, nibble, 4)     # K shared between workgroups
    assert full == least > 0 and full % (128 * 4096 * 4) == 0
    assert sizes(1, 4096, 4096, 4, nibble, 4) == sizes(1024, 14336, 4096, 4, nibble, 4) == (0, 0)


@pytest.mark.parametrize("m,n,k", [(32760, 5120, 13824), (131072, 3072, 12288), (2000000, 4096, 4096)])
def test_the_decoded_activations_are_bounded(lib, m, n, k):
    # 512 MB of them and one more row of tiles for every part, whatever the token count; the weights are decoded whole
    part = (512 << 20) + 256 * k * 2
    size = lib.oq_packed_linear_workspace_bytes(m, n, k, 6, _lib.OQ_CODES_U8, 6)
    assert operand_order(n, k) < size <= part + operand_order(n, k) and size < operand_order(m, k) + operand_order(n, k)
    size = lib.oq_packed_linear_int8_workspace_bytes(4 * m, n, k)
    assert operand_order(n, k, 1) < size <= part + operand_order(n, k, 1)


PARTS = [   # (tokens, rows, values, weight bits, parts of K that a launch adds up in fp32; 0: four wavefronts' parts in one launch)
    (65, 8192, 12288, 2, 8), (65, 8192, 16384, 4, 8), (1259, 280, 8448, 4, 8), (100, 4608, 8192, 3, 7), (256, 2048, 8192, 2, 7),
    (128, 3072, 8192, 4, 7), (512, 1152, 8192, 4, 6), (87, 4864, 9728, 3, 6), (200, 3072, 16384, 2, 5), (200, 3072, 8192, 4, 5),
    (200, 4608, 4608, 2, 0), (67, 8856, 3328, 3, 0), (1912, 2160, 6656, 2, 0), (256, 14336, 8192, 4, 0), (512, 8192, 8192, 4, 0),
    (2048, 2048, 8192, 4, 0)]


@pytest.mark.parametrize("abits", [4, 6])
@pytest.mark.parametrize("m,n,k,wbits,parts", PARTS)
def test_64x64_tiles_do_not_lessen_the_partial_sums(lib, m, n, k, wbits, parts, abits):
    """The fewer partial sums, the larger their error (512 x 1152 x 8192 in fp32: 2.5e-7 of the result with six, 3.7e-7 with four)."""
    fmt = _lib.OQ_CODES_U8 if abits > 4 else _lib.OQ_CODES_NIBBLE
    assert lib.oq_packed_linear_workspace_bytes(m, n, k, wbits, fmt, abits) == 4 * m * n * parts


@pytest.mark.parametrize("m,n,k", [(829, 3568, 12608), (1217, 1552, 6464), (5807, 680, 15936), (772, 4888, 2048), (299, 14224, 8000), (4668, 880, 5312)])
def test_64x64_tiles_take_no_whole_numbers_into_fp32(lib, m, n, k):
    assert lib.oq_packed_linear_int8_workspace_bytes(m, n, k) == operand_order(m, k, 1) + operand_order(n, k, 1)


@pytest.mark.parametrize("m,k,block,built", [
    (2442, 4096, 4096, True), (1396, 7168, 1024, True), (26042, 384, 128, True), (19532, 512, 8, True),         # 25.4 -> 23.7, 31.6 -> 24.6, 45 -> 32, 35 -> 31 us
    (4608, 14336, 2048, True), (4883, 4096, 8, True), (13021, 1536, 512, True), (26042, 768, 256, True),         # 204 -> 78, 26.0 -> 25.1, 40 -> 34, 49 -> 41
    (2442, 4096, 8, False), (3907, 2560, 512, False), (698, 14336, 512, False), (13021, 768, 8, False),          # 15.5 -> 22.7, 21.0 -> 24.5, 21.7 -> 23.7, 25.1 -> 25.6
    (9766, 1024, 128, False), (2048, 4096, 4096, False), (20000, 8192, 8192, False), (20000, 4100, 4, False)])   # 21.1 -> 24.3, 21.2 -> 23.7, no such kernel
def test_large_quantizer_calls_build_a_plan_where_that_is_faster(m, k, block, built):
    import torch

    from orbitquant_amd import ops

    for dtype, sixteen_bit in ((torch.bfloat16, True), (torch.float16, True), (torch.float32, False)):
        rows = torch.empty(m, k, dtype=dtype, device="meta")
        assert ops._worth_a_plan(rows, 16, block, block ** -0.5) == (built and sixteen_bit)


@pytest.mark.parametrize("block,factor,built", [(4096, 1 / 64, True), (4096.0, 1 / 64, True), (64.0, 1 / 8, False), (4096, 1e-60, False),
                                                (4096, 1e60, False), (4096, float("inf"), False), (4096, float("nan"), False), (4096, 0.0, False)])
def test_a_plan_built_for_a_call_refuses_nothing(block, factor, built):
    """A plan needs a factor that is positive and finite as the float it is handed over as; the kernel without one does not."""
    import torch

    from orbitquant_amd import ops

    assert ops._worth_a_plan(torch.empty(2442, 4096, dtype=torch.bfloat16, device="meta"), 16, block, factor) == built


@pytest.mark.parametrize("m,k,block,built", [(8_388_607, 8192, 1024, True), (8_388_608, 8192, 1024, False), (16_000_000, 8192, 1024, False),
                                             (8_388_608, 512, 8, True), (67_108_863, 8, 8, True), (67_108_864, 8, 8, False)])
def test_a_plan_is_built_only_for_launches_of_fewer_than_2_to_the_32_threads(m, k, block, built):
    import torch

    from orbitquant_amd import ops

    assert ops._worth_a_plan(torch.empty(m, k, dtype=torch.bfloat16, device="meta"), 16, block, block ** -0.5) == built
