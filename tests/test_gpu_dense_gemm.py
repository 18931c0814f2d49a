"""GPU tests of the GEMM that decodes both operands first (csrc/dense_gemm.hip, csrc/operand_order.hip): the same
operand values summed in the same order as the packed GEMM's launches that do not share K, so the same bits, for every
tile, at ragged sizes; and the rule that chooses it depends on the workspace the caller brings."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    if not torch.cuda.is_available():
        pytest.skip("needs an AMD GPU")
    from orbitquant_amd import _lib

    lib = _lib.load()
    assert lib.oq_device_ok() == 0, lib.oq_last_error()
    return torch.device("cuda:0")


def operands(dev, m, k, n, wbits, abits, seed):
    g = torch.Generator(device=dev)
    g.manual_seed(seed)
    codes = torch.randint(0, 1 << abits, (m, k), device=dev, generator=g, dtype=torch.uint8)
    if abits <= 4:
        codes = codes[:, ::2] | (codes[:, 1::2] << 4)
    return dict(
        codes=codes.contiguous(), norms=torch.rand(m, device=dev, generator=g) + 0.5,
        acents=torch.randn(1 << abits, device=dev, generator=g) * 0.02, wcents=torch.randn(1 << wbits, device=dev, generator=g) * 0.02,
        packed=torch.randint(0, 256, ((n * k * wbits + 7) // 8,), device=dev, generator=g, dtype=torch.uint8),
        rn=(torch.rand(n, device=dev, generator=g) + 0.5).to(torch.bfloat16), bias=torch.randn(n, device=dev, generator=g))


def multiply(o, m, k, n, wbits, abits, dtype, output_map=None):
    from orbitquant_amd import ops

    return ops.packed_linear(o["codes"], o["norms"], o["acents"], o["packed"], o["rn"], o["wcents"], code_format="nibble" if abits <= 4 else "u8",
                             activation_bits=abits, weight_bits=wbits, out_features=n, in_features=k, bias=o["bias"], output_dtype=dtype,
                             output_map=output_map)


A_TABLE = [-128, -79, -62, -48, -36, -25, -15, -5, 0, 15, 25, 36, 48, 62, 79, 127]


def looked_up(packed, rows, k, table):
    """The values of two 4-bit codes per byte, in 64 bits."""
    return table.double()[torch.stack((packed & 15, packed >> 4), dim=-1).long()].view(rows, k)


@pytest.mark.parametrize("tile", [0, 1, 2, 3])
@pytest.mark.parametrize("m,k,n,wbits,abits,dtype,mapped", [
    (300, 64, 264, 4, 4, torch.bfloat16, False), (257, 192, 520, 3, 3, torch.float16, False), (512, 1024, 512, 2, 4, torch.bfloat16, True),
    (129, 576, 1000, 6, 6, torch.float32, False), (65, 128, 72, 8, 8, torch.float16, True)])
def test_same_bits_as_the_packed_gemm(dev, library_switch, tile, m, k, n, wbits, abits, dtype, mapped):
    from orbitquant_amd import ops

    o = operands(dev, m, k, n, wbits, abits, seed=m + n)
    table = ops.activation_table(torch.nn.functional.gelu, dtype, dev) if mapped else None
    library_switch("OQ_GEMM_TILE", 0)
    library_switch("OQ_DENSE_GEMM", "never")
    want = multiply(o, m, k, n, wbits, abits, dtype, table)
    library_switch("OQ_DENSE_GEMM", tile)
    assert torch.equal(multiply(o, m, k, n, wbits, abits, dtype, table), want)


@pytest.mark.parametrize("tile,n", [(0, 4088), (0, 4728), (1, 3064), (2, 2040), (2, 2616)])
def test_last_round_of_workgroups_in_parts(dev, library_switch, tile, n):
    """More than 256 tiles and a last round that is at most half full: its tiles are cut into two parts or four, of which
    some lie wholly past the matrix (seventeen rows of tiles, four rows in the last; columns likewise)."""
    from orbitquant_amd import ops

    m, k = 4100, 192
    o = operands(dev, m, k, n, 3, 4, seed=n)
    library_switch("OQ_GEMM_TILE", 0)
    library_switch("OQ_DENSE_GEMM", "never")
    want = multiply(o, m, k, n, 3, 4, torch.float32)
    library_switch("OQ_DENSE_GEMM", tile)
    assert torch.equal(multiply(o, m, k, n, 3, 4, torch.float32), want)
    o = operands(dev, m, k, n, 4, 4, seed=n + 1)
    table = torch.tensor(A_TABLE, dtype=torch.int8, device=dev)
    got = ops.packed_linear_int8(o["codes"], o["norms"], table, o["packed"], o["rn"], table, scale=0.01, out_features=n, in_features=k,
                                 output_dtype=torch.float32)
    sums = (looked_up(o["codes"], m, k, table) @ looked_up(o["packed"], n, k, table).T).float()
    assert torch.equal(got, sums * (o["norms"] * 0.01)[:, None] * o["rn"].float())


def test_chosen_for_large_problems_only_and_only_with_a_workspace(dev):
    from orbitquant_amd import _lib, ops

    lib = _lib.load()
    m, k, n = 4104, 3072, 9216
    want_bytes = lib.oq_packed_linear_workspace_bytes(m, n, k, 4, 0, 6)
    assert want_bytes == (-(-m // 32) + n // 32) * (k // 64) * 4096
    assert lib.oq_packed_linear_workspace_bytes(128, n, k, 4, 0, 6) < want_bytes // 8
    o = operands(dev, m, k, n, 4, 6, seed=3)
    with_workspace = multiply(o, m, k, n, 4, 6, torch.bfloat16)
    out = torch.empty_like(with_workspace)
    dt = ops._DTYPES
    for workspace, size in ((None, 0), (torch.empty(4096, dtype=torch.uint8, device=dev), 4096)):   # none, too small
        rc = lib.oq_packed_linear(o["codes"].data_ptr(), 0, o["norms"].data_ptr(), o["acents"].data_ptr(), 6, o["packed"].data_ptr(), 4,
                                  o["rn"].data_ptr(), o["wcents"].data_ptr(), o["bias"].data_ptr(), dt[torch.float32], m, n, k, out.data_ptr(),
                                  dt[torch.bfloat16], None if workspace is None else workspace.data_ptr(), size,
                                  torch.cuda.current_stream().cuda_stream)
        assert rc == 0 and torch.equal(out, with_workspace)


@pytest.mark.parametrize("tile", [0, 3])
@pytest.mark.parametrize("wbits,abits,mapped", [(3, 4, False), (6, 6, True)])
def test_activations_decoded_in_parts(dev, library_switch, tile, wbits, abits, mapped):
    """More rows than are decoded at a time: two parts, the second one ragged."""
    from orbitquant_amd import _lib, ops

    m, k, n = 16640 + 33, 16384, 264
    fmt = _lib.OQ_CODES_U8 if abits > 4 else _lib.OQ_CODES_NIBBLE
    o = operands(dev, m, k, n, wbits, abits, seed=abits)
    table = ops.activation_table(torch.nn.functional.gelu, torch.bfloat16, dev) if mapped else None
    library_switch("OQ_GEMM_TILE", 0)
    library_switch("OQ_DENSE_GEMM", "never")
    want = multiply(o, m, k, n, wbits, abits, torch.bfloat16, table)
    library_switch("OQ_DENSE_GEMM", tile)
    size = _lib.load().oq_packed_linear_workspace_bytes(m, n, k, wbits, fmt, abits)
    assert size < (-(-m // 32) + -(-n // 32)) * (k // 64) * 4096
    assert torch.equal(multiply(o, m, k, n, wbits, abits, torch.bfloat16, table), want)


def test_int8_activations_decoded_in_parts(dev, library_switch):
    from orbitquant_amd import _lib, ops

    m, k, n = 32768 + 97, 16448, 72
    o = operands(dev, m, k, n, 4, 4, seed=9)
    table = torch.tensor(A_TABLE, dtype=torch.int8, device=dev)
    library_switch("OQ_DENSE_GEMM", 1)
    assert _lib.load().oq_packed_linear_int8_workspace_bytes(m, n, k) < (-(-m // 32) + -(-n // 32)) * -(-k // 128) * 4096
    got = ops.packed_linear_int8(o["codes"], o["norms"], table, o["packed"], o["rn"], table, scale=0.01, out_features=n, in_features=k,
                                 output_dtype=torch.float32)
    w = looked_up(o["packed"], n, k, table)
    for start in (0, 16000, 32000):   # around the seam, and the ends
        rows = slice(start, start + 1000)
        sums = (looked_up(o["codes"][rows], len(got[rows]), k, table) @ w.T).float()
        assert torch.equal(got[rows], sums * (o["norms"][rows] * 0.01)[:, None] * o["rn"].float())


@pytest.mark.parametrize("m,k,n,wbits,abits,decoded", [
    (2040, 4096, 4096, 6, 6, True), (4608, 3072, 12288, 3, 4, True),
    (6564, 2560, 520, 8, 6, False), (2048, 14336, 4096, 3, 4, False)])   # packed: 128 x 96 tiles, K shared inside
def test_with_and_without_a_workspace_as_the_rules_choose(dev, m, k, n, wbits, abits, decoded):
    from orbitquant_amd import _lib, ops

    lib = _lib.load()
    o = operands(dev, m, k, n, wbits, abits, seed=m)
    fmt = _lib.OQ_CODES_U8 if abits > 4 else _lib.OQ_CODES_NIBBLE
    asked = (-(-m // 32) + -(-n // 32)) * (k // 64) * 4096
    assert lib.oq_packed_linear_workspace_bytes(m, n, k, wbits, fmt, abits) == (asked if decoded else 0)
    with_workspace, room = torch.empty(m, n, device=dev), torch.empty(asked, dtype=torch.uint8, device=dev)
    without = torch.empty_like(with_workspace)
    for out, workspace, size in ((with_workspace, room.data_ptr(), asked), (without, None, 0)):
        rc = lib.oq_packed_linear(o["codes"].data_ptr(), fmt, o["norms"].data_ptr(), o["acents"].data_ptr(), abits, o["packed"].data_ptr(), wbits,
                                  o["rn"].data_ptr(), o["wcents"].data_ptr(), o["bias"].data_ptr(), _lib.OQ_F32, m, n, k, out.data_ptr(), _lib.OQ_F32,
                                  workspace, size, torch.cuda.current_stream().cuda_stream)
        assert rc == 0
    assert torch.equal(without, with_workspace)
    index = ops.unpack_lowbit(o["packed"], wbits, n * k).view(n, k).long()
    codes = o["codes"].long() if abits > 4 else torch.stack((o["codes"] & 15, o["codes"] >> 4), dim=-1).view(m, k).long()
    a, w = o["acents"].bfloat16().double()[codes], o["wcents"].bfloat16().double()[index]   # the tables hold bf16
    factor = o["norms"].double()[:, None] * o["rn"].double()
    exact = (a @ w.T) * factor + o["bias"].double()
    # K additions and four more operations in fp32; a quarter of the additions where four wavefronts share K
    bound = ((a.abs() @ w.abs().T) * factor + o["bias"].double().abs()) * ((k if decoded else k // 4 + 4) + 4) * 2.0 ** -24
    assert bool(((with_workspace.double() - exact).abs() <= bound).all())
    if not decoded:   # at K = 14336 four partial sums leave 7.3e-8, one running sum 2.3e-7
        assert float((with_workspace.double() - exact).norm() / exact.norm()) < 1e-7


@pytest.mark.parametrize("tile", [0, 1, 2, 3])
@pytest.mark.parametrize("m,k,n", [(65, 64, 72), (300, 192, 264), (257, 1088, 520)])
def test_int8_pair_sums_integers_exactly(dev, library_switch, tile, m, k, n):
    import orbitquant_packed_matmul as package

    o = operands(dev, m, k, n, 4, 4, seed=m)
    library_switch("OQ_DENSE_GEMM", tile)
    a_table = torch.tensor([-128, -79, -62, -48, -36, -25, -15, -5, 0, 15, 25, 36, 48, 62, 79, 127], dtype=torch.int8, device=dev)
    w_table = a_table.flip(0).contiguous()
    got = package.matmul_packed_w4a4_int8(o["codes"], o["packed"], o["norms"], o["rn"], a_table, w_table, activation_scale=0.005, weight_scale=0.004,
                                          out_features=n, in_features=k, bias=o["bias"].half(), output_dtype=torch.float16)
    value = lambda packed, rows, table: table.double()[torch.stack((packed & 15, packed >> 4), dim=-1).long()].view(rows, k)
    sums = value(o["codes"], m, a_table) @ value(o["packed"].view(n, k // 2), n, w_table).T
    exact = sums * (o["norms"].double() * (0.005 * 0.004))[:, None] * o["rn"].double() + o["bias"].half().double()
    # one rounding of the sum, three of products, one of the addition (2^-24 each, of terms no larger than |exact| +
    # |bias| in the addition), then half an ulp of fp16
    bound = exact.abs() * 2.0 ** -11 + (exact.abs() + o["bias"].abs().double()) * 2.0 ** -20 + 2.0 ** -24
    assert bool(((got.double() - exact).abs() <= bound).all())


@pytest.mark.parametrize("tile", [0, 1, 2, 3])
@pytest.mark.parametrize("m,k,n,table", [
    (65, 64, 72, A_TABLE), (300, 192, 264, A_TABLE), (257, 16384, 520, list(range(112, 128))),   # sums beyond 2^24
    (65, 131008, 8, [-128] * 15 + [-127])])                                                      # ... and near 2^31
def test_int8_kernel_itself(dev, library_switch, tile, m, k, n, table):
    """`ops.packed_linear_int8` and nothing in its place: the sums are the integers, rounded once to fp32.  The bf16
    kernel rounds each partial sum, which from 2^24 on is another result."""
    from orbitquant_amd import ops

    o = operands(dev, m, k, n, 4, 4, seed=m + k)
    library_switch("OQ_DENSE_GEMM", tile)
    table = torch.tensor(table, dtype=torch.int8, device=dev)
    ones, unit = torch.ones(m, device=dev), torch.ones(n, dtype=torch.bfloat16, device=dev)
    got = ops.packed_linear_int8(o["codes"], ones, table, o["packed"], unit, table, scale=1.0, out_features=n, in_features=k,
                                 output_dtype=torch.float32)
    assert got is not None
    want = (looked_up(o["codes"], m, k, table) @ looked_up(o["packed"], n, k, table).T).float()
    assert torch.equal(got, want)
    if k == 16384:
        library_switch("OQ_DENSE_GEMM", "never")
        in_bf16 = ops.packed_linear(o["codes"], ones, table.float(), o["packed"], unit, table.float(), code_format="nibble", activation_bits=4,
                                    weight_bits=4, out_features=n, in_features=k, output_dtype=torch.float32)
        assert not torch.equal(in_bf16, want)


def test_int8_pair_takes_the_integer_kernel_by_itself(dev):
    import orbitquant_packed_matmul as package
    from orbitquant_amd import _lib, ops

    m, k, n = 1024, 4096, 14336
    o = operands(dev, m, k, n, 4, 4, seed=1)
    table = torch.tensor(list(range(112, 128)), dtype=torch.int8, device=dev)
    assert _lib.load().oq_packed_linear_int8_workspace_bytes(m, n, k) > 0
    direct = ops.packed_linear_int8(o["codes"], o["norms"], table, o["packed"], o["rn"], table, scale=0.5, out_features=n, in_features=k,
                                    output_dtype=torch.bfloat16)
    assert direct is not None
    got = package.matmul_packed_w4a4_int8(o["codes"], o["packed"], o["norms"], o["rn"], table, table, activation_scale=0.5, weight_scale=1.0,
                                          out_features=n, in_features=k, output_dtype=torch.bfloat16)
    assert torch.equal(got, direct)
    rows = slice(1000, 1024)
    sums = (looked_up(o["codes"][rows], 24, k, table) @ looked_up(o["packed"], n, k, table).T).float()
    want = sums * (o["norms"][rows] * 0.5)[:, None] * o["rn"].float()   # the epilogue's fp32 products, in its order
    assert torch.equal(got[rows], want.bfloat16())


def test_int8_kernel_says_what_it_does_not_take(dev):
    from orbitquant_amd import _lib, ops

    lib = _lib.load()
    m, k, n = 2048, 4096, 4096
    need = lib.oq_packed_linear_int8_workspace_bytes(m, n, k)
    assert need > 0
    o = operands(dev, m, k, n, 4, 4, seed=2)
    table = torch.tensor(A_TABLE, dtype=torch.int8, device=dev)
    out, ws = torch.empty(m, n, device=dev), torch.empty(need, dtype=torch.uint8, device=dev)

    def call(rows=m, workspace=ws.data_ptr(), size=need, codes=o["codes"].data_ptr(), activation_table=table.data_ptr()):
        return lib.oq_packed_linear_int8(codes, o["norms"].data_ptr(), 1.0, activation_table, o["packed"].data_ptr(), o["rn"].data_ptr(),
                                         table.data_ptr(), None, 0, rows, n, k, out.data_ptr(), _lib.OQ_F32, workspace, size,
                                         torch.cuda.current_stream().cuda_stream)

    assert call() == 0 and call(rows=0) == 0
    invalid, unsupported = call(codes=None), call(rows=64)
    assert invalid != 0 and unsupported not in (0, invalid)
    assert call(activation_table=None) == invalid
    assert call(workspace=None, size=0) == call(size=need - 1) == call(workspace=ws.data_ptr() + 8, size=need - 8) == invalid
    assert call(codes=o["codes"].data_ptr() + 8) == unsupported
    assert ops.packed_linear_int8(o["codes"][:64], o["norms"][:64], table, o["packed"], o["rn"], table, scale=1.0, out_features=n, in_features=k) is None


@pytest.mark.parametrize("dense,tile", [("never", 0), ("never", 1), ("never", 3), ("never", 4), (0, None), (1, None), (2, None), (3, None)])
@pytest.mark.parametrize("m,k,n,wbits", [(9, 64, 8, 2), (33, 256, 264, 3), (129, 192, 520, 4), (257, 1280, 200, 6), (65, 512, 72, 8)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_floating_activations_from_operand_order(dev, library_switch, dense, tile, m, k, n, wbits, dtype):
    from orbitquant_amd import ops

    library_switch("OQ_DENSE_GEMM", dense)
    if tile is not None:
        library_switch("OQ_GEMM_TILE", tile)
    o = operands(dev, m, k, n, wbits, 4, seed=m + k)
    g = torch.Generator(device=dev)
    g.manual_seed(k)
    x = torch.randn(m, k, device=dev, generator=g).to(dtype)
    got = ops.matmul_packed_weight_values(x, o["packed"], o["rn"], o["wcents"], bits=wbits, out_features=n, in_features=k, bias=o["bias"],
                                          token_scale=o["norms"])
    index = ops.unpack_lowbit(o["packed"], wbits, n * k).view(n, k).long()
    w = o["wcents"].to(dtype).double()[index]   # the tables hold values of the activations' type
    factor = o["norms"].double()[:, None] * o["rn"].double()
    exact = (x.double() @ w.T) * factor + o["bias"].double()
    # K additions and three more operations in fp32, then half an ulp of the output type
    magnitude = (x.double().abs() @ w.abs().T) * factor + o["bias"].double().abs()
    bound = magnitude * (k + 4) * 2.0 ** -24 + exact.abs() * (2.0 ** -11 if dtype == torch.float16 else 2.0 ** -8) + 2.0 ** -25
    assert bool(((got.double() - exact).abs() <= bound).all())


@pytest.mark.parametrize("m,k,n,wbits", [(3416, 3072, 2352, 2), (2700, 3072, 2992, 8), (4608, 3072, 3072, 6), (1024, 4096, 4096, 3)])
def test_bf16_values_sum_alike_with_and_without_a_workspace(dev, m, k, n, wbits):
    """As the rules choose: beside packed launches that share K between wavefronts (the first two), decoded first (the
    third), neither (the last)."""
    from orbitquant_amd import _lib, ops

    o = operands(dev, m, k, n, wbits, 4, seed=m)
    x = torch.randn(m, k, device=dev, generator=torch.Generator(device=dev).manual_seed(n)).bfloat16()
    with_workspace = ops.matmul_packed_weight_values(x, o["packed"], o["rn"], o["wcents"], bits=wbits, out_features=n, in_features=k, bias=o["bias"])
    out = torch.empty_like(with_workspace)
    rc = _lib.load().oq_matmul_packed_weight(x.data_ptr(), _lib.OQ_BF16, None, o["packed"].data_ptr(), wbits, o["rn"].data_ptr(), o["wcents"].data_ptr(),
                                             o["bias"].data_ptr(), _lib.OQ_F32, m, n, k, out.data_ptr(), _lib.OQ_BF16, None, 0,
                                             torch.cuda.current_stream().cuda_stream)
    assert rc == 0 and torch.equal(out, with_workspace)


@pytest.fixture
def no_memory_from(monkeypatch):
    """`no_memory_from(size)`: workspaces of that size and more cannot be allocated."""
    from orbitquant_amd import ops

    real = torch.empty

    def limit_to(limit):
        def empty(size, *args, **kwargs):
            if isinstance(size, int) and size >= limit:
                raise torch.OutOfMemoryError("no memory")
            return real(size, *args, **kwargs)

        monkeypatch.setattr(ops.torch, "empty", empty)

    return limit_to


def test_without_memory_for_the_decoded_operands(dev, no_memory_from):
    """A warning, and the launch without them; memory that the call needed all along stays an error."""
    import orbitquant_packed_matmul as package
    from orbitquant_amd import ops

    o = operands(dev, 4608, 3072, 12288, 3, 4, seed=1)
    linear = lambda: multiply(o, 4608, 3072, 12288, 3, 4, torch.bfloat16)
    x = {dtype: torch.randn(4608, 3072, device=dev).to(dtype) for dtype in (torch.bfloat16, torch.float16)}
    v = operands(dev, 1, 3072, 3072, 6, 4, seed=2)
    values = lambda dtype: ops.matmul_packed_weight_values(x[dtype], v["packed"], v["rn"], v["wcents"], bits=6, out_features=3072, in_features=3072)
    t = operands(dev, 2048, 4096, 4096, 4, 4, seed=3)
    table = torch.tensor(A_TABLE, dtype=torch.int8, device=dev)
    pair = lambda: package.matmul_packed_w4a4_int8(t["codes"], t["packed"], t["norms"], t["rn"], table, table, activation_scale=0.05, weight_scale=0.04,
                                                   out_features=4096, in_features=4096)
    short = operands(dev, 128, 14336, 4096, 4, 4, seed=4)
    want = [linear(), values(torch.bfloat16), values(torch.float16), pair()]
    copy = 4608 * 3072 * 2
    no_memory_from(copy + 1)
    with pytest.warns(RuntimeWarning, match="workspace"):
        assert torch.equal(linear(), want[0])
    with pytest.warns(RuntimeWarning, match="workspace"):
        assert torch.equal(values(torch.bfloat16), want[1])   # the activations' copy fits: the weights stay packed
    no_memory_from(4 << 20)
    with pytest.raises(torch.OutOfMemoryError):
        values(torch.bfloat16)
    with pytest.raises(torch.OutOfMemoryError):               # K shared between workgroups
        multiply(short, 128, 14336, 4096, 4, 4, torch.bfloat16)
    # the same operands in another order of additions: the results differ by roundings to the output type
    with pytest.warns(RuntimeWarning, match="workspace"):
        torch.testing.assert_close(values(torch.float16).float(), want[2].float(), rtol=2.0 ** -10, atol=1e-3)
    with pytest.warns(RuntimeWarning, match="workspace"):
        torch.testing.assert_close(pair().float(), want[3].float(), rtol=2.0 ** -7, atol=1e-3 * float(want[3].float().abs().max()))


def same_bits(a, b):
    """Equal, NaN where the other is NaN."""
    return torch.equal(a.isnan(), b.isnan()) and torch.equal(a.nan_to_num(0.0), b.nan_to_num(0.0))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("tile", [0, 1, 2, 3])
def test_infinities_and_nan_in_values_stay_in_their_rows(dev, library_switch, tile, dtype):
    from orbitquant_amd import ops

    m, k, n = 263, 192, 264
    o = operands(dev, m, k, n, 4, 4, seed=21)
    x = torch.randn(m, k, device=dev, generator=torch.Generator(device=dev).manual_seed(3)).to(dtype)
    x[1, 5], x[64, 0], x[200, 191], x[262, 100] = float("nan"), float("inf"), -float("inf"), float("nan")   # (the last row is repeated as padding)
    call = lambda: ops.matmul_packed_weight_values(x, o["packed"], o["rn"], o["wcents"], bits=4, out_features=n, in_features=k, bias=o["bias"],
                                                   token_scale=o["norms"])
    library_switch("OQ_GEMM_TILE", 0)
    library_switch("OQ_DENSE_GEMM", "never")
    want = call()
    library_switch("OQ_DENSE_GEMM", tile)
    got = call()
    touched = torch.zeros(m, dtype=torch.bool, device=dev)
    touched[[1, 64, 200, 262]] = True
    assert torch.equal((~got.isfinite()).any(dim=1), touched) and bool(got[[1, 262]].isnan().all())
    assert same_bits(got, want)


@pytest.mark.parametrize("tile", [0, 1, 2, 3])
def test_infinities_and_nan_in_token_norms_and_bias(dev, library_switch, tile):
    from orbitquant_amd import ops

    m, k, n = 263, 192, 264
    o = operands(dev, m, k, n, 4, 4, seed=22)
    o["norms"][[0, 130, 262]] = torch.tensor([float("nan"), float("inf"), 0.0], device=dev)
    o["bias"][[7, 263]] = torch.tensor([float("inf"), float("nan")], device=dev)
    library_switch("OQ_GEMM_TILE", 0)
    library_switch("OQ_DENSE_GEMM", "never")
    want = multiply(o, m, k, n, 4, 4, torch.float32)
    library_switch("OQ_DENSE_GEMM", tile)
    got = multiply(o, m, k, n, 4, 4, torch.float32)
    assert same_bits(got, want) and bool(got[0].isnan().all()) and bool(got[:, 263].isnan().all())
    table = torch.tensor(A_TABLE, dtype=torch.int8, device=dev)
    integers = ops.packed_linear_int8(o["codes"], o["norms"], table, o["packed"], o["rn"], table, scale=0.5, out_features=n, in_features=k,
                                      bias=o["bias"], output_dtype=torch.float32)
    sums = (looked_up(o["codes"], m, k, table) @ looked_up(o["packed"], n, k, table).T).float()
    exact = (sums * (o["norms"] * 0.5)[:, None] * o["rn"].float()).double() + o["bias"].double()
    assert torch.equal(integers.isfinite(), exact.float().isfinite()) and torch.equal(integers.isnan(), exact.isnan())
    finite = exact.isfinite()   # (the last product and the addition round once or twice)
    magnitude = (exact.abs() + 2 * o["bias"].double().abs())[finite]
    assert bool(((integers.double() - exact).abs()[finite] <= magnitude * 2.0 ** -23).all())


@pytest.mark.parametrize("integers", [False, True])
def test_a_captured_large_problem_computes_what_the_eager_call_does(dev, integers):
    import orbitquant_packed_matmul as package
    from orbitquant_amd import _lib

    lib = _lib.load()
    m, k, n = 2040, 4096, 4096
    o = operands(dev, m, k, n, 4 if integers else 6, 4 if integers else 6, seed=5)
    table = torch.tensor(A_TABLE, dtype=torch.int8, device=dev)
    if integers:
        assert lib.oq_packed_linear_int8_workspace_bytes(m, n, k) > 0
        call = lambda: package.matmul_packed_w4a4_int8(o["codes"], o["packed"], o["norms"], o["rn"], table, table, activation_scale=0.05, weight_scale=0.04,
                                                       out_features=n, in_features=k)
    else:
        assert lib.oq_packed_linear_workspace_bytes(m, n, k, 6, _lib.OQ_CODES_U8, 6) > lib.oq_packed_linear_least_workspace_bytes(m, n, k, 6, _lib.OQ_CODES_U8, 6)
        call = lambda: multiply(o, m, k, n, 6, 6, torch.bfloat16)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        call()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = call()
    for seed in range(4):
        fresh = operands(dev, m, k, n, 4 if integers else 6, 4 if integers else 6, seed=10 + seed)
        for name in ("codes", "norms"):
            o[name].copy_(fresh[name])
        graph.replay()
        torch.cuda.synchronize()
        replayed = out.clone()
        assert torch.equal(replayed, call())
