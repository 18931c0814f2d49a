"""GPU tests of the plan-based rotate+quantize kernel (oq_rotate_plan_build + the rotate_plan
argument of oq_rotate_quantize): codes, norms and values must equal the CPU oracle bit for bit,
and therefore the plain kernel, on every configuration dimension, every block size the kernel is
instantiated for, every output form, and on rows that take its slow paths (tiny or non-finite
values, codebooks without a cell table)."""

from __future__ import annotations

import numpy as np
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


def constants(dev, k, block, bits):
    from oracle import oracle_np

    perm, signs, h, inv = oracle_np.rpbh_constants(k, 0, block)
    from parity_util import reference_tables

    cents, bounds = reference_tables(k, bits)
    t = dict(perm=torch.from_numpy(perm.astype(np.int32)).to(dev), signs=torch.from_numpy(signs.astype(np.int8)).to(dev),
             bounds=torch.from_numpy(bounds).to(dev), cents=torch.from_numpy(cents).to(dev))
    return perm, signs, h, inv, cents, bounds, t


def both_kernels(x, t, h, inv, **kw):
    from orbitquant_amd import ops

    plan = ops.rotate_plan(t["perm"], t["signs"], t["bounds"], block_size=h, inv_sqrt_block=float(inv))
    fast = ops.rotate_quantize(x, t["perm"], t["signs"], t["bounds"], block_size=h, eps=1e-10, inv_sqrt_block=float(inv),
                               plan=plan, **kw)
    plain = ops.rotate_quantize(x, t["perm"], t["signs"], t["bounds"], block_size=h, eps=1e-10, inv_sqrt_block=float(inv), **kw)
    return fast, plain


def make_rows(m, k, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(m, k, generator=g)
    x[torch.rand(m, k, generator=g) < 0.01] *= 20
    x[3] = 0
    x[5, ::2] = 0
    return x.to(dtype)


CONFIG_DIMS = [(1152, 64), (1152, "paper"), (4608, "paper"), (3072, "paper"), (12288, "paper"), (5120, "paper"),
               (13824, "paper"), (4096, "paper"), (14336, "paper")]


@pytest.mark.parametrize("k,block", CONFIG_DIMS)
@pytest.mark.parametrize("dtype,bits", [(torch.bfloat16, 4), (torch.float16, 3), (torch.float32, 4), (torch.bfloat16, 6)])
def test_plan_kernel_equals_oracle_on_config_dims(dev, k, block, dtype, bits):
    from oracle import oracle_c

    perm, signs, h, inv, cents, bounds, t = constants(dev, k, block, bits)
    m = 37
    x = make_rows(m, k, dtype, seed=k + bits)
    (codes, _, norms), (codes_plain, _, norms_plain) = both_kernels(x.to(dev), t, h, inv, code_format="u8")
    want_codes, want_norms = oracle_c.rotate_quantize(x.float().numpy(), perm, signs, bounds, h, 1e-10, inv)
    assert np.array_equal(codes.cpu().numpy(), want_codes)
    assert np.array_equal(norms.cpu().numpy().view(np.int32), want_norms.view(np.int32))
    assert torch.equal(codes, codes_plain) and torch.equal(norms, norms_plain)


@pytest.mark.parametrize("log_h", range(3, 13))
def test_every_block_size(dev, log_h):
    from oracle import oracle_c

    h = 1 << log_h
    k = max(h, 8) * 3
    for dtype in (torch.bfloat16, torch.float32):
        perm, signs, hh, inv, cents, bounds, t = constants(dev, k, h, 4)
        x = make_rows(19, k, dtype, seed=log_h)
        (packed, _, norms), (packed_plain, _, _) = both_kernels(x.to(dev), t, h, inv, code_format="nibble")
        want_codes, want_norms = oracle_c.rotate_quantize(x.float().numpy(), perm, signs, bounds, h, 1e-10, inv)
        want_packed = (want_codes[:, 0::2] | (want_codes[:, 1::2] << 4)).astype(np.uint8)
        assert np.array_equal(packed.cpu().numpy(), want_packed), (h, dtype)
        assert np.array_equal(norms.cpu().numpy().view(np.int32), want_norms.view(np.int32))
        assert torch.equal(packed, packed_plain)


@pytest.mark.parametrize("log_h", range(3, 13))
def test_every_block_size_in_byte_codes_and_weight_indices(dev, log_h):
    """What a lane holds after the last stages (16 and 32 lanes apart) is not its own slots: codes are put back as they
    are packed, by emitter and width.  The other weight widths have their own packing, 1000 rows their own kernel."""
    from oracle import oracle_c, oracle_np
    from orbitquant_amd import ops

    h = 1 << log_h
    k = max(h, 8) * 3
    perm, signs, hh, inv, cents, bounds, t = constants(dev, k, h, 6)
    for m in (19, 1100):
        x = make_rows(m, k, torch.float16, seed=log_h)
        (codes, _, _), _ = both_kernels(x.to(dev), t, h, inv, code_format="u8")
        want, _ = oracle_c.rotate_quantize(x.float().numpy(), perm, signs, bounds, h, 1e-10, inv)
        assert np.array_equal(codes.cpu().numpy(), want), (h, m)
    for bits in (3, 4, 6, 8):
        edges = np.linspace(-3, 3, 2 ** bits - 1).astype(np.float32) / np.float32(np.sqrt(k))
        w = torch.randn(9, k, generator=torch.Generator().manual_seed(bits))
        packed, norms = ops.quantize_weight(w.to(dev), t["perm"], t["signs"], torch.from_numpy(edges).to(dev), bits=bits, block_size=h,
                                            eps=1e-10, inv_sqrt_block=float(inv))
        want_packed, want_norms, _ = oracle_np.quantize_weight(w.numpy(), perm, signs, edges, h, 1e-10, bits, norm_order="sumsq_v1")
        assert np.array_equal(packed.cpu().numpy(), want_packed), (h, bits)
        assert torch.equal(norms.cpu(), want_norms)


@pytest.mark.parametrize("k,h", [(520, 8), (1048, 8), (2056, 8), (24 * 64, 64), (17 * 128, 128), (9 * 256, 256)])
def test_ragged_rows(dev, k, h):
    """Rows that are not a multiple of 512: the last unit has idle lanes."""
    from oracle import oracle_c

    perm, signs, hh, inv, cents, bounds, t = constants(dev, k, h, 4)
    x = make_rows(33, k, torch.bfloat16, seed=k)
    (codes, _, norms), _ = both_kernels(x.to(dev), t, h, inv, code_format="u8")
    want_codes, want_norms = oracle_c.rotate_quantize(x.float().numpy(), perm, signs, bounds, h, 1e-10, inv)
    assert np.array_equal(codes.cpu().numpy(), want_codes)
    assert np.array_equal(norms.cpu().numpy().view(np.int32), want_norms.view(np.int32))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("k,h", [(1536, 512), (6144, 2048)])
def test_gather_that_repeats_positions(dev, dtype, k, h):
    """A gather that is no permutation has no sign per input position: the kernel applies the signs by slot."""
    from oracle import oracle_c

    perm, signs, hh, inv, cents, bounds, t = constants(dev, k, h, 4)
    perm = perm.copy()
    perm[1::3] = perm[0::3][: len(perm[1::3])]
    t["perm"] = torch.from_numpy(perm.astype(np.int32)).to(dev)
    x = make_rows(21, k, dtype, seed=h)
    (codes, _, norms), (codes_plain, _, _) = both_kernels(x.to(dev), t, h, inv, code_format="u8")
    want_codes, want_norms = oracle_c.rotate_quantize(x.float().numpy(), perm, signs, bounds, h, 1e-10, inv)
    assert np.array_equal(codes.cpu().numpy(), want_codes)
    assert np.array_equal(norms.cpu().numpy().view(np.int32), want_norms.view(np.int32))
    assert torch.equal(codes, codes_plain)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_rows_that_take_the_ieee_division(dev, dtype):
    """Tiny values, tiny and huge norms, infinities and NaNs: the row-level test must send these
    rows to the plain division, and the result must still be the specification's."""
    from oracle import oracle_c

    k, h = 1024, 256
    perm, signs, hh, inv, cents, bounds, t = constants(dev, k, h, 4)
    x = make_rows(40, k, torch.float32, seed=1)
    tiny = 1e-30 if dtype != torch.float16 else 6e-8
    x[1, 7] = tiny                      # one tiny value in an ordinary row
    x[2] *= 1e-28 if dtype != torch.float16 else 1e-4   # a row of tiny values
    x[4] *= 1e12 if dtype != torch.float16 else 30.0    # a huge norm
    x[6, 100] = float("inf")
    x[7, 5] = float("nan")
    x[8] = 0
    x[8, 9] = -tiny
    if dtype == torch.bfloat16:
        x[9, 3] = 1e-39                 # a bf16 denormal
    x = x.to(dtype)
    (codes, _, norms), (codes_plain, _, norms_plain) = both_kernels(x.to(dev), t, h, inv, code_format="u8")
    with np.errstate(all="ignore"):
        want_codes, want_norms = oracle_c.rotate_quantize(x.float().numpy(), perm, signs, bounds, h, 1e-10, inv)
    assert torch.equal(codes, codes_plain)
    assert np.array_equal(codes.cpu().numpy(), want_codes)
    got = norms.cpu().numpy()
    assert np.array_equal(np.isnan(got), np.isnan(want_norms))
    ok = ~np.isnan(want_norms)
    assert np.array_equal(got[ok].view(np.int32), want_norms[ok].view(np.int32))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("k,h", [(1024, 1024), (9216, 1024), (8192, 1024), (2048, 2048), (14336, 2048), (4096, 4096), (8192, 4096), (12288, 4096), (16384, 4096)])
@pytest.mark.parametrize("m,bits", [(1, 4), (12, 3), (12, 6)])
def test_blocks_shared_by_wavefronts(dev, k, h, m, bits, dtype):
    """Few rows: two to eight wavefronts a block, eight or sixteen values each; slow rows, and a codebook without cells."""
    from oracle import oracle_c

    perm, signs, hh, inv, cents, bounds, t = constants(dev, k, h, bits)
    x = make_rows(16, k, torch.float32, seed=k + bits)[:m]
    if m > 1:
        x[1, 7] = 1e-30 if dtype != torch.float16 else 6e-8
        x[2] *= 1e12 if dtype != torch.float16 else 30.0
        x[4, 100] = float("inf")
        x[6, 5] = float("nan")
    x = x.to(dtype)
    fmt = "nibble" if bits <= 4 else "u8"
    for table in (bounds, np.sort(np.concatenate([bounds[:-1], bounds[:1] * (1 + 1e-7)])).astype(np.float32)):
        t["bounds"] = torch.from_numpy(table).to(dev)
        (codes, _, norms), (codes_plain, _, _) = both_kernels(x.to(dev), t, h, inv, code_format=fmt)
        with np.errstate(all="ignore"):
            want, want_norms = oracle_c.rotate_quantize(x.float().numpy(), perm, signs, table, h, 1e-10, inv)
        if fmt == "nibble":
            want = (want[:, 0::2] | (want[:, 1::2] << 4)).astype(np.uint8)
        assert np.array_equal(codes.cpu().numpy(), want) and torch.equal(codes, codes_plain)
        got, ok = norms.cpu().numpy(), ~np.isnan(want_norms)
        assert np.array_equal(np.isnan(got), ~ok) and np.array_equal(got[ok].view(np.int32), want_norms[ok].view(np.int32))


@pytest.mark.parametrize("levels", [2, 3, 5, 16, 64, 100, 256])
def test_any_codebook_size_and_awkward_boundaries(dev, levels):
    """Boundary sets for which no cell table exists (more than 64 levels, clustered boundaries)
    take the binary search over the folded thresholds."""
    from oracle import oracle_np

    k, h = 2048, 512
    perm, signs, hh, inv = oracle_np.rpbh_constants(k, 0, h)
    g = np.random.default_rng(levels)
    bounds = np.sort(g.normal(0, 0.03, levels - 1)).astype(np.float32)
    if levels == 16:
        bounds[5] = np.nextafter(bounds[4], np.float32(1))  # two boundaries one ulp apart
    t = dict(perm=torch.from_numpy(perm.astype(np.int32)).to(dev), signs=torch.from_numpy(signs.astype(np.int8)).to(dev),
             bounds=torch.from_numpy(bounds).to(dev))
    x = make_rows(21, k, torch.bfloat16, seed=levels)
    (codes, _, _), (codes_plain, _, _) = both_kernels(x.to(dev), t, h, inv, code_format="u8")
    want, _ = oracle_np.quantize_codes(x.float().numpy(), perm, signs, bounds, h, 1e-10, inv)
    assert np.array_equal(codes.cpu().numpy(), want)
    assert torch.equal(codes, codes_plain)


def test_values_on_exact_boundaries(dev):
    """A rotated value that lands exactly on a boundary belongs to the lower code; the folded
    thresholds must keep that for a factor that is not a power of two (block 512)."""
    from oracle import oracle_np

    k, h = 512, 512
    perm, signs, hh, inv = oracle_np.rpbh_constants(k, 0, h)
    x = np.zeros((64, k), np.float32)
    x[np.arange(64), np.arange(64) * 7 % k] = 1.0   # one-hot rows: every rotated value is +-1/sqrt(512) exactly
    rot = np.float32(1.0) * np.float32(inv)
    bounds = np.array([-rot, np.nextafter(-rot, np.float32(0)), 0.0, np.nextafter(rot, np.float32(0)), rot], np.float32)
    t = dict(perm=torch.from_numpy(perm.astype(np.int32)).to(dev), signs=torch.from_numpy(signs.astype(np.int8)).to(dev),
             bounds=torch.from_numpy(bounds).to(dev))
    (codes, _, _), (codes_plain, _, _) = both_kernels(torch.from_numpy(x).to(dev), t, h, inv, code_format="u8")
    want, _ = oracle_np.quantize_codes(x, perm, signs, bounds, h, 1e-10, inv)
    assert set(np.unique(want)) == {0, 4}   # -rot is not above the boundary -rot: code 0; +rot is above four: code 4
    assert np.array_equal(codes.cpu().numpy(), want) and torch.equal(codes, codes_plain)


@pytest.mark.parametrize("values", ["scaled", "unit_bf16"])
def test_value_outputs(dev, values):
    k, h = 3072, 1024
    perm, signs, hh, inv, cents, bounds, t = constants(dev, k, h, 4)
    for dtype in (torch.bfloat16, torch.float32):
        x = make_rows(23, k, dtype, seed=2).to(dev)
        fast, plain = both_kernels(x, t, h, inv, code_format="u8", values=values, centroids=t["cents"])
        for a, b in zip(fast, plain):
            assert torch.equal(a, b)
        fast, plain = both_kernels(x, t, h, inv, code_format=None, values=values, centroids=t["cents"])
        assert fast[0] is None and torch.equal(fast[1], plain[1]) and torch.equal(fast[2], plain[2])


def test_plan_for_another_shape_is_loud(dev):
    from orbitquant_amd import ops

    perm, signs, h, inv, cents, bounds, t = constants(dev, 1024, 256, 4)
    other = constants(dev, 1024, 512, 4)
    wrong = ops.rotate_plan(other[6]["perm"], other[6]["signs"], other[6]["bounds"], block_size=512, inv_sqrt_block=float(other[3]))
    x = make_rows(32, 1024, torch.bfloat16, seed=3).to(dev)
    lib_codes = torch.full((32, 1024), 0xAB, dtype=torch.uint8, device=dev)
    from orbitquant_amd import _lib

    lib = _lib.load()
    norms = torch.full((32,), -1.0, device=dev)
    rc = lib.oq_rotate_quantize(x.data_ptr(), 2, 32, 1024, t["perm"].data_ptr(), t["signs"].data_ptr(), t["bounds"].data_ptr(),
                                None, 16, 256, 1e-10, float(inv), wrong.data_ptr(), lib_codes.data_ptr(), 0, None, 0,
                                norms.data_ptr(), None)
    torch.cuda.synchronize()
    assert rc == 0
    # the kernel does not walk a plan built for another block size: no codes, and NaN norms, so that
    # whatever is computed from this call's outputs is NaN instead of looking like a result
    assert bool((lib_codes == 0xAB).all()) and bool(torch.isnan(norms).all())
    # the Python wrapper knows what the plan was built for and refuses it before any launch
    with pytest.raises(ValueError, match="rotate plan was built for"):
        ops.rotate_quantize(x, t["perm"], t["signs"], t["bounds"], block_size=256, eps=1e-10, inv_sqrt_block=float(inv),
                            code_format="u8", plan=wrong)


def test_layer_uses_the_plan_and_matches_the_two_call_path(dev):
    from orbitquant_amd import OrbitLinear, ops, recipe

    torch.manual_seed(0)
    lin = torch.nn.Linear(1152, 256)
    layer = OrbitLinear.from_linear(lin, config=recipe("w4a4")).to(dev)
    assert layer._rotation_plan is not None and layer._rotation_plan.device.type == "cuda"
    x = make_rows(300, 1152, torch.bfloat16, seed=4).to(dev)
    y = layer(x)
    codes, _, norms = ops.rotate_quantize(x, layer._rotation_permutation, layer._rotation_signs,
                                          layer._activation_codebook_boundaries, block_size=layer.rotation.block_size,
                                          eps=layer.activation_eps, inv_sqrt_block=layer.rotation.normalization,
                                          code_format="nibble")
    want = ops.packed_linear(codes, norms, layer._activation_codebook_centroids, layer.packed_weight_indices,
                             layer.row_norms, layer._weight_codebook_centroids, code_format="nibble", activation_bits=4,
                             weight_bits=4, out_features=256, in_features=1152, bias=layer.bias.to(torch.bfloat16),
                             output_dtype=torch.bfloat16)
    assert torch.equal(y, want)


@pytest.mark.parametrize("m", [1, 32])
def test_a_kept_plan_of_an_earlier_layout_is_loud(dev, m):
    """The layout with signs merged into two sets of gather entries had the first byte 0x4c.  A plan of it holds other
    things at the places that are read now."""
    from orbitquant_amd import _lib, ops

    perm, signs, h, inv, cents, bounds, t = constants(dev, 2048, 256, 4)
    plan = ops.rotate_plan(t["perm"], t["signs"], t["bounds"], block_size=256, inv_sqrt_block=float(inv))
    earlier = plan.clone()
    assert bytes(plan[:4].tolist()) != b"LPQO"
    earlier[:4] = torch.tensor(list(b"LPQO"), dtype=torch.uint8, device=dev)
    x = make_rows(32, 2048, torch.bfloat16, seed=3)[:m].to(dev)
    for kept, loud in ((plan, False), (earlier, True)):
        codes, _, norms = ops.rotate_quantize(x, t["perm"], t["signs"], t["bounds"], block_size=256, eps=1e-10, inv_sqrt_block=float(inv),
                                              code_format="u8", plan=kept)
        assert bool(torch.isnan(norms).all()) == loud
    weight = torch.randn(8, 2048, device=dev)
    packed, weight_norms = torch.zeros(8 * 2048 // 2, dtype=torch.uint8, device=dev), torch.zeros(8, dtype=torch.bfloat16, device=dev)
    assert _lib.load().oq_quantize_weight(weight.data_ptr(), _lib.OQ_F32, 8, 2048, earlier.data_ptr(), t["bounds"].data_ptr(), 16, 256, 1e-10, float(inv), 4,
                                          packed.data_ptr(), weight_norms.data_ptr(), torch.cuda.current_stream().cuda_stream) == 0
    assert bool(torch.isnan(weight_norms).all()) and not packed.any()


def test_a_layer_pickled_with_an_earlier_plan(dev):
    """A module saved whole by a build whose plans were 2048 bytes shorter computes what it did."""
    import io

    from orbitquant_amd import OrbitLinear, recipe

    torch.manual_seed(0)
    layer = OrbitLinear.from_linear(torch.nn.Linear(1152, 256), config=recipe("w4a4")).to(dev)
    x = make_rows(40, 1152, torch.bfloat16, seed=4).to(dev)
    want = layer(x)
    for cut in (0, 2048):
        layer._rotation_plan = layer._rotation_plan[: layer._rotation_plan.numel() - cut].clone()
        file = io.BytesIO()
        torch.save(layer, file)
        file.seek(0)
        restored = torch.load(file, weights_only=False)
        assert torch.equal(restored(x), want) and torch.equal(restored(x[:1]), want[:1])


@pytest.mark.parametrize("m", [1, 12])
def test_shared_blocks_refuse_a_plan_for_another_shape(dev, m):
    """Few rows check the plan behind their first requests: still no codes, and NaN norms."""
    from orbitquant_amd import _lib, ops

    _, _, _, inv, _, _, t = constants(dev, 4096, 4096, 4)
    _, _, _, other_inv, _, _, other = constants(dev, 2048, 2048, 4)
    wrong = ops.rotate_plan(other["perm"], other["signs"], other["bounds"], block_size=2048, inv_sqrt_block=float(other_inv))
    x = make_rows(16, 4096, torch.bfloat16, seed=5)[:m].contiguous().to(dev)
    codes, norms = torch.full((m, 2048), 0xAB, dtype=torch.uint8, device=dev), torch.full((m,), -1.0, device=dev)
    rc = _lib.load().oq_rotate_quantize(x.data_ptr(), 2, m, 4096, t["perm"].data_ptr(), t["signs"].data_ptr(), t["bounds"].data_ptr(), None, 16,
                                        4096, 1e-10, float(inv), wrong.data_ptr(), codes.data_ptr(), 1, None, 0, norms.data_ptr(), None)
    torch.cuda.synchronize()
    assert rc == 0 and bool((codes == 0xAB).all()) and bool(torch.isnan(norms).all())


@pytest.mark.parametrize("which", ["perm", "signs"])
def test_few_rows_with_an_unaligned_permutation(dev, which):
    """The shared form reads the permutation and the signs in pieces of sixteen and eight bytes; others take another kernel."""
    from oracle import oracle_c

    perm, signs, h, inv, _, bounds, t = constants(dev, 4096, 4096, 4)
    x = make_rows(8, 4096, torch.bfloat16, seed=6)
    t[which] = torch.cat([t[which][:1], t[which]])[1:]
    assert t[which].data_ptr() % 8 != 0
    (codes, _, norms), (plain, _, _) = both_kernels(x.to(dev), t, h, inv, code_format="u8")
    want, want_norms = oracle_c.rotate_quantize(x.float().numpy(), perm, signs, bounds, h, 1e-10, inv)
    assert torch.equal(codes, plain) and np.array_equal(codes.cpu().numpy(), want)
    assert np.array_equal(norms.cpu().numpy().view(np.int32), want_norms.view(np.int32))


@pytest.mark.parametrize("k,h", [(1152, 64), (3072, 1024), (4096, 4096), (8192, 8192), (13824, 512), (104, 8)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("gather", ["bijective", "repeated"])
@pytest.mark.parametrize("start", ["aligned", "shifted"])
def test_a_plan_built_for_the_call_changes_nothing(dev, k, h, dtype, gather, start, monkeypatch):
    """One is built just where it can be used: not for a block beyond 4096, fp32 rows, or rows off a 16-byte boundary.  Also for a
    gather that repeats positions, whose signs are applied behind it."""
    from orbitquant_amd import ops

    _, _, _, inv, _, _, t = constants(dev, k, h, 4)
    if gather == "repeated":
        t["perm"][5] = t["perm"][9]
    x = make_rows(40, k, dtype, seed=k).to(dev)
    if start == "shifted":
        x = torch.cat([x.view(-1)[:1], x.view(-1)])[1:].view(40, k)
    assert (x.data_ptr() % 16 == 0) == (start == "aligned")
    call = lambda: ops.rotate_quantize(x, t["perm"], t["signs"], t["bounds"], block_size=h, eps=1e-10, inv_sqrt_block=float(inv), code_format="nibble")
    built, build = [], ops.rotate_plan
    monkeypatch.setattr(ops, "rotate_plan", lambda *args, **kw: built.append(build(*args, **kw)) or built[-1])
    want, _, norms = call()
    assert not built
    monkeypatch.setattr(ops, "_PLAN_FROM_VALUES", 1)
    got, _, got_norms = call()
    assert len(built) == (dtype != torch.float32 and h <= 4096 and start == "aligned")
    for plan in built:
        assert plan[32:36].cpu().numpy().view(np.uint32) == (gather == "bijective")
    assert torch.equal(got, want) and torch.equal(got_norms, norms)


def test_without_memory_for_a_plan_built_for_the_call(dev, monkeypatch):
    from orbitquant_amd import ops

    _, _, h, inv, _, _, t = constants(dev, 384, 128, 4)
    x = make_rows(40, 384, torch.bfloat16, seed=7).to(dev)
    call = lambda: ops.rotate_quantize(x, t["perm"], t["signs"], t["bounds"], block_size=128, eps=1e-10, inv_sqrt_block=float(inv), code_format="nibble")
    want, _, norms = call()
    asked = []

    def none_left(*args, **kw):
        asked.append(args)
        raise torch.OutOfMemoryError("no memory")

    monkeypatch.setattr(ops, "_PLAN_FROM_VALUES", 1)
    monkeypatch.setattr(ops, "rotate_plan", none_left)
    got, _, got_norms = call()
    assert len(asked) == 1 and torch.equal(got, want) and torch.equal(got_norms, norms)


@pytest.mark.parametrize("k,h", [(4096, 4096), (3072, 1024), (14336, 2048), (16384, 4096)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("perm_off,signs_off", [(1, 0), (0, 1), (2, 4), (3, 7)])
def test_few_rows_share_blocks_wherever_the_permutation_lies(dev, k, h, dtype, perm_off, signs_off):
    """Elements off an aligned address do not send a call to the slower kernel.  What tells them apart: blocks are shared on the
    signs themselves, which are here the opposite of those that the plan has, and the other kernel takes the plan's."""
    from oracle import oracle_c
    from orbitquant_amd import ops

    perm, signs, _, inv, _, bounds, t = constants(dev, k, h, 4)
    x = make_rows(8, k, dtype, seed=k)
    plan = ops.rotate_plan(t["perm"], t["signs"], t["bounds"], block_size=h, inv_sqrt_block=float(inv))
    off = lambda tensor, by: torch.cat([tensor[:by], tensor])[by:]
    p, s = off(t["perm"], perm_off), off(-t["signs"], signs_off)
    assert p.data_ptr() % 16 == 4 * perm_off and s.data_ptr() % 16 == signs_off
    codes, _, norms = ops.rotate_quantize(x.to(dev), p, s, t["bounds"], block_size=h, eps=1e-10, inv_sqrt_block=float(inv), code_format="u8", plan=plan)
    want, want_norms = oracle_c.rotate_quantize(x.float().numpy(), perm, -signs, bounds, h, 1e-10, inv)
    assert np.array_equal(codes.cpu().numpy(), want) and np.array_equal(norms.cpu().numpy().view(np.int32), want_norms.view(np.int32))


def test_copies_that_the_plans_launch_cannot_fill_are_refused(dev):
    from orbitquant_amd import ops

    _, _, _, inv, _, _, t = constants(dev, 384, 128, 4)
    build = lambda *copies: ops.rotate_plan(t["perm"], t["signs"], t["bounds"], block_size=128, inv_sqrt_block=float(inv), copies=copies)
    perm, signs = torch.empty_like(t["perm"]), torch.empty_like(t["signs"])
    build(perm, signs)
    assert torch.equal(perm, t["perm"]) and torch.equal(signs, t["signs"])
    wide = torch.zeros(768, dtype=torch.int32, device=dev)
    for wrong in ((perm[:383], signs), (perm, signs[1:]), (perm.long(), signs), (perm, signs.float()), (perm.cpu(), signs), (perm, signs.cpu()),
                  (wide[::2], signs), (signs, perm), (perm,), (perm, signs, signs), (None, signs)):
        with pytest.raises((ValueError, TypeError, AttributeError)):
            build(*wrong)
    assert not bool(wide.any()) and torch.equal(perm, t["perm"])
