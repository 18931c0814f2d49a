"""GPU tests of oq_quantize_weight (the weight side of a layer made on the device): the packed
index stream and the bf16 row norms must equal the oracle's (`oracle_np.quantize_weight` with the
kernel's summation order for the row norm) byte for byte, for the five recipes at the reference's
own test dimension, at the configuration dimensions, for every packing width and input dtype,
with zero rows, and whatever the row tiling.  Against the oracle with torch's norm (the
reference's host path) the norms must agree after bf16 rounding almost everywhere and the
indices everywhere except at boundary ties."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import oracle_np as o
from parity_util import reference_tables

pytestmark = pytest.mark.gpu

RECIPES = {"w4a4": (4, 4), "w3a3": (3, 3), "w2a4": (2, 4), "w2a3": (2, 3), "w4a6": (4, 6)}


@pytest.fixture(scope="module")
def dev():
    if not torch.cuda.is_available():
        pytest.skip("needs an AMD GPU")
    from orbitquant_amd import _lib

    lib = _lib.load()
    assert lib.oq_device_ok() == 0, lib.oq_last_error()
    return torch.device("cuda:0")


def gpu_quantize(dev, w, perm, signs, bounds, block, inv, bits, row_tile=None):
    from orbitquant_amd import ops

    return ops.quantize_weight(w.to(dev), torch.from_numpy(perm.astype(np.int32)).to(dev), torch.from_numpy(signs).to(dev),
                               torch.from_numpy(bounds).to(dev), bits=bits, block_size=block, eps=1e-10,
                               inv_sqrt_block=float(inv), row_tile=row_tile)


@pytest.mark.parametrize("recipe", sorted(RECIPES))
def test_five_recipes_at_the_reference_test_dimension(dev, recipe):
    # tests/test_paper_reference_oracle.py:122-203 of the reference: dim 24 (block 8), seed 29
    wbits, _ = RECIPES[recipe]
    k, n = 24, 13
    perm, signs, block, inv = o.rpbh_constants(k, 29, "paper")
    _, bounds = reference_tables(k, wbits)
    w = torch.randn(n, k, generator=torch.Generator().manual_seed(29))
    w[4] = 0
    packed, norms = gpu_quantize(dev, w, perm, signs, bounds, block, inv, wbits)
    want_packed, want_norms, _ = o.quantize_weight(w.numpy(), perm, signs, bounds, block, 1e-10, wbits, norm_order="sumsq_v1")
    assert np.array_equal(packed.cpu().numpy(), want_packed)
    assert torch.equal(norms.cpu(), want_norms)
    assert float(norms[4]) == 0.0
    # the host path of the product (torch's norm) on this small case: identical
    host_packed, host_norms, _ = o.quantize_weight(w.numpy(), perm, signs, bounds, block, 1e-10, wbits)
    assert np.array_equal(packed.cpu().numpy(), host_packed) and torch.equal(norms.cpu(), host_norms)


@pytest.mark.parametrize(("n", "k", "bits", "dtype"), [
    (4608, 1152, 4, torch.float32),    # c2 fc1
    (1152, 4608, 4, torch.bfloat16),   # c2 fc2
    (1024, 3072, 3, torch.float32),    # c3 (a slab of rows)
    (512, 12288, 3, torch.float16),    # c3 fc2, block 4096
    (512, 5120, 4, torch.bfloat16),    # c4 fc1
    (256, 13824, 4, torch.float32),    # c4 fc2
    (1024, 4096, 2, torch.float32),    # c5 q / k
    (512, 14336, 3, torch.bfloat16),   # c5 down, block 2048
    (300, 1152, 6, torch.float32),
    (77, 2048, 8, torch.float32),
    (64, 1024, 1, torch.float32),
    (50, 520, 5, torch.float32),       # ragged row length, block 8
])
def test_configuration_dimensions(dev, n, k, bits, dtype):
    perm, signs, block, inv = o.rpbh_constants(k, 0, "paper")
    _, bounds = reference_tables(k, bits) if bits in (2, 3, 4, 6, 8) else o.lloyd_max_tables(k, bits)
    gen = torch.Generator().manual_seed(n + k + bits)
    w = (torch.randn(n, k, generator=gen) * 0.02).to(dtype)
    w[n // 3] = 0
    w[n // 2, ::3] *= 40
    packed, norms = gpu_quantize(dev, w, perm, signs, bounds, block, inv, bits)
    want_packed, want_norms, want_idx = o.quantize_weight(w.float().numpy(), perm, signs, bounds, block, 1e-10, bits,
                                                         norm_order="sumsq_v1")
    assert torch.equal(norms.cpu(), want_norms)
    got_idx = o.unpack_bits(packed.cpu().numpy(), bits, n * k).reshape(n, k)
    assert int(np.count_nonzero(got_idx != want_idx)) == 0
    assert np.array_equal(packed.cpu().numpy(), want_packed)
    # row tiling writes the same stream
    tiled, tiled_norms = gpu_quantize(dev, w, perm, signs, bounds, block, inv, bits, row_tile=37 if (37 * k * bits) % 8 == 0 else 40)
    assert torch.equal(tiled, packed) and torch.equal(tiled_norms, norms)
    # against torch's norm: the same up to ties
    host_packed, host_norms, host_idx = o.quantize_weight(w.float().numpy(), perm, signs, bounds, block, 1e-10, bits)
    assert int((norms.cpu().view(torch.int16) != host_norms.view(torch.int16)).sum()) <= max(1, n // 500)
    assert int(np.count_nonzero(got_idx != host_idx)) <= max(2, n * k // 200000)


def test_layer_built_from_a_gpu_weight_matches_the_host_built_layer(dev):
    from orbitquant_amd import OrbitLinear, recipe

    torch.manual_seed(3)
    lin = torch.nn.Linear(1152, 384)
    host = OrbitLinear.from_linear(lin, config=recipe("w4a4"))
    device_built = OrbitLinear.from_linear(lin.to(dev), config=recipe("w4a4"))
    assert device_built.packed_weight_indices.device.type == "cuda"
    assert torch.equal(device_built.row_norms.cpu(), host.row_norms)
    differing = int((device_built.packed_weight_indices.cpu() != host.packed_weight_indices).sum())
    assert differing <= 2   # ties only (the two paths sum a row's squares in different orders)
    x = torch.randn(64, 1152, generator=torch.Generator().manual_seed(1)).to(torch.bfloat16).to(dev)
    y_dev = device_built(x)
    y_host = host.to(dev)(x)
    assert float((y_dev.float() - y_host.float()).abs().max()) <= 0.05 * float(y_host.float().abs().max())


def test_argument_checks(dev):
    from orbitquant_amd import _lib

    lib = _lib.load()
    w = torch.zeros(4, 1024, device=dev)
    bounds = torch.zeros(15, device=dev)
    plan = torch.zeros(int(lib.oq_rotate_plan_bytes(1024)), dtype=torch.uint8, device=dev)
    packed = torch.zeros(4 * 1024 // 2, dtype=torch.uint8, device=dev)
    norms = torch.zeros(4, dtype=torch.bfloat16, device=dev)

    def call(k=1024, block=256, bits=4, levels=16, w_ptr=None):
        return lib.oq_quantize_weight(w.data_ptr() if w_ptr is None else w_ptr, 0, 4, k, plan.data_ptr(), bounds.data_ptr(), levels,
                                      block, 1e-10, 0.0625, bits, packed.data_ptr(), norms.data_ptr(), None)

    assert call(bits=9) == 1 and call(levels=17) == 1 and call(block=48) == 1
    assert call(k=1020, block=4) == 2      # block below 8: no kernel
    assert call(block=4) == 2
    assert call(w_ptr=w.data_ptr() + 4) == 1
    assert call() == 0                      # a zero plan has the wrong magic: no indices are written, the row norms are NaN
    torch.cuda.synchronize()
    assert not packed.any() and bool(torch.isnan(norms.float()).all())


@pytest.mark.parametrize("bits", [2, 3, 4, 6, 8])
@pytest.mark.parametrize("k", [24, 1152, 4096])
def test_rows_of_any_magnitude_and_any_start_of_the_stream(dev, bits, k):
    """Rows that the fast quotient takes and rows that it leaves to the IEEE division (norms beyond 2^20 and below
    eps, values below 2^-80 beside ordinary ones), in one stream and from starts that are not multiples of eight."""
    n = 11
    perm, signs, block, inv = o.rpbh_constants(k, 5, "paper")
    bounds = np.linspace(-3, 3, 2 ** bits - 1).astype(np.float32) / np.float32(np.sqrt(k))
    w = torch.randn(n, k, generator=torch.Generator().manual_seed(k + bits))
    w[1] *= 2.0 ** 24
    w[2] *= 2.0 ** -40
    w[3] *= 2.0 ** -100
    w[4] = 0
    w[5, ::3] *= 2.0 ** -90
    w[6, 1:] = 0
    w[7] *= 2.0 ** 14
    w[8] *= torch.linspace(-100, 0, k).exp2()
    want_packed, want_norms, _ = o.quantize_weight(w.numpy(), perm, signs, bounds, block, 1e-10, bits, norm_order="sumsq_v1")
    for row_tile in (None, 1):
        packed, norms = gpu_quantize(dev, w, perm, signs, bounds, block, inv, bits, row_tile=row_tile)
        assert np.array_equal(packed.cpu().numpy(), want_packed) and torch.equal(norms.cpu(), want_norms)


def test_a_weight_without_rows(dev):
    from orbitquant_amd import OrbitLinear, OrbitQuantConfig

    perm, signs, block, inv = o.rpbh_constants(64, 5, "paper")
    bounds = np.linspace(-0.3, 0.3, 15).astype(np.float32)
    packed, norms = gpu_quantize(dev, torch.empty(0, 64), perm, signs, bounds, block, inv, 4)
    assert packed.shape == (0,) and packed.dtype == torch.uint8 and norms.shape == (0,) and norms.dtype == torch.bfloat16
    layer = OrbitLinear.from_weight(torch.empty(0, 64, device=dev), bias=None, config=OrbitQuantConfig())
    assert layer.packed_weight_indices.numel() == 0 and layer.row_norms.shape == (0,)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_rows_with_infinities_and_nan(dev, dtype):
    """Their norms are not finite, so they take the IEEE division: a NaN has no boundary below it (the oracle's search
    sorts it last), a finite value over an infinite norm is zero.  The rows beside them are what they are alone."""
    k, bits = 1152, 4
    perm, signs, block, inv = o.rpbh_constants(k, 5, "paper")
    bounds = np.linspace(-3, 3, 2 ** bits - 1).astype(np.float32) / np.float32(np.sqrt(k))
    w = torch.randn(7, k, generator=torch.Generator().manual_seed(9)).to(dtype)
    w[1, 3], w[3, 1000], w[5, 0], w[5, 1] = float("nan"), float("inf"), -float("inf"), float("inf")
    packed, norms = gpu_quantize(dev, w, perm, signs, bounds, block, inv, bits)
    want_packed, want_norms, _ = o.quantize_weight(w.float().numpy(), perm, signs, bounds, block, 1e-10, bits, norm_order="sumsq_v1")
    assert torch.equal(norms.cpu().isnan(), want_norms.isnan()) and torch.equal(norms.cpu().nan_to_num(0.0), want_norms.nan_to_num(0.0))
    got, want = packed.cpu().numpy().reshape(7, -1), want_packed.reshape(7, -1)
    codes = lambda rows: np.stack((rows & 15, rows >> 4), axis=-1)
    for row in (1, 3, 5):
        assert np.array_equal(codes(got[row]), np.where(codes(want[row]) == 15, 0, codes(want[row])))
    for row in (0, 2, 4, 6):
        assert np.array_equal(got[row], want[row])
        alone, _ = gpu_quantize(dev, w[row : row + 1], perm, signs, bounds, block, inv, bits)
        assert torch.equal(alone, packed.view(7, -1)[row])


@pytest.mark.parametrize("kind", ["crowded", "repeated", "wide", "two"])
def test_boundaries_with_and_without_cells(dev, kind):
    """Boundaries too close for one cell each, equal ones, far apart ones, a single one; weights that sit on them."""
    k, n = 512, 40
    perm, signs, block, inv = o.rpbh_constants(k, 0, "paper")
    _, bounds = reference_tables(k, 4)
    bounds = {"crowded": np.sort(np.concatenate([bounds[:8], bounds[7] * (1 + np.arange(7) * 1e-6)])), "repeated": np.repeat(bounds[::2], 2)[:15],
              "wide": bounds * np.float32(40), "two": bounds[7:8]}[kind].astype(np.float32)
    w = torch.randn(n, k, generator=torch.Generator().manual_seed(3))
    w[3] = 0                                        # every value is zero
    w[5] = 0
    w[5, 9] = 1.0                                   # every value is +-1/sqrt(block)
    packed, norms = gpu_quantize(dev, w, perm, signs, bounds, block, inv, 4)
    want_packed, want_norms, _ = o.quantize_weight(w.numpy(), perm, signs, bounds, block, 1e-10, 4, norm_order="sumsq_v1")
    assert np.array_equal(packed.cpu().numpy(), want_packed) and torch.equal(norms.cpu(), want_norms)


@pytest.mark.parametrize("k", [24, 1152, 4096])
@pytest.mark.parametrize("change", ["activation codebook", "one boundary", "signed zero", "none"])
def test_a_plan_over_other_boundaries_decides_nothing(dev, k, change):
    """The indices are those of the call's own boundaries, whatever boundaries the plan was built from."""
    from orbitquant_amd import _lib, ops

    lib = _lib.load()
    n, bits = 21, 4
    perm, signs, block, inv = o.rpbh_constants(k, 5, "paper")
    bounds = (np.linspace(-2.5, 2.5, 15) / np.sqrt(k)).astype(np.float32)
    bounds[7] = 0.0
    other = bounds.copy()
    if change == "activation codebook":
        other = (bounds * np.float32(1.4) + np.float32(0.1 / np.sqrt(k))).astype(np.float32)
    elif change == "one boundary":
        other[11] = np.nextafter(other[11], np.float32(1))
    elif change == "signed zero":
        other[7] = -0.0
    w = torch.randn(n, k, generator=torch.Generator().manual_seed(k)).bfloat16()
    w[2] = 0
    t = lambda a: torch.from_numpy(a).to(dev)
    plan = ops.rotate_plan(t(perm.astype(np.int32)), t(signs), t(other), block_size=block, inv_sqrt_block=float(inv))
    weight, mine = w.to(dev), t(bounds)
    packed = torch.zeros(n * k * bits // 8, dtype=torch.uint8, device=dev)
    norms = torch.zeros(n, dtype=torch.bfloat16, device=dev)
    assert lib.oq_quantize_weight(weight.data_ptr(), _lib.OQ_BF16, n, k, plan.data_ptr(), mine.data_ptr(), 16, block, 1e-10, float(inv), bits,
                                  packed.data_ptr(), norms.data_ptr(), torch.cuda.current_stream().cuda_stream) == 0
    want_packed, want_norms, _ = o.quantize_weight(w.float().numpy(), perm, signs, bounds, block, 1e-10, bits, norm_order="sumsq_v1")
    assert np.array_equal(packed.cpu().numpy(), want_packed) and torch.equal(norms.cpu(), want_norms)


@pytest.mark.parametrize("bits", [2, 4, 6])
@pytest.mark.parametrize(("k", "dtype"), [(4096, torch.bfloat16), (2048, torch.float32), (12288, torch.float16), (13824, torch.bfloat16), (14336, torch.float32), (5120, torch.bfloat16)])
def test_rows_with_thresholds_of_their_own_equal_divided_ones(dev, k, dtype, bits):
    """Long rows compare with boundaries that carry the row's norm; a plan over other boundaries has every value divided
    and searched.  The same indices, for norms and values of every size, a boundary at zero, and values next to boundaries."""
    from orbitquant_amd import ops

    n = 96
    perm, signs, block, inv = o.rpbh_constants(k, 2, "paper")
    levels = 1 << bits
    bounds = (np.linspace(-2.4, 2.4, levels - 1) / np.sqrt(k)).astype(np.float32)
    bounds[levels // 2 - 1] = 0.0
    g = torch.Generator().manual_seed(k + bits)
    w = torch.randn(n, k, generator=g)
    w[:40] *= 10.0 ** torch.linspace(-6 if dtype == torch.float16 else -30, 3 if dtype == torch.float16 else 8, 40)[:, None]
    w[40] = 0
    w[41, 1:] = 0                                    # every value is +-1 / sqrt(block) of the row's norm
    w[42] = torch.round(w[42])                       # few distinct sums, many of them zero
    w[43, ::2] = 0
    w = w.to(dtype).to(dev)
    t = lambda a: torch.from_numpy(a).to(dev)
    args = (w, t(perm.astype(np.int32)), t(signs), t(bounds))
    kw = dict(bits=bits, block_size=block, eps=1e-10, inv_sqrt_block=float(inv))
    other = ops.rotate_plan(*args[1:3], t((bounds * np.float32(1.3)).astype(np.float32)), block_size=block, inv_sqrt_block=float(inv))
    packed, norms = ops.quantize_weight(*args, **kw)
    divided, divided_norms = ops.quantize_weight(*args, **kw, plan=other)
    assert torch.equal(packed, divided) and torch.equal(norms, divided_norms)
    rows = [0, 20, 39, 41, 42, 95]
    want, _, _ = o.quantize_weight(w[rows].float().cpu().numpy(), perm, signs, bounds, block, 1e-10, bits, norm_order="sumsq_v1")
    assert np.array_equal(packed.view(n, -1)[rows].cpu().numpy().reshape(-1), want)


def cell_of(v, scale, offset):
    """The cell of a value in a plan's table: one fused multiply-add, one rounding to 0..255."""
    place = (v.astype(np.float64) * np.float64(scale) + np.float64(offset)).astype(np.float32)
    return np.clip(np.rint(place), 0, 255).astype(np.int64)


@pytest.mark.parametrize(("k", "folds"), [(4096, True), (2048, True), (3072, False)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_which_rows_have_thresholds_of_their_own(dev, k, dtype, folds):
    """What tells the two ways apart: the place of a value in the table is rounded once from the rotated value, or from the divided
    one.  In a plan whose cells without a boundary hold 0 and 15 in turn the two differ for values between two cells.  Rows of
    few values a wavefront are divided, and so are rows whose division needs the compiler's (here: norms above 2^20)."""
    from orbitquant_amd import ops

    n, bits, levels = 2048, 4, 16
    perm, signs, block, inv = o.rpbh_constants(k, 2, "paper")
    bounds = (np.linspace(0.7, 1.3, levels - 1) / np.sqrt(k)).astype(np.float32)
    w = torch.randn(n, k, generator=torch.Generator().manual_seed(k)).to(dtype)
    w[n // 2 :] *= 2.0 ** 30
    t = lambda a: torch.from_numpy(a).to(dev)
    args = (w.to(dev), t(perm.astype(np.int32)), t(signs), t(bounds))
    kw = dict(block_size=block, inv_sqrt_block=float(inv))
    plan = ops.rotate_plan(*args[1:], **kw).clone()
    blob = plan.cpu().numpy()
    scale, offset = blob[40:48].view(np.float32)
    cells = blob[-2048:].view([("bound", np.float32), ("below", np.uint32)])
    empty = np.isinf(cells["bound"])
    assert blob[36:40].view(np.uint32) == 256 and empty.sum() == 256 - (levels - 1)
    cells["below"][empty] = 15 * (np.arange(256) & 1)[empty]
    packed, _ = ops.quantize_weight(*args, bits=bits, eps=1e-10, plan=t(blob), **kw)
    got = packed.cpu().numpy().reshape(n, -1)
    got = np.stack([got & 15, got >> 4], axis=-1).reshape(n, k)

    x32 = w.float().numpy()
    norm = np.sqrt(o.sumsq_v1(x32)).astype(np.float32).reshape(n, 1)
    folded = cell_of(o.rotate(x32, perm, signs, block, np.float32(1)), np.float32(scale) * (np.float32(inv) / norm), offset)
    divided = cell_of(o.rotate(x32, perm, signs, block, inv) / norm, scale, offset)
    differ = empty[folded] & empty[divided] & (cells["below"][folded] != cells["below"][divided])   # (the others have a boundary to compare with)
    divides = np.arange(n)[:, None] >= (n // 2 if folds else 0)
    assert differ[: n // 2].any() and differ[n // 2 :].any()   # (some five each)
    assert np.array_equal(got[differ], cells["below"][np.where(divides, divided, folded)][differ])


@pytest.mark.parametrize("bits", [(4, 4), (3, 4)])
def test_a_converted_layer_has_what_a_built_one_has(dev, bits):
    """One plan where weights and activations share a codebook, constants in storages of their own."""
    import io

    from orbitquant_amd import OrbitLinear, OrbitQuantConfig

    config = OrbitQuantConfig(weight_bits=bits[0], activation_bits=bits[1])
    w = torch.randn(136, 384, generator=torch.Generator().manual_seed(4)).bfloat16().to(dev)
    for layer in (OrbitLinear.from_weight(w, bias=None, config=config), OrbitLinear.from_weight(w, bias=None, config=config)):
        built = OrbitLinear(in_features=384, out_features=136, config=config, bias=None, packed_weight_indices=layer.packed_weight_indices,
                            row_norms=layer.row_norms)
        for (name, a), (other, b) in zip(layer.named_buffers(), built.named_buffers()):
            assert name == other and a.dtype == b.dtype and torch.equal(a, b), name
        torch.save(layer, io.BytesIO())
        layer._rotation_signs.neg_()      # (a layer's constants are its own: the next one is not made of them)


def test_a_layer_of_constants_in_one_buffer_can_be_saved(dev):
    import io

    from orbitquant_amd import OrbitLinear, OrbitQuantConfig, layers

    config = OrbitQuantConfig(weight_bits=4, activation_bits=4)
    made = OrbitLinear.from_weight(torch.randn(136, 384).bfloat16().to(dev), bias=None, config=config)
    constants = layers._on_device(made._constants(), made.row_norms.device)
    layer = OrbitLinear(in_features=384, out_features=136, config=config, bias=None, packed_weight_indices=made.packed_weight_indices,
                        row_norms=made.row_norms, constants=constants)
    file = io.BytesIO()
    torch.save(layer, file)
    file.seek(0)
    restored = torch.load(file, weights_only=False)
    x = torch.randn(5, 384).bfloat16().to(dev)
    assert torch.equal(restored(x), made(x)) and torch.equal(layer(x), made(x))
