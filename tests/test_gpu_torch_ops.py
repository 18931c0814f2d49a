"""The custom ops' compiled implementation against the Python one it hands unusual calls to: the same results, the same
refusals."""

from __future__ import annotations

import subprocess
import sys
from pathlib import Path

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def layer():
    if not torch.cuda.is_available():
        pytest.skip("needs an AMD GPU")
    from orbitquant_amd import OrbitLinear, recipe

    torch.manual_seed(0)
    return OrbitLinear.from_linear(torch.nn.Linear(384, 136), config=recipe("w4a4")).cuda()


def arguments(layer, x, **changed):
    a = dict(x=x, permutation=layer._rotation_permutation, signs=layer._rotation_signs, act_centroids=layer._activation_codebook_centroids,
             act_boundaries=layer._activation_codebook_boundaries, packed_weight_indices=layer.packed_weight_indices, row_norms=layer.row_norms,
             weight_centroids=layer._weight_codebook_centroids, bias=layer.bias.to(x.dtype), block_size=layer.rotation.block_size,
             eps=layer.activation_eps, inv_sqrt_block=layer.rotation.normalization, activation_bits=4, weight_bits=4, out_features=136,
             input_map=None, output_map=None, rotate_plan=layer._rotation_plan)
    return {**a, **changed}


def both(a):
    op = torch.ops.orbitquant_amd
    return op.quantized_linear(**a), op.quantized_linear_general(**a)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("shape", [(1, 384), (384,), (3, 7, 384), (0, 384), (130, 384)])
def test_same_results(layer, shape, dtype):
    x = torch.randn(*shape, device="cuda").to(dtype)
    for changed in ({}, {"bias": None}, {"rotate_plan": None}, {"rotate_plan": layer._rotation_plan.clone()}, {"bias": layer.bias.double().float()},
                    {"row_norms": torch.stack([layer.row_norms, layer.row_norms], 1)[:, 0]}):
        got, want = both(arguments(layer, x, **changed))
        assert got.dtype == dtype and got.shape == want.shape == (*shape[:-1], 136) and torch.equal(got, want)


def test_views_and_tables(layer):
    from orbitquant_amd import ops

    x = torch.randn(64, 768, device="cuda").bfloat16()
    table = ops.activation_table(torch.nn.functional.gelu, torch.bfloat16, "cuda")
    for view in (x[:, ::2], x[:, 384:], x[::2, :384], x.t()[:384].t()):
        got, want = both(arguments(layer, view, input_map=table, output_map=table))
        assert torch.equal(got, want)


@pytest.mark.parametrize("wrong", [
    {"signs": torch.ones(383, dtype=torch.int8)}, {"permutation": torch.arange(384)}, {"row_norms": torch.ones(136)}, {"weight_bits": 3},
    {"packed_weight_indices": torch.zeros(10, dtype=torch.uint8)}, {"bias": torch.zeros(5)}, {"input_map": torch.zeros(65536, dtype=torch.float16)},
    {"rotate_plan": torch.zeros(16, dtype=torch.uint8)}])
def test_same_refusals(layer, wrong):
    a = arguments(layer, torch.randn(8, 384, device="cuda").bfloat16(), **{k: v.cuda() if isinstance(v, torch.Tensor) else v for k, v in wrong.items()})
    op = torch.ops.orbitquant_amd
    for call in (op.quantized_linear, op.quantized_linear_general):
        with pytest.raises(ValueError):
            call(**a)


def test_a_plan_of_another_shape_is_refused(layer):
    from orbitquant_amd import ops

    other = ops.rotate_plan(layer._rotation_permutation, layer._rotation_signs, layer._activation_codebook_boundaries, block_size=64, inv_sqrt_block=0.125)
    with pytest.raises(ValueError, match="built for"):
        torch.ops.orbitquant_amd.quantized_linear(**arguments(layer, torch.randn(8, 384, device="cuda").bfloat16(), rotate_plan=other))


@pytest.mark.parametrize("m", [1, 40, 200])
def test_group_equals_its_members(layer, m):
    from orbitquant_amd import OrbitLinear, OrbitLinearGroup, recipe

    torch.manual_seed(1)
    linears = [layer] + [OrbitLinear.from_linear(torch.nn.Linear(384, n, bias=False), config=recipe("w4a4")).cuda() for n in (64, 8)]
    x = torch.randn(2, m, 384, device="cuda").bfloat16()
    for view in (x, x.transpose(0, 1)):
        for got, l in zip(OrbitLinearGroup(*linears)(view), linears):
            assert torch.equal(got, l(view))


def test_under_fake_tensors(layer):
    from torch._subclasses.fake_tensor import FakeTensorMode

    with FakeTensorMode(allow_non_fake_inputs=True) as mode:
        y = layer(mode.from_tensor(torch.empty(3, 384, dtype=torch.bfloat16, device="meta")).to("cuda"))
        assert y.shape == (3, 136) and y.dtype == torch.bfloat16


def test_constants_made_under_capture_are_not_one_buffer(monkeypatch):
    """A captured copy would read the pinned buffer again at each replay, when it holds something else: there the copies
    are the blocking ones, which a capture refuses."""
    from orbitquant_amd import layers

    tensors = {"a": torch.arange(5, dtype=torch.int32), "b": torch.ones(3)}
    device = torch.device("cuda:0")

    def shared():
        there = layers._on_device(tensors, device)
        assert all(torch.equal(there[name].cpu(), t) for name, t in tensors.items())
        return there["a"].untyped_storage().data_ptr() == there["b"].untyped_storage().data_ptr()

    assert shared()
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
    assert not shared()


def test_layers_are_made_and_moved_under_a_default_device():
    """`torch.device("cuda")` as a context: what torch makes without a device is on the GPU, pinned memory is not."""
    from orbitquant_amd import OrbitLinear, recipe

    config = recipe("w4a4")
    host = OrbitLinear.from_linear(torch.nn.Linear(384, 136), config=config)
    weight = torch.randn(136, 384, device="cuda").bfloat16()
    want = OrbitLinear.from_weight(weight, bias=None, config=config)   # (and the caches are filled)
    x = torch.randn(3, 384, device="cuda").bfloat16()
    with torch.device("cuda"):
        got = OrbitLinear.from_weight(weight, bias=None, config=config)
        assert torch.equal(got(x), want(x)) and torch.equal(got.to(torch.bfloat16).cuda()(x), want(x))
        assert host.cuda()(x).shape == (3, 136)


def test_without_the_compiled_module():
    """Forwards of every kind are those of the general implementations, where they raised (another process: the ops are
    registered when the package is imported)."""
    program = """
import sys
sys.modules["orbitquant_amd._torch_ops"] = None      # importing it raises ImportError
import torch
from orbitquant_amd import OrbitLinear, OrbitLinearGroup, RTNInt4Linear, recipe
torch.manual_seed(0)
linears = [OrbitLinear.from_linear(torch.nn.Linear(384, n), config=recipe("w4a4")).cuda() for n in (136, 64)]
adaln = RTNInt4Linear.from_linear(torch.nn.Linear(384, 136), config=recipe("w4a4")).cuda()
for m in (1, 40):
    x = torch.randn(m, 384, device="cuda").bfloat16()
    alone = [l(x) for l in linears]
    assert all(torch.equal(a, b) for a, b in zip(OrbitLinearGroup(*linears)(x), alone)) and alone[0].shape == (m, 136)
    general = torch.ops.orbitquant_amd.adaln_int4_linear_general
    assert torch.equal(adaln(x), general(x, adaln.packed_weight, adaln.scales, adaln.bias, 136, 384, adaln.group_size))
"""
    done = subprocess.run([sys.executable, "-c", program], cwd=Path(__file__).resolve().parent.parent, capture_output=True, text=True, timeout=100)
    assert done.returncode == 0, done.stderr
    assert "RuntimeWarning" in done.stderr


def test_group_entries_of_other_forms(layer):
    """What is no tuple of six tensors and plain numbers is the Python implementation's to take or to refuse."""
    import numpy as np

    from orbitquant_amd import ops

    x = torch.randn(5, 384, device="cuda").bfloat16()
    entry = (layer.packed_weight_indices, layer.row_norms, layer._weight_codebook_centroids, 4, 136, None)

    def call(*weights):
        return ops.quantized_linear_group(
            x, layer._rotation_permutation, layer._rotation_signs, layer._activation_codebook_boundaries, layer._activation_codebook_centroids,
            weights, block_size=layer.rotation.block_size, eps=layer.activation_eps, inv_sqrt_block=layer.rotation.normalization,
            activation_bits=4, plan=layer._rotation_plan)

    want, = call(entry)
    for other in (list(entry), (*entry[:3], np.int64(4), np.int32(136), None)):
        got, same = call(other, entry)
        assert torch.equal(got, want) and torch.equal(same, want)
    for wrong in ((*entry, None), entry[:5]):
        with pytest.raises(ValueError, match="unpack"):
            call(entry, wrong)
    with pytest.raises(AttributeError):
        call((None, *entry[1:]))


@pytest.mark.parametrize("how", ["from_weight", "moved", "cast"])
def test_layers_are_saved_whole(how):
    """torch.save takes a module, or its buffers, only where no storage is viewed as more than one type."""
    import copy
    import io

    from orbitquant_amd import OrbitLinear, recipe

    torch.manual_seed(0)
    weight = torch.randn(136, 384)
    layer = OrbitLinear.from_weight(weight.cuda() if how == "from_weight" else weight, bias=None, config=recipe("w4a6")).cuda()
    if how == "cast":
        layer = layer.to(torch.bfloat16)
    x = torch.randn(5, 384, device="cuda").bfloat16()
    for saved in (layer, dict(layer.named_buffers()), layer.state_dict()):
        file = io.BytesIO()
        torch.save(saved, file)
        file.seek(0)
        restored = torch.load(file, weights_only=False)
        if saved is layer:
            assert torch.equal(restored(x), layer(x))
        else:
            assert all(torch.equal(t, saved[name]) and t.dtype == saved[name].dtype for name, t in restored.items())
    assert torch.equal(copy.deepcopy(layer)(x), layer(x))
