"""A layer that was built or moved on one stream is complete for every other stream when the call returns, as a torch
module is: nothing of it may still be on its way (its permutation is a table of gather indices)."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

K, N = 4096, 320


@pytest.fixture(scope="module")
def source():
    if not torch.cuda.is_available():
        pytest.skip("needs an AMD GPU")
    torch.manual_seed(0)
    return torch.nn.Linear(K, N)


def made(how: str, source):
    from orbitquant_amd import OrbitLinear, recipe

    config = recipe("w4a4")
    if how == "converted":
        return OrbitLinear.from_weight(source.weight.detach().cuda().bfloat16(), bias=None, config=config)
    if how == "converted on the host":   # (a type the GPU's quantizer does not take)
        return OrbitLinear.from_weight(source.weight.detach().cuda().double(), bias=None, config=config)
    if how == "empty":
        return OrbitLinear.empty_from_linear(torch.nn.Linear(K, N, device="cuda"), config=config)
    if how == "moved":
        return OrbitLinear.from_linear(source, config=config).cuda()
    return OrbitLinear.from_linear(source.cuda(), config=config).to(torch.bfloat16)


@pytest.mark.parametrize("how", ["converted", "converted on the host", "empty", "moved", "cast"])
def test_a_layer_is_complete_when_the_call_returns(source, how, monkeypatch):
    from orbitquant_amd import layers

    work = torch.randn(8192, 8192, device="cuda", dtype=torch.bfloat16)
    on_device = layers._on_device

    def behind_other_work(tensors, device):
        for _ in range(20):   # some 20 ms
            work @ work
        return on_device(tensors, device)

    made(how, source)         # (the caches of rotations and codebooks, and of pinned memory, are filled)
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    monkeypatch.setattr(layers, "_on_device", behind_other_work)
    with torch.cuda.stream(side):
        layer = made(how, source)
        assert side.query()
    monkeypatch.undo()
    torch.cuda.current_stream().wait_stream(side)
    for x in (torch.randn(1, K, device="cuda").bfloat16(), torch.randn(40, K, device="cuda").bfloat16()):
        here = layer(x)
        other = torch.cuda.Stream()
        other.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(other):
            there = layer(x)
        torch.cuda.current_stream().wait_stream(other)
        assert torch.equal(here, there)


def test_a_capture_refuses_to_make_or_move_a_layer(source):
    """Its constants come from host memory, which a captured copy would read again at each replay.  The capture itself
    goes on, and replays what else was given to it."""
    from orbitquant_amd import OrbitLinear, recipe

    layer = made("converted", source)
    config = recipe("w4a4")
    weight, moved = source.weight.detach().cuda(), made("converted", source)
    x = torch.randn(4, K, device="cuda").bfloat16()
    want = layer(x)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        with pytest.raises(RuntimeError, match="captur"):
            OrbitLinear.from_weight(weight, bias=None, config=config)
        with pytest.raises(RuntimeError, match="captur"):
            moved.to(torch.bfloat16)
        y = layer(x)
    for _ in range(3):
        y.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want) and torch.equal(made("converted", source)(x), want)


def test_a_capture_refuses_the_first_conversion_of_a_width(source):
    """Nothing of its constants has been made yet, and nothing may be pinned there: refused like any other, and the capture goes on."""
    from orbitquant_amd import OrbitLinear, layers, recipe

    layer, config = made("converted", source), recipe("w4a4")
    x, weight = torch.randn(4, K, device="cuda").bfloat16(), torch.randn(40, 1352, device="cuda").bfloat16()
    want = layer(x)
    torch.cuda.synchronize()
    layers._conversion_constants.cache_clear()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        with pytest.raises(RuntimeError, match="captur"):
            OrbitLinear.from_weight(weight, bias=None, config=config)
        y = layer(x)
    for _ in range(3):
        y.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want)
    assert OrbitLinear.from_weight(weight, bias=None, config=config)(torch.randn(2, 1352, device="cuda")).shape == (2, 40)
