"""What a call does when there is no memory for its workspace (CPU: the allocation is made to fail)."""

from __future__ import annotations

import warnings

import pytest
import torch

from orbitquant_amd import ops


@pytest.fixture
def memory(monkeypatch):
    """`memory(limit)`: allocations of more than `limit` bytes fail from now on; the sizes asked for."""
    real, asked = torch.empty, []

    def limit_to(limit):
        def empty(size, *args, **kwargs):
            asked.append(size)
            if size > limit:
                raise torch.OutOfMemoryError("no memory")
            return real(size, *args, **kwargs)

        monkeypatch.setattr(ops.torch, "empty", empty)
        return asked

    return limit_to


LIKE = torch.zeros(1)


def test_a_workspace_that_fits(memory):
    asked = memory(4096)
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        address, size, owner = ops._workspace(4096, LIKE, lambda: pytest.fail("nothing smaller is looked for"))
    assert (address, size) == (owner.data_ptr(), 4096) and asked == [4096]
    assert ops._workspace(0, LIKE) == (None, 0, None)


def test_running_out_is_an_error_where_the_call_has_nothing_smaller(memory):
    memory(100)
    for smaller in ((), (4096,)):
        with pytest.raises(torch.OutOfMemoryError):
            ops._workspace(4096, LIKE, lambda: smaller)


@pytest.mark.parametrize("limit,sizes,got", [(2000, (1000, 0), 1000), (100, (1000, 0), 0), (100, (0,), 0)])
def test_a_smaller_workspace_is_taken_and_said(memory, limit, sizes, got):
    memory(limit)
    with pytest.warns(RuntimeWarning, match="workspace of 4096 bytes"):
        address, size, owner = ops._workspace(4096, LIKE, lambda: sizes)
    assert size == got and (address is None) == (owner is None) == (got == 0)


def test_running_out_of_the_last_size_raises(memory):
    memory(100)
    with pytest.warns(RuntimeWarning), pytest.raises(torch.OutOfMemoryError):
        ops._workspace(4096, LIKE, lambda: (1000,))
