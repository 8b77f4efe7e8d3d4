"""Arguments of the Python entry points, checked before anything reaches the
GPU: stand-ins with a tensor's attributes take the place of device tensors."""
import weakref
from collections import deque
from types import SimpleNamespace

import pytest
import torch

from rns_llm_amd import HipRNSBackend
from rns_llm_amd.backends.hip_backend import RNSWorkspace


def matrix(rows, cols, dtype=torch.int8):
    return SimpleNamespace(is_cuda=True, ndim=2, is_contiguous=lambda: True, dtype=dtype, device="cuda:0",
                           shape=(rows, cols), numel=lambda: rows * cols)


def backend():
    return object.__new__(HipRNSBackend)  # no GPU here


@pytest.mark.parametrize("held", [list, tuple, deque, lambda r: dict(enumerate(r)).values()],
                         ids=["list", "tuple", "deque", "values"])
def test_requests_in_any_sized_container(held):
    """Anything with a length that can be iterated: the checks go on to what
    is wrong with the requests themselves."""
    prepared = SimpleNamespace(k=64)
    with pytest.raises(ValueError, match="widths"):
        backend().matmul_prepared_fused_requests(held([matrix(1, 64), matrix(2, 32)]), prepared)
    with pytest.raises(ValueError, match="dtypes"):
        backend().matmul_prepared_fused_requests(held([matrix(1, 64), matrix(2, 64, torch.int16)]), prepared)


@pytest.mark.parametrize("moduli", [torch.tensor([255, 253, 251]), ["255", "253", "251"], (255.0, 253.0, 251.0),
                                    iter((255, 253, 251))], ids=["tensor", "text", "float", "iterator"])
def test_unprepared_moduli_become_integers(moduli):
    """The set keys the cache of device constants: a fresh tensor's elements
    would be a new entry on every call."""
    mods = backend()._wide_operands(matrix(4, 64), matrix(64, 8), moduli)
    assert mods == (255, 253, 251) and all(type(m) is int for m in mods)


def test_a_workspace_keeps_the_scratch_it_grew_from():
    """A captured graph holds the address of the scratch it ran with: a later
    call that needs a larger one must not let go of it."""
    workspace = RNSWorkspace(accumulators=torch.zeros(64, dtype=torch.uint8), output=torch.zeros((1, 1), dtype=torch.int64),
                             channels=4, m=1, n=1)
    kept = []
    for nbytes in (128, 100, 512):
        kept.append(weakref.ref(workspace.accumulators))
        assert HipRNSBackend._scratch(workspace, nbytes).numel() >= nbytes
    assert all(ref() is not None for ref in kept)
    assert workspace.accumulators.numel() == 512 and len({id(ref()) for ref in kept}) == 2  # 64, 128
    del workspace
    assert all(ref() is None for ref in kept)
