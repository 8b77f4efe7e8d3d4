"""Residue planes by channel units: one channel of a tile per workgroup, the
last one to finish reconstructs.  Integer outputs are exact, so every check is
an equality; float outputs are compared with the kernel that holds all channels
in a wave, whose epilogue is the same."""
from __future__ import annotations

import pytest
import torch

from oracle import rns_oracle as ro
from rns_llm_amd import HipRNSBackend

pytestmark = pytest.mark.gpu

MODULI = (255, 253, 251, 247, 241, 239)
SMALL, LARGE = (11, 2, 1, 0), (11, 4, 2, 0)  # 64 x 64 and 128 x 128 tiles
MFMA = (2, 2, 1, 4)


def operands(m, n, k, channels, dtype=torch.int16):
    gen = torch.Generator().manual_seed(m * 7 + n * 3 + k + channels)
    most = 127 if dtype == torch.int8 else 32767 if channels == 6 else 2047
    a = torch.randint(-most, most + 1, (m, k), generator=gen)
    w = torch.randint(-most, most + 1, (n, k), generator=gen)
    # sums below 2^53: float64 products are exact
    exact = (a.double() @ w.double().t()).to(torch.int64)
    return a.to(dtype).cuda(), w.to(torch.int16).cuda(), exact


@pytest.mark.parametrize("plan", [None, SMALL, LARGE])
@pytest.mark.parametrize("m, n, k, channels", [
    (17, 64, 64, 5),       # one K step; one tile, few rows
    (64, 64, 128, 6),      # whole tiles of the small form, one pair of steps
    (65, 65, 190, 6),      # one past a tile; three steps: half a pair at the end
    (77, 1531, 1000, 5),   # ragged everywhere, odd output rows: no paired stores
    (128, 256, 320, 6),    # whole tiles of both forms, five steps
    (129, 130, 257, 5),    # one past the large tile; the last step holds one value
    (300, 514, 576, 6),
])
def test_channel_units_are_exact(m, n, k, channels, plan):
    a, w, exact = operands(m, n, k, channels)
    backend = HipRNSBackend()
    prepared = backend.prepare_weight_nk(w, MODULI[:channels])
    workspace = backend.create_workspace(device=a.device, channels=channels, m=m, n=n, k=k)
    for _ in range(2):  # the counters are left as they were found
        out = backend.matmul_prepared_fused(a, prepared, workspace=workspace, plan=plan)
        assert torch.equal(out.cpu(), exact)


@pytest.mark.parametrize("plan", [SMALL, LARGE])
@pytest.mark.parametrize("out_dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("m, n", [(128, 256), (77, 131)])
def test_channel_units_float_outputs(m, n, out_dtype, plan):
    a, w, _ = operands(m, n, 448, 6)
    backend = HipRNSBackend()
    prepared = backend.prepare_weight_nk(w, MODULI)
    gen = torch.Generator().manual_seed(3)
    epilogue = dict(a_scale=torch.tensor([3e-5], device="cuda"),
                    w_scale=(torch.rand((n,), generator=gen) * 1e-4).cuda(),
                    bias=torch.randn((n,), generator=gen).cuda())
    want, got = (torch.empty((m, n), dtype=out_dtype, device="cuda") for _ in range(2))
    backend.matmul_prepared_fused(a, prepared, plan=MFMA, out=want, **epilogue)
    backend.matmul_prepared_fused(a, prepared, plan=plan, out=got, **epilogue)
    assert torch.equal(got, want)


@pytest.mark.parametrize("plan", [None, SMALL, LARGE])
@pytest.mark.parametrize("m, n, k", [(96, 640, 1024), (200, 515, 513)])
def test_channel_units_adaptive_prefix(m, n, k, plan):
    """Units past the prefix the activations need end at once.  Prefixes of
    different lengths alternate on one workspace, so a ticket that one call
    left would end the next one early."""
    gen = torch.Generator().manual_seed(k)
    w = torch.randint(-32767, 32768, (n, k), generator=gen)
    w[0, 0] = 32767
    backend = HipRNSBackend()
    prepared = backend.prepare_weight_adaptive_nk(w.to(torch.int16).cuda(), MODULI, min_channels=2)
    workspaces = {6: backend.create_workspace(device=torch.device("cuda"), channels=6, m=m, n=n, k=k)}
    seen = []
    for most in (1, 32767, 2000, 1, 2000, 32767):
        a = torch.randint(-most, most + 1, (m, k), generator=gen)
        out, meta = backend.matmul_prepared_adaptive_fused(a.to(torch.int16).cuda(), prepared, return_metadata=True,
                                                           workspace_by_channels=workspaces, plan=plan)
        channels, bound, capacity = ro.adaptive_select(a.numpy(), 32767, MODULI, min_channels=2)
        assert dict(meta) == {"channels": channels, "bound": bound, "capacity": capacity}
        assert torch.equal(out.cpu(), (a.double() @ w.double().t()).to(torch.int64))
        seen.append(channels)
    assert seen[:3] == ([4, 6, 5] if k == 1024 else [4, 5, 5])


def test_channel_units_replayed():
    a, w, exact = operands(160, 1536, 1024, 6)
    backend = HipRNSBackend()
    prepared = backend.prepare_weight_nk(w, MODULI)
    workspace = backend.create_workspace(device=a.device, channels=6, m=160, n=1536, k=1024)
    backend.matmul_prepared_fused(a, prepared, workspace=workspace)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = backend.matmul_prepared_fused(a, prepared, workspace=workspace)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out.cpu(), exact)


def test_channel_units_without_an_exchange_area():
    """A workspace with room for the planes alone: the same product by a kernel
    that needs no exchange."""
    import ctypes

    from rns_llm_amd import _native

    m, n, k = 160, 1536, 1024
    a, w, exact = operands(m, n, k, 6)
    backend = HipRNSBackend()
    prepared = backend.prepare_weight_nk(w, MODULI)
    lib = _native.lib()
    mfma = _native.Plan(2, 2, 1, 4, 1, 0)
    small = lib.rnsmx_prepared_workspace_bytes(m, k, n, 6, ctypes.byref(mfma))
    assert small < lib.rnsmx_prepared_workspace_bytes(m, k, n, 6, None)
    workspace = torch.zeros((small,), dtype=torch.uint8, device="cuda")
    out = torch.empty((m, n), dtype=torch.int64, device="cuda")
    mods = _native.make_moduli(MODULI)
    _native.check(lib.rnsmx_matmul_prepared_fused(
        a.data_ptr(), _native.INT16, m, k, n, prepared.packed.data_ptr(), ctypes.byref(mods), None, 0, None, None,
        None, workspace.data_ptr(), small, out.data_ptr(), torch.cuda.current_stream().cuda_stream))
    assert torch.equal(out.cpu(), exact)
