"""Packed weights by byte products (int8 and int16 activations): the decode
kernel over fragments, waves and ragged rows, the tiles over ragged edges, K
steps that fill no trip and K splits, float outputs, and sets too small for
the product, against the exact product taken to the set's centered range."""
import ctypes
from math import prod

import numpy as np
import pytest
import torch

from oracle import rns_oracle as ro
from rns_llm_amd import _native

pytestmark = pytest.mark.gpu

DENSE6 = (255, 253, 251, 247, 241, 239)


def operands(m, k, n, dtype, seed):
    gen = torch.Generator().manual_seed(seed)
    lim = 128 if dtype == torch.int8 else 32768
    a = torch.randint(-lim, lim, (m, k), generator=gen, dtype=torch.int32).to(dtype)
    w = torch.randint(-32768, 32768, (n, k), generator=gen, dtype=torch.int32).to(torch.int16)
    # the largest sums of every byte product, both signs
    a[0], w[0] = -lim, -32768
    a[m // 2, ::2], w[n // 2] = lim - 1, 32767
    return a, w, torch.from_numpy(ro.exact_matmul(a.numpy(), w.t().numpy()))


def run(backend, a, w, moduli, plan, **kw):
    prepared = backend.prepare_weight_packed_nk(w.cuda(), moduli)
    ws = backend.create_workspace(device=torch.device("cuda"), channels=len(moduli), m=a.shape[0], n=w.shape[0])
    first = backend.matmul_prepared_fused(a.cuda(), prepared, workspace=ws, plan=plan, **kw).clone()
    # a second call on the same workspace (counters left at zero)
    assert torch.equal(first, backend.matmul_prepared_fused(a.cuda(), prepared, workspace=ws, plan=plan, **kw))
    return first.cpu()


# rows of 16-byte chunks that end inside a step, that are copied to padded
# ones (777, 100 int8), and K below and above a round of chunks
@pytest.mark.parametrize("k,n", [(1000, 77), (777, 16), (100, 33), (64, 15), (2176, 40)])
@pytest.mark.parametrize("m", [1, 7, 8, 9, 16, 17, 32, 33, 64])
@pytest.mark.parametrize("dtype", [torch.int8, torch.int16])
def test_decode_rows(backend, m, k, n, dtype):
    per = 16 if dtype == torch.int8 else 8
    if m > 4 * per:
        pytest.skip("more tokens than four fragments hold")
    a, w, want = operands(m, k, n, dtype, m + k)
    frags = 1 if m <= per else 2 if m <= 2 * per else 4
    for ks in (1, 3, 4):
        assert torch.equal(run(backend, a, w, DENSE6, (9, frags, 1, ks)), want)
    assert torch.equal(run(backend, a, w, DENSE6, None), want)


# one tile and several with ragged edges; 1, 3, 5, 8 and 18 K steps
@pytest.mark.parametrize("m,k,n", [(1, 64, 1), (130, 192, 200), (65, 300, 97), (257, 512, 385), (128, 1100, 192)])
@pytest.mark.parametrize("mb", [4, 8])
@pytest.mark.parametrize("dtype", [torch.int8, torch.int16])
def test_tiles(backend, m, k, n, mb, dtype):
    a, w, want = operands(m, k, n, dtype, m + k + mb)
    assert torch.equal(run(backend, a, w, DENSE6, (10, mb, 1, 0)), want)


# the longest K whose int32 sums hold: every middle product of the weight's and
# the activations' bytes is 2^14, twice per K index, 2145386496 of 2^31 - 1
@pytest.mark.parametrize("plan", [None, (9, 4, 1, 1), (9, 4, 1, 4), (10, 4, 1, 0), (10, 8, 1, 0), (10, 8, 1, 0, 4)], ids=str)
@pytest.mark.parametrize("dtype", [torch.int8, torch.int16])
def test_longest_k(backend, plan, dtype):
    lim = 128 if dtype == torch.int8 else 32768
    for k in (65472, 65471, 65473):
        a, w = (torch.empty((3, k), dtype=t) for t in (dtype, torch.int16))
        for x, top in ((a, lim), (w, 32768)):
            x[0], x[1], x[2] = -top, top - 1, torch.arange(k) % (2 * top) - top
        want = torch.from_numpy(ro.exact_matmul(a.numpy(), w.t().numpy()))
        if k == 65473 and plan is not None:
            with pytest.raises(ValueError, match="65472"):
                run(backend, a, w, DENSE6, plan)
        else:
            assert torch.equal(run(backend, a, w, DENSE6, plan), want)


@pytest.mark.parametrize("splits,tail", [(2, 0), (3, 0), (8, 0), (2, 1)])
@pytest.mark.parametrize("mb", [4, 8])
@pytest.mark.parametrize("dtype", [torch.int8, torch.int16])
def test_tiles_split_over_k(backend, mb, splits, tail, dtype):
    m, k, n = 70, 2100, 200
    a, w, want = operands(m, k, n, dtype, splits)
    assert torch.equal(run(backend, a, w, DENSE6, (10, mb, 1, 0, splits, tail)), want)


@pytest.mark.parametrize("plan", [None, (10, 4, 1, 0), (10, 8, 1, 0, 2)], ids=str)
@pytest.mark.parametrize("out_dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("dtype", [torch.int8, torch.int16])
def test_float_outputs(backend, plan, out_dtype, dtype):
    m, k, n = 20, 1024, 130
    a, w, want = operands(m, k, n, dtype, 5)
    gen = torch.Generator().manual_seed(9)
    a_scale, w_scale = torch.tensor([3e-5]), torch.rand((n,), generator=gen) * 1e-4
    bias = torch.randn((n,), generator=gen)
    out = torch.empty((m, n), dtype=out_dtype, device="cuda")
    got = run(backend, a, w, DENSE6, plan, out=out, a_scale=a_scale.cuda(), w_scale=w_scale.cuda(), bias=bias.cuda())
    ref = ((want.float() * a_scale.view(1, 1)) * w_scale.unsqueeze(0) + bias).to(out_dtype)
    bits = torch.int32 if out_dtype == torch.float32 else torch.int16
    assert torch.equal(got.view(bits), ref.view(bits))


@pytest.mark.parametrize("moduli", [(255, 253, 251, 247), (2, 3), (254, 253, 251), DENSE6[:5]], ids=str)
@pytest.mark.parametrize("m", [5, 40, 200])
@pytest.mark.parametrize("dtype", [torch.int8, torch.int16])
def test_sets_too_small_for_the_product(backend, moduli, m, dtype):
    p = prod(moduli)
    a, w, want = operands(m, 512, 70, dtype, m)
    r = np.mod(want.numpy(), p)
    r = np.where(r > p >> 1, r - p, r)
    assert torch.equal(run(backend, a, w, moduli, None), torch.from_numpy(r))
    assert torch.equal(run(backend, a, w, moduli, (10, 8, 1, 0, 2)), torch.from_numpy(r))


# both sides of where a few int16 rows take the channel rows: rows that are
# copied (K no multiple of 8) in one, two and four blocks; 17 to 32 rows from
# K = 1400 or 2000; one column past one round of workgroups
@pytest.mark.parametrize("m,k,n", [(4, 1001, 40), (5, 1001, 40), (12, 1001, 40), (4, 1000, 40), (12, 1000, 40), (17, 1396, 40),
                                   (32, 1404, 40), (32, 1992, 40), (17, 2000, 40), (17, 2000, 4096), (17, 2000, 4097)])
@pytest.mark.parametrize("channels", [3, 4, 6])
def test_rows_on_both_sides_of_the_channel_rows(backend, m, k, n, channels):
    moduli = DENSE6[:channels]
    p = prod(moduli)
    a, w, want = operands(m, k, n, torch.int16, m + k)
    r = torch.remainder(want, p)
    assert torch.equal(run(backend, a, w, moduli, None), torch.where(r > p >> 1, r - p, r))


@pytest.mark.parametrize("m", [3, 40, 200])
def test_adaptive_prefix(backend, m):
    a, w, want = operands(m, 512, 70, torch.int16, m)
    for b_max in (127, 32767):
        w8 = w.clamp(-b_max, b_max)
        adaptive = backend.prepare_weight_adaptive_nk(w8.cuda(), DENSE6, min_channels=3, packed=True)
        out, meta = backend.matmul_prepared_adaptive_fused(a.cuda(), adaptive, return_metadata=True)
        c, bound, cap = ro.adaptive_select(a.numpy(), b_max, DENSE6, min_channels=3)
        assert dict(meta) == {"channels": c, "bound": bound, "capacity": cap}
        assert torch.equal(out.cpu(), torch.from_numpy(ro.exact_matmul(a.numpy(), w8.t().numpy())))


def test_replays_of_a_captured_split(backend):
    """A K split under capture: each replay equals the eager result, with
    eager calls on the same workspace between them."""
    a, w, want = operands(70, 2048, 200, torch.int16, 3)
    prepared = backend.prepare_weight_packed_nk(w.cuda(), DENSE6)
    ws = backend.create_workspace(device=torch.device("cuda"), channels=6, m=70, n=200)
    x, plan = a.cuda(), (10, 4, 1, 0, 4)
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        backend.matmul_prepared_fused(x, prepared, workspace=ws, plan=plan)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        backend.matmul_prepared_fused(x, prepared, workspace=ws, plan=plan)
    for _ in range(3):
        ws.output.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(ws.output.cpu(), want)
        assert torch.equal(backend.matmul_prepared_fused(x, prepared, workspace=ws, plan=plan).cpu(), want)


@pytest.mark.parametrize("m", [70, 130])
@pytest.mark.parametrize("dtype", [torch.int8, torch.int16])
def test_split_without_an_exchange_area(backend, m, dtype):
    """A workspace with room for the planes alone: the same product, unsplit."""
    k, n = 4096, 200
    a, w, want = operands(m, k, n, dtype, m)
    prepared = backend.prepare_weight_packed_nk(w.cuda(), DENSE6)
    lib, mods = _native.lib(), _native.make_moduli(DENSE6)
    whole = _native.Plan(10, 4, 1, 0, 1, 0)
    small = lib.rnsmx_packed_workspace_bytes(m, k, n, 6, ctypes.byref(whole))
    assert small < lib.rnsmx_packed_workspace_bytes(m, k, n, 6, None)
    x = a.cuda()
    workspace = torch.zeros((small,), dtype=torch.uint8, device="cuda")
    out = torch.empty((m, n), dtype=torch.int64, device="cuda")
    _native.check(lib.rnsmx_matmul_packed_fused(
        x.data_ptr(), _native.dtype_code(dtype), m, k, n, prepared.packed.data_ptr(), ctypes.byref(mods), None, 0, None,
        None, None, workspace.data_ptr(), small, out.data_ptr(), torch.cuda.current_stream().cuda_stream))
    assert torch.equal(out.cpu(), want)


@pytest.mark.parametrize("m", [1, 8, 20, 70])
def test_outputs_over_the_activations(backend, m):
    """Float outputs written where the int16 activations lie, and int64 ones
    that begin inside them: as into another buffer."""
    k = n = 512
    a, w, want = operands(m, k, n, torch.int16, m)
    prepared = backend.prepare_weight_packed_nk(w.cuda(), DENSE6)
    scales = dict(a_scale=torch.tensor([3e-5], device="cuda"), w_scale=torch.full((n,), 1e-4, device="cuda"))
    out = torch.empty((m, n), dtype=torch.float16, device="cuda")
    backend.matmul_prepared_fused(a.cuda(), prepared, out=out, **scales)
    buffer = torch.empty((5 * m * k,), dtype=torch.int16, device="cuda")
    for _ in range(5):
        x = buffer[:m * k].view(m, k).copy_(a)
        got = backend.matmul_prepared_fused(x, prepared, out=x.view(torch.float16), **scales)
        assert torch.equal(got, out)
        x.copy_(a)
        ws = backend.create_workspace(device=x.device, channels=6, m=m, n=n, k=k)
        ws.output = buffer[m * k - 64:m * k - 64 + 4 * m * n].view(torch.int64).view(m, n)
        assert torch.equal(backend.matmul_prepared_fused(x, prepared, workspace=ws).cpu(), want)


def test_plans_refused(backend):
    a, w, _ = operands(20, 64, 16, torch.int32, 1)
    prepared = backend.prepare_weight_packed_nk(w.cuda(), DENSE6)
    for dtype, plan in ((torch.int32, (10, 8, 1, 0)), (torch.int32, (9, 4, 1, 1)), (torch.int16, (9, 2, 1, 1)),
                        (torch.int16, (9, 4, 1, 5)), (torch.int16, (10, 3, 1, 0)), (torch.int16, (9, 4, 1, 1, 2))):
        with pytest.raises(ValueError):
            backend.matmul_prepared_fused(a.clamp(-9, 9).to(dtype).cuda(), prepared, plan=plan)
