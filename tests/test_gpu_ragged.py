"""Products of plain integers where rows are not 16-byte aligned: int8
activations copied to padded rows (prepared weights, fixed and adaptive, next
to a plan that asks for residue planes), and the unprepared product, whose B
is encoded from [K, N] straight into fragments."""
import pytest
import torch

from oracle import rns_oracle as ro

pytestmark = pytest.mark.gpu

DENSE4 = (255, 253, 251, 247)
DENSE6 = DENSE4 + (241, 239)


def ints(shape, lim, dtype, seed):
    gen = torch.Generator().manual_seed(seed)
    x = torch.randint(-lim - 1, lim + 1, shape, generator=gen, dtype=torch.int64)
    x[0], x[-1, ::2] = -lim - 1, lim
    return x.to(dtype)


def exact(a, b):
    return torch.from_numpy(ro.exact_matmul(a.numpy(), b.numpy()))


@pytest.mark.parametrize("k", [100, 777, 1001, 2055])
@pytest.mark.parametrize("m", [1, 4, 5, 96, 300])
def test_int8_rows_padded(backend, m, k):
    n = 200
    a, b = ints((m, k), 127, torch.int8, m + k), ints((k, n), 126, torch.int8, k)
    want = exact(a, b)
    prepared = backend.prepare_weight(b.cuda(), DENSE4)
    ws = backend.create_workspace(device=torch.device("cuda"), channels=4, m=m, n=n, k=k)
    for _ in range(2):
        assert torch.equal(backend.matmul_prepared_fused(a.cuda(), prepared, workspace=ws).cpu(), want)
    # a forced plan on such rows keeps the residue planes
    assert torch.equal(backend.matmul_prepared_fused(a.cuda(), prepared, plan=(8, 0, 0, 0) if (k + 63) // 64 % 4 == 0
                                                     else (2, 2, 1, 0)).cpu(), want)
    adaptive = backend.prepare_weight_adaptive(b.cuda(), DENSE4, min_channels=2)
    out, meta = backend.matmul_prepared_adaptive_fused(a.cuda(), adaptive, return_metadata=True)
    c, bound, cap = ro.adaptive_select(a.numpy(), int(b.to(torch.int32).abs().max()), DENSE4, min_channels=2)
    assert dict(meta) == {"channels": c, "bound": bound, "capacity": cap}
    assert torch.equal(out.cpu(), want)


# one fragment, ragged fragments and rows, a K split, more rows than columns
@pytest.mark.parametrize("m,k,n", [(1, 1, 1), (3, 65, 17), (40, 130, 63), (5, 2100, 70), (257, 64, 129), (64, 4096, 96)])
@pytest.mark.parametrize("dtype", [torch.int8, torch.int16, torch.int32])
def test_unprepared(backend, m, k, n, dtype):
    lim = 127 if dtype == torch.int8 else 32767
    if dtype == torch.int32:
        lim = 90000  # past int16, within the 6-channel set
    a, b = ints((m, k), lim, dtype, m), ints((k, n), lim, dtype, n)
    want = exact(a, b)
    backend.reset_stats()
    got = backend.matmul_wide(a.cuda(), b.cuda(), DENSE6)
    assert backend.stats_snapshot() == {"encode_centered_calls": 2, "encode_centered_values": a.numel() + b.numel(),
                                        "fused_gemm_calls": 1, "fused_gemm_channels_6": 1}
    assert torch.equal(got.cpu(), want)
    ws = backend.create_workspace(device=torch.device("cuda"), channels=6, m=m, n=n)
    for _ in range(2):
        out = backend.matmul_wide_fused(a.cuda(), b.cuda(), DENSE6, lut_channels=2, workspace=ws)
        assert out.data_ptr() == ws.output.data_ptr() and torch.equal(out.cpu(), want)
    # the residues, through the planes
    res = backend.matmul_wide(a.cuda(), b.cuda(), DENSE6, decode=False)
    assert torch.equal(backend.decode_garner(res.contiguous(), DENSE6).cpu(), want)


@pytest.mark.parametrize("moduli", [(2, 3), (16, 15, 7, 11), (254, 253)], ids=str)
@pytest.mark.parametrize("dtype", [torch.int8, torch.int16])
def test_unprepared_residues_of_every_value(backend, moduli, dtype):
    """B holds every int8 value, and int16 values up to both ends, against a
    row of ones and one of zeros: the product is the value taken to the
    centered range of the set."""
    values = torch.arange(-128, 128) if dtype == torch.int8 else torch.arange(-32768, 32768, 7)
    a = torch.ones((2, 1), dtype=dtype)
    a[1] = 0
    b = values.to(dtype).view(1, -1)
    p = 1
    for m in moduli:
        p *= m
    r = values % p
    want = torch.where(r > p // 2, r - p, r)
    got = backend.matmul_wide(a.cuda(), b.cuda(), moduli).cpu()
    assert torch.equal(got[0], want) and not got[1].any()


def test_unprepared_refusals(backend):
    a, b = ints((4, 64), 9, torch.int8, 1).cuda(), ints((64, 8), 9, torch.int8, 2).cuda()
    for bad in (lambda: backend.matmul_wide(a, b.to(torch.int16), DENSE4), lambda: backend.matmul_wide(a, b[:32].contiguous(), DENSE4),
                lambda: backend.matmul_wide(a, b.t(), DENSE4), lambda: backend.matmul_wide(a, b, (255, 51)),
                lambda: backend.matmul_wide(a, b, (255,)), lambda: backend.matmul_wide_fused(a, b, DENSE4, lut_channels=3),
                lambda: backend.matmul_wide(a.float(), b.float(), DENSE4)):
        with pytest.raises(ValueError):
            bad()
    # an empty batch
    assert backend.matmul_wide(a[:0], b, DENSE4).shape == (0, 8)


@pytest.mark.parametrize("dtype", [torch.int8, torch.int16])
@pytest.mark.parametrize("where", ["output", "accumulators"])
@pytest.mark.parametrize("operand", ["a", "b"])
def test_operands_inside_the_workspace(backend, operand, where, dtype):
    """An operand that lies where the outputs or the scratch will be."""
    m, k, n = 64, 128, 96
    a, b = ints((m, k), 126, dtype, 3), ints((k, n), 126, dtype, 4)
    ws = backend.create_workspace(device=torch.device("cuda"), channels=6, m=m, n=n)
    want = exact(a, b)
    # grown to this shape's size, so that the next call keeps the buffer
    assert torch.equal(backend.matmul_wide_fused(a.cuda(), b.cuda(), DENSE6, workspace=ws).cpu(), want)
    x, y = a.cuda(), b.cuda()
    for _ in range(5):
        at = getattr(ws, where).view(-1).view(torch.int8)
        at = at[at.numel() // 2 // 16 * 16:] if where == "accumulators" else at
        inside = at[:(x if operand == "a" else y).nbytes].view(dtype).view((x if operand == "a" else y).shape)
        pair = (inside.copy_(x), y) if operand == "a" else (x, inside.copy_(y))
        assert torch.equal(backend.matmul_wide_fused(*pair, DENSE6, workspace=ws).cpu(), want)
        ws.accumulators.zero_()  # its counters were written over
