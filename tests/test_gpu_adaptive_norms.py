"""The adaptive prefix where a row norm needs more than 31 bits: large int32
activations, and int16 ones over a long K.  The norms lie on both sides of the
bits that change sign or word; metadata and products against the oracle."""
import pytest
import torch

from oracle import rns_oracle as ro

pytestmark = pytest.mark.gpu

DENSE6 = (255, 253, 251, 247, 241, 239)
NORMS = (2 ** 31 - 1, 2 ** 31, 2 ** 31 + 12345, 2 ** 32 - 1, 2 ** 32, 2 ** 32 + 2 ** 31 - 1, 2 ** 32 + 2 ** 31, 2 ** 34 - 1)


def check(backend, a, w, packed):
    adaptive = backend.prepare_weight_adaptive_nk(w.cuda(), DENSE6, min_channels=2, packed=packed)
    out, meta = backend.matmul_prepared_adaptive_fused(a.cuda(), adaptive, return_metadata=True)
    channels, bound, capacity = ro.adaptive_select(a.numpy(), int(w.to(torch.int32).abs().max()), DENSE6, min_channels=2)
    assert dict(meta) == {"channels": channels, "bound": bound, "capacity": capacity}
    assert torch.equal(out.cpu(), torch.from_numpy(ro.exact_matmul(a.numpy(), w.t().numpy())))


@pytest.mark.parametrize("norm", NORMS)
@pytest.mark.parametrize("m", [1, 3, 40, 200, 300])
@pytest.mark.parametrize("packed", [False, True])
def test_int32_rows(backend, m, norm, packed):
    k, n = 128, 70
    gen = torch.Generator().manual_seed(m)
    a = torch.randint(-1000, 1001, (m, k), generator=gen, dtype=torch.int32)
    row, left = a[m // 2], norm
    row.zero_()
    for i in range(k):  # values up to 2^30, both signs, that sum to the norm
        part = min(left, 2 ** 30)
        row[i] = part if i % 2 else -part
        left -= part
    w = torch.randint(-127, 128, (n, k), generator=gen, dtype=torch.int32).to(torch.int8)
    check(backend, a, w, packed)


@pytest.mark.parametrize("m", [2, 30])
@pytest.mark.parametrize("k", [65535, 65536, 66000])
def test_int16_rows_of_a_long_k(backend, m, k):
    gen = torch.Generator().manual_seed(k)
    a = torch.randint(-9, 10, (m, k), generator=gen, dtype=torch.int32).to(torch.int16)
    a[m - 1] = -32768
    w = torch.randint(-9, 10, (3, k), generator=gen, dtype=torch.int32).to(torch.int8)
    for packed in (False, True):
        check(backend, a, w, packed)
