"""Reconstruction by fractions, the GEMM epilogue's way from channel sums to
the signed integer (up to 6 channels; more take the mixed-radix digits).

On the CPU the arithmetic is restated with every double operation rounded
once from the exact rational (what an fma does) and compared with the
remainder of the exact value, at sums over the whole int32 range and outputs
at both ends of the centered range; on the GPU every kernel family runs sets
with an even modulus and sums that wrap, shorter prefixes included."""
from fractions import Fraction
from math import prod

import numpy as np
import pytest
import torch

from oracle import rns_oracle as ro

SETS = [(255, 253, 251, 247, 241, 239), (255, 253, 251, 247, 241), (255, 253, 251, 247), (254, 253, 251, 247),
        (255, 254, 253, 251, 247, 241), (255, 253, 251), (2, 3), (128, 3, 5), (251,), (253, 255)]


def weights(moduli, parts):
    """The rows of the weighted sum and its starting phase, as doubles."""
    p = prod(moduli)
    rows = [[], [], []][:parts]
    for m in moduli:
        k = pow(p // m, -1, m) if len(moduli) > 1 else 1
        rest = Fraction(k - m if 2 * k > m else k)
        for r in range(parts):
            if r < parts - 1:
                unit = Fraction(1, 2 ** (20 * (r + 1)))
                f = round(float(rest / m) / float(unit)) * unit
            else:
                f = Fraction(float(rest / m))
            rows[r].append(f)
            rest -= f * m
    half = (p - 1) >> 1
    return rows, p, half, Fraction((half + 0.25) / p)


def reconstruct(v, moduli):
    parts = 2 if len(moduli) <= 4 else 3
    rows, p, half, turn = weights(moduli, parts)
    rounded = lambda x: Fraction(float(x))  # noqa: E731
    z = Fraction(0)
    for r in range(parts - 1):
        for x, f in zip(v, rows[r]):
            exact = z + x * f
            z = rounded(exact)
            assert z == exact  # the leading rows lose nothing
        z -= z.__floor__()
    s = turn
    for x, f in zip(v, rows[-1]):
        s = rounded(s + x * f)
    z = rounded(z + s)
    z -= z.__floor__()
    magic = Fraction(6755399441055744 - half)
    return int(rounded(z * p + magic) - 6755399441055744)


def centered(x, p):
    r = x % p
    return r - p if r > p >> 1 else r


@pytest.mark.parametrize("moduli", SETS, ids=str)
def test_fractions_equal_the_centered_remainder(moduli):
    p, rng = prod(moduli), np.random.default_rng(len(moduli) * 1000 + moduli[0])
    ends = [0, 1, -1, p >> 1, (p >> 1) - 1, -((p - 1) >> 1), -((p - 1) >> 1) + 1, (p >> 1) // 2]
    values = ends + [int(rng.integers(-(p >> 1), (p >> 1) + 1)) for _ in range(200)]
    for y in values:
        y = centered(y, p)
        for how in range(4):
            # sums congruent to y: small, at both ends of int32, anywhere
            v = []
            for m in moduli:
                r = y % m
                lo, hi = (-2 ** 31 - r) // m + 1, (2 ** 31 - 1 - r) // m
                t = [0, lo, hi, int(rng.integers(lo, hi + 1))][how]
                v.append(r + t * m)
            assert all(-2 ** 31 <= x < 2 ** 31 for x in v)
            assert reconstruct(v, moduli) == y


def _wrapped(a, w_nk, moduli):
    """The exact product reduced to the centered range of the set."""
    p = prod(moduli)
    return torch.from_numpy(np.vectorize(lambda x: centered(int(x), p), otypes=[np.int64])(
        ro.exact_matmul(a.numpy(), w_nk.t().numpy())))


# one plan of every family whose epilogue differs: stream (LDS and register
# epilogue), MFMA, 256 x 64 and 256 x 96 LDS tiles (4 channels, K % 256 = 0),
# residue-plane LDS tiles (int16)
@pytest.mark.gpu
@pytest.mark.parametrize("plan,dtype", [((1, 1, 1, 4), torch.int8), ((1, 1, 1, 1), torch.int8), ((2, 2, 1, 0), torch.int8),
                                        ((3, 0, 0, 0), torch.int8), ((7, 0, 0, 0), torch.int8),
                                        ((8, 0, 0, 0), torch.int16)], ids=str)
@pytest.mark.parametrize("moduli", [(254, 253, 251, 247), (16, 15, 7, 11), (255, 254, 253, 251, 247, 241)], ids=str)
def test_even_and_undersized_sets_on_every_family(backend, plan, dtype, moduli):
    if len(moduli) > 4 and plan[0] in (3, 7):
        pytest.skip("tiles for up to 4 channels")
    gen = torch.Generator().manual_seed(plan[0] * 7 + len(moduli))
    lim = 128 if dtype == torch.int8 else 32768
    m, k, n = 37, 512, 70
    a = torch.randint(-lim, lim, (m, k), generator=gen, dtype=torch.int32).to(dtype)
    w = torch.randint(-lim, lim, (n, k), generator=gen, dtype=torch.int32).to(dtype)
    a[0], w[0] = -lim, -lim  # the largest sums
    a[1] = lim - 1
    prepared = backend.prepare_weight_nk(w.cuda(), moduli)
    got = backend.matmul_prepared_fused(a.cuda(), prepared, plan=plan).cpu()
    assert torch.equal(got, _wrapped(a, w, moduli))


@pytest.mark.gpu
@pytest.mark.parametrize("m", [3, 40, 300])
@pytest.mark.parametrize("moduli,dtype,expect", [((253, 254, 255, 251), torch.int8, 2), ((253, 254, 255, 251), torch.int8, 3),
                                                 ((255, 254, 253, 251, 247, 241), torch.int16, 3),
                                                 ((255, 254, 253, 251, 247, 241), torch.int16, 5)], ids=str)
def test_shorter_prefixes(backend, m, moduli, dtype, expect):
    """The device's prefix (its rows derived in the kernel) on every family
    that takes m: the range of the activations sets the prefix."""
    k, n = 512, 75
    lim, b_max = {(torch.int8, 2): (1, 20), (torch.int8, 3): (127, 60), (torch.int16, 3): (100, 100),
                  (torch.int16, 5): (32767, 1000)}[dtype, expect]
    gen = torch.Generator().manual_seed(m + expect)
    a = torch.randint(-lim, lim + 1, (m, k), generator=gen, dtype=torch.int32).to(dtype)
    w = torch.randint(-b_max, b_max + 1, (n, k), generator=gen, dtype=torch.int32).to(dtype)
    a[0], w[0, 0] = lim, b_max
    c, bound, _ = ro.adaptive_select(a.numpy(), b_max, moduli, min_channels=2)
    assert c == expect
    # every sum that fits the prefix's bound, largest ones among them
    w[1], a[m - 1] = b_max, -lim
    adaptive = backend.prepare_weight_adaptive_nk(w.cuda(), moduli, min_channels=2)
    out, meta = backend.matmul_prepared_adaptive_fused(a.cuda(), adaptive, return_metadata=True)
    assert meta["channels"] == expect and meta["bound"] == bound
    assert torch.equal(out.cpu(), torch.from_numpy(ro.exact_matmul(a.numpy(), w.t().numpy())))


# float outputs: whole tiles with rows of 4 columns (four columns per store),
# rows of 66 and 70 (one column per store) and edges, every tile family
@pytest.mark.gpu
@pytest.mark.parametrize("n", [64, 66, 70, 100, 192])
@pytest.mark.parametrize("out_dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("plan,dtype", [((2, 2, 1, 0), torch.int8), ((5, 3, 1, 4), torch.int8), ((3, 0, 0, 0), torch.int8),
                                        ((7, 0, 0, 0), torch.int8), ((8, 0, 0, 0), torch.int16)], ids=str)
def test_float_rows(backend, plan, dtype, out_dtype, n):
    m, k = 261, 256
    moduli = (255, 253, 251, 247) if dtype == torch.int8 else (255, 253, 251, 247, 241, 239)
    gen = torch.Generator().manual_seed(n)
    lim = 128 if dtype == torch.int8 else 32768
    a = torch.randint(-lim, lim, (m, k), generator=gen, dtype=torch.int32).to(dtype)
    w = torch.randint(-lim, lim, (n, k), generator=gen, dtype=torch.int32).to(dtype)
    scale, w_scale = torch.tensor([1e-3]), torch.rand((n,), generator=gen) * 1e-3
    bias = torch.randn((n,), generator=gen)
    prepared = backend.prepare_weight_nk(w.cuda(), moduli)
    exact = torch.from_numpy(ro.exact_matmul(a.numpy(), w.t().numpy()))
    for b in (bias, None):
        out = torch.empty((m, n), dtype=out_dtype, device="cuda")
        backend.matmul_prepared_fused(a.cuda(), prepared, plan=plan, out=out, a_scale=scale.cuda(), w_scale=w_scale.cuda(),
                                      bias=None if b is None else b.cuda())
        ref = (exact.float() * scale.view(1, 1)) * w_scale.unsqueeze(0)
        ref = (ref if b is None else ref + b).to(out_dtype)
        bits = torch.int32 if out_dtype == torch.float32 else torch.int16
        assert torch.equal(out.cpu().view(bits), ref.view(bits))
