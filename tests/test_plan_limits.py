"""Sizes at which a kernel's addressing ends: the host refuses its plan.
Workspaces made for other calls: the host takes a plan that fits them.  And
arguments that a C caller can get wrong: an error code, not the process."""
import ctypes
import os
import subprocess
import sys

import pytest
import torch

from rns_llm_amd import _native

LDS_TILES = 10  # byte-product tiles (include/rnsmx.h)


def test_byte_product_planes_stay_below_32_bit_offsets():
    """Rows of an activation plane are addressed by 32-bit offsets: M rows of
    kp rounded up to 128 bytes must end below 2^32 - 256."""
    lib = _native.lib()
    for k, limit in ((4096, 4096), (4033, 4096), (4100, 4224)):
        most = ((1 << 32) - 257) // limit
        for mb in (4, 8):
            plan = _native.Plan(LDS_TILES, mb, 1, 0, 1, 0)
            assert lib.rnsmx_packed_workspace_bytes(most, k, 64, 6, ctypes.byref(plan)) > 2 * most * limit
            assert lib.rnsmx_packed_workspace_bytes(most + 1, k, 64, 6, ctypes.byref(plan)) == -1
        # an automatic plan still serves them, by residue channels
        assert lib.rnsmx_packed_workspace_bytes(most + 1, k, 64, 6, None) > 0


def room(query, m, n, k, channels, plan=None):
    return query(m, k, n, channels, None if plan is None else ctypes.byref(_native.Plan(*plan)))


# (M, N, K, channels) on both sides of where an automatic plan takes channel
# units (kind 11), and their two tiles; None: the plan without them
@pytest.mark.parametrize("shape,units", [
    ((16, 4096, 4096, 6), None), ((17, 4096, 4096, 6), (11, 2, 1, 0)),           # rows
    ((17, 768, 768, 6), None),                                                   # short K: the stream kernel
    ((64, 2304, 768, 5), (11, 2, 1, 0)), ((160, 1536, 1024, 6), (11, 2, 1, 0)),
    ((200, 515, 513, 6), (11, 2, 1, 0)), ((40, 12288, 4096, 6), (11, 4, 2, 0)),
    ((512, 768, 768, 6), None), ((300, 514, 576, 6), None), ((512, 12288, 4096, 6), None),
    # 128 x 128 units of which a few start a second round, at 14, 16 and 17 K steps; 18 steps; more of them
    ((203, 2757, 896, 6), None), ((72, 5691, 1008, 6), None), ((203, 2757, 1088, 6), None),
    ((72, 5691, 1152, 6), (11, 4, 2, 0)), ((132, 4416, 1024, 6), (11, 4, 2, 0)),
    ((512, 2048, 5120, 6), None),                                                # past four workgroups per CU
], ids=str)
def test_where_channel_units_are_taken(shape, units):
    """Read from the room the automatic plan asks for: the units' exchange of a
    byte per channel and element, or that of the plan rnsmx_gemm_plan gives."""
    lib = _native.lib()
    query, (m, n, k, channels) = lib.rnsmx_prepared_workspace_bytes, shape
    other = _native.Plan()
    _native.check(lib.rnsmx_gemm_plan(m, n, k, channels, 0, ctypes.byref(other)))
    rooms = {plan: room(query, *shape, plan=plan) for plan in ((11, 2, 1, 0), (11, 4, 2, 0), other.as_tuple())}
    taken = rooms.pop(units or other.as_tuple())
    assert room(query, *shape) == taken and taken not in rooms.values()  # so the room tells which


# N = 12288: 128 tiles of 64 x 96; K of no whole 256, so that int32 activations
# (the channel form) never split
@pytest.mark.parametrize("shape,splits", [
    ((17, 12288, 4160), 2), ((64, 12288, 4160), 2), ((65, 12288, 4160), 1), ((64, 12384, 4160), 1),
    ((64, 6144, 4160), 4), ((64, 6240, 4160), 2), ((128, 3072, 4160), 4),       # one round of 256
    ((64, 4096, 4160), 4), ((64, 4096, 4032), 2),                               # 16 K steps in each of four
    ((64, 4096, 2112), 2), ((64, 4096, 1984), 1),                               # ... of two
    ((32, 12288, 4160), 2), ((16, 12288, 4160), 1),                             # int16 rows to 16 tokens, int8 to 32
], ids=str)
def test_where_byte_products_split_k(shape, splits):
    query, (m, n, k) = _native.lib().rnsmx_packed_workspace_bytes, shape
    rooms = {s: room(query, *shape, 6, plan=(10, 4, 1, 0, s, 0)) for s in (1, 2, 4)}
    assert room(query, *shape, 6) == rooms[splits]
    assert len(set(rooms.values())) == 3


def runs_in(lib, mods, dtype, m, k, n, nbytes):
    """Whether a packed product accepts a workspace of nbytes.  Without a GPU a
    call that passes its checks ends at the launch, which reads nothing."""
    fake = 1 << 20
    return lib.rnsmx_matmul_packed_fused(fake, dtype, m, k, n, fake, ctypes.byref(mods), None, 0, None, None, None,
                                         fake, nbytes, fake, None) != _native.ESPACE


@pytest.mark.skipif(torch.cuda.is_available(), reason="calls that pass the checks would launch on made-up pointers")
@pytest.mark.parametrize("k,n", [(2048, 64), (2048, 333), (4096, 4096), (4096, 12288), (8192, 768)])
@pytest.mark.parametrize("moduli", [(255, 253, 251), (255, 253, 251, 247, 241, 239)], ids=len)
def test_a_packed_workspace_serves_fewer_rows(moduli, k, n):
    """The room that residue channels of `most` rows take serves every call of
    up to `most` rows: a byte product whose K split needs more runs unsplit."""
    lib = _native.lib()
    mods = _native.make_moduli(moduli)
    for most in (24, 48, 64, 128, 256, 512, 1024):
        # the planes and row terms of residue channels, the counters and the row norms
        up = lambda v: (v + 255) // 256 * 256  # noqa: E731
        planes = up(2 * len(moduli) * most * k + 4 * len(moduli) * ((most + 63) // 64 * 64 + 64))
        room = _native.SPLIT_TICKETS * 4 + max(planes, up(16 * k * 16 if most <= 32 else 0)) + up(8 * (most + 1))
        for m in (1, 9, 17, 24, 33, 48, 64, 65, 128, 200, 256, 512, 1024):
            if m <= most:
                for dtype in (_native.INT8, _native.INT16):
                    assert runs_in(lib, mods, dtype, m, k, n, room), (most, m, dtype)


@pytest.mark.skipif(torch.cuda.is_available(), reason="calls that pass the checks would launch on made-up pointers")
def test_requests_stay_clear_of_the_staging_buffer():
    lib, mods = _native.lib(), _native.make_moduli((255, 253, 251, 247))
    staging, k, rows = 1 << 20, 64, (3, 2)

    def code(*at):
        return lib.rnsmx_matmul_requests((ctypes.c_void_p * 2)(*at), (ctypes.c_int32 * 2)(*rows), 2, _native.INT8, k, 16,
                                         1 << 22, ctypes.byref(mods), 0, staging, 1 << 23, 1 << 30, 1 << 24, None)

    end = staging + 5 * k
    for at in ((staging, end), (end, staging), (end - 1, end + 512), (end, staging - 2 * k + 1)):
        assert code(*at) == _native.EINVAL and b"staging" in lib.rnsmx_last_error()
    for at in ((end, end + 3 * k), (staging - 3 * k, end), (end + 16, staging - 2 * k)):
        assert code(*at) == _native.ELAUNCH  # no device: every check passed


@pytest.mark.skipif(torch.cuda.is_available(), reason="calls that pass the checks would launch on made-up pointers")
@pytest.mark.parametrize("dtype,size", [(_native.INT8, 1), (_native.INT16, 2)])
def test_unprepared_operands_stay_clear_of_what_is_written(dtype, size):
    lib, mods = _native.lib(), _native.make_moduli((255, 253, 251, 247))
    m, k, n, ws = 32, 64, 48, 1 << 24
    need = lib.rnsmx_wide_workspace_bytes(m, k, n, 4)

    def code(a=1 << 20, b=1 << 21, out=1 << 22, width=k):
        return lib.rnsmx_matmul_wide(a, b, dtype, m, width, n, ctypes.byref(mods), ws, need, out, None)

    assert code() == _native.ELAUNCH  # no device: every check passed
    for bad in (dict(a=ws), dict(b=ws + need - 16), dict(a=ws + 16 - size * m * k), dict(b=ws + 1 - size * k * n)):
        assert code(**bad) == _native.EINVAL and b"workspace" in lib.rnsmx_last_error()
    assert code(b=ws - size * k * n) == _native.ELAUNCH and code(a=ws + (need + 15) // 16 * 16) == _native.ELAUNCH
    # int8 rows are read in place where K is a multiple of 16; others are copied first
    over = (1 << 22) + 16
    assert code(a=over) == (_native.EINVAL if size == 1 else _native.ELAUNCH)
    assert code(a=over, width=k - 1) == _native.ELAUNCH
    assert code(b=over) == _native.ELAUNCH


UNFILLED = """
import ctypes, sys
from rns_llm_amd import _native
lib, fake = _native.lib(), 1 << 20
for values in ((0, 0), (0, 251), (251, 0, 1), (1, 1), (-3, 5), (4, 2, 0, 0, 0, 0)):
    print(values, flush=True)
    mods = _native.Moduli(channels=len(values))
    mods.moduli[:len(values)] = values
    lib.rnsmx_matmul_prepared_fused(fake, _native.INT8, 4, 64, 16, fake, ctypes.byref(mods), None, 0, None, None, None,
                                    fake, 1 << 30, fake, None)
"""


@pytest.mark.skipif(torch.cuda.is_available(), reason="calls that pass the checks would launch on made-up pointers")
def test_a_set_that_was_never_initialised_ends_no_process():
    """A moduli block whose channels are set but whose constants are not: an
    error code (the launch's, without a GPU), and the process goes on."""
    path = os.pathsep.join(p for p in sys.path if p)
    done = subprocess.run([sys.executable, "-c", UNFILLED], env=dict(os.environ, PYTHONPATH=path), capture_output=True,
                          text=True, timeout=120)
    assert done.returncode == 0, done.stdout + done.stderr
