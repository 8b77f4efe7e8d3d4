"""Sizes at which a kernel's addressing ends: the host refuses its plan."""
import ctypes

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
