"""The constants by which the kernel for at most 64 columns (oz2_skinny.hip) reduces A' modulo m, as the library
computes them, for every modulus that a descriptor may hold and every dot product of A's balanced bytes with the
weights. CPU only."""
import ctypes

import numpy as np
import pytest

from oztt_amd.device import hip


class NarrowModulus(ctypes.Structure):
    _fields_ = [("w", ctypes.c_uint32 * 2), ("magic", ctypes.c_uint32), ("init", ctypes.c_int), ("mneg", ctypes.c_int)]


@pytest.mark.parametrize("m1", range(2, 256))
def test_residue_bytes(m1):
    c = NarrowModulus()
    hip().oz_rule_narrow_modulus(m1, ctypes.byref(c))
    w = np.array(list(c.w), np.uint32).view(np.int8).astype(np.int64)
    assert all((int(x) - pow(256, j, m1)) % m1 == 0 for j, x in enumerate(w))
    m = (1 << 24) - c.mneg
    assert m % m1 == 0 and 128 <= m <= 255 and np.abs(w).max() <= m // 2
    assert c.magic < 1 << 24
    top = 8 * 128 * 127  # |A' bytes| <= 128, |weights| <= 127
    dot = np.arange(-top, top + 1, dtype=np.int64)
    u = dot + c.init
    v = u + dot
    assert v.min() >= 0 and v.max() < 1 << 20 and u.max() < 1 << 24
    q = (v * c.magic) >> 32
    x = (q * c.mneg + u) & 0xFFFFFF  # the low 24 bits of v_mad_u32_u24
    byte = ((x & 0xFF) ^ 0x80) - 0x80
    assert np.all((byte - dot) % m1 == 0)
    # products with B's residues stay within 127^2, the pass's bound on its sums
    assert np.abs(byte).max() <= (127 if m != 128 else 128)
    assert np.abs(byte).max() * (m1 // 2) <= 127 * 127
