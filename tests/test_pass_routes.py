"""Which way a whole Scheme II INT8 pass goes (oz2_pass.hip), by the library's own rules on 256 compute units, on either
side of their lines. CPU only."""
import ctypes

import pytest

from oztt_amd.device import hip, moduli_desc

CUS = 256
TABLE = [255, 254, 253, 251, 247, 241, 239, 233, 229, 227, 223, 217, 211, 199, 197, 193, 191]


# at most 64 columns without A's planes: the parts of K, 0 where the planes stay
@pytest.mark.parametrize("M,N,K,S,nd,parts", [
    (8192, 64, 8192, 15, 3, 2), (8192, 65, 8192, 15, 3, 0), (8192, 64, 1023, 15, 3, 0), (8192, 64, 8192, 15, 4, 0),
    (8192, 1, 1024, 16, 3, 2), (8192, 64, 8192, 17, 3, 0), (16384, 64, 1024, 15, 3, 1), (6081, 64, 1024, 15, 3, 2),
    (6080, 64, 1024, 15, 3, 0), (12225, 64, 1024, 15, 3, 1), (12224, 64, 1024, 15, 3, 0),
    (8192, 64, 2048, 4, 3, 2), (8192, 64, 2048, 3, 3, 0),           # few moduli
    (6144, 64, 2048, 6, 3, 2), (6144, 64, 2048, 5, 3, 0), (12288, 24, 2048, 5, 3, 0), (16384, 24, 2048, 4, 3, 1),
])
def test_narrow_pass(M, N, K, S, nd, parts):
    assert hip().oz_rule_narrow_parts(CUS, ctypes.byref(moduli_desc(TABLE[:S], nd)), M, N, K) == parts


def test_narrow_pass_of_two_even_moduli():
    assert hip().oz_rule_narrow_parts(CUS, ctypes.byref(moduli_desc([255, 254, 253, 252, 251, 247], 3)), 8192, 64, 2048) == 0
