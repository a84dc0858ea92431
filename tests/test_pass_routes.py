"""Which way a whole Scheme II INT8 pass goes (oz2_pass.hip), by the library's own rules on 256 compute units, on either
side of their lines. CPU only."""
import ctypes

import pytest

from oztt_amd.device import crt_desc, hip, moduli_desc

CUS = 256
TABLE = [255, 254, 253, 251, 247, 241, 239, 233, 229, 227, 223, 217, 211, 199, 197, 193, 191, 181, 179, 173, 167, 163, 157, 151]
PREP, FUSED, PART = 1, 2, 4


def route(M, N, K, S=15, nd=3, moduli=None, nw=None):
    moduli = moduli or TABLE[:S]
    md, cd = moduli_desc(moduli, nd), crt_desc(TABLE[:len(moduli)], {3: 54, 4: 70, 5: 90}[nd], nd)
    cd.nw = cd.nw if nw is None else nw
    return hip().oz_rule_pass(CUS, ctypes.byref(md), ctypes.byref(cd), M, N, K)


# at most 64 columns without A's planes: the parts of K, 0 where the planes stay
@pytest.mark.parametrize("M,N,K,S,nd,parts", [
    (8192, 64, 8192, 15, 3, 2), (8192, 65, 8192, 15, 3, 0), (8192, 64, 1023, 15, 3, 0), (8192, 64, 8192, 15, 4, 0),
    (8192, 1, 1024, 16, 3, 2), (8192, 64, 8192, 17, 3, 0), (16384, 64, 1024, 15, 3, 1), (6081, 64, 1024, 15, 3, 2),
    (6080, 64, 1024, 15, 3, 0), (12225, 64, 1024, 15, 3, 1), (12224, 64, 1024, 15, 3, 0),
    (8192, 64, 2048, 4, 3, 2), (8192, 64, 2048, 3, 3, 0),           # few moduli
    (6144, 64, 2048, 6, 3, 2), (6144, 64, 2048, 5, 3, 0), (12288, 24, 2048, 5, 3, 0), (16384, 24, 2048, 4, 3, 1),
])
def test_narrow_pass(M, N, K, S, nd, parts):
    assert route(M, N, K, S, nd) // PART == parts


def test_two_even_moduli():
    even2 = [255, 254, 253, 252, 251, 247]
    assert route(8192, 64, 2048, moduli=even2) == 0 and route(128, 128, 128, moduli=even2) == 0


@pytest.mark.parametrize("M,N,K,S,nd,want", [
    (128, 128, 128, 15, 3, PREP), (9, 9, 1, 15, 3, PREP), (40, 31, 256, 24, 5, PREP), (128, 128, 257, 15, 3, 0),
    (256, 4000, 512, 15, 3, PREP), (256, 3839, 512, 15, 3, 0), (255, 4000, 512, 15, 3, 0), (256, 4000, 513, 15, 3, 0),
    (256, 4000, 512, 18, 4, 0),
    (2048, 1024, 256, 15, 3, PREP | FUSED), (2047, 960, 256, 15, 3, PREP), (2048, 1024, 257, 15, 3, 0),
    (2048, 2048, 320, 15, 3, PREP), (1500, 1409, 64, 15, 3, PREP | FUSED), (4096, 4096, 256, 15, 3, PREP | FUSED),
    (4096, 4096, 256, 18, 4, PREP | FUSED), (4096, 4096, 256, 21, 5, PREP),   # 7 limbs
])
def test_short_inner_dimension(M, N, K, S, nd, want):
    assert route(M, N, K, S, nd) == want


def test_accumulators_that_the_reconstruction_refuses():
    for nw, want in ((2, PREP), (3, PREP), (4, PREP | FUSED), (8, PREP | FUSED), (9, PREP)):
        assert route(1500, 1409, 64, nw=nw) == want
