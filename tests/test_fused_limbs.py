"""The CRT accumulator of the fused products and reconstruction (oz2_gemm_crt.hip), emulated on the CPU:
V = sum_s C_s W_s in limbs of w bits, t = rint(V / M) from an FP64 estimate, C' = V - t M. Every
intermediate that the kernel holds in a double must be an integer of at most 2^53, the estimate must be
within the threshold delta = 2^-20 of V / M, and C' must be the C_s's exact integer."""
import ctypes
from fractions import Fraction
from math import prod

import numpy as np
import pytest

from oztt_amd.device import crt_desc, hip

MODULI = [255, 254, 253, 251, 247, 241, 239, 233, 229, 227, 223, 217, 211, 199, 197, 193]


def fma(a, b, c):
    return float(Fraction(a) * Fraction(b) + Fraction(c))


@pytest.mark.parametrize("S", [8, 14, 15, 16])
@pytest.mark.parametrize("K", [64, 128, 192, 256])
def test_limbs_hold_every_step(S, K):
    moduli = MODULI[:S]
    M = prod(moduli)
    w = 52 - (S * K * 127 * 127).bit_length()
    L = max(4, -(-M.bit_length() // w))
    assert 4 <= L <= 6
    mask = (1 << w) - 1
    limbs = lambda v: [(v >> (w * l)) & mask for l in range(L)]  # noqa: E731
    assert M >> (w * L) == 0
    W = [pow(M // m % m, -1, m) * (M // m) for m in moduli]
    Mw, Md = limbs(M), float(M)
    rng = np.random.default_rng(S + K)
    big = K * 127 * 127
    for trial in range(400):
        if trial < 4:  # the largest sums, all signs alike and alternating
            C = [big if trial == 0 or (trial > 1 and (s + trial) % 2) else -big for s in range(S)]
        elif trial < 40:  # integers next to the ends and to zero, through any representative
            target = int(rng.choice([M // 2, M // 2 - M + 1, 0, 1, -1, M // 2 - 1])) if trial % 2 else int(rng.integers(-9, 9))
            C = [target % m - m * int(rng.integers(0, 2)) for m in moduli]
        else:
            C = [int(rng.integers(-big, big + 1)) for _ in moduli]
        V = sum(c * x for c, x in zip(C, W))
        x = [sum(c * limbs(y)[l] for c, y in zip(C, W)) for l in range(L)]
        assert max(map(abs, x)) <= 1 << 52
        vd = float(x[-1])
        for l in range(L - 2, -1, -1):
            vd = fma(vd, 2.0 ** w, float(x[l]))
        q = vd * (1.0 / Md)
        assert abs(Fraction(q) - Fraction(V, M)) < Fraction(1, 1 << 21)
        t = round(q)
        y = [a - t * b for a, b in zip(x, Mw)]
        assert max(map(abs, y)) <= 1 << 53
        got = sum(v << (w * l) for l, v in enumerate(y))
        if abs(q - t) > 0.5 - (2.0 ** -20 + 2.0 / Md):  # settled exactly by the kernel
            got -= M if got > M // 2 else -M if got <= M // 2 - M else 0
        assert M // 2 - M < got <= M // 2
        assert all((got - c) % m == 0 for c, m in zip(C, moduli))


TABLE = MODULI + [191, 181, 179, 173, 167, 163, 157, 151]


def limbs_of(S, K):
    """The kernel's own answer: width and number of limbs, or None where it does not take the moduli."""
    w, n = ctypes.c_int(), ctypes.c_int()
    ok = hip().oz_rule_fused_limbs(ctypes.byref(crt_desc(TABLE[:S], 54, 3)), K, ctypes.byref(w), ctypes.byref(n))
    return (w.value, n.value) if ok else None


def test_the_rule_is_the_one_emulated():
    for S in (8, 14, 15, 16):
        for K in (64, 128, 192, 256):
            w = 52 - (S * K * 127 * 127).bit_length()
            assert limbs_of(S, K) == (w, max(4, -(-prod(MODULI[:S]).bit_length() // w)))


@pytest.mark.parametrize("S", range(1, 25))
def test_every_accepted_quotient_is_within_the_threshold(S):
    M = prod(TABLE[:S])
    taken = [K for K in range(64, 131072 + 1, 64) if limbs_of(S, K)]
    rng = np.random.default_rng(S)
    for K in taken[-1:]:  # the longest: the smallest width and the largest quotients
        w, L = limbs_of(S, K)
        big = K * 127 * 127
        assert S * big << w <= 1 << 52 and M >> (w * L) == 0
        assert Fraction((2 * L + 8) * S * big, 1 << 53) < Fraction(1, 1 << 20)
        mask = (1 << w) - 1
        W = [pow(M // m % m, -1, m) * (M // m) for m in TABLE[:S]]
        for trial in range(60):
            C = [int(rng.integers(-big, big + 1)) if trial % 2 else big * int(rng.choice([-1, 1])) for _ in W]
            vd = 0.0
            for l in range(L - 1, -1, -1):
                vd = fma(vd, 2.0 ** w, float(sum(c * ((x >> (w * l)) & mask) for c, x in zip(C, W))))
            V = sum(c * x for c, x in zip(C, W))
            assert abs(Fraction(vd * (1.0 / float(M))) - Fraction(V, M)) < Fraction(1, 1 << 20)
