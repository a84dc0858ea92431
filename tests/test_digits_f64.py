"""The residue generator's A' for nd = 3 (split_integer3 in oztt_amd/csrc/oz2_residue.hpp), which follows the
reference's binary32 digit procedure through binary64 operations, against that procedure itself (load_triple
and make_digits in oz_tf32.hpp / oz2_residue.hpp, restated here operation by operation in float32). CPU only:
both sides are restatements, so this shows that the one sequence equals the other; that the kernels hold them is what
tests/test_gpu_stages.py (against the oracle) and tests/test_gpu_far_elements.py show."""
import numpy as np

F = np.float32


def two_sum_fast(a, b):
    s = a + b
    return s, b - (s - a)


def reference(x, d):
    """A' = d0 2^40 + d1 2^20 + d2 by the binary32 procedure."""
    u = x.view(np.uint64)
    w1, w0 = (u >> np.uint64(32)).astype(np.int64), (u & np.uint64(0xFFFFFFFF)).astype(np.int64)
    sgn = np.where(w1 & 0x80000000, -1.0, 1.0)
    E = (w1 >> 20) & 0x7FF
    a = 0x400000 | ((w1 & 0xFFFFF) << 2) | (w0 >> 30)
    rem = w0 & 0x3FFFFFFF
    up = rem >= 0x20000000
    a = a + up
    r = rem - up * 0x40000000
    b, c = r >> 7, r & 0x7F
    e = E - 1075 + d
    hi = np.ldexp(sgn * a, e + 30).astype(F)
    mid = np.ldexp(sgn * b, e + 7).astype(F)
    lo = np.ldexp(sgn * c, e).astype(F)
    zero = E == 0
    hi, mid, lo = (np.where(zero, F(0), v) for v in (hi, mid, lo))
    digits = []
    for i in range(3):
        if i:
            hi, mid, lo = (v * F(2**20) for v in (hi, mid, lo))
            s3, e4 = two_sum_fast(mid, lo)
            s5, e6 = two_sum_fast(hi, s3)
            hi = s5
            mid, lo = two_sum_fast(e6, e4)
        t = np.rint(hi)
        hi = hi - t
        digits.append(t.astype(np.int64))
    return (digits[0] << 40) + (digits[1] << 20) + digits[2]


def split_integer3(x, d):
    return integer_and_sum(x, d)[0]


def integer_and_sum(x, d):
    """The kernel's sequence: A', and T, whose upper word says whether the sequence holds."""
    u = x.view(np.int64)
    r = ((u & 0xFFFFFFFF) << 34) >> 34  # bits 0..29, signed
    h0 = np.ldexp((u - r).view(np.float64), d)
    v0 = np.ldexp(x, d)
    m0 = v0 - h0
    t0 = np.rint(h0)
    g = h0 - t0
    s3 = m0.astype(F).astype(np.float64)
    s5 = (g + s3).astype(F).astype(np.float64)
    T1 = s5 + 1.5 * 2.0**32
    hi2 = s5 - (T1 - 1.5 * 2.0**32)
    mid = ((g + m0) - s5).astype(F).astype(np.float64)
    f = (hi2 + mid).astype(F)
    fb = (f.astype(np.float64) * 2.0**40 + 12582912.0).astype(F).view(np.int32).astype(np.int64)  # one rounding: exact below 2^53
    T = T1 + t0
    return ((T.view(np.uint64) << np.uint64(20)).view(np.int64)) + (fb - 0x4B400000), T


def check(x, d):
    with np.errstate(over="ignore", under="ignore"):
        a, b = reference(x, d), split_integer3(x, d)
    bad = np.flatnonzero(a != b)
    assert not bad.size, (x[bad[:3]].tolist(), d[bad[:3]].tolist() if np.ndim(d) else d, a[bad[:3]], b[bad[:3]])


def test_random_elements():
    """Elements from the row's maximum (up to 2^20 after scaling) down past the last digit."""
    rng = np.random.default_rng(1)
    for top in (8, 13, 16, 20):  # b - 40
        for _ in range(4):
            n = 400000
            x = rng.uniform(-1, 1, n) * np.exp2(rng.integers(-70, 1, n).astype(float))
            check(x, np.int64(top))
            check(np.copysign(rng.uniform(0.5, 1, n), rng.uniform(-1, 1, n)), np.int64(top))


def test_halves_and_their_neighbours():
    """Digits at and next to ties, in either stage, with the low bits of x next to the limbs' own rounding."""
    rng = np.random.default_rng(2)
    n = 300000
    for pos in range(-45, 4):  # the scaled value's first digit boundary falls at every bit of x
        k = rng.integers(0, 2**12, n).astype(float) + 0.5
        low = np.exp2(-rng.integers(1, 42, n).astype(float)) * rng.integers(-3, 4, n)
        x = np.ldexp(np.copysign(k + low, rng.uniform(-1, 1, n)), pos)
        check(x, np.int64(rng.integers(0, 21)))
    # bit patterns: long runs of ones and zeros around the limbs' boundaries (bits 30, 29, 7)
    m = np.zeros(n, np.uint64)
    for b in (0, 1, 5, 6, 7, 8, 28, 29, 30, 31, 40, 51):
        m ^= rng.integers(0, 2, n).astype(np.uint64) << np.uint64(b)
    m ^= rng.integers(0, 2, n).astype(np.uint64) * np.uint64(0x1FFFFFFF)
    m ^= rng.integers(0, 2, n).astype(np.uint64) * np.uint64(0xFFFFFC0000000)
    m &= np.uint64((1 << 52) - 1)
    for e in range(-60, 1):
        x = ((np.uint64(1023 + e) << np.uint64(52)) | m).view(np.float64)
        check(np.where(rng.integers(0, 2, n) == 1, x, -x), np.int64(rng.integers(0, 21)))


def test_zero_and_extremes():
    x = np.array([0.0, -0.0, 5e-324, -2.0**-1022, 2.0**-1060, 1.0, -1.0, 2.0**-41, 2.0**-40, -2.0**-20])
    for d in (0, 16, 20, 142):
        check(x[:5] if d > 20 else x, np.int64(d))


def test_far_elements_are_told_apart():
    """Every element that Far passes has the procedure's A', whatever its size and delta, and no element below 2^30
    (what the scale leaves, unless a range flag is raised) is sent through the procedure."""
    rng = np.random.default_rng(3)
    n = 400000
    for spread in (40, 120, 2000):
        x = rng.integers(0, 2**64, n, dtype=np.uint64).view(np.float64).copy()  # infinities and NaN among them
        u = x.view(np.uint64)
        near_range = rng.random(n) < 0.8
        E = np.clip(1023 + rng.integers(-spread, spread + 1, n), 0, 2047).astype(np.uint64)
        u[near_range] = (u[near_range] & np.uint64((1 << 63) | ((1 << 52) - 1))) | (E[near_range] << np.uint64(52))
        x[:16] = [np.inf, -np.inf, np.nan, -np.nan, 0.0, -0.0, 5e-324, 1.7976931348623157e308, 2.0**31, -(2.0**31), 2.0**30,
                  2.0**32, -(2.0**32), 1.5 * 2.0**32, -1.5 * 2.0**32, -(2.0**33)]
        d = rng.integers(-60, 60, n)
        some = rng.random(n) < 0.1
        d[some] = rng.integers(-1100, 1100, int(some.sum()))
        d[:16] = 0
        with np.errstate(all="ignore"):
            got, T = integer_and_sum(x, d)
            want = reference(x, d)
            size = np.abs(np.ldexp(x, d))
        hi = T.view(np.uint64) >> np.uint64(32)
        passed = (hi >= 0x41F00000) & (hi < 0x42000000) & (d < 541)
        assert 0.01 < passed.mean() < 0.99
        bad = np.flatnonzero(passed & (got != want))
        assert not bad.size, (x[bad[:3]], d[bad[:3]])
        assert passed[(size < 2.0**30) & (d < 541)].all()
