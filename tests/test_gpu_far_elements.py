"""Residue planes of elements that the scale flags (infinities, NaN, values above the largest BF16 and what shares
their row or column, nothing of which has a place in the digits): still those of the binary32 digit procedure, for
which oz2_digits_f32 gives the digits and layout 0 the even modulus. Bit for bit, in every blocked splitter."""
import numpy as np
import pytest

from oztt_amd.device import from_blocks, moduli_desc

pytestmark = pytest.mark.gpu

MODULI = [255, 254, 253, 251, 7, 13, 193]
SHIFT = 14  # b = 54, three digits


def spoilt(rng, n, k):
    """n x k, rows of every kind between ordinary ones."""
    X = rng.uniform(-1, 1, (n, k))
    X[0, k - 1] = np.inf
    X[2, 0] = np.nan
    X[3, k // 2] = 2.0 ** 130
    X[5] *= 2.0 ** 140                                                    # nothing but elements above the range
    X[6] *= np.exp2(rng.integers(0, 60, k))                               # digits of 2^30 and more beside an infinity
    X[6, 0] = -np.inf
    X[8] *= np.exp2(rng.integers(-60, 1020, k))
    X[8, k - 1] = -np.nan
    X[9] = 2.0 ** -1060
    X[10, 0] = 2.0 ** 128
    X[n - 1, k - 1] = np.inf
    return X


def procedure_planes(dev, bX, rows, cols, mode, bd, shape):
    """The planes (MODULI x rows x cols) from the procedure's digits."""
    out = dev.alloc(12 * rows * cols)
    dev.digits(bX, rows, cols, cols, mode, bd, 3, out)
    dig = dev.download(out, np.float32, 3 * rows * cols).reshape(rows, cols, 3).astype(np.float64)
    i = np.clip(np.nan_to_num(dig, nan=0.0), -2**31, 2**31 - 1).astype(np.int64).view(np.uint64)  # as the GPU converts
    y = (i[..., 0] << np.uint64(40)) + (i[..., 1] << np.uint64(20)) + i[..., 2] + np.uint64(0x8080808080808080)
    a = [(((y >> np.uint64(8 * j)) & np.uint64(255)).astype(np.int64) - 128) for j in range(8)]  # balanced bytes
    prow, pld = -(-rows // 64) * 64, -(-cols // 64) * 64
    row0 = dev.alloc(len(MODULI) * prow * pld)
    dev.split_int8(bX, rows, cols, cols, mode, bd, moduli_desc(MODULI, 3), row0, 0, prow, pld, prow * pld)
    chain = dev.download(row0, np.int8, len(MODULI) * prow * pld).reshape(len(MODULI), prow, pld)[:, :rows, :cols]
    want = np.zeros((len(MODULI),) + shape, np.int8)
    for s, m in enumerate(MODULI):
        r = sum(a[j] * (pow(256, j, m)) for j in range(8)) % m
        r = np.where(r > m // 2, r - m, r)
        r = chain[s] if m % 2 == 0 else r
        if mode == 0:
            want[s, :rows, :cols] = r
        else:
            want[s, :cols, :rows] = r.T
    return want


# A (rows) and B (columns), in 4 elements per lane (oz2_split_pair_int8, few blocks), in 16 (more blocks), ragged
# and whole blocks, and one operand at a time (oz2_split_int8)
@pytest.mark.parametrize("M,N,K", [(40, 27, 100), (64, 64, 64), (1100, 1056, 1030), (2048, 1024, 1024)])
def test_far_elements(dev, M, N, K):
    rng = np.random.default_rng(M + N + K)
    A, B = spoilt(rng, M, K), np.ascontiguousarray(spoilt(rng, N, K).T)
    md, S = moduli_desc(MODULI, 3), len(MODULI)
    Mg, Ng, Kg = -(-M // 16) * 16, -(-N // 16) * 16, -(-K // 64) * 64
    bA, bB, dA, dB = dev.upload(A), dev.upload(B), dev.alloc(4 * M), dev.alloc(4 * N)
    fl = dev.upload(np.zeros(2, np.uint32))
    dev.scale_pair(bA, M, K, K, bB, N, N, 1, SHIFT, dA, dB, fl)
    assert tuple(dev.download(fl, np.uint32, 2)) == (7, 7)
    wA = procedure_planes(dev, bA, M, K, 0, dA, (Mg, Kg))
    wB = procedure_planes(dev, bB, K, N, 1, dB, (Ng, Kg))
    pA, pB = dev.alloc(S * Mg * Kg), dev.alloc(S * Ng * Kg)

    def check(what):
        for p, R, want in ((pA, Mg, wA), (pB, Ng, wB)):
            got = from_blocks(dev.download(p, np.int8, S * R * Kg).reshape(S, R * Kg), R, Kg)
            np.testing.assert_array_equal(got, want, err_msg=what)

    dev.split_pair_int8(bA, M, K, K, dA, bB, N, N, dB, md, pA, pB, Mg, Ng, Kg)
    check("pair")
    dev.fill_u32(pA, 0x55555555, S * Mg * Kg // 4)
    dev.fill_u32(pB, 0x55555555, S * Ng * Kg // 4)
    dev.split_int8(bA, M, K, K, 0, dA, md, pA, 2, Mg, Kg, Mg * Kg)
    dev.split_int8(bB, K, N, N, 1, dB, md, pB, 3, Ng, Kg, Ng * Kg)
    check("one operand")
    for x in list(dev.bufs):
        x.free()
    dev.bufs.clear()


def test_deltas_of_a_callers_own(dev):
    # scaled far beyond the digits, and subnormal elements (zero to the procedure) scaled up to where they would have some
    M, N, K = 18, 17, 70
    rng = np.random.default_rng(1)
    A, B = rng.uniform(-1, 1, (M, K)), rng.uniform(-1, 1, (K, N))
    A[0], B[:, 1] = 2.0 ** -1030, 2.0 ** -1040
    d = np.array([1030, 28, 29, 30, 31, 60, 100, 170, 200, -300, -1200, 541, 540, 14, 14, 14, 14, 14], np.int32)
    bA, bB, dA, dB = dev.upload(A), dev.upload(B), dev.upload(d), dev.upload(np.roll(d, 1)[:N].copy())
    Mg, Ng, Kg, S = 32, 32, 128, len(MODULI)
    pA, pB = dev.alloc(S * Mg * Kg), dev.alloc(S * Ng * Kg)
    dev.split_pair_int8(bA, M, K, K, dA, bB, N, N, dB, moduli_desc(MODULI, 3), pA, pB, Mg, Ng, Kg)
    for p, R, want in ((pA, Mg, procedure_planes(dev, bA, M, K, 0, dA, (Mg, Kg))),
                       (pB, Ng, procedure_planes(dev, bB, K, N, 1, dB, (Ng, Kg)))):
        got = from_blocks(dev.download(p, np.int8, S * R * Kg).reshape(S, R * Kg), R, Kg)
        np.testing.assert_array_equal(got, want)
    for x in list(dev.bufs):
        x.free()
    dev.bufs.clear()
