"""The whole Scheme II INT8 pass where it takes steps together, against the same pass run stage by stage
(checked against the oracle elsewhere), bit for bit: products and reconstruction in one kernel
(oz2_gemm_crt.hip: short K, large results), normalization and residues in one (oz2_prep.hip: short K),
and the range flags that the last kernel hands over."""
import ctypes

import numpy as np
import pytest

import oztt_amd as oz
from oztt_amd.device import crt_desc, hip, moduli_desc

pytestmark = pytest.mark.gpu


def operands(M, N, K, seed, phi):
    rng = np.random.default_rng(seed)
    A = rng.uniform(-0.5, 0.5, (M, K)) * np.exp(phi * rng.normal(0, 1, (M, K)))
    B = rng.uniform(-0.5, 0.5, (K, N)) * np.exp(phi * rng.normal(0, 1, (K, N)))
    A[1] = 0.0                      # zero rows and columns: C' = 0
    B[:, 2] = 0.0
    A[3] = 0.0
    A[3, 0] = 1.0                   # single elements
    A[4] = np.abs(A[4]) + 1e-3      # parallel to column 5: sums near the bound
    B[:, 5] = A[4]
    A[6] = -A[4]
    A[7] *= 2.0 ** -600             # maxima below the range: a flag, no digits, zeros
    B[:, 8] *= 2.0 ** -500
    if M > 9:
        A[8] *= 2.0 ** -125 / np.abs(A[8]).max()   # the smallest exponents that results have (2^-252 and less)
    if N > 9:
        B[:, 9] *= 2.0 ** -125 / np.abs(B[:, 9]).max()
    return A, B


PREP, FUSED, PART = 1, 2, 4  # ways of a pass (oz_rules.hip)


@pytest.mark.parametrize("M,N,K,phi,width", [
    (1500, 1409, 64, 0.5, 0), (2048, 1024, 128, 0.5, 0), (1473, 1472, 250, 1.0, 0), (1440, 1473, 193, 2.0, 0),
    (700, 3300, 1, 0.5, 0), (1500, 1409, 256, 0.5, 30), (1500, 1409, 256, 4.0, 60), (1500, 1409, 256, 0.5, 66),
    (1409, 1500, 100, 2.0, 70),
])
def test_fused_pass_equals_the_stages(dev, M, N, K, phi, width):
    A, B = operands(M, N, K, M + K, phi)
    assert pass_equals_stages(dev, A, B, M, N, K, width) == PREP | FUSED


# deltas and planes in one launch (oz2_prep.hip): 4 elements per lane up to K = 256, 8 up to 512, bands and
# blocks with padding, 3 to 5 digits
@pytest.mark.parametrize("M,N,K,width", [
    (9, 9, 1, 0), (17, 33, 64, 0), (100, 60, 33, 0), (128, 128, 128, 0), (300, 65, 256, 66), (40, 31, 200, 84),
    (256, 4000, 512, 0), (3900, 300, 449, 0), (2048, 2049, 300, 30),
    (70, 90, 256, 86), (9, 17, 1, 80),
])
def test_prepared_pass_equals_the_stages(dev, M, N, K, width):
    A, B = operands(M, N, K, M + K, 1.0)
    assert pass_equals_stages(dev, A, B, M, N, K, width) & PREP


# at most 64 columns (oz2_skinny.hip): K in one part and in two, uneven halves, ragged rows, columns and K,
# elements in 16-byte pairs (odd K here) and single ones, few moduli, and 17 of them and more (not taken)
@pytest.mark.parametrize("M,N,K,phi,width", [
    (6081, 64, 1024, 0.5, 0), (6100, 9, 1089, 1.0, 0), (8191, 33, 1027, 2.0, 0), (12290, 61, 1100, 0.5, 0),
    (12225, 64, 1025, 0.5, 30), (6144, 64, 1152, 0.5, 40), (6081, 63, 1999, 4.0, 0), (6144, 17, 1024, 0.5, 66),
    (8191, 33, 1027, 0.5, 0), (6081, 63, 1999, 0.5, 0),
])
def test_narrow_pass_equals_the_stages(dev, M, N, K, phi, width):
    A, B = operands(M, N, K, M + K, phi)
    # (17 moduli by the spread of the elements, and by the width)
    taken = width != 66 and phi not in (2.0, 4.0)
    assert pass_equals_stages(dev, A, B, M, N, K, width) // PART == (0 if not taken else 1 if M > 12224 else 2)


def test_range_flags(dev):
    # the flags of a pass are its own: set by one, clear again in the next; infinities, maxima below 2^-126 and
    # above the largest BF16 on either side, through every route of the pass
    for M, N, K in [(64, 48, 100), (64, 48, 700), (1500, 1409, 64), (2048, 2048, 512), (6100, 20, 1030)]:
        A, B = operands(M, N, K, 5, 0.5)
        bad = A.copy()
        bad[0, 0], bad[5, K - 1], bad[9, 0] = np.inf, 2.0**130, 1.0
        tiny = B.copy()
        tiny[:, 1] = 2.0**-200
        # (A's row 7 and B's column 8 of operands() are below 2^-126 already)
        clean = A.copy(), B.copy()
        clean[0][7], clean[1][:, 8] = 1.0, 1.0
        plan = clean
        for X, Y, want in [(clean[0], clean[1], (0, 0)), (bad, clean[1], (4 | 1 | 2, 0)), (clean[0], tiny, (0, 2)),
                           (clean[0], clean[1], (0, 0))]:
            pass_equals_stages(dev, X, Y, M, N, K, 0, plan, want)


# Rows and columns with a range flag: infinities, NaN, values above the largest BF16, alone and beside values whose
# scaled digits do not fit (the even modulus of such elements is no residue of their A'). One size of every route; of
# the narrow one both parts of K, few moduli, and 2 as the even one.
@pytest.mark.parametrize("M,N,K,width,moduli", [
    (100, 90, 120, 0, None), (300, 4000, 512, 0, None), (300, 300, 700, 0, None), (1500, 1409, 64, 0, None),
    (1500, 1409, 200, 66, None), (300, 65, 256, 84, None), (6100, 20, 1030, 0, None), (12290, 64, 1100, 0, None), (6081, 64, 1999, 0, None), (6100, 33, 1024, 30, None),
    (6144, 17, 1100, 0, [255, 253, 251, 247, 2, 241, 239, 233, 229, 227, 223, 217, 211, 199, 197, 193]),
    (8192, 24, 1100, 0, [255, 254, 253, 251]),
    (6144, 9, 1100, 0, [255, 253, 251, 247, 241, 239, 233, 229, 227, 223, 217, 211, 199, 197, 193]),
])
def test_flagged_operands_equal_the_stages(dev, M, N, K, width, moduli):
    A, B = operands(M, N, K, M + K, 0.5)
    rng = np.random.default_rng(K)
    for X, n, axis in ((A, K, 0), (B.T, K, 1)):
        X[0, n - 1], X[3, n // 2] = np.inf, np.nan
        if len(X) < 16:
            continue
        X[9, 0] = 2.0 ** 130
        X[10] *= 2.0 ** 140
        X[11] *= np.exp2(rng.integers(0, 60, n))
        X[11, 0] = -np.inf
        X[12] *= np.exp2(rng.integers(-60, 1000, n))
        X[13] = 2.0 ** -1060
        X[15, n - 1] = 2.0 ** 128
    A[M - 1, K - 1], A[M // 2, K // 2] = np.nan, -np.inf  # by themselves in their rows and K blocks
    way = pass_equals_stages(dev, A, B, M, N, K, width, operands(M, N, K, 1, 0.5), moduli=moduli)
    assert way == (PREP | FUSED if M == 1500 else PREP if K <= 512 else 0 if M == 300 else PART if M > 12224 else 2 * PART)


# One such element per row, beside values that its flag leaves larger than the scale would: their digits hold, but not in
# the bytes that the narrow kernel makes of A' (the even modulus again). Between 2^2 and 2^20, in rows that have the flag's
# element in the first K block, the last, and the middle one (K in two parts for the last two).
@pytest.mark.parametrize("M,N,K", [(12290, 64, 1100), (6100, 20, 1030), (8192, 64, 2048)])
@pytest.mark.parametrize("log2", [2, 6, 7, 8, 9, 12, 16, 20])
def test_flagged_rows_with_large_values_equal_the_stages(dev, M, N, K, log2):
    A, B = operands(M, N, K, M + K, 0.5)
    rows = np.arange(9, M, 97)
    A[rows] *= 2.0 ** log2
    A[rows, np.array([0, K // 2, K - 1])[rows % 3]] = np.array([np.inf, 2.0 ** 130, np.nan])[rows % 3]
    assert pass_equals_stages(dev, A, B, M, N, K, 0, operands(M, N, K, 1, 0.5)) // PART in (1, 2)


def pass_equals_stages(dev, A, B, M, N, K, width, plan=None, want_flags=None, moduli=None):
    # width 0: the plan; up to 60 bits: the plan at that width; above: the moduli for it, in four or five digits (the
    # planner stops at 16 moduli)
    PA, PB = plan or (A, B)
    if width > 60:
        p, b, nd = oz.choose_moduli_int8(K, 24, width), width, -(-width // 20)
    else:
        p = oz.plan2_int8(PA.ravel(), PB.ravel(), M, N, K, fixed_bits=width)
        b, nd = p.b, p.nd
    moduli = moduli or [p.m[i] for i in range(p.S)]
    S = len(moduli)
    md, cd = moduli_desc(moduli, nd), crt_desc(moduli, b, nd)
    lda, ldb, ldc = K + 3, N + 5, N + 7
    a, b = np.zeros((M, lda)), np.zeros((K, ldb))
    a[:, :K], b[:, :N] = A, B
    bA, bB = dev.upload(a), dev.upload(b)
    bC = dev.upload(np.full((M, ldc), -7.0))
    fl = dev.alloc(16)
    need = dev.gemm_f64_workspace(M, N, K, S)
    work = dev.alloc(need)
    dev.gemm_f64(bA, lda, bB, ldb, bC, ldc, M, N, K, md, cd, fl, work, need)
    got = dev.download(bC, np.float64, M * ldc).reshape(M, ldc)
    # the stages
    Mg, Ng, Kg = -(-M // 256) * 256, -(-N // 256) * 256, -(-K // 64) * 64
    dA, dB, f2 = dev.alloc(4 * M), dev.alloc(4 * N), dev.upload(np.zeros(2, np.uint32))
    pA, pB, dg, out = dev.alloc(S * Mg * Kg), dev.alloc(S * Ng * Kg), dev.alloc(S * Mg * Ng), dev.alloc(8 * M * N)
    dev.scale_pair(bA, M, K, lda, bB, N, ldb, 1, cd.shift, dA, dB, f2)
    dev.split_pair_int8(bA, M, K, lda, dA, bB, N, ldb, dB, md, pA, pB, Mg, Ng, Kg)
    dev.gemm_digits(pA, pB, dg, Mg, Ng, Kg, S, Ng, Mg * Kg, Ng * Kg, Mg * Ng, cd)
    dev.crt_digits(dg, M, N, Ng, Mg * Ng, cd, dA, dB, out, N)
    want = dev.download(out, np.float64, M * N).reshape(M, N)
    if plan is None:
        assert not want[1].any() and not want[:, 2].any()
    np.testing.assert_array_equal(got[:, :N].view(np.uint64), want.view(np.uint64))
    assert np.all(got[:, N:] == -7.0)
    flags = dev.download(fl, np.uint32, 2)
    np.testing.assert_array_equal(flags, dev.download(f2, np.uint32, 2))
    if want_flags:
        assert tuple(flags) == want_flags
    for x in (bA, bB, bC, fl, work, dA, dB, f2, pA, pB, dg, out):
        x.free()
    dev.bufs.clear()
    return hip().oz_rule_pass(256, ctypes.byref(md), ctypes.byref(cd), M, N, K)
