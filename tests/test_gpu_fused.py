"""The whole Scheme II INT8 pass where it computes products and reconstruction in one kernel
(oz2_gemm_crt.hip: short K, large results), against the same pass run stage by stage through the digits
(checked against the oracle elsewhere), bit for bit."""
import numpy as np
import pytest

import oztt_amd as oz
from oztt_amd.device import crt_desc, moduli_desc

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
    A[7] *= 2.0 ** -600             # results below the normal range once multiplied
    B[:, 8] *= 2.0 ** -500
    return A, B


@pytest.mark.parametrize("M,N,K,phi,width", [
    (1500, 1409, 64, 0.5, 0), (2048, 1024, 128, 0.5, 0), (1473, 1472, 250, 1.0, 0), (1440, 1473, 193, 2.0, 0),
    (700, 3300, 1, 0.5, 0), (1500, 1409, 256, 0.5, 30), (1500, 1409, 256, 4.0, 60),
])
def test_fused_pass_equals_the_stages(dev, M, N, K, phi, width):
    A, B = operands(M, N, K, M + K, phi)
    p = oz.plan2_int8(A.ravel(), B.ravel(), M, N, K, fixed_bits=width)
    moduli = [p.m[i] for i in range(p.S)]
    md, cd = moduli_desc(moduli, p.nd), crt_desc(moduli, p.b, p.nd)
    lda, ldb, ldc = K + 3, N + 5, N + 7
    a, b = np.zeros((M, lda)), np.zeros((K, ldb))
    a[:, :K], b[:, :N] = A, B
    bA, bB = dev.upload(a), dev.upload(b)
    bC = dev.upload(np.full((M, ldc), -7.0))
    fl = dev.alloc(16)
    need = dev.gemm_f64_workspace(M, N, K, p.S)
    work = dev.alloc(need)
    dev.gemm_f64(bA, lda, bB, ldb, bC, ldc, M, N, K, md, cd, fl, work, need)
    got = dev.download(bC, np.float64, M * ldc).reshape(M, ldc)
    # the stages
    Mg, Ng, Kg = -(-M // 256) * 256, -(-N // 256) * 256, -(-K // 64) * 64
    dA, dB, f2 = dev.alloc(4 * M), dev.alloc(4 * N), dev.upload(np.zeros(2, np.uint32))
    pA, pB, dg, out = dev.alloc(p.S * Mg * Kg), dev.alloc(p.S * Ng * Kg), dev.alloc(p.S * Mg * Ng), dev.alloc(8 * M * N)
    dev.scale_pair(bA, M, K, lda, bB, N, ldb, 1, cd.shift, dA, dB, f2)
    dev.split_pair_int8(bA, M, K, lda, dA, bB, N, ldb, dB, md, pA, pB, Mg, Ng, Kg)
    dev.gemm_digits(pA, pB, dg, Mg, Ng, Kg, p.S, Ng, Mg * Kg, Ng * Kg, Mg * Ng, cd)
    dev.crt_digits(dg, M, N, Ng, Mg * Ng, cd, dA, dB, out, N)
    want = dev.download(out, np.float64, M * N).reshape(M, N)
    assert not want[1].any() and not want[:, 2].any()
    np.testing.assert_array_equal(got[:, :N].view(np.uint64), want.view(np.uint64))
    assert np.all(got[:, N:] == -7.0)
    np.testing.assert_array_equal(dev.download(fl, np.uint32, 2), dev.download(f2, np.uint32, 2))
    for x in (bA, bB, bC, fl, work, dA, dB, f2, pA, pB, dg, out):
        x.free()
    dev.bufs.clear()
