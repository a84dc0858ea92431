"""What the whole Scheme II INT8 pass refuses, on every route that it can take."""
import numpy as np
import pytest

from oztt_amd.device import crt_desc, moduli_desc

pytestmark = pytest.mark.gpu

MODULI = [255, 254, 253, 251, 247, 241, 239, 233, 229, 227, 223, 217, 211, 199, 197]

# products and reconstruction in one kernel; normalization and residues in one; stage by stage; at most 64 columns
ROUTES = [(1500, 1409, 64), (100, 90, 120), (300, 300, 700), (6100, 20, 1030)]


class Pass:
    """Operands, a result filled with 3 and flags filled with 99 on the device, and the call."""

    def __init__(self, dev, M, N, K):
        rng = np.random.default_rng(M + N + K)
        self.dev, self.shape = dev, (M, N, K)
        self.A, self.B = rng.uniform(-1, 1, (M, K)), rng.uniform(-1, 1, (K, N))
        self.A[3, 0] = np.inf
        self.B[1, 2] = 2.0 ** 130
        self.md, self.cd = moduli_desc(MODULI, 3), crt_desc(MODULI, 54, 3)

    def run(self):
        dev, (M, N, K) = self.dev, self.shape
        bA, bB, bC = dev.upload(self.A), dev.upload(self.B), dev.upload(np.full(M * N, 3.0))
        fl = dev.upload(np.full(2, 99, np.uint32))
        need = dev.gemm_f64_workspace(M, N, K, len(MODULI))
        work = dev.alloc(need)
        try:
            dev.gemm_f64(bA, K, bB, N, bC, N, M, N, K, self.md, self.cd, fl, work, need)
            refused = None
        except RuntimeError as e:
            refused = str(e)
        got = dev.download(bC, np.float64, M * N), tuple(dev.download(fl, np.uint32, 2))
        for x in list(dev.bufs):
            x.free()
        dev.bufs.clear()
        return refused, *got


@pytest.mark.parametrize("M,N,K", ROUTES)
@pytest.mark.parametrize("nw", [0, 2, 3, 9])
def test_accumulator_words(dev, M, N, K, nw):
    # 15 moduli: S M takes 122 bits, four words
    p = Pass(dev, M, N, K)
    p.cd.nw = nw
    refused, C, flags = p.run()
    assert refused and "oz2_crt_digits_f64" in refused
    assert np.all(C == 3.0)
    assert flags == (4, 1)  # the refusal comes after the scale: what it found, as in a pass that runs
    p.cd.nw = 4
    p.A[3, 0] = p.B[1, 2] = 1.0
    assert p.run()[2] == (0, 0)  # and the next pass finds nothing of it


@pytest.mark.parametrize("M,N,K", ROUTES)
@pytest.mark.parametrize("nw", [4, 8])
def test_accumulator_words_that_hold(dev, M, N, K, nw):
    p = Pass(dev, M, N, K)
    p.cd.nw = nw
    refused, C, flags = p.run()
    assert refused is None and flags == (4, 1)
    assert not np.any(C == 3.0)
