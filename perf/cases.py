"""What is timed when the framework's speed is looked at: FP64 products C = A B by the Ozaki schemes,
over the sizes and options its users bring, and not only the benchmark's.

Three kinds of programs are stood for:

  "pass"      a program that keeps FP64 matrices in GPU memory and a plan for them, and calls the C ABI's
              whole Scheme II INT8 pass on them (oz2_gemm_f64): C stays on the GPU, calls are queued.
  "scheme1",  the same for Scheme I and for Scheme II on the FP8 matrix cores, whose stages such a
  "fp8"       program calls one by one (scale, split, products, reconstruction).
  "host"      a program that calls Context.gemm on its own host arrays (the drop-in interface).
  "resident"  a program that uploads its operands once (Context.upload) and reads every product back.

Inputs follow the evaluation's distribution, (U(0,1) - 0.5) exp(phi N(0,1)).

Every result is defined bit for bit: the integer products are exact, Scheme II reconstructs the exact
integer product of the scaled operands and rounds it once, and Scheme I is the reference's own sequence
of operations. So tolerance() is "exact" for every case.
"""
import math

import numpy as np
import torch

import oztt_amd as oz
from oztt_amd import device as ozd


def listed():
    return [
        # the smallest call of the evaluation's tables (128^3): five launches, nothing but latency
        {"name": "pass_128", "kind": "pass", "m": 128, "n": 128, "k": 128, "phi": 0.5, "pad": 0},
        # the benchmark's small configuration, one product of a medium dense step
        {"name": "pass_1024", "kind": "pass", "m": 1024, "n": 1024, "k": 1024, "phi": 0.5, "pad": 0},
        # sizes that fit no tile, operands that are windows of larger matrices
        {"name": "pass_ragged", "kind": "pass", "m": 1000, "n": 700, "k": 1500, "phi": 1.0, "pad": 10},
        # the trailing update of a blocked LU, Cholesky or QR: a large matrix, a panel's inner dimension
        {"name": "pass_update", "kind": "pass", "m": 4096, "n": 4096, "k": 256, "phi": 0.5, "pad": 0},
        # a matrix on a block of vectors (subspace iteration, many right-hand sides)
        {"name": "pass_block_vectors", "kind": "pass", "m": 8192, "n": 64, "k": 8192, "phi": 0.5, "pad": 0},
        # inner products of two sets of long vectors (Gram and overlap matrices)
        {"name": "pass_gram", "kind": "pass", "m": 256, "n": 256, "k": 32768, "phi": 0.5, "pad": 0},
        # the benchmark's headline, the largest
        {"name": "pass_8192", "kind": "pass", "m": 8192, "n": 8192, "k": 8192, "phi": 0.5, "pad": 0},
        # Scheme I with automatic slices, the benchmark's INT8 configuration
        {"name": "scheme1_int8_4096", "kind": "scheme1", "format": "INT8", "slices": 0, "m": 4096, "n": 4096, "k": 4096, "phi": 1.0},
        # Scheme I, BF16 digits (radix 64), fixed slices: the benchmark's long inner dimension at a smaller size
        {"name": "scheme1_bf16_long", "kind": "scheme1", "format": "BF16", "slices": 8, "m": 1024, "n": 1024, "k": 8192, "phi": 4.0},
        # Scheme II on the FP8 matrix cores at the smallest size of the reference's large tables
        {"name": "fp8_3520", "kind": "fp8", "m": 3520, "n": 3520, "k": 3520, "phi": 2.0},
        # the drop-in call on host arrays: validation, planning, both transfers
        {"name": "host_600", "kind": "host", "format": "INT8", "m": 600, "n": 400, "k": 500, "phi": 0.5},
        # operands kept on the GPU, the product read back each time
        {"name": "resident_2048", "kind": "resident", "format": "INT8", "m": 2048, "n": 2048, "k": 2048, "phi": 0.5},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    # a whole pass twice as often as each of the others
    kind = rng.choice(["pass"] * 6 + ["scheme1"] * 2 + ["fp8", "host", "resident"])
    phi = rng.choice([0.5, 0.5, 1.0, 2.0])
    if kind == "pass":
        # shapes from cubes to updates, block vectors and Gram matrices: every extent by itself
        lo, hi, most, kmax = 48, 8192, 4096.0**3, 32768
    elif kind in ("scheme1", "fp8"):
        lo, hi, most, kmax = 100, 4096, 3000.0**3, 8192
    else:
        lo, hi, most, kmax = 64, 2000, 1500.0**3, 3000
    while True:
        c = {"kind": kind, "m": _log(rng, lo, hi), "n": _log(rng, lo, hi), "k": _log(rng, lo, kmax), "phi": phi}
        if rng.random() < 0.4:  # some of them multiples of the tiles
            c.update({x: -(-c[x] // 64) * 64 for x in "mnk"})
        if float(c["m"]) * c["n"] * c["k"] <= most and c["k"] * max(c["m"], c["n"]) <= 2**26:
            break
    if kind == "pass":
        c["pad"] = rng.choice([0, 0, 0, 6, 17])
    elif kind == "scheme1":
        c["format"], c["slices"] = rng.choice([("INT8", 0), ("INT8", 7), ("BF16", 8), ("BFP8", 10)])
    elif kind in ("host", "resident"):
        c["format"] = "INT8"
    return c


# ---- inputs -----------------------------------------------------------------------------------------

_DEV = None


def _device():
    """The program's device handle: one stream, as one thread of a program has."""
    global _DEV
    if _DEV is None:
        _DEV = ozd.Device(0)
    return _DEV


_CTX = None


def _context():
    global _CTX
    if _CTX is None:
        _CTX = oz.Context()
    return _CTX


class _Ptr:
    """A torch tensor as the device wrapper's buffer."""

    def __init__(self, t):
        import ctypes

        self.t, self.ptr = t, ctypes.c_void_p(t.data_ptr())

    def offset(self, nbytes):
        import ctypes

        return ctypes.c_void_p(self.t.data_ptr() + int(nbytes))


def _operands(case, seed):
    g = torch.Generator(device="cuda:0").manual_seed(int(seed) * 2654435761 % (1 << 62))

    def matrix(rows, cols):
        u = torch.rand((rows, cols), dtype=torch.float64, device="cuda:0", generator=g) - 0.5
        z = torch.randn((rows, cols), dtype=torch.float64, device="cuda:0", generator=g)
        return u * torch.exp(case["phi"] * z)

    return matrix(case["m"], case["k"]), matrix(case["k"], case["n"])


def _bytes(n):
    return torch.empty(max(int(n), 256), dtype=torch.uint8, device="cuda:0")


def _window(x, pad):
    """x as a window of a matrix `pad` columns wider."""
    if not pad:
        return x.contiguous()
    w = torch.zeros((x.shape[0], x.shape[1] + pad), dtype=x.dtype, device=x.device)
    w[:, : x.shape[1]] = x
    return w


def prepare(case, seed):
    M, N, K, kind = case["m"], case["n"], case["k"], case["kind"]
    A, B = _operands(case, seed)
    s = {"case": case}
    if kind == "host":
        s["a"], s["b"] = A.cpu().numpy().ravel(), B.cpu().numpy().ravel()
        s["options"] = oz.Options(scheme=oz.Scheme.II, format=oz.Format[case["format"]])
        s["c"] = np.empty(M * N)
        _context()
        return s
    ha, hb = A.cpu().numpy().ravel(), B.cpu().numpy().ravel()
    if kind == "resident":
        ctx = _context()
        s["a"], s["b"] = ctx.upload(ha, M, K), ctx.upload(hb, K, N)
        s["options"] = oz.Options(scheme=oz.Scheme.II, format=oz.Format[case["format"]])
        s["c"] = np.empty(M * N)
        return s
    dev = _device()
    s["flags"] = _Ptr(torch.zeros(4, dtype=torch.int32, device="cuda:0"))
    if kind == "pass":
        p = oz.plan2_int8(ha, hb, M, N, K)
        moduli = [p.m[i] for i in range(p.S)]
        s["md"], s["cd"] = ozd.moduli_desc(moduli, p.nd), ozd.crt_desc(moduli, p.b, p.nd)
        pad = case["pad"]
        s["A"], s["B"] = _Ptr(_window(A, pad)), _Ptr(_window(B, pad))
        s["C"] = _Ptr(torch.zeros((M, N + pad), dtype=torch.float64, device="cuda:0"))
        s["work_bytes"] = dev.gemm_f64_workspace(M, N, K, p.S)
        s["work"] = _Ptr(_bytes(s["work_bytes"]))
        return s
    # the stages' operands and planes: rows in tiles of 256, K in blocks of 64
    Mg, Ng, Kg = -(-M // 256) * 256, -(-N // 256) * 256, -(-K // 64) * 64
    s["A"], s["B"] = _Ptr(A), _Ptr(B)
    s["C"] = _Ptr(torch.zeros((M, N), dtype=torch.float64, device="cuda:0"))
    s["dA"], s["dB"] = _Ptr(_bytes(4 * M)), _Ptr(_bytes(4 * N))
    s["geometry"] = Mg, Ng, Kg
    if kind == "scheme1":
        fmt = oz.Format[case["format"]]
        p = oz.plan1(ha, hb, M, N, K, case["slices"], fmt)
        # radix, digit bound, rounding of the maxima, exponent target and product kind of the format
        radix, dmax, ceil, nshift, signmag = {"INT8": (254, 127, 1, -1, 1), "BF16": (64, 32, 0, -1, 0), "BFP8": (64, 32, 0, -1, 0)}[case["format"]]
        s["fmt"] = radix, dmax, ceil, nshift
        s["p"] = p.p
        s["desc"] = ozd.Oz1ReconDesc(p.p, radix, signmag, p.nsmall, p.Whi, p.Wlo, p.qw)
        planes, outs = p.p, 4 * p.p
    else:
        s["dd"], s["gd"], s["cd"], s["terms"] = oz.plan2_fp8_device(ha, hb, M, N, K, execution_set=True)
        planes, outs = s["gd"].nplanes, 2 * s["gd"].nout
    s["pA"], s["pB"] = _Ptr(_bytes(planes * Mg * Kg)), _Ptr(_bytes(planes * Ng * Kg))
    s["products"] = _Ptr(_bytes(outs * Mg * Ng))
    return s


def run(s):
    case = s["case"]
    M, N, K, kind = case["m"], case["n"], case["k"], case["kind"]
    if kind == "host":
        _context().gemm(s["a"], s["b"], s["c"], M, N, K, s["options"])
        return s["c"]
    if kind == "resident":
        _context().gemm_resident(s["a"], s["b"], s["c"], s["options"])
        return s["c"]
    dev = _device()
    if kind == "pass":
        pad = case["pad"]
        dev.gemm_f64(s["A"], K + pad, s["B"], N + pad, s["C"], N + pad, M, N, K, s["md"], s["cd"], s["flags"], s["work"], s["work_bytes"])
        return s["C"].t, s["flags"].t
    Mg, Ng, Kg = s["geometry"]
    if kind == "scheme1":
        radix, dmax, ceil, nshift = s["fmt"]
        dev.scale_pair(s["A"], M, K, K, s["B"], N, N, ceil, nshift, s["dA"], s["dB"], s["flags"])
        dev.oz1_split_pair(s["A"], M, K, K, s["dA"], s["B"], N, N, s["dB"], s["p"], radix, dmax, s["pA"], s["pB"], Mg, Ng, Kg)
        dev.oz1_gemm_diag(s["pA"], s["pB"], s["products"], Mg, Ng, Kg, s["p"], Ng, Mg * Kg, Ng * Kg, Mg * Ng, dmax)
        dev.oz1_recon(s["products"], M, N, Ng, Mg * Ng, s["desc"], s["dA"], s["dB"], s["C"], N)
        return s["C"].t, s["flags"].t
    dev.scale_pair(s["A"], M, K, K, s["B"], N, N, 1, s["cd"].shift, s["dA"], s["dB"], s["flags"])
    dev.split_digits_pair(s["A"], M, K, K, s["dA"], s["B"], N, N, s["dB"], s["dd"], s["pA"], s["pB"], Mg, Ng, Kg)
    dev.gemm_groups_f8(s["pA"], s["pB"], s["products"], Mg, Ng, Kg, s["gd"], 1, Ng, Mg * Kg, Ng * Kg, Mg * Ng)
    dev.crt_terms(s["products"], M, N, Ng, Mg * Ng, len(s["terms"]), s["terms"], s["cd"], s["dA"], s["dB"], s["C"], N)
    return s["C"].t, s["flags"].t


# Exact products that the schemes need for one FP64 product: moduli of Scheme II INT8 and digit products of
# its FP8 route (both to a few, by the inputs), slice pairs of Scheme I (36 for 8 slices).
_PRODUCTS = {"pass": 15, "host": 15, "resident": 15, "fp8": 34, "scheme1": 36}


def work(case):
    M, N, K = case["m"], case["n"], case["k"]
    products = _PRODUCTS[case["kind"]]
    if case["kind"] == "scheme1" and case["slices"]:
        products = case["slices"] * (case["slices"] + 1) // 2
    return {"bytes": 8 * (M * K + K * N + M * N), "flops": 2 * M * N * K * products}


def tolerance(case):
    return "exact"


def exact(case, seed):
    A, B = _operands(case, seed)
    C = A @ B
    if case["kind"] in ("host", "resident"):
        return C.cpu().numpy().ravel()
    if case.get("pad"):
        C = torch.nn.functional.pad(C, (0, case["pad"]))
    return C, None
