"""The code generated for the kernels that copy operands into LDS by inline asm, besides those of
test_gemm_asm.py: M0, which the copy sets itself, serves nothing else, and nothing spills (scratch accesses
would enter the counts that the copies' waits rely on)."""
import re
import subprocess

import pytest

from oztt_amd import build as B

SOURCES = {"oz_gemm_tiles.hip": "gemm_i8_", "oz2_gemm_crt.hip": "gemm_crt_kernel", "oz2_skinny.hip": "skinny_kernel"}


@pytest.mark.parametrize("src", sorted(SOURCES))
def test_m0_and_spills(src, tmp_path):
    out = tmp_path / "x.s"
    cmd = [B.HIPCC, *B.HIP_FLAGS, *B.HIP_SOURCES[src], "--cuda-device-only", "-S", str(B.CSRC / src), "-o", str(out)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    asm = out.read_text()
    body = [l.strip() for l in asm.split("\n") if l.strip() and not l.strip().startswith(";")]
    m0 = [i for i, l in enumerate(body) if re.search(r"\bm0\b", l) and not l.startswith(".")]
    assert all(re.match(r"s_mov_b32 m0, (s\d+|vcc_lo|vcc_hi)$", body[i]) for i in m0)
    assert all(body[i + 1].startswith("global_load_lds_dwordx4") for i in m0)
    assert sum(l.startswith("global_load_lds") for l in body) == len(m0)
    meta = re.findall(r"\.name:\s+(_Z\S*" + SOURCES[src] + r"\S*)\s.*?\.private_segment_fixed_size:\s+(\d+).*?"
                      r"\.vgpr_spill_count:\s+(\d+)", asm, re.S)
    assert meta and all(p == "0" and s == "0" for _, p, s in meta), meta


@pytest.mark.parametrize("src,stem", [("oz_scale.hip", "scale_pair_kernel"), ("oz2_prep.hip", "prep_kernel"),
                                      ("oz2_split.hip", "split_"), ("oz2_crt.hip", "crt_digits_kernel")])
def test_no_spills(src, stem, tmp_path):
    # kernels whose registers are held down by launch bounds, or close to a step of the occupancy
    out = tmp_path / "x.s"
    cmd = [B.HIPCC, *B.HIP_FLAGS, *B.HIP_SOURCES[src], "--cuda-device-only", "-S", str(B.CSRC / src), "-o", str(out)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    meta = re.findall(r"\.name:\s+(_Z\S*" + stem + r"\S*)\s.*?\.private_segment_fixed_size:\s+(\d+).*?"
                      r"\.vgpr_spill_count:\s+(\d+)", out.read_text(), re.S)
    assert meta and all(p == "0" and s == "0" for _, p, s in meta), meta
