"""The tile grids divide a tile index by a tile count from the device: ee_tile_div.h's f32
quotient with its correction equals the integer division whatever the last bit of the hardware's
reciprocal, and the uncorrected product, which is wrong from about two million tiles on (a C of 64 GB),
is shown to fail."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "triton-kernels-optimization_amd", "csrc")
SRC = os.path.join(HERE, "tile_div_check.cpp")

pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")


def _run(tmp_path, src):
    exe = tmp_path / "tile_div_check"
    subprocess.run(["g++", "-std=c++17", "-O2", "-fopenmp", "-ffp-contract=off", "-fno-fast-math", "-I", CSRC, str(src),
                    "-o", str(exe)], check=True)
    return subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)


def test_tile_div_is_the_integer_division(tmp_path):
    out = _run(tmp_path, SRC)
    assert out.returncode == 0 and "mismatches 0" in out.stdout, out.stdout


def test_the_uncorrected_product_is_caught(tmp_path):
    text = open(SRC).read()
    call = "tile_div_rcp((int)i, t, rt)"
    assert call in text
    src = tmp_path / "variant.cpp"
    src.write_text(text.replace(call, "(int)(((float)(int)i + 0.5f) * rt)"))
    out = _run(tmp_path, src)
    assert out.returncode != 0 and "mismatch i" in out.stdout


def test_the_grids_divide_by_it():
    src = open(os.path.join(CSRC, "common", "ee_gemm_dev.h")).read()
    body = src[src.index("EE_DEV int tile_div("):]
    assert "tile_div_rcp(i, t," in body[:body.index("}")]
