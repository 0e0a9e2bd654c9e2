"""The random stream's device code itself, jne_rng.h, built for the host and compared with
the oracle's stream bit for bit (CPU): 2 ln(u1) for every u1 the stream can produce, the
quadrant turn near the angles where a sign of zero could differ, and the Philox block
function.  Built with the clang that compiles the device code: gcc turns -fma(a, b, c) into
fma(-a, b, -c), which has the other zero.  The square root rests on v_rsq_f32's own
results, so it is checked on the GPU (test_rng_check_gpu.py)."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(ROOT, "johansen-null-eigenspectra_amd", "csrc")
CLANG = shutil.which("amdclang++") or shutil.which("clang++", path="/opt/rocm/llvm/bin")


def build(tmp_path, csrc=CSRC):
    dev, ora, exe = (str(tmp_path / n) for n in ("dev.o", "oracle.o", "forms"))
    flags = ["-O2", "-mfma", "-ffp-contract=off", "-c"]
    subprocess.run([CLANG, "-std=c++17", *flags, "-I", os.path.join(HERE, "hip_stub"), "-I", csrc,
                    os.path.join(HERE, "stream_forms.cpp"), "-o", dev], check=True)
    subprocess.run(["gcc", "-std=c11", *flags, "-I", os.path.join(ROOT, "oracle"),
                    os.path.join(HERE, "stream_forms_oracle.c"), "-o", ora], check=True)
    subprocess.run(["g++", dev, ora, "-o", exe, "-lm", "-lpthread"], check=True)
    return exe


needs_compilers = pytest.mark.skipif(CLANG is None or shutil.which("gcc") is None, reason="no clang or gcc")


@needs_compilers
def test_the_device_stream_equals_the_oracle(tmp_path):
    res = subprocess.run([build(tmp_path)], capture_output=True, text=True, timeout=300)
    assert res.returncode == 0 and res.stdout.count(" 0/") == 3, res.stdout + res.stderr


@needs_compilers
@pytest.mark.parametrize("was,wrong,differ", [("& 0xFF800000u", "& 0xFF000000u", "radius"),
                                              ("0x1.05c61p-51f", "0x1.05c61p-52f", "radius"),
                                              ("0x80000000u, 0xD2)", "0x80000000u, 0x78)", "turn"),
                                              ("k1 += kPhiloxW1", "k1 += kPhiloxW0", "philox")])
def test_a_wrong_form_is_seen(tmp_path, was, wrong, differ):
    """The comparison fails for a wrong mask, constant, sign table or key schedule."""
    text = open(os.path.join(CSRC, "jne_rng.h")).read()
    assert text.count(was) == 1
    (tmp_path / "jne_rng.h").write_text(text.replace(was, wrong))
    (tmp_path / "out").mkdir()
    res = subprocess.run([build(tmp_path / "out", str(tmp_path))], capture_output=True, text=True, timeout=300)
    assert res.returncode == 1 and f"{differ} 0/" not in res.stdout, res.stdout + res.stderr
