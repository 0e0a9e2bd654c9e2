"""The normal transform's square root at every radius word (all 2^32), on the GPU."""
import json
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
TOOL = os.path.join(ROOT, "johansen-null-eigenspectra_amd", "bin", "jne_rng_check")


@pytest.mark.gpu
def test_every_root_is_correctly_rounded():
    res = subprocess.run([TOOL], capture_output=True, text=True, timeout=60)
    assert res.returncode in (0, 1), res.stderr
    got = json.loads(res.stdout)
    assert res.returncode == 0 and got["differ"] == 0 and got["words"] == 1 << 32, got
