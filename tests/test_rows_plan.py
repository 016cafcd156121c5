"""The host-side rules of the denoiser's row kernel (gartus_amd/csrc/rows_plan.h): which layers take it. CPU
only: the rules are compiled with g++ through tests/rows_plan_shim.cpp."""
import ctypes as C
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent


@pytest.fixture(scope="module")
def shim(tmp_path_factory):
    out = tmp_path_factory.mktemp("shim") / "librowsplan.so"
    subprocess.run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-o", str(out),
                    str(ROOT / "tests" / "rows_plan_shim.cpp")], check=True)
    return C.CDLL(str(out))


def test_an_encoder_layer_of_80_to_32_takes_the_row_kernel(shim):
    """k_conv takes twice as long on it at 1920x1080. Only that forward layer has an instance of 80 channels."""
    assert shim.shim_rows_frags(0, 80, 32, 0) == 2
    assert shim.shim_rows_frags(0, 80, 32, 1) == 0
    assert all(shim.shim_rows_frags(0, 80, c, 0) == 0 for c in (16, 48, 64, 80, 96, 112, 128))
