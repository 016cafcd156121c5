"""The traversal's own arithmetic (gartus_amd/csrc/device.h) against the compiler's operators, bit for bit, on the
device. Reciprocals and roots are enumerated: every mantissa of every exponent they claim. A quotient has two operands:
every mantissa of the divisor (or, for a constant divisor, of the numerator) meets one numerator of each listed
exponent."""
import ctypes as C
from pathlib import Path

import numpy as np
import pytest
import torch  # before the libraries load: one HIP runtime per process

pytestmark = pytest.mark.gpu

LIB = Path(__file__).resolve().parent / "libdevice_math_probe.so"


@pytest.fixture(scope="module")
def probe():
    if not LIB.exists():
        from gartus_amd import build
        build.build_math_probe()
    lib = C.CDLL(str(LIB))
    p, u = C.c_void_p, C.c_uint32
    lib.probe_unary.argtypes = [C.c_int, u, u, p]
    lib.probe_div.argtypes = [u, u, u, C.c_float, p]
    lib.probe_div31.argtypes = [u, p, p, u]
    lib.probe_normalized.argtypes = [p, p, u]
    torch.cuda.synchronize()
    return lib


def _mismatches(launches):
    """What launches(counter address) counted."""
    bad = torch.zeros(1, dtype=torch.int64, device="cuda")
    torch.cuda.synchronize()
    launches(C.c_void_p(bad.data_ptr()))
    torch.cuda.synchronize()
    return int(bad.item())


def test_reciprocals_are_the_operators(probe):
    def run(bad):
        for e in range(127 - 96, 127 + 126):  # rcp_rn: 2^-96 <= |d| < 2^126
            for sign in (0, 1):
                assert probe.probe_unary(0, e, sign, bad) == 0
        for e in range(127 - 96, 255):        # reciprocal: to the largest number
            assert probe.probe_unary(1, e, 0, bad) == 0
    assert _mismatches(run) == 0


def test_roots_are_the_operators(probe):
    assert _mismatches(lambda bad: [probe.probe_unary(2, e, 0, bad) for e in range(255)]) == 0


@pytest.mark.parametrize("divisor,numerator", [(0, 0), (0, -101), (0, 100), (-60, 0), (-96, -90), (60, -27), (100, 120),
                                               (125, 125), (125, 0), (-52, 60)])
def test_quotients_are_the_operators(probe, divisor, numerator):
    """Divisors 2^divisor .. 2^(divisor + 1), numerators 2^numerator ..; the quotients are normal numbers."""
    assert _mismatches(lambda bad: [probe.probe_div(127 + divisor, 127 + numerator, seed, 0.0, bad)
                                    for seed in range(8)]) == 0


@pytest.mark.parametrize("divisor", [float(np.float32(np.pi)), float(np.float32(2 * np.pi)), 3.0, 7.0, 33.0, 2047.0,
                                     2048.0, 16777215.0])
def test_quotients_of_constants_are_the_operators(probe, divisor):
    """Pi, 2 pi and environment widths under every numerator of 2^-60 to 2^31."""
    assert _mismatches(lambda bad: [probe.probe_div(0, 127 + e, 1, divisor, bad) for e in range(-60, 32)]) == 0


def test_index_quotients_are_exact(probe):
    rng = np.random.default_rng(1)
    top = (1 << 31) - 1
    divisors = [1, 2, 3, 5, 7, 641, 1919, 1920, 2047, 2048, 2049, 65535, 65537, 2073600, (1 << 30) - 1, 1 << 30,
                (1 << 30) + 1, top, 1 << 31] + [int(d) for d in rng.integers(1, 1 << 31, 40)]
    for d in divisors:
        k = rng.integers(0, top // d + 1, 2000, dtype=np.int64) * d
        n = np.concatenate([k - 1, k, k + 1, k + d - 1, [0, 1, d - 1, d, d + 1, top - 1, top],
                            rng.integers(0, 1 << 31, 2000)])
        n = np.unique(n[(n >= 0) & (n <= top)]).astype(np.uint32)
        src = torch.from_numpy(n.view(np.int32)).cuda()
        out = torch.zeros((len(n), 2), dtype=torch.int32, device="cuda")
        torch.cuda.synchronize()
        assert probe.probe_div31(d, C.c_void_p(src.data_ptr()), C.c_void_p(out.data_ptr()), len(n)) == 0
        torch.cuda.synchronize()
        got = out.cpu().numpy().view(np.uint32)
        np.testing.assert_array_equal(got[:, 0], n // np.uint32(d), err_msg=f"d = {d}")
        np.testing.assert_array_equal(got[:, 1], n % np.uint32(d), err_msg=f"d = {d}")


def test_normalized_is_the_quotient_by_the_length(probe):
    """Signs of zeros included; infinities and NaN as the operators make them."""
    rng = np.random.default_rng(2)
    v = rng.standard_normal((200_000, 3)) * np.exp2(rng.uniform(-40, 60, (200_000, 1)))
    v *= rng.choice([0.0, -0.0, 1.0, 1.0, 1.0, 2.0 ** -20], v.shape)
    edges = [0.0, -0.0, 1e-20, 1e-17, 1.0, -3e19, 3e38, -np.inf, np.inf, np.nan]
    grid = np.stack(np.meshgrid(edges, edges, edges), -1).reshape(-1, 3)
    v = np.concatenate([v, grid]).astype(np.float32)
    src = torch.from_numpy(v).cuda()
    out = torch.zeros((len(v), 2, 3), device="cuda")
    torch.cuda.synchronize()
    assert probe.probe_normalized(C.c_void_p(src.data_ptr()), C.c_void_p(out.data_ptr()), len(v)) == 0
    torch.cuda.synchronize()
    got, want = out[:, 0].cpu().numpy(), out[:, 1].cpu().numpy()
    np.testing.assert_array_equal(got, want)
    same = ~np.isnan(want)
    np.testing.assert_array_equal(got.view(np.uint32)[same], want.view(np.uint32)[same])
