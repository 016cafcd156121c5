"""The host-side rules of the denoiser's row kernel (gartus_amd/csrc/rows_plan.h): which layers take it, and
how a launch is split. CPU only: the rules are compiled with g++ through tests/rows_plan_shim.cpp."""
import ctypes as C
import subprocess
from pathlib import Path

import pytest

from test_gpu_denoise import LONG_BATCH

ROOT = Path(__file__).resolve().parent.parent


@pytest.fixture(scope="module")
def shim(tmp_path_factory):
    out = tmp_path_factory.mktemp("shim") / "librowsplan.so"
    subprocess.run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-o", str(out),
                    str(ROOT / "tests" / "rows_plan_shim.cpp")], check=True)
    lib = C.CDLL(str(out))
    lib.shim_rows_frags.argtypes = [C.c_int] * 4 + [C.c_int64]
    return lib


def _frags(shim, ca, cb, cout, grad, n, h, w):
    return shim.shim_rows_frags(ca, cb, cout, int(grad), n * -(-h // 4) * -(-w // 64))


def test_an_encoder_layer_of_80_to_32_takes_the_row_kernel(shim):
    """k_conv takes twice as long on it at 1920x1080. Only that forward layer has an instance of 80 channels."""
    for size in ((1, 8, 12), (1, 1080, 1920)):
        assert _frags(shim, 0, 80, 32, False, *size) == 2
        assert _frags(shim, 0, 80, 32, True, *size) == 0
        assert all(_frags(shim, 0, 80, c, False, *size) == 0 for c in (16, 48, 64, 80, 96, 112, 128))


@pytest.mark.parametrize("grad", [False, True], ids=["forward", "gradient"])
def test_small_images_take_the_faster_kernel(shim, grad):
    """Forward layers of 64 channels, and layers whose output channels need a second launch, stay with k_conv on
    images where it is faster; the others, and all of them on a 1920x1080 frame, take the row kernel."""
    for cin, couts in ((64, (48, 80, 112) if grad else (32, 48, 64, 80, 96, 112, 128)), (16, (80, 112)), (32, (80, 112)), (48, (80, 112)),
                       (96, (48, 80, 112))):
        for cout in couts:
            assert _frags(shim, 0, cin, cout, grad, 1, 32, 48) == 0, (cin, cout)
            assert _frags(shim, 0, cin, cout, grad, 1, 1080, 1920) > 0, (cin, cout)
    for cin, couts in ((16, (16, 32, 48, 64, 96, 128)), (32, (16, 32, 48, 64, 96, 128)), (48, (16, 32, 48, 64, 96, 128)),
                       (64, (16, 32, 64, 96, 128) if grad else (16,)), (96, (16, 32, 64, 96, 128))):
        for cout in couts:
            assert _frags(shim, 0, cin, cout, grad, 1, 2, 2) > 0, (cin, cout)


def test_lines_between_the_kernels_follow_k_convs_blocks(shim):
    """The same layer on both sides of its line, where k_conv changes its groups too (256 tiles)."""
    assert _frags(shim, 0, 64, 64, False, 1, 128, 128) == 0 and _frags(shim, 0, 64, 64, False, 1, 200, 256) == 2
    assert _frags(shim, 0, 64, 32, False, 1, 256, 384) == 0 and _frags(shim, 0, 64, 32, False, 1, 360, 640) == 2
    assert _frags(shim, 0, 64, 112, True, 1, 256, 256) == 0 and _frags(shim, 0, 64, 112, True, 1, 256, 384) == 2
    assert [_frags(shim, 0, 64, 16, False, 1, h, w) for h, w in ((128, 128), (200, 256), (360, 640))] == [2, 0, 2]


@pytest.mark.parametrize("cin", [16, 32, 48, 64, 96])
def test_48_output_channels_are_one_launch(shim, cin):
    """In groups of two fragments and one, the input was read twice: slower than k_conv on large images."""
    assert _frags(shim, 0, cin, 48, False, 1, 1080, 1920) == _frags(shim, 0, cin, 48, True, 16, 256, 256) == 3


def test_concatenations_with_an_instance(shim):
    """A decoder layer has as many output channels as its skip part."""
    for ca, cb in ((48, 32), (64, 32), (64, 48), (96, 64)):
        assert [c for c in range(16, 129, 16) if _frags(shim, ca, cb, c, False, 1, 1080, 1920)] == [cb]
    for ca, cb in ((32, 16), (96, 32), (80, 48), (128, 96), (112, 80)):
        assert _frags(shim, ca, cb, cb, False, 1, 1080, 1920) == 0


@pytest.mark.parametrize("level", [0, 1])
@pytest.mark.parametrize("waves", [1024, 2048, 4096], ids=["1-wave", "2-waves", "4-waves"])
def test_the_long_batch_reaches_every_part_of_the_walk(shim, level, waves):
    """The batch of test_gpu_denoise.py's long segments, on 256 CUs of 1, 2 or 4 waves a SIMD, for every number of
    output groups (four waves a SIMD: layers of 16 channels, four groups at most): several segments of more rows than
    the fragment ring holds (at most five), a shorter last one, and waves that walk more than one tile."""
    n, h, w = LONG_BATCH[0], LONG_BATCH[1] >> level, LONG_BATCH[2] >> level
    out = (C.c_int * 4)()
    for groups in range(1, 5 if waves == 4096 else 9):
        shim.shim_rows_split(n, h, w, groups, waves, out)
        rows, segs, strips, blocks = out
        assert segs >= 2 and rows >= 12 and 0 < h - (segs - 1) * rows < rows, (groups, list(out))
        if (level, waves, groups) != (1, 4096, 1):  # 16->16 and 16->32 below the full resolution: a tile a wave
            tiles_at_once = 8 * 4 * (blocks // groups)
            assert n * segs * strips > tiles_at_once, (groups, list(out))


@pytest.mark.parametrize("n,h,w", [(1, 1, 1), (1, 2, 15), (1, 64, 16), (3, 17, 17), (1, 1088, 1920), (16, 256, 256),
                                   (1, 4, 200000), (512, 2, 2)])
def test_a_split_covers_the_image(shim, n, h, w):
    out = (C.c_int * 4)()
    for groups in (1, 2, 3, 7):
        for waves in (1024, 4096):
            shim.shim_rows_split(n, h, w, groups, waves, out)
            rows, segs, strips, blocks = out
            assert rows % 2 == 0 and (segs - 1) * rows < h <= segs * rows and (strips - 1) * 16 < w <= strips * 16
            assert blocks % groups == 0 and 0 < blocks <= max(waves // 32, groups)
