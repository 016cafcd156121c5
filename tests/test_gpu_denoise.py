"""The denoiser's MFMA kernels against the float64 oracle (oracle/denoise_ref.py).

The oracle rounds to bf16 wherever the GPU stores bf16 (bf16=True), so the
remaining differences come from fp32 accumulation order, which moves an
occasional bf16 rounding by one step (2^-8 relative) and propagates through
later layers. Tolerances:
  - network output z: |z_gpu - z_ref| <= 0.02 + 0.02 |z_ref| for 99.5% of
    values; mean absolute difference below 2^-8 (one bf16 step at 1) times
    sqrt(number of convolutions), the growth of independent one-step
    rounding flips over the network's depth;
  - loss: 1e-3 relative;
  - gradients: per convolution, ||g_gpu - g_ref|| / ||g_ref|| below
    1% times sqrt(number of convolutions) (the backward chain of the deepest
    layer crosses every convolution twice), and cosine similarity above
    0.998. A transposed weight, a wrong tap or a lost term gives errors of
    order one.
"""
import sys

import numpy as np
import pytest

import denoise_ref as dr
from gartus_amd import abi
from gartus_amd.denoiser import Denoiser

pytestmark = pytest.mark.gpu


def say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


def _problem(levels, channels, n, h, w, seed):
    rng = np.random.default_rng(seed)
    net = dr.Net(levels, channels)
    # a He-like scale keeps activations O(1) through the layers
    p = np.zeros(net.nparams)
    for i, (cin, cout, _) in enumerate(net.convs):
        w0, b0 = net.offsets[i]
        p[w0:b0] = rng.normal(scale=np.sqrt(2.0 / (9 * cin)), size=b0 - w0)
        p[b0:b0 + cout] = rng.normal(scale=0.05, size=cout)
    # input channels 9..15 and output channels 3..15 are padding
    w0, b0 = net.offsets[0]
    p[w0:b0].reshape(net.convs[0][1], 9, 16)[:, :, 9:] = 0.0
    w0, b0 = net.offsets[-1]
    p[w0:b0].reshape(16, 9, net.convs[-1][0])[3:] = 0.0
    p[b0 + 3:b0 + 16] = 0.0
    net.params = dr.bf16(p)  # the GPU's bf16 copy is then exact
    beauty = rng.gamma(1.0, 1.0, (n, h, w, 3)).astype(np.float32)
    albedo = rng.uniform(0, 1, (n, h, w, 3)).astype(np.float32)
    normal = rng.uniform(0, 1, (n, h, w, 3)).astype(np.float32)
    target = rng.gamma(1.0, 1.0, (n, h, w, 3)).astype(np.float32)
    return net, beauty, albedo, normal, target


# the last case pads 21 x 30 to 24 x 32: the output convolution writes radiance for the image
# inside the padded tensor only
CASES = [(2, (16, 16), 2, 16, 16), (3, (32, 48, 16), 1, 20, 28), (5, (32, 48, 64, 96, 128), 2, 32, 48),
         (3, (32, 48, 16), 2, 21, 30)]


def _check_forward_and_gradients(gpu_context, levels, channels, n, h, w, loss):
    say(f"denoiser levels {levels} channels {channels} batch {n}x{h}x{w} loss {loss}")
    net, b, a, nr, t = _problem(levels, channels, n, h, w, seed=levels)
    dn = Denoiser(gpu_context, levels, channels, loss=loss)
    assert dn.param_count == net.nparams
    dn.set_params(net.params.astype(np.float32))
    np.testing.assert_array_equal(dn.get_params(), net.params.astype(np.float32))

    loss_ref, g_ref, z_ref = dr.loss_and_gradients(net, b.astype(np.float64), a.astype(np.float64),
                                                   nr.astype(np.float64), t.astype(np.float64), bf=True,
                                                   kind=loss)
    rad_gpu = dn.infer(b, a, nr)
    rad_ref = dr.radiance(z_ref, h, w)
    # compare in the network's output space, z = log1p(radiance) where z >= 0
    zg, zr = np.log1p(rad_gpu), np.log1p(rad_ref)
    err = np.abs(zg - zr)
    assert np.mean(err <= 0.02 + 0.02 * np.abs(zr)) > 0.995, f"max {err.max()}"
    assert err.mean() < 2.0 ** -8 * np.sqrt(len(net.convs)), err.mean()

    loss_gpu, g_gpu = dn.loss_and_gradients(b, a, nr, t)
    assert loss_gpu == pytest.approx(loss_ref, rel=1e-3)
    for i, (cin, cout, _) in enumerate(net.convs):
        w0, b0 = net.offsets[i]
        for name, sl in (("w", slice(w0, b0)), ("b", slice(b0, b0 + cout))):
            gr, gg = g_ref[sl], g_gpu[sl].astype(np.float64)
            nref = np.linalg.norm(gr)
            if nref == 0.0:
                assert np.linalg.norm(gg) < 1e-12
                continue
            rel = np.linalg.norm(gg - gr) / nref
            cos = gg @ gr / (np.linalg.norm(gg) * nref)
            assert rel < 0.01 * np.sqrt(len(net.convs)) and cos > 0.998, \
                f"conv {i} {name}: rel {rel:.4f} cos {cos:.6f}"
    dn.close()


@pytest.mark.parametrize("loss", [abi.GT_DENOISE_LOSS_REL_L2, abi.GT_DENOISE_LOSS_L1_TONEMAP], ids=["rel-l2", "l1"])
@pytest.mark.parametrize("levels,channels,n,h,w", CASES)
def test_forward_and_gradients_match_oracle(gpu_context, levels, channels, n, h, w, loss):
    _check_forward_and_gradients(gpu_context, levels, channels, n, h, w, loss)


# Channel pairs of the row kernel's instances and of the layers beside them, forward and backward, at widths below, at
# and beyond a strip of 16 columns and more strips than a block's four waves. These images are small: the launches have
# segments of 1 to 8 rows, one a wave, and the layers that take k_conv on small images (rows_frags) take it here. Longer
# segments and several of them a wave: test_long_segments_match_single_images.
@pytest.mark.parametrize("levels,channels,n,h,w", [
    (2, (32, 48), 1, 2, 2), (2, (32, 48), 3, 17, 15), (2, (32, 64), 1, 6, 130), (2, (48, 64), 1, 66, 18),
    (2, (48, 64), 1, 64, 260), (2, (64, 96), 2, 10, 34), (2, (96, 128), 1, 5, 33), (2, (96, 128), 1, 131, 16),
    (2, (32, 80), 1, 36, 34), (2, (80, 32), 1, 34, 70)])
def test_row_kernel_shapes_match_oracle(gpu_context, levels, channels, n, h, w):
    _check_forward_and_gradients(gpu_context, levels, channels, n, h, w, abi.GT_DENOISE_LOSS_REL_L2)


# The gradient of the decoder's concatenation: 80 channels from 32 in one launch, 112 from 48 in one of six fragments
# and one of the odd seventh, at a full resolution where every wave of the chip has a segment. (The oracle takes about
# 20 and 50 s here.)
@pytest.mark.parametrize("channels", [(32, 48), (48, 64)], ids=["cat80", "cat112"])
def test_concatenation_gradients_match_oracle(gpu_context, channels):
    _check_forward_and_gradients(gpu_context, 2, channels, 1, 128, 2048, abi.GT_DENOISE_LOSS_REL_L2)


def test_gradients_are_deterministic(gpu_context):
    net, b, a, nr, t = _problem(3, (32, 48, 16), 2, 24, 24, seed=9)
    dn = Denoiser(gpu_context, 3, (32, 48, 16))
    dn.set_params(net.params.astype(np.float32))
    l1, g1 = dn.loss_and_gradients(b, a, nr, t)
    l2, g2 = dn.loss_and_gradients(b, a, nr, t)
    assert l1 == l2
    np.testing.assert_array_equal(g1, g2)
    dn.close()


def test_training_reduces_loss(gpu_context):
    """Adam steps on a fixed synthetic task (target = the clean version of a
    noisy beauty) must drive the loss down."""
    rng = np.random.default_rng(5)
    n, h, w = 4, 32, 32
    clean = np.repeat(np.repeat(rng.uniform(0.2, 2.0, (n, h // 8, w // 8, 3)), 8, axis=1), 8, axis=2)
    noisy = clean * rng.gamma(4.0, 0.25, clean.shape)
    albedo = np.clip(clean / 2.0, 0, 1)
    normal = np.full(clean.shape, 0.5)
    args = [x.astype(np.float32) for x in (noisy, albedo, normal, clean)]
    dn = Denoiser(gpu_context, 3, (32, 48, 64), seed=2)
    first = dn.train_step(*args, lr=2e-3)
    for _ in range(60):
        last = dn.train_step(*args, lr=2e-3)
    assert np.isfinite(last) and last < 0.5 * first, (first, last)
    dn.close()


@pytest.mark.parametrize("levels,channels,n,h,w", CASES[1:])
def test_halves_network_matches_oracle(gpu_context, levels, channels, n, h, w):
    """beauty_halves: two half-sample renders packed as log1p of their mean
    and the log difference (channels 9-11), which here carry weight."""
    say(f"denoiser with beauty halves, levels {levels} batch {n}x{h}x{w}")
    net, b, a, nr, t = _problem(levels, channels, n, h, w, seed=20 + levels)
    rng = np.random.default_rng(30 + levels)
    w0, b0 = net.offsets[0]
    wts = net.params[w0:b0].reshape(net.convs[0][1], 9, 16).copy()
    wts[:, :, 9:12] = dr.bf16(rng.normal(scale=0.2, size=wts[:, :, 9:12].shape))
    net.params[w0:b0] = wts.ravel()
    b2 = rng.gamma(1.0, 1.0, (n, h, w, 3)).astype(np.float32)
    dn = Denoiser(gpu_context, levels, channels, halves=True)
    dn.set_params(net.params.astype(np.float32))
    loss_ref, g_ref, z_ref = dr.loss_and_gradients(net, b.astype(np.float64), a.astype(np.float64),
                                                   nr.astype(np.float64), t.astype(np.float64), bf=True,
                                                   beauty_b=b2.astype(np.float64))
    halves = np.stack([b, b2])
    zg, zr = np.log1p(dn.infer(halves, a, nr)), np.log1p(dr.radiance(z_ref, h, w))
    err = np.abs(zg - zr)
    assert np.mean(err <= 0.02 + 0.02 * np.abs(zr)) > 0.995, f"max {err.max()}"
    loss_gpu, g_gpu = dn.loss_and_gradients(halves, a, nr, t)
    # relative L2 divides by the squared prediction (+0.01), so the bf16-level output differences
    # already bounded above move it more than they move L1
    assert loss_gpu == pytest.approx(loss_ref, rel=1e-2)
    w0, b0 = net.offsets[0]
    gr, gg = g_ref[w0:b0], g_gpu[w0:b0].astype(np.float64)
    rel = np.linalg.norm(gg - gr) / np.linalg.norm(gr)
    cos = gg @ gr / (np.linalg.norm(gg) * np.linalg.norm(gr))
    assert rel < 0.01 * np.sqrt(len(net.convs)) and cos > 0.998, (rel, cos)  # the bar of the test above
    # the first convolution's gradient reaches the difference channels
    assert np.abs(gg.reshape(-1, 9, 16)[:, :, 9:12]).max() > 0
    dn.close()


# A batch of small images whose layers the row kernel walks in long segments, with a shorter last one, several tiles a
# wave (test_rows_plan.py checks that it does).
LONG_BATCH = (512, 132, 96)
LONG_CHANNELS = [(16, 64), (32, 48), (32, 64), (32, 80), (32, 112), (48, 64), (48, 80), (48, 96), (64, 96), (64, 112),
                 (80, 32), (96, 48), (96, 80), (96, 128), (112, 16)]


@pytest.mark.parametrize("channels", LONG_CHANNELS, ids=lambda c: f"{c[0]}-{c[1]}")
def test_long_segments_match_single_images(gpu_context, channels):
    """A network's images do not depend on the batch they come in: bit for bit the images of a batch of one, whose
    layers run in short segments or through k_conv and match the oracle above. The gradients are the mean of the single
    ones (the batch's scale is a power of two): a data gradient sums in another order in k_conv, so that at most about
    2^-9 of its bf16 values round the other way by 2^-8, 2^-8 * 2^-4.5 = 1.7e-4 of its norm a layer, over six layers in
    a row below 2e-3; weight gradients sum in fp32 in another order, below 1e-4."""
    import torch
    n, h, w = LONG_BATCH
    say(f"denoiser levels 2 channels {channels} batch {n}x{h}x{w}")
    net, *images = _problem(2, channels, 4, h, w, seed=7)
    dn = Denoiser(gpu_context, 2, channels, loss=abi.GT_DENOISE_LOSS_REL_L2)
    dn.set_params(net.params.astype(np.float32))
    one = [torch.from_numpy(x).cuda() for x in images]
    many = [x.repeat(n // 4, 1, 1, 1) for x in one]
    torch.cuda.synchronize()

    singles = [dn.infer(*(x[k:k + 1] for x in one[:3])) for k in range(4)]
    batch = dn.infer(*many[:3])
    gpu_context.synchronize()
    single = torch.cat(singles)
    assert torch.isfinite(single).all() and single.std() > 0
    assert torch.equal(batch.reshape(n // 4, 4, h, w, 3), single.expand(n // 4, 4, h, w, 3))

    parts = [dn.loss_and_gradients(*(x[k:k + 1] for x in one)) for k in range(4)]
    loss, grads = dn.loss_and_gradients(*many)
    assert loss == pytest.approx(np.mean([p[0] for p in parts]), rel=1e-5)
    g, ref = np.asarray(grads, np.float64), np.mean([np.asarray(p[1], np.float64) for p in parts], axis=0)
    for i, (cin, cout, _) in enumerate(net.convs):
        w0, b0 = net.offsets[i]
        rel = np.linalg.norm(g[w0:b0 + cout] - ref[w0:b0 + cout]) / np.linalg.norm(ref[w0:b0 + cout])
        assert rel < 2e-3, f"conv {i} {cin}->{cout}: {rel:.2e}"
    dn.close()
