"""Gradients of the warm-start U-Net at the sizes where its kernels' tiles
end: one voxel at the coarsest level, sides that leave partial row tiles and
partial x segments of the weight gradients' blocks (128 voxels along x), and
rows of one and two voxels.  Against the float64 oracle with the bounds of
tests/test_gpu_unet.py (BF16 activations: about three digits), and the same
bits in a second call, since every sum has a fixed order."""
import os
import sys

import numpy as np
import pytest

import artss_amd
import cases

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "oracle"))
import unet_ref as U  # noqa: E402
from test_gpu_unet import _bf16, _flat, _rel, _unflat  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("X,Y,Z", [(8, 8, 8), (136, 8, 16), (16, 40, 8), (8, 136, 8), (72, 16, 24)])
def test_gradients_match_reference(X, Y, Z):
    dom = artss_amd.Domain(cases.ns_taylor_green(n=16, levels=2, steps=1))
    rng = np.random.default_rng(X * 1000 + Y)
    p = U.init_params(seed=X + Z)
    for n, *_ in U.LAYERS:
        p[n + ".W"] = _bf16(p[n + ".W"])
        p[n + ".b"] = 0.05 * rng.standard_normal(p[n + ".b"].shape)
    x, target = rng.standard_normal((Z, Y, X, 2)), rng.standard_normal((Z, Y, X, 1))
    net = artss_amd.UNet(dom, seed=1)
    net.set_params(_flat(p))
    xb = artss_amd.Buffer(dom, x.astype(np.float32))
    tb = artss_amd.Buffer(dom, target.astype(np.float32))
    loss, g = net.gradients(xb, tb)
    loss_ref, g_ref = U.loss_and_grad(p, x, target)
    assert abs(loss - loss_ref) <= 3e-2 * loss_ref
    gg = _unflat(g.astype(np.float64))
    for n, *_ in U.LAYERS:
        for key in (n + ".W", n + ".b"):
            a, b = gg[key].reshape(-1), g_ref[key].reshape(-1)
            cos = float(a @ b / max(np.linalg.norm(a) * np.linalg.norm(b), 1e-30))
            print(key, "rel err %.3g cos %.5f" % (_rel(a, b), cos))
            assert cos > 0.995 and _rel(a, b) < 0.1, key
    again, g2 = net.gradients(xb, tb)
    assert again == loss and np.array_equal(g, g2)
    assert net.gradients(xb, tb, want_grads=False)[0] == loss


def test_forward_of_a_large_volume_matches_its_corners():
    """The marching kernel of the last upsampling layer serves large volumes
    only.  An output voxel depends on inputs at most 40 voxels away (8 at the
    coarsest level and its upsampling, 8 + 4 + 3 at the finer ones, rounded up
    to whole coarse voxels), so the two far corners of a large volume with
    partial tiles must repeat in 96-voxel boxes cut from it, which take the
    small volumes' kernel.  The two sum in different orders in FP32: a BF16
    activation may differ by one rounding (2^-8), in each of eight layers."""
    X, Y, Z = 168, 136, 136
    dom = artss_amd.Domain(cases.ns_taylor_green(n=16, levels=2, steps=1))
    rng = np.random.default_rng(11)
    net = artss_amd.UNet(dom, seed=3)
    p = U.init_params(seed=5)
    for n, *_ in U.LAYERS:
        p[n + ".W"] = rng.standard_normal(p[n + ".W"].shape) * np.sqrt(2.0 / (27 * p[n + ".W"].shape[-2]))
    net.set_params(_flat(p))
    x = rng.standard_normal((Z, Y, X, 2)).astype(np.float32)

    def forward(v):
        out = artss_amd.Buffer(dom, np.zeros(v.shape[:3] + (1,), np.float32))
        net.forward(artss_amd.Buffer(dom, np.ascontiguousarray(v)), out)
        return out.download()[..., 0]

    whole = forward(x)
    assert np.isfinite(whole).all() and np.any(whole)
    low, high = forward(x[:96, :96, :96]), forward(x[-96:, -96:, -96:])
    for part, ref in ((low[:48, :48, :48], whole[:48, :48, :48]), (high[-48:, -48:, -48:], whole[-48:, -48:, -48:])):
        err = float(np.linalg.norm(part - ref) / np.linalg.norm(ref))
        print("relative difference", err)
        assert err < np.sqrt(8) * 2.0 ** -8
