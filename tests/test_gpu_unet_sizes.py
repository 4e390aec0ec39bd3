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
