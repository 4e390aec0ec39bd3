"""The fills that ride along with an operator or with other fields' fills.

Advection with its fill in the same launch against the separate fill (taken
where the output array is one of the velocities), and the projection's three
fills in one launch against artss_apply_boundary on each field: the same bits
on boxes of one wavefront, one cell more, and ragged ones, with obstacles
(touching ones make the fill take the general path), periodic, and on the
two-dimensional fill that reads the ghost layer.
"""
import numpy as np
import pytest

import artss_amd
import cases
import refxml

pytestmark = pytest.mark.gpu

TOUCHING = [(0.25, 0.5, 0.0, 0.375, 0.5, 0.75), (0.5, 0.75, 0.25, 0.5, 0.25, 0.5)]


def _plume(n, obstacles=()):
    return cases.plume(n=n, levels=1, steps=2, dt=0.01, obstacles=list(obstacles), hrr=3.0, open_top=True)


CASES = {
    "16x16x16": lambda: _plume((16, 16, 16)),
    "65x5x3": lambda: _plume((65, 5, 3)),
    "66x20x24_obstacle": lambda: _plume((66, 20, 24), TOUCHING[:1]),
    "40x16x24_touching": lambda: _plume((40, 16, 24), TOUCHING),
    "130x36x30": lambda: _plume((130, 36, 30), TOUCHING[1:]),
    "periodic": lambda: cases.ns_taylor_green(n=20, levels=1, steps=2),
    "cavity_2d": lambda: bytes(refxml.load("ns_cavity")["xml"]).decode(),
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_fills_match_separate_launches(name):
    dom = artss_amd.Domain(CASES[name]())
    size = dom.info(0)["size"]
    rng = np.random.default_rng(size)
    vel = [rng.uniform(-3, 3, size) for _ in range(3)]
    src = rng.standard_normal(size)
    for ft in (0, 1, 2, 3, 4, 5):
        u, v, w, f = (dom.field(x) for x in (vel[0], vel[1], vel[2], src))
        out = dom.field(vel[0])  # cells nothing writes: as in the array that is overwritten below
        dom.sl_advect(out, f, u, v, w, ft)
        apart = out.download()
        dom.sl_advect(u, f, u, v, w, ft)
        assert np.array_equal(apart, u.download()), ft
    p = dom.field(src)
    a = [dom.field(x) for x in vel]
    dom.projection(a[0], a[1], a[2], a[0], a[1], a[2], p)
    for q, ft in zip(a, (1, 2, 3)):
        once = q.download()
        dom.apply_boundary(q, ft, 0)
        assert np.array_equal(once, q.download()), ft
