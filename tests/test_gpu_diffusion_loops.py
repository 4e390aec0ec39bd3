"""The one-launch diffusion iterations against the oracle, bit for bit, where
their cases change: iteration counts of either parity (which array holds the
last iterate, with `in` and `out` as the loop leaves them), loops that stop
in the middle of an enqueued batch, none at all, boxes that give the
Gauss-Seidel tiles 2, 4 and 8 planes with partial last tiles, odd rows (the
two-launch form), obstacles against a wall, and periodic patches whose ghosts
follow obstacle cells."""
import numpy as np
import pytest

import artss_amd
import artss_xml
import cases
import oracle_py as O

pytestmark = pytest.mark.gpu

OBST = [(0.25, 0.5, 0.0, 0.375, 0.5, 0.75), (0.5, 0.75, 0.25, 0.5, 0.25, 0.5), (0.75, 1.0, 0.5, 0.75, 0.25, 0.5)]
PERIODIC = '<boundary field="T" patch="front,back,left,right,bottom,top" type="periodic" />'


def _domain(n, obstacles=OBST, periodic=False):
    xml = cases.plume(n=n, levels=1, steps=2, dt=0.01, obstacles=obstacles, hrr=3.0)
    if periodic:
        xml = xml.replace('<boundary field="T" patch="front,back,top,left,right" type="dirichlet" value="293.15" />'
                          '<boundary field="T" patch="bottom" type="neumann" value="0.0" />', PERIODIC)
        assert PERIODIC in xml
    return artss_amd.Domain(xml), O.Domain(artss_xml.parse(xml)), artss_xml.parse(xml)["dt"]


def _compare(n, method, max_iter, tol, turbulent, **kw):
    dom, odom, dt = _domain(n, **kw)
    rng = np.random.default_rng(sum(n) + max_iter)
    o, i, b = (rng.standard_normal(odom.size(0)) for _ in range(3))
    ev = 1e-2 * np.abs(rng.standard_normal(odom.size(0))) if turbulent else None
    go, gi = dom.field(o), dom.field(i)
    it_g, res_g = dom.diffuse(method, go, gi, dom.field(b), 1e-3, dom.field(ev) if turbulent else None, artss_amd.T,
                              max_iter, tol, 1.0)
    it_o, res_o = odom.diffuse(method, o, i, b, 1e-3, ev, dt, max_iter, tol, 1.0, artss_amd.T)
    assert it_g == it_o
    # the update norm is a sum in another order over at most n cells
    assert abs(res_g - res_o) <= 1e-12 * max(res_o, 1e-300) * odom.size(0) ** 0.5
    assert np.array_equal(go.download(), o) and np.array_equal(gi.download(), i)
    return it_g


@pytest.mark.parametrize("method", ["Jacobi", "ColoredGaussSeidel"])
@pytest.mark.parametrize("max_iter", [0, 1, 2, 3, 4, 5, 9])
def test_iteration_counts(method, max_iter):
    assert _compare((18, 12, 14), method, max_iter, 0.0, True) == max_iter


@pytest.mark.parametrize("method", ["Jacobi", "ColoredGaussSeidel"])
@pytest.mark.parametrize("n", [(8, 8, 8), (23, 17, 9), (64, 20, 31), (61, 50, 33), (126, 44, 40)])
@pytest.mark.parametrize("turbulent", [False, True])
def test_to_tolerance(method, n, turbulent):
    assert _compare(n, method, 100, 1e-8, turbulent) > 2


@pytest.mark.parametrize("n", [(130, 130, 67), (66, 70, 90)])
def test_deep_tiles(n):
    assert _compare(n, "ColoredGaussSeidel", 3, 0.0, True) == 3


@pytest.mark.parametrize("method", ["Jacobi", "ColoredGaussSeidel"])
@pytest.mark.parametrize("max_iter", [3, 4])
def test_periodic_with_obstacles(method, max_iter):
    wall = [(0.0, 0.25, 0.25, 0.5, 0.25, 0.5), (0.5, 0.75, 0.0, 0.25, 0.5, 0.75)]
    assert _compare((16, 16, 16), method, max_iter, 0.0, False, obstacles=wall, periodic=True) == max_iter
