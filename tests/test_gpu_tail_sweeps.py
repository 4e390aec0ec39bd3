"""The register sweeps of the single-workgroup multigrid kernel against the
one-launch-per-operator schedule, bit for bit, at the sizes where their
dispatch changes: a coarse level of 1024 cells (one cell per thread), just
above (two), 2048, and above 2048 (the plain sweeps); odd sides; and levels
with obstacles next to periodic patches, where a fluid cell reads a ghost
copied from an obstacle cell and the plain sweeps must run."""
import numpy as np
import pytest

import artss_amd
import cases

pytestmark = pytest.mark.gpu

BOX = [(0.25, 0.5, 0.0, 0.375, 0.5, 0.75)]
WALL = [(0.0, 0.25, 0.25, 0.5, 0.25, 0.5)]  # against the x = 0 patch


def _plume(n, obstacles=(), **kw):
    return cases.plume(n=n, levels=2, steps=2, dt=0.01, obstacles=obstacles, hrr=3.0, open_top=True, **kw)


def _periodic(n, boxes):
    x = cases.ns_taylor_green(n=8, levels=2, steps=2)
    for a, m in zip("xyz", n):
        x = x.replace("<n%s> 8 </n%s>" % (a, a), "<n%s> %d </n%s>" % (a, m, a))
    return x.replace('<obstacles enabled="No"/>', cases.obstacles_xml(boxes))


CASES = {
    "1024": lambda: _plume((32, 16, 16)),
    "1024_obstacle": lambda: _plume((32, 16, 16), BOX),
    "1088": lambda: _plume((34, 16, 16), BOX),
    "2048": lambda: _plume((32, 32, 16), BOX),
    "2304": lambda: _plume((36, 32, 16), BOX),
    "odd_693": lambda: _plume((23, 19, 15), BOX),
    "smallest": lambda: _plume((8, 8, 8)),
    "periodic": lambda: _periodic((24, 16, 20), []),
    "periodic_obstacle_at_patch": lambda: _periodic((16, 16, 16), WALL),
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_tail_matches_plain_schedule(name):
    xml = CASES[name]()
    dt = float(xml.split("<dt>")[1].split("</dt>")[0])
    rng = np.random.default_rng(len(name))
    out = []
    for mode, tail in ((0, 0), (1, 4096), (2, 4096)):
        dom = artss_amd.Domain(xml)
        size = dom.size(0)
        if not out:
            p0, rhs = 0.01 * rng.standard_normal(size), rng.standard_normal(size)
        mg = dom.multigrid()
        mg.set_schedule(mode, tail)
        assert mode == 0 or mg.tail_level() < dom.levels
        p, b = dom.field(p0), dom.field(rhs)
        cycles = [mg.pressure(p, b, t * dt) for t in (2, 3, 4)]
        out.append((cycles, p.download(), mg.residual(p, b)))
    for cycles, p, res in out[1:]:
        assert cycles == out[0][0] and res == out[0][2]
        assert np.array_equal(p, out[0][1]), np.abs(p - out[0][1]).max()
