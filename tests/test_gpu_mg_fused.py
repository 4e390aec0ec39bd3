"""The V-cycle's fused level kernels at the edges of their tiles.

FP64: fields bit-identical to the one-launch-per-operator schedule, at sizes
that leave partial tiles along every axis, odd level sizes, one and two
columns of tiles, obstacles on tile edges and behind periodic faces.  FP32
(GCR's preconditioner): its GCR must reach the target in as many iterations as
with the FP64 V-cycle of the same sweeps, up to one, and give the same
pressure: the target bounds the error of p by tol / lambda_min(lap), about
pi^2 / 4 on these boxes of unit height with p = 0 on top.
"""
import zlib

import numpy as np
import pytest

import artss_amd
import cases

pytestmark = pytest.mark.gpu

BOX = [(0.25, 0.5, 0.0, 0.375, 0.5, 0.75)]


def _relax(xml, n):
    return xml.replace("<n_relax> 4 </n_relax>", "<n_relax> %d </n_relax>" % n)


def _periodic_box(n):
    xml = cases.plume(n=n, levels=2, steps=2, dt=0.01, obstacles=[(0.0, 0.25, 0.25, 0.75, 0.0, 0.5)], hrr=3.0)
    return xml.replace('<boundary field="p" patch="front,back,bottom,top,left,right" type="neumann" value="0.0" />',
                       '<boundary field="p" patch="front,back,bottom,top,left,right" type="periodic" />')


# (rows of 64 cells below 16384: the small tile, from there on the large one)
FP64 = {
    "partial_tiles": lambda: cases.plume(n=(132, 20, 28), X=(0.0, 2.0), levels=2, steps=2, dt=0.01, hrr=3.0,
                                         open_top=True),
    "odd_levels": lambda: cases.plume(n=(70, 14, 22), levels=2, steps=2, dt=0.01, hrr=3.0, open_top=True),
    "one_column": lambda: cases.plume(n=(16, 24, 40), levels=2, steps=2, dt=0.01, obstacles=BOX, hrr=3.0),
    "periodic": lambda: cases.ns_taylor_green(n=36, levels=2, steps=2),
    "periodic_obstacle": lambda: _periodic_box((32, 32, 32)),
    "large_partial": lambda: cases.plume(n=(72, 92, 94), levels=2, steps=2, dt=0.01, obstacles=BOX, hrr=3.0),
    "large_one_column": lambda: cases.plume(n=(40, 128, 132), levels=2, steps=2, dt=0.01, hrr=3.0, open_top=True),
}


@pytest.mark.parametrize("n_relax", [1, 3, 5])
@pytest.mark.parametrize("name", sorted(FP64))
def test_fp64_matches_one_launch_per_operator(name, n_relax):
    xml = _relax(FP64[name](), n_relax)
    size = artss_amd.Domain(xml, device=-1).info(0)["size"]
    rng = np.random.default_rng(zlib.crc32(name.encode()))
    p0, rhs = 0.01 * rng.standard_normal(size), rng.standard_normal(size)
    states = []
    for mode in (0, 1, 2):
        dom = artss_amd.Domain(xml)
        mg = dom.multigrid()
        mg.set_schedule(mode, 0 if mode == 0 else 3000)
        gp, grhs = dom.field(p0), dom.field(rhs)
        got = []
        for _ in range(3):
            mg.vcycle(gp, grhs)
            got.append(gp.download())
        states.append(got)
    for got in states[1:]:
        for q, ref in enumerate(states[0]):
            assert np.array_equal(got[q], ref), (name, n_relax, q, np.abs(got[q] - ref).max())


@pytest.mark.parametrize("n,X,levels,obstacles,sweeps",
                         [((64, 32, 32), 2.0, 3, BOX, 1), ((64, 32, 32), 2.0, 3, BOX, 3), ((136, 24, 40), 2.0, 3, BOX, 3),
                          ((136, 24, 40), 2.0, 3, [], 1), ((40, 20, 24), 1.0, 3, [], 1), ((128, 92, 96), 1.0, 4, [], 1),
                          ((64, 128, 128), 1.0, 4, BOX, 1), ((64, 128, 128), 1.0, 4, BOX, 3)])
def test_mixed_preconditioner_matches_fp64(n, X, levels, obstacles, sweeps):
    xml = _relax(cases.plume(n=n, X=(0.0, X), levels=levels, steps=3, dt=0.01, obstacles=obstacles, hrr=3.0,
                             source_x=0.75 * X, open_top=True), sweeps)
    tol = 1e-9
    out = {}
    for method, pair in ((1, None), (2, sweeps), (2, 2)):
        s = artss_amd.Solver(xml)
        s.set_mg_schedule(2, 4096)
        s.set_pressure_mode(True, tol, 400)
        s.set_pressure_method(method)
        if pair:
            s.set_mixed_sweeps(pair, pair)
        counts = []
        for step in (1, 2, 3):
            s.step(step * 0.01)
            c = s.counters()
            assert 0 <= c["residual"] <= tol
            counts.append(c["vcycles"])
        out[method, pair] = s.field("p"), counts
    (p1, c1), (p2, c2), (p3, c3) = out[1, None], out[2, sweeps], out[2, 2]
    print("iterations", c1, c2, c3, "p differs by", np.linalg.norm(p2 - p1), np.linalg.norm(p3 - p1))
    # the first right-hand side that is not zero is the last step's
    assert c1[:2] == c2[:2] == c3[:2] == [0, 0] and c1[2] > 0
    assert abs(c1[2] - c2[2]) <= 1, (c1, c2)
    inner = [np.ascontiguousarray(p.reshape(n[2] + 2, n[1] + 2, n[0] + 2)[1:-1, 1:-1, 1:-1]) for p in (p1, p2, p3)]
    # |lap(p - q)| <= 2 tol; half of pi^2 / 4 covers the discrete eigenvalue and the obstacle
    bound = 2 * tol / (0.5 * np.pi ** 2 / 4)
    for p in inner[1:]:
        assert np.linalg.norm(p - inner[0]) <= bound, np.linalg.norm(p - inner[0])
