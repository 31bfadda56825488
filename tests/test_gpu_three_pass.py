"""The three-pass FP64 evaluations (the y transform divided between the x and
z passes) at the splits where they can go wrong: the shortest rows and columns,
a last tile of one, two and three k1, one, two and four k1 per z workgroup,
lanes that divide unevenly over a stage (28 = 4 x 7, 105 = 7 x 15 on 8 threads,
126 on 14), the longest and shortest radices of y (16 x 8, 6 x 3, 10 x 10), all
fields in one x workgroup (n1 = 128) and one. Against the oracle at the parity
bar (1e-10) and against the staged LDS passes at 1e-13 of max|potential|, the
bound the other register passes are held to. The trial-point and signed forms
by two iterations of the minimizers that use no other against the staged
passes: rounding differences of 1e-14 that two line searches may amplify a
thousandfold, 1e-10 of each energy. (The Newton form divides a difference of
gradients by a small step; the converged truncated-Newton solves hold it.)"""
import numpy as np
import pytest

from oracle import profess_oracle as O
from tests.test_gpu_lengths import LAT, _run, pa  # noqa: F401

pytestmark = pytest.mark.gpu

GRIDS = [(18, 16, 16), (20, 18, 28), (24, 25, 105), (36, 112, 126), (128, 32, 18), (126, 28, 20), (100, 100, 24),
         (42, 128, 30), (28, 160, 16), (120, 50, 27), (54, 81, 120), (30, 49, 128), (192, 42, 150), (162, 63, 27), (60, 75, 24),
         (36, 21, 63)]


@pytest.mark.parametrize("grid", GRIDS)
@pytest.mark.parametrize("kind", ["wt", "wt4", "spin"])
def test_three_pass(pa, monkeypatch, grid, kind):  # noqa: F811
    print(grid, kind, flush=True)
    n1, n2, n3 = grid
    lat = LAT * (0.24 * np.array(grid))[None, :]
    cell = O.Cell(lat, n1, n2, n3)
    ne = 0.027 * cell.vol
    rng = np.random.default_rng(n1 + 7 * n2 + 31 * n3)
    rho = 0.027 * (1.0 + 0.3 * (2.0 * rng.random(cell.shape) - 1.0))
    vion = rng.random(cell.shape) - 0.5
    if kind == "spin":
        rho = np.stack([0.55 * rho, 0.45 * rho[::-1]])
    pot, et = _run(pa, grid, kind, rho, vion, ne, lat)
    monkeypatch.setenv("OFD_GENERIC", "1")
    p0, e0 = _run(pa, grid, kind, rho, vion, ne, lat)
    monkeypatch.delenv("OFD_GENERIC")
    assert np.max(np.abs(pot - p0)) <= 1e-13 * np.max(np.abs(p0))
    assert np.all(np.abs(et - e0) <= 1e-12 * np.abs(e0) + 1e-12)
    f = O.Functional(kinetic=4, alpha=0.9 if kind == "wt4" else -100.0, beta=0.7 if kind == "wt4" else -100.0)
    sysm = O.System(cell, f.resolve(ne, cell.vol), vion)
    ref, er = (O.calculate_potential_plus_spin if kind == "spin" else O.calculate_potential_plus)(rho, sysm)
    assert np.max(np.abs(pot - ref)) <= 1e-10 * np.max(np.abs(ref))
    assert np.all(np.abs(et - er) <= 1e-10 * np.abs(er) + 1e-12)


@pytest.mark.parametrize("dir_type", [2, 3])
@pytest.mark.parametrize("grid", [(20, 24, 18), (128, 28, 25)])
def test_three_pass_minimizer_forms(pa, monkeypatch, grid, dir_type):  # noqa: F811
    print(grid, dir_type, flush=True)
    n1, n2, n3 = grid
    lat = LAT * (0.24 * np.array(grid))[None, :]
    vol = abs(np.linalg.det(lat))
    x = [np.arange(n) * (2.0 * np.pi / n) for n in (n3, n2, n1)]
    vion = 0.3 * (np.cos(x[0])[:, None, None] + np.sin(x[1])[None, :, None] * np.cos(x[2])[None, None, :])
    rho = np.full((n3, n2, n1), 0.027)

    def solve():
        s = pa.OFDSystem(lat, grid, 0.027 * vol)
        s.set_ion_terms(vion)
        out = pa.ProjNormRhoMinimization(s, rho, dir_type=dir_type, max_iter=2)
        s.close()
        return out

    r1, e1, _, _ = solve()
    monkeypatch.setenv("OFD_GENERIC", "1")
    r0, e0, _, _ = solve()
    assert np.all(np.abs(e1 - e0) <= 1e-10 * np.abs(e0) + 1e-12)
    assert np.max(np.abs(r1 - r0)) <= 1e-10 * np.max(r0)
