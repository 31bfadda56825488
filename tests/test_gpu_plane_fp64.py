"""FP64 evaluations of the plane shapes that the three passes leave (y lengths
32, 64 and 128 with rows as long and z lengths of 192 and 256; WGC on 128 x 128
planes; two spin channels on 32 x 32): fused x + y pass, z, y back, and the x
inverse, which is the general one on rows of 128. Split and whole planes, the
shortest z column and the longest. Against the staged LDS passes at 1e-13 of
max|potential|, the bound the other register passes are held to, and against
the oracle at the parity bar (1e-10)."""
import numpy as np
import pytest

from oracle import profess_oracle as O
from tests import wgc_tables as W

pytestmark = pytest.mark.gpu

LAT = np.array([[1.0, 0.2, 0.1], [0.3, 1.0, 0.0], [-0.2, 0.4, 1.0]]).T
CASES = [((128, 128, 192), "wt"), ((128, 128, 192), "wt4"), ((64, 64, 256), "wt"), ((64, 64, 256), "wt4"),
         ((32, 32, 192), "wt"), ((128, 128, 24), "wgc"), ((32, 32, 24), "spin"), ((32, 32, 24), "spin4")]


def system(grid, kind, **kw):
    """A skew system of its grid and kind and its electron count."""
    import profess_amd as pa
    lat = LAT * (0.24 * np.array(grid))[None, :]
    ne = 0.027 * abs(np.linalg.det(lat))
    opts = dict(kinetic=5, gamma=2.7) if kind == "wgc" else dict(alpha=0.9, beta=0.7) if kind[-1] == "4" else {}
    s = pa.OFDSystem(lat, grid, ne, **opts, **kw)
    if kind.startswith("spin"):
        s.set_spin(2, fixed_mag=True)
    if kind == "wgc":
        p = s.params
        s.set_wgc_table(*W.for_params(p["alpha"], p["beta"], p["gamma"]))
    return s, ne


@pytest.mark.parametrize("grid,kind", CASES)
def test_fp64_plane_passes(monkeypatch, grid, kind):
    import profess_amd as pa
    print(grid, kind, flush=True)
    rng = np.random.default_rng(grid[0] + grid[2])
    res = {}
    for name, env in (("default", {}), ("whole", {"OFD_PLANE_SPLIT": "1"}), ("staged", {"OFD_GENERIC": "1"})):
        for k in ("OFD_PLANE_SPLIT", "OFD_GENERIC"):
            monkeypatch.delenv(k, raising=False)
        for k, v in env.items():
            monkeypatch.setenv(k, v)
        s, ne = system(grid, kind)
        if name == "default":
            rho = 0.027 * (1.0 + 0.3 * (2.0 * rng.random(s.shape) - 1.0))
            vion = rng.random(s.shape) - 0.5
            if s.nspin == 2:
                rho = np.stack([0.55 * rho, 0.45 * rho[::-1]])
        s.set_ion_terms(vion)
        res[name] = pa.CalculatePotentialPlus(s, rho)
        s.close()
    p0, e0 = res["staged"]
    for name in ("default", "whole"):
        pot, et = res[name]
        assert np.max(np.abs(pot - p0)) <= 1e-13 * np.max(np.abs(p0)), name
        assert np.all(np.abs(et - e0) <= 1e-12 * np.abs(e0) + 1e-12), name
    if kind == "wgc":   # the oracle's spline fill is the slow part: the other kinds pin the passes
        return
    cell = O.Cell(LAT * (0.24 * np.array(grid))[None, :], *grid)
    ab = 0.9 if kind[-1] == "4" else -100.0, 0.7 if kind[-1] == "4" else -100.0
    sysm = O.System(cell, O.Functional(kinetic=4, alpha=ab[0], beta=ab[1]).resolve(ne, cell.vol), vion)
    ref, er = (O.calculate_potential_plus_spin if s.nspin == 2 else O.calculate_potential_plus)(rho, sysm)
    pot, et = res["default"]
    assert np.max(np.abs(pot - ref)) <= 1e-10 * np.max(np.abs(ref))
    assert np.all(np.abs(et - er) <= 1e-10 * np.abs(er) + 1e-12)
