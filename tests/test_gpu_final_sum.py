"""The final sum of the workgroups' energy partials where its thread count
changes: rows of 200 points take four rows a workgroup, so n2 n3 / 4 partials,
here 4096 (two rounds of 256 threads, the last size of that form), 4320 and
8192 (part of and exactly one round of 1024) and 8269 (a second round of 77).
The ion-electron energy is a plain sum of products: against numpy at 1e-13 of
the sum of magnitudes (30 levels of pairwise rounding are 3e-15, the point
products add 4e-16). All energies against the staged passes, whose partials are
grouped otherwise, at the bound of the other register passes."""
import numpy as np
import pytest

from tests.test_gpu_lengths import LAT, _run, pa  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("grid", [(200, 128, 128), (200, 128, 135), (200, 128, 256), (200, 135, 245)])
def test_final_sum(pa, monkeypatch, grid):  # noqa: F811
    print(grid, flush=True)
    n1, n2, n3 = grid
    lat = LAT * (0.24 * np.array(grid))[None, :]
    vol = abs(np.linalg.det(lat))
    rng = np.random.default_rng(n2 + n3)
    rho = 0.027 * (1.0 + 0.3 * (2.0 * rng.random((n3, n2, n1)) - 1.0))
    vion = rng.random((n3, n2, n1)) - 0.5
    _, et = _run(pa, grid, "wt", rho, vion, 0.027 * vol, lat)
    p, dv = rho * vion, vol / rho.size
    assert abs(et[2] - p.sum() * dv) <= 1e-13 * np.abs(p).sum() * dv
    monkeypatch.setenv("OFD_GENERIC", "1")
    _, e0 = _run(pa, grid, "wt", rho, vion, 0.027 * vol, lat)
    assert np.all(np.abs(et - e0) <= 1e-12 * np.abs(e0) + 1e-12)
