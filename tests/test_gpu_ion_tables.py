"""The B-spline table and force stencils at the sizes where their indexing can
go wrong: axes shorter than the stencil (it wraps more than once), of exactly
two bins, with a last bin of one point, rows longer than one pass of a wave
(n1 > 256), the shortest and longest splines, and ions outside the cell
[0, 1). Against the oracle at the bounds of the other ion tests: the potential
within 1e-11 and the forces within 1e-10 of their maximum."""
import numpy as np
import pytest

from oracle import profess_oracle as O

pytestmark = pytest.mark.gpu

CASES = [((12, 20, 21), 10), ((12, 10, 14), 16), ((20, 40, 42), 10), ((288, 18, 20), 10), ((24, 21, 25), 4),
         ((18, 9, 8), 4), ((90, 48, 45), 16)]


@pytest.mark.parametrize("grid,order", CASES)
def test_spline_tables(grid, order):
    import profess_amd as pa
    print(grid, order, flush=True)
    lat = np.diag(0.4 * np.array(grid)) + 0.3 * np.array([[0, 1, 0], [0, 0, 1], [1, 0, 0]])
    cell = O.Cell(lat, *grid)
    rng = np.random.default_rng(5)
    frac = rng.random((7, 3))
    frac[0] = [0.0, 0.0, 0.0]
    frac[1] = [-0.3, 1.2, 0.999]
    mg, v = O.synthetic_recpot_values(3, 1.2)
    psp = O.make_psp(mg, v)
    s = pa.OFDSystem(lat, grid, 21.0)
    s.build_ion_potential([(mg, v, frac)], spline_order=order)
    ref = O.ion_potential(cell, [(psp, frac)], order)
    assert np.max(np.abs(s.ion_potential() - ref)) <= 1e-11 * np.max(np.abs(ref))
    rho = 21.0 / cell.vol * (1 + 0.2 * rng.random(cell.shape))
    fr = O.ion_forces(cell, [(psp, frac)], rho, order)
    assert np.max(np.abs(pa.IonElectronForcesSpline(s, rho) - fr)) <= 1e-10 * np.max(np.abs(fr)) + 1e-14
    s.close()
