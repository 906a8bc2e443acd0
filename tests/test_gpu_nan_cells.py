"""A NaN cell in a mixture block or a block built from its grid, in the fast forms: the
clipping of a reconstructed value hands on a NaN of the cell to the right of a face, as
the reference's comparisons do, so that the step over it ends as in the reference
arithmetic, with the same counts of bad cells (none of its neighbours is spared)."""
import numpy as np
import pytest

import eilmer4_amd as e4
from eilmer4_amd.fvcore import BCType, Face, FlowSolverException
from eilmer4_amd.lib import E4hipError
from test_oracle_geometry import curvy_grid

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(33, 9, 7), (40, 12, 1)])
@pytest.mark.parametrize("what,quantity", [("grid", 4), ("grid", 1), ("mixture", 1), ("grid mixture", 1)])
@pytest.mark.parametrize("flux", ["ausmdv", "adaptive_hanel_ausmdv"])
def test_ends_as_in_reference_arithmetic(gpu, n, what, quantity, flux):
    ni, nj, nk = n
    dims = 2 if nk == 1 else 3
    rng = np.random.default_rng(11)
    nc = ni * nj * nk
    v = 20.0 * rng.standard_normal((3, nc))
    if dims == 2:
        v[2] = 0.0
    if "mixture" in what:
        gas = e4.ThermallyPerfectGas.from_json()
        T = 900.0 + 100.0 * rng.random(nc)
        Y = rng.random((5, nc)) + 0.05
        Y /= Y.sum(axis=0)
        U0, guess = gas.encode(0.2 + 0.05 * rng.random(nc), gas.energy(T, Y), *v, Y), (T,)
    else:
        gas = e4.IdealGas()
        rho, u, _ = gas.rho_u_a_from_pT(1.0e5 * (0.9 + 0.2 * rng.random(nc)), 300.0 * (0.9 + 0.2 * rng.random(nc)))
        U0, guess = gas.encode(rho, u, *v), ()
    cells = np.zeros((nk, nj, ni), bool)
    cells[nk // 2, 4::6, 3::7] = True
    bad = U0.copy()
    bad[quantity, cells.ravel()] = np.nan
    grid = curvy_grid(ni, nj, nk, seed=5)
    if dims == 2:
        grid = grid[0].copy()
        grid[..., 2] = 0.0
    ends = {}
    for precision in ("fp64_exact", "fp64", "mixed"):
        b = e4.SFluidBlock.from_grid(gas, grid) if "grid" in what else e4.SFluidBlock(gas, dims, ni, nj, nk, 0.1, 0.1, 0.1)
        for face in list(Face)[:2 * dims]:
            b.set_bc(face, BCType.periodic, None)
        sim = e4.Simulation([b], e4.GlobalConfig(precision_mode=e4.PrecisionMode[precision],
                                                 flux_calculator=e4.FluxCalculator[flux], max_invalid_cells=nc))
        b.upload(U0, *guess)
        with pytest.raises(E4hipError):              # the upload says so, and leaves the state in place
            b.upload(bad, *guess)
        sim.state.dt_global = 1.0e-8
        stopped = False
        try:
            sim.gasdynamic_explicit_increment_with_fixed_grid()
        except FlowSolverException:
            stopped = True
        ends[precision] = (stopped, sim.last_bad_cells)
        b.destroy()
    assert ends["fp64"] == ends["fp64_exact"]
    assert ends["mixed"] == ends["fp64_exact"]
