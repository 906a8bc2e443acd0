"""The plain FP64 form's sound speed at the ends of the square root's range: cells that
decode to T = 0 (a = 0) and to an infinite energy (a = inf).  An upload reports such cells
and leaves them in place; a step over them ends as it does in the reference arithmetic,
with the same count of bad cells.  AUSM+-up takes the mean of the two sides' sound speeds
and HLLC and Roe their wave speeds from them, so a NaN in place of either would change
the faces around the cell.

Only how the step ends is compared, not its states: a stage sets a cell whose energy is
not above zero to 200 K, and around zero a rounding decides that.
"""
import numpy as np
import pytest

import eilmer4_amd as e4
from eilmer4_amd.fvcore import BCType, Face, FlowSolverException
from eilmer4_amd.lib import E4hipError

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(33, 9, 7), (40, 12, 1)])
@pytest.mark.parametrize("flux,energy", [("ausm_plus_up", 0.0), ("hllc", np.inf), ("roe", np.inf)])
def test_same_as_reference_arithmetic(gpu, n, flux, energy):
    ni, nj, nk = n
    dims = 2 if nk == 1 else 3
    gas = e4.IdealGas()
    rng = np.random.default_rng(11)
    nc = ni * nj * nk
    rho, u, _ = gas.rho_u_a_from_pT(1.0e5 * (0.9 + 0.2 * rng.random(nc)), 300.0 * (0.9 + 0.2 * rng.random(nc)))
    v = 20.0 * rng.standard_normal((3, nc))
    if dims == 2:
        v[2] = 0.0
    U0 = gas.encode(rho, u, *v).reshape(5, nk, nj, ni).copy()
    cells = np.zeros((nk, nj, ni), bool)
    cells[nk // 2, 4::6, 3::7] = True            # alone, inside the block and at tile edges
    U0[1:4, cells] = 0.0
    U0[4, cells] = energy
    U0 = np.ascontiguousarray(U0.reshape(5, nc))
    ends = []
    for precision in ("fp64_exact", "fp64"):
        b = e4.SFluidBlock(gas, dims, ni, nj, nk, 0.1, 0.1, 0.1)
        for face in list(Face)[:2 * dims]:
            b.set_bc(face, BCType.periodic, None)
        sim = e4.Simulation([b], e4.GlobalConfig(precision_mode=e4.PrecisionMode[precision],
                                                 flux_calculator=e4.FluxCalculator[flux], max_invalid_cells=nc))
        if energy == 0.0:
            with pytest.raises(E4hipError):
                b.upload(U0)
        else:
            try:
                b.upload(U0)
            except E4hipError:
                pass
        sim.state.dt_global = 1.0e-6
        stopped = False
        try:
            sim.gasdynamic_explicit_increment_with_fixed_grid()
        except FlowSolverException:
            stopped = True
        ends.append((stopped, sim.last_bad_cells[0], b.download()))
        b.destroy()
    (stop0, bad0, U), (stop1, bad1, Uf) = ends
    assert (stop0, bad0) == (stop1, bad1)
    if not stop0:
        assert np.all(np.isfinite(U)) and np.all(np.isfinite(Uf))
