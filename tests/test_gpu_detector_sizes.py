"""The shock detector's tiles: a wave is a row of 62 cells with a lane beyond it on
either side, a workgroup eight rows, marching up to 16 planes.  Sizes at those
edges, with ghosts that copy a cell of the block (wall, extrapolation, periodic)
and ghosts that do not (inflow), one step of adaptive_hanel_ausmdv on a rough
field where a good part of the cells are shock points.

fp64_exact is bit-identical to the oracle (a single wrong indicator changes a
flux); the fast form's detector compares squares, so its bar is that of the
plain form after one step, 1e-12."""
import numpy as np
import pytest

import eilmer4_amd as e4
import pyoracle as O
from eilmer4_amd.fvcore import BCType, Face
from parity_helpers import rel_err

pytestmark = pytest.mark.gpu

PAIRS = [(Face.west, Face.east), (Face.south, Face.north), (Face.bottom, Face.top)]
SIZES = [(2, 2, 2), (61, 7, 3), (62, 8, 4), (63, 9, 5), (64, 2, 17), (124, 3, 16), (125, 17, 2), (3, 3, 33),
         (62, 8, 1), (63, 9, 1), (130, 3, 1), (2, 2, 1)]


@pytest.mark.parametrize("kinds", ["wall", "extrapolate", "periodic", "inflow"])
@pytest.mark.parametrize("n", SIZES)
def test_step_matches_oracle(n, kinds):
    ni, nj, nk = n
    dims = 2 if nk == 1 else 3
    gas = e4.IdealGas()
    rng = np.random.default_rng(ni * 10000 + nj * 100 + nk)
    nc = ni * nj * nk
    rho, u, _ = gas.rho_u_a_from_pT(1.0e5 * (0.7 + 0.6 * rng.random(nc)), 300.0 * (0.7 + 0.6 * rng.random(nc)))
    U0 = gas.encode(rho, u, *(90.0 * rng.standard_normal((2, nc))), (90.0 if dims == 3 else 0.0) * rng.standard_normal(nc))
    fs = gas.flowstate(1.0e5, 300.0, (700.0, 60.0, 30.0 if dims == 3 else 0.0))
    ob = O.Block(O.Gas.ideal(), dims, ni, nj, nk, 0.1, 0.1, 0.1)
    ob.set_config(flux_calc=int(e4.FluxCalculator.adaptive_hanel_ausmdv))
    bcs = {}
    for d, pair in enumerate(PAIRS[:dims]):
        for side, face in enumerate(pair):
            bcs[face] = {"wall": (BCType.slip_wall, None), "extrapolate": (BCType.extrapolate, None),
                         "periodic": (BCType.periodic, None),
                         "inflow": (BCType.inflow, fs) if side == 0 else (BCType.extrapolate, None)}[kinds]
            ob.set_bc(int(face), int(bcs[face][0]), bcs[face][1])
    ob.set_U(U0)
    dt, _, _ = ob.determine_dt(1e-3, 0.3, False)
    assert ob.step(dt)[0] == 0
    Uo = ob.get_U()
    for precision in ("fp64_exact", "fp64"):
        db = e4.SFluidBlock(gas, dims, ni, nj, nk, 0.1, 0.1, 0.1)
        for face, (kind, state) in bcs.items():
            db.set_bc(face, kind, state)
        db.upload(U0)
        sim = e4.Simulation([db], e4.GlobalConfig(precision_mode=e4.PrecisionMode[precision]))
        sim.state.dt_global = dt
        sim.gasdynamic_explicit_increment_with_fixed_grid()
        U = db.download()
        db.destroy()
        if precision == "fp64_exact":
            assert np.array_equal(U, Uo), rel_err(U, Uo)
        else:
            assert rel_err(U, Uo).max() <= 1.0e-12, rel_err(U, Uo)
