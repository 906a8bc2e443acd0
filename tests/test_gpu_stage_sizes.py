"""The ideal-gas stage kernel at the edges of its tiles (32 x 8 columns) and chunks:
halo cells that lie in the block, copy a cell of it (wall, extrapolation, periodic)
or have a ghost state of their own (inflow, connected faces), with one, two, three
and all planes to a workgroup, for a flux with and without the shock indicator and
for a formula of its own.

fp64_exact is bit-identical to the oracle.  The plain form regroups the arithmetic:
a cell's update is some 300 roundings of 1.1e-16 of terms no larger than a few times
its state, so after a step it is within 1e-12 of the oracle's norm."""
import numpy as np
import pytest

import eilmer4_amd as e4
import pyoracle as O
from eilmer4_amd.fvcore import BCType, Face
from parity_helpers import rel_err

pytestmark = pytest.mark.gpu

PAIRS = [(Face.west, Face.east), (Face.south, Face.north), (Face.bottom, Face.top)]
SIZES = [(2, 2, 2), (31, 7, 4), (32, 8, 5), (33, 9, 6), (64, 3, 7), (65, 17, 3), (3, 16, 9), (33, 9, 1), (64, 16, 1)]


@pytest.mark.parametrize("kinds", ["wall", "extrapolate", "periodic", "inflow", "connected"])
@pytest.mark.parametrize("n", SIZES)
def test_step_matches_oracle(gpu, monkeypatch, n, kinds):
    ni, nj, nk = n
    dims = 2 if nk == 1 else 3
    gas = e4.IdealGas()
    rng = np.random.default_rng(ni * 10000 + nj * 100 + nk)
    nc = ni * nj * nk
    rho, u, _ = gas.rho_u_a_from_pT(1.0e5 * (0.7 + 0.6 * rng.random(nc)), 300.0 * (0.7 + 0.6 * rng.random(nc)))
    vz = (90.0 if dims == 3 else 0.0) * rng.standard_normal(nc)
    U0 = gas.encode(rho, u, *(90.0 * rng.standard_normal((2, nc))), vz)
    fs = gas.flowstate(1.0e5, 300.0, (700.0, 60.0, 30.0 if dims == 3 else 0.0))

    def bcs(b):
        for pair in PAIRS[:dims]:
            for side, face in enumerate(pair):
                kind = {"wall": BCType.slip_wall, "extrapolate": BCType.extrapolate, "periodic": BCType.periodic,
                        "inflow": BCType.extrapolate if side else BCType.inflow}.get(kinds)
                if kind is not None:
                    b.set_bc(face if isinstance(b, e4.SFluidBlock) else int(face),
                             kind if isinstance(b, e4.SFluidBlock) else int(kind),
                             fs if kind == BCType.inflow else None)
            if kinds == "connected":
                if isinstance(b, e4.SFluidBlock):
                    e4.connect_blocks(b, pair[1], b, pair[0], 0)
                else:
                    O.connect_blocks(b, int(pair[1]), b, int(pair[0]), 0)

    for flux in ("ausmdv", "adaptive_hanel_ausmdv", "hllc"):
        ob = O.Block(O.Gas.ideal(), dims, ni, nj, nk, 0.1, 0.1, 0.1)
        ob.set_config(flux_calc=int(e4.FluxCalculator[flux]))
        bcs(ob)
        ob.set_U(U0)
        dt, _, _ = ob.determine_dt(1e-3, 0.3, False)
        if kinds == "connected":
            assert O.multi_step([ob], dt)[0] == 0
        else:
            assert ob.step(dt)[0] == 0
        Uo = ob.get_U()
        for precision in ("fp64_exact", "fp64"):
            for height in (1, 2, 3, nk):
                if height > nk:
                    continue
                monkeypatch.setenv("E4HIP_KCHUNK", str(height))
                db = e4.SFluidBlock(gas, dims, ni, nj, nk, 0.1, 0.1, 0.1)
                bcs(db)
                db.upload(U0)
                sim = e4.Simulation([db], e4.GlobalConfig(precision_mode=e4.PrecisionMode[precision],
                                                          flux_calculator=e4.FluxCalculator[flux]))
                sim.state.dt_global = dt
                sim.gasdynamic_explicit_increment_with_fixed_grid()
                U = db.download()
                db.destroy()
                what = (flux, precision, height, rel_err(U, Uo))
                if precision == "fp64_exact":
                    assert np.array_equal(U, Uo), what
                else:
                    assert rel_err(U, Uo).max() <= 1.0e-12, what
