"""The time-step reduction over more blocks than are read back at once (128): the limiting
cell in the first block, at either side of that edge and in the last, with and without the
rescaling of a CFL number that is too large.  Equal to the oracle's per-block values
combined: the smallest dt_allow and the largest cfl_max."""
import numpy as np
import pytest

import eilmer4_amd as e4
import pyoracle as O

pytestmark = pytest.mark.gpu

NBLK, NI, NJ = 131, 4, 3


@pytest.mark.parametrize("limiting", [0, 127, 128, NBLK - 1])
def test_matches_oracle(gpu, limiting):
    gas = e4.IdealGas()
    rng = np.random.default_rng(limiting)
    og = O.Gas.ideal()
    obs, dbs = [], []
    for n in range(NBLK):
        nc = NI * NJ
        rho, u, _ = gas.rho_u_a_from_pT(1.0e5 * (0.9 + 0.2 * rng.random(nc)), 300.0 * (0.9 + 0.2 * rng.random(nc)))
        v = 50.0 * rng.standard_normal((2, nc))
        if n == limiting:
            v[0, rng.integers(nc)] = 2500.0
        U = gas.encode(rho, u, v[0], v[1], np.zeros(nc))
        ob, db = O.Block(og, 2, NI, NJ, 1, 0.1, 0.1, 1.0), e4.SFluidBlock(gas, 2, NI, NJ, 1, 0.1, 0.1, 1.0)
        ob.set_config()
        ob.set_U(U)
        db.upload(U)
        obs.append(ob)
        dbs.append(db)
    sim = e4.Simulation(dbs, e4.GlobalConfig(precision_mode=e4.PrecisionMode.fp64_exact))
    for dt, check in ((1.0e-5, False), (1.0e-5, True), (1.0e-3, True)):
        per = [ob.determine_dt(dt, 0.5, check) for ob in obs]
        dt_allow, cfl_max = sim.block_dt(dt, check)
        assert (dt_allow, cfl_max) == (min(p[0] for p in per), max(p[1] for p in per)), (dt, check)
        if not check:
            assert min(range(NBLK), key=lambda n: per[n][0]) == limiting
    for db in dbs:
        db.destroy()
