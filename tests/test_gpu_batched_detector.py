"""The shock detector's one launch over the blocks of a batched stage: joined 2D and 3D
blocks of unequal odd sizes about its tiles (rows of 62 cells, eight rows), one step of
adaptive_hanel_ausmdv on a rough field against the oracle.

fp64_exact is bit-identical (a wrong indicator changes a flux); the plain form's bar after
one step is 1e-12."""
import numpy as np
import pytest

import eilmer4_amd as e4
import pyoracle as O
from eilmer4_amd.fvcore import BCType, Face
from parity_helpers import rel_err

pytestmark = pytest.mark.gpu

SIZES = {2: [(61, 9, 1), (63, 9, 1), (3, 9, 1), (130, 9, 1), (62, 9, 1)],
         3: [(61, 13, 5), (64, 13, 5), (2, 13, 5), (125, 13, 5)]}


@pytest.mark.parametrize("dims", [2, 3, "2 and 3"])
def test_step_matches_oracle(gpu, dims):
    gas = e4.IdealGas()
    rng = np.random.default_rng(21)
    chains = [SIZES[d] for d in ((2, 3) if dims == "2 and 3" else (dims,))]
    for precision in ("fp64_exact", "fp64"):
        obs, dbs = [], []
        for sizes in chains:
            d = 2 if sizes[0][2] == 1 else 3
            oc, dc = [], []
            for n in sizes:
                nc = n[0] * n[1] * n[2]
                rho, u, _ = gas.rho_u_a_from_pT(1.0e5 * (0.7 + 0.6 * rng.random(nc)), 300.0 * (0.7 + 0.6 * rng.random(nc)))
                v = 90.0 * rng.standard_normal((3, nc))
                if d == 2:
                    v[2] = 0.0
                U = gas.encode(rho, u, *v)
                ob, db = O.Block(O.Gas.ideal(), d, *n, 0.1, 0.1, 0.1), e4.SFluidBlock(gas, d, *n, 0.1, 0.1, 0.1)
                ob.set_config(flux_calc=int(e4.FluxCalculator.adaptive_hanel_ausmdv))
                for face in list(Face)[:2 * d]:
                    if face in (Face.east, Face.west):
                        continue
                    kind = BCType.slip_wall if face in (Face.south, Face.bottom) else BCType.extrapolate
                    ob.set_bc(int(face), int(kind), None)
                    db.set_bc(face, kind, None)
                ob.set_U(U)
                db.upload(U)
                oc.append(ob)
                dc.append(db)
            for k in range(len(sizes)):
                O.connect_blocks(oc[k], int(Face.east), oc[(k + 1) % len(sizes)], int(Face.west), 0)
                e4.connect_blocks(dc[k], Face.east, dc[(k + 1) % len(sizes)], Face.west, 0)
            obs += oc
            dbs += dc
        dt = 2.0e-5
        assert O.multi_step(obs, dt)[0] == 0
        sim = e4.Simulation(dbs, e4.GlobalConfig(precision_mode=e4.PrecisionMode[precision], batch_blocks=True))
        sim.state.dt_global = dt
        sim.gasdynamic_explicit_increment_with_fixed_grid()
        for ob, db in zip(obs, dbs):
            U, Uo = db.download(), ob.get_U()
            if precision == "fp64_exact":
                assert np.array_equal(U, Uo), rel_err(U, Uo)
            else:
                assert rel_err(U, Uo).max() <= 1.0e-12, rel_err(U, Uo)
        for db in dbs:
            db.destroy()
