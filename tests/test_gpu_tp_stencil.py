"""Mixture face kernels: waves whose stencils all lie in their own block are read
through scalar bases, the others position by position.  Blocks of two to a few
cells across and rows around the wave's 64 lanes, with every kind of ghost that
is a cell of the block (wall, extrapolation, periodic) and one that is not
(inflow), against the oracle.

Tolerance: the bar of the mixture steps (1e-10 relative to each quantity's
maximum): the same algorithm, another library's logarithm."""
import numpy as np
import pytest

import eilmer4_amd as e4
import pyoracle as O
from eilmer4_amd import workloads
from eilmer4_amd.fvcore import BCType, Face
from parity_helpers import rel_err

pytestmark = pytest.mark.gpu

PAIRS = [(Face.west, Face.east), (Face.south, Face.north), (Face.bottom, Face.top)]


@pytest.mark.parametrize("kinds", ["wall", "extrapolate", "periodic", "inflow"])
@pytest.mark.parametrize("n", [(2, 3, 5), (3, 2, 2), (64, 2, 3), (63, 3, 2), (65, 2, 2), (5, 67, 2), (31, 4, 1)])
def test_steps_match_oracle(n, kinds):
    ni, nj, nk = n
    dims = 2 if nk == 1 else 3
    gas = e4.ThermallyPerfectGas.from_json()
    rng = np.random.default_rng(ni * 100 + nj * 10 + nk)
    nc = ni * nj * nk
    T = 900.0 + 700.0 * rng.random(nc)
    Y = rng.random((5, nc)) + 0.05
    Y /= Y.sum(axis=0)
    U0 = gas.encode(0.2 + 0.1 * rng.random(nc), gas.energy(T, Y), *(80.0 * rng.standard_normal((2, nc))),
                    (80.0 if dims == 3 else 0.0) * rng.standard_normal(nc), Y)
    fs = gas.flowstate(2.0e4, 1000.0, (200.0, 30.0, 10.0 if dims == 3 else 0.0), [0.7, 0.2, 0.05, 0.03, 0.02])
    og = O.Gas.from_json("therm-perf-5-species-air.json")
    ob = O.Block(og, dims, ni, nj, nk, 0.1, 0.1, 0.1)
    ob.set_config(flux_calc=O.AUSMDV)
    db = e4.SFluidBlock(gas, dims, ni, nj, nk, 0.1, 0.1, 0.1)
    for d, pair in enumerate(PAIRS[:dims]):
        for side, face in enumerate(pair):
            kind, state = {"wall": (BCType.slip_wall, None), "extrapolate": (BCType.extrapolate, None),
                           "periodic": (BCType.periodic, None),
                           "inflow": (BCType.inflow, fs) if side == 0 else (BCType.extrapolate, None)}[kinds]
            ob.set_bc(int(face), int(kind), state)
            db.set_bc(face, kind, state)
    ob.set_U(U0, T)
    sim = e4.Simulation([db], e4.GlobalConfig(flux_calculator=e4.FluxCalculator.ausmdv))
    db.upload(U0, T)
    dt, _, _ = ob.determine_dt(1e-3, 0.25, False)
    for _ in range(2):
        assert ob.step(dt)[0] == 0
        sim.state.dt_global = dt
        sim.gasdynamic_explicit_increment_with_fixed_grid()
    err = rel_err(db.download(), ob.get_U())
    db.destroy()
    assert err.max() <= 1.0e-10, err
