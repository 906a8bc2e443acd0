"""Blocks built from their grid at the edges of the face launch: workgroups of 128
faces, the directions' faces in turn, runs of workgroups dealt to eight dies; stencil
positions that are cells, copy one (wall, extrapolation, periodic) or have a state of
their own (inflow, connected faces), down to two cells in a direction.

fp64_exact is bit-identical to the oracle.  The plain form regroups some 300
roundings of 1.1e-16 per cell, of terms no larger than a few times its state: within
1e-12 of the oracle's norm after a step."""
import numpy as np
import pytest

import eilmer4_amd as e4
import pyoracle as O
from eilmer4_amd.fvcore import BCType, Face
from parity_helpers import rel_err
from test_gpu_geometry import _device_from_grid, _inflow, _mixed_bcs, _oracle_from_grid, _U0
from test_oracle_geometry import curvy_grid

pytestmark = pytest.mark.gpu

PAIRS = [(Face.west, Face.east), (Face.south, Face.north), (Face.bottom, Face.top)]
SIZES = [(2, 2, 2), (3, 2, 5), (127, 2, 2), (128, 3, 2), (31, 17, 4), (2, 64, 3), (2, 2, 1), (129, 8, 1)]


@pytest.mark.parametrize("kinds", ["mixed", "wall", "periodic", "connected"])
@pytest.mark.parametrize("n", SIZES)
def test_step_matches_oracle(gpu, n, kinds):
    ni, nj, nk = n
    dims = 2 if nk == 1 else 3
    gas = e4.IdealGas()
    g = curvy_grid(ni, nj, nk, seed=5)
    if dims == 2:
        g = g[0].copy()
        g[..., 2] = 0.0
    U0 = _U0(gas, (nk, nj, ni), 6)
    kind = {"wall": BCType.slip_wall, "periodic": BCType.periodic}.get(kinds)
    bcs = _mixed_bcs(dims) if kinds == "mixed" else {f: kind for pair in PAIRS[:dims] for f in pair if kind is not None}
    fs_in = _inflow(gas)
    for flux in ("ausmdv", "adaptive_hanel_ausmdv"):
        fc = e4.flux_calculator_from_name(flux)
        ob = _oracle_from_grid(g, U0, bcs, fs_in, fc)
        if kinds == "connected":
            for lo, hi in PAIRS[:dims]:
                O.connect_blocks(ob, int(hi), ob, int(lo), 0)
        dt = 1.0e-7
        assert O.multi_step([ob], dt)[0] == 0
        Uo = ob.get_U()
        for precision in ("fp64_exact", "fp64"):
            db = _device_from_grid(gas, g, U0, bcs, fs_in)
            if kinds == "connected":
                for lo, hi in PAIRS[:dims]:
                    e4.connect_blocks(db, hi, db, lo, 0)
            sim = e4.Simulation([db], e4.GlobalConfig(flux_calculator=fc, precision_mode=e4.PrecisionMode[precision]))
            sim.state.dt_global = dt
            sim.gasdynamic_explicit_increment_with_fixed_grid()
            U = db.download()
            db.destroy()
            if precision == "fp64_exact":
                assert np.array_equal(U, Uo), (flux, rel_err(U, Uo))
            else:
                assert rel_err(U, Uo).max() <= 1.0e-12, (flux, rel_err(U, Uo))
