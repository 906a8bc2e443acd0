"""Blocks with more cells than 32-bit byte offsets reach: E4HIP_WIDE_OFFSETS gives small
blocks the route of such a block through the face kernels of mixtures and of blocks
built from their grid.  It changes how a cell is addressed and not what is computed, so
every value must be the same, bit for bit."""
import numpy as np
import pytest

import eilmer4_amd as e4
from eilmer4_amd.fvcore import BCType, Face
from test_oracle_geometry import curvy_grid

pytestmark = pytest.mark.gpu

PAIRS = [(Face.west, Face.east), (Face.south, Face.north), (Face.bottom, Face.top)]


@pytest.mark.parametrize("kinds", ["wall", "periodic", "inflow", "connected"])
@pytest.mark.parametrize("n", [(2, 2, 2), (65, 3, 4), (5, 67, 2), (31, 9, 1)])
@pytest.mark.parametrize("what", ["mixture", "grid", "grid mixture"])
def test_same_bits(gpu, monkeypatch, what, n, kinds):
    ni, nj, nk = n
    dims = 2 if nk == 1 else 3
    rng = np.random.default_rng(ni * 10000 + nj * 100 + nk)
    nc = ni * nj * nk
    v = 80.0 * rng.standard_normal((3, nc))
    inflow_v = (700.0, 60.0, 30.0 if dims == 3 else 0.0)
    if dims == 2:
        v[2] = 0.0
    if "mixture" in what:
        gas = e4.ThermallyPerfectGas.from_json()
        T = 900.0 + 700.0 * rng.random(nc)
        Y = rng.random((5, nc)) + 0.05
        Y /= Y.sum(axis=0)
        state = gas.encode(0.2 + 0.1 * rng.random(nc), gas.energy(T, Y), *v, Y), T
        fs = gas.flowstate(2.0e4, 1000.0, inflow_v, [0.7, 0.2, 0.05, 0.03, 0.02])
    else:
        gas = e4.IdealGas()
        rho, u, _ = gas.rho_u_a_from_pT(1.0e5 * (0.7 + 0.6 * rng.random(nc)), 300.0 * (0.7 + 0.6 * rng.random(nc)))
        state = (gas.encode(rho, u, *v),)
        fs = gas.flowstate(1.0e5, 300.0, inflow_v)
    grid = curvy_grid(ni, nj, nk, seed=5)
    if dims == 2:
        grid = grid[0].copy()
        grid[..., 2] = 0.0
    for precision in ("fp64_exact", "fp64", "mixed"):
        for flux in ("ausmdv", "adaptive_hanel_ausmdv"):
            out = []
            for wide in ("0", "1"):
                monkeypatch.setenv("E4HIP_WIDE_OFFSETS", wide)
                b = e4.SFluidBlock.from_grid(gas, grid) if "grid" in what else e4.SFluidBlock(gas, dims, ni, nj, nk, 0.1, 0.1, 0.1)
                for pair in PAIRS[:dims]:
                    if kinds == "connected":
                        e4.connect_blocks(b, pair[1], b, pair[0], 0)
                        continue
                    for side, face in enumerate(pair):
                        kind = {"wall": BCType.slip_wall, "periodic": BCType.periodic,
                                "inflow": BCType.extrapolate if side else BCType.inflow}[kinds]
                        b.set_bc(face, kind, fs if kind == BCType.inflow else None)
                sim = e4.Simulation([b], e4.GlobalConfig(precision_mode=e4.PrecisionMode[precision],
                                                         flux_calculator=e4.flux_calculator_from_name(flux)))
                b.upload(*state)           # (decoded in the configured precision)
                for _ in range(2):
                    sim.state.dt_global = 1.0e-7
                    sim.gasdynamic_explicit_increment_with_fixed_grid()
                out.append(b.download())
                b.destroy()
            assert np.all(np.isfinite(out[0]))
            assert np.array_equal(out[0], out[1]), (precision, flux)
