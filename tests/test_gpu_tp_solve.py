"""The fast modes' temperature solve (tp_newton_fast) from good, far-off and
misleading guesses: it evaluates the ends of its bracket only when it has to,
and must end where the reference's solve ends.

Tolerance: both solves stop at a last step below 1e-6 K, so each root is within
1e-6 K of the curve's (a bisection step; Newton steps leave far less): 2e-6 K
between them, plus rounding (1e-12 T)."""
import numpy as np
import pytest

import eilmer4_amd as e4
import pyoracle as O
from eilmer4_amd import workloads

pytestmark = pytest.mark.gpu

GUESSES = {
    "exact": lambda T: T,
    "near": lambda T: T * 1.01,
    "inside the bracket, above": lambda T: T + 480.0,
    "inside the bracket, below": lambda T: np.maximum(T - 480.0, 25.0),
    "root at the bracket's end": lambda T: T - 500.0 + 1.0e-4,
    "outside the bracket, above": lambda T: T + 700.0,
    "outside the bracket, below": lambda T: np.maximum(T - 2500.0, 60.0),
    "uniform 300 K": lambda T: np.full_like(T, 300.0),
    "uniform 20000 K": lambda T: np.full_like(T, 20000.0),
    "in the first blend": lambda T: np.full_like(T, 1000.0),
    "one cell in 64 off": lambda T: np.where(np.arange(T.size) % 64 == 7, T + 900.0, T),
}


@pytest.mark.parametrize("name", sorted(GUESSES))
def test_decode_from_guess(name):
    gas = e4.ThermallyPerfectGas.from_json()
    ni, nj, nk = 13, 11, 9                     # 1287 cells: a last wave of 7 lanes
    geom, fields, _, _ = workloads.thermally_perfect_box_3d(gas, n=16)
    U, T = workloads.initial_U_tp(gas, fields)
    n = ni * nj * nk
    U, T = np.ascontiguousarray(U[:, :n]), T[:n].copy()
    Tg = np.maximum(GUESSES[name](T), 21.0)
    ob = O.Block(O.Gas.from_json("therm-perf-5-species-air.json"), 3, ni, nj, nk, 1.0, 1.0, 1.0)
    ob.set_config()
    ob.set_U(U, Tg)
    blk = e4.SFluidBlock(gas, 3, ni, nj, nk, 1.0, 1.0, 1.0)
    e4.Simulation([blk], e4.GlobalConfig(precision_mode=e4.PrecisionMode.fp64))
    blk.upload(U, Tg)
    fs = blk.download(with_fs=True)[1]
    blk.destroy()
    To = ob.get_fs()[2]
    assert np.all(np.abs(fs[2] - To) <= 2.0e-6 + 1.0e-12 * To), np.max(np.abs(fs[2] - To))
