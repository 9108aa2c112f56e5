"""The chunk heights chosen by the library (omhd_step.hip default_rows: one per
pass, from 1 row up, by the number of chunks) against a height given by the
caller: the same bits, at sizes where the chosen heights and the last chunk's
remainder differ."""
import numpy as np
import pytest

from omhd_testlib import smooth_state
from test_oracle_golden import bits_equal

pytestmark = pytest.mark.gpu


def run(U, shape, rows, walls, resistive):
    from openmhd_amd import Solver

    nx, ny, nz = shape
    bc = ("periodic", "wall" if walls else "periodic", "periodic")[:3 if nz else 2]
    s = Solver(nx, ny, 0.1, nz=nz, cfl=0.4, lm_type=2, bc=bc, rows_per_wave=rows,
               resistivity=(1.0 / 60, 1.0 / 1000, 4.0) if resistive else None)
    s.upload(U)
    dts, _ = s.step(3, trace=True)
    V = s.download()
    s.close()
    return dts, V


@pytest.mark.parametrize("shape,walls,resistive", [
    ((4, 4, 0), False, False), ((61, 9, 0), True, False), ((1030, 61, 0), True, False),
    ((700, 1500, 0), False, False), ((2200, 2100, 0), False, False),
    ((61, 5, 4), True, False), ((7, 40, 33), False, True), ((130, 70, 50), True, False), ((121, 96, 80), True, True)])
def test_chosen_heights(shape, walls, resistive):
    nx, ny, nz = shape
    U = smooth_state(np.random.default_rng(nx + ny), nx + 2, ny + 2, *([nz + 2] if nz else []))
    a, b = run(U, shape, 0, walls, resistive), run(U, shape, 11, walls, resistive)
    assert bits_equal(a[0], b[0]) and bits_equal(a[1], b[1])


def test_ensemble_heights():
    from openmhd_amd import Ensemble, Solver
    from openmhd_amd.solver import make_config

    sizes = [(6, 5), (61, 40), (200, 77)]
    e = Ensemble([make_config(nx, ny, 0.1) for nx, ny in sizes])
    Us = [smooth_state(np.random.default_rng(i), nx + 2, ny + 2) for i, (nx, ny) in enumerate(sizes)]
    for i, U in enumerate(Us):
        e.upload(i, U)
    e.step(3)
    for i, ((nx, ny), U) in enumerate(zip(sizes, Us)):
        s = Solver(nx, ny, 0.1, rows_per_wave=11)
        s.upload(U)
        s.step(3)
        assert bits_equal(e.download(i), s.download())
        s.close()
    e.close()
