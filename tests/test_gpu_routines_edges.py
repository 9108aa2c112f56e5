"""The separate routines at the edges of their index ranges (csrc/omhd_dropin.hip:
one lane per cell of a box, x fastest, whatever the direction): extents of one,
two and three cells, lines longer than a workgroup, and for set_dt more cells
than one round of workgroups.  Bit for bit against the oracle, what a routine
leaves unwritten included."""
import ctypes as C

import numpy as np
import pytest

from omhd_testlib import farr, ptr, random_prim, prim_to_cons
from test_oracle_golden import bits_equal

pytestmark = pytest.mark.gpu

SHAPES = [(2, 7, 1), (7, 2, 1), (261, 3, 1), (3, 70, 5), (70, 3, 5), (5, 6, 2), (4, 3, 67), (33, 18, 17)]


def dirs(shape):
    return [d for d in (1, 2, 3) if shape[d - 1] > 1]


@pytest.mark.parametrize("shape", SHAPES)
def test_limiter_and_flux(oracle, shape):
    from openmhd_amd import api

    rng = np.random.default_rng(sum(shape))
    wk = np.asfortranarray(rng.standard_normal(shape))
    VL, VR = (np.asfortranarray(random_prim(rng, shape)) for _ in range(2))
    for d in dirs(shape):
        for t in range(5):
            out = [np.full(shape, v, order="F") for v in (7.0, -7.0, 7.0, -7.0)]
            api.limiter(wk, out[0], out[1], shape[0], shape[1], d, t, shape[2])
            oracle.limiter(wk, out[2], out[3], d, t)
            assert bits_equal(out[0], out[2]) and bits_equal(out[1], out[3])
        F1, F2 = np.full(shape + (9,), np.nan, order="F"), np.full(shape + (9,), np.nan, order="F")
        api.flux_solver(F1, VL, VR, 1.7, *shape[:2], d, 3, shape[2])
        oracle.flux_solver(F2, VL, VR, 1.7, d, 3)
        assert bits_equal(F1, F2)


@pytest.mark.parametrize("shape", [s for s in SHAPES if 2 not in s])
@pytest.mark.parametrize("bc", (0, 1))
def test_face_pairs(oracle, shape, bc):
    from openmhd_amd import api
    from openmhd_amd._lib import lib

    rng = np.random.default_rng(sum(shape) + bc)
    sg = rng.choice((-1.0, 1.0), (6, 9))
    A, L, R = (np.asfortranarray(rng.standard_normal(shape + (9,))) for _ in range(3))
    B, L2, R2 = A.copy(order="F"), L.copy(order="F"), R.copy(order="F")
    api._bc_u(A, *shape, [bc] * 6, sg)
    oracle.L.or_bc_u(ptr(B), *shape, (C.c_int * 6)(*[bc] * 6), ptr(sg))
    assert bits_equal(A, B)
    for d in dirs(shape):
        lo, hi = sg[2 * d - 2].copy(), sg[2 * d - 1].copy()
        assert lib.omhd_bc_face(ptr(L), ptr(R), *shape, d, bc, ptr(lo), ptr(hi)) == 0
        oracle.L.or_bc_face(ptr(L2), ptr(R2), *shape, d, bc, ptr(lo), ptr(hi))
        assert bits_equal(L, L2) and bits_equal(R, R2)


@pytest.mark.parametrize("shape", [(3, 3, 1), (261, 4, 1), (1031, 700, 1), (90, 80, 90)])
def test_set_dt(oracle, shape):
    from openmhd_amd import OMHDError, api

    rng = np.random.default_rng(shape[0])
    W = random_prim(rng, shape)
    fast = tuple(max(n - 2, 0) for n in shape)  # the last interior cell holds the maximum
    W[fast + (0,)] = 50.0
    U, V = np.asfortranarray(prim_to_cons(W)), farr(*shape, 4)
    oracle.u2v(U, V)
    nd = 2 if shape[2] == 1 else 3
    _, vm, dt = oracle.set_dt(U, V, 0.1, 0.4, nd)
    assert bits_equal(api.set_dt(U, V, 0.1, 0.4, *shape, nd), [vm, dt]) and vm > 50.0
    V[fast + (3,)] = np.nan  # the pressure: no speed of that cell is a number
    with pytest.raises(OMHDError):
        api.set_dt(U, V, 0.1, 0.4, *shape, nd)


def test_calls_from_many_threads(oracle):
    """u2v and set_dt share a bounded number of result slots: more threads than
    slots, each with its own arrays, some with a cell that u2v reports."""
    from concurrent.futures import ThreadPoolExecutor

    from openmhd_amd import OMHDError, api

    shape = (40, 30, 1)

    def one(t):
        rng = np.random.default_rng(t)
        W = random_prim(rng, shape)
        U, V, V2 = np.asfortranarray(prim_to_cons(W)), farr(*shape, 4), farr(*shape, 4)
        oracle.u2v(U, V2)
        want = oracle.set_dt(U, V2, 0.1, 0.4, 2)[1:]
        bad = U.copy(order="F")
        bad[t % 38 + 1, 3, 0, 3] = -5.0  # energy: a negative pressure
        for _ in range(4):
            api.u2v(U, V, *shape)
            assert bits_equal(V, V2) and bits_equal(api.set_dt(U, V, 0.1, 0.4, *shape), want)
            with pytest.raises(OMHDError) as e:
                api.u2v(bad, V, *shape)
            assert e.value.code == 1 and e.value.cell[0] == t % 38 + 2
        return True

    with ThreadPoolExecutor(80) as ex:
        assert all(ex.map(one, range(80)))


@pytest.mark.parametrize("shape", [(4, 4, 1), (131, 5, 1), (1031, 700, 1), (90, 80, 90), (4, 5, 6)])
def test_first_dt_of_a_solver(oracle, shape):
    """The CFL reduction after an upload (omhd_step.hip k_cfl: 64 cells of a row
    per wavefront, a bounded grid), its maximum in the last interior cell."""
    from openmhd_amd import Solver

    rng = np.random.default_rng(shape[1])
    W = random_prim(rng, shape)
    W[..., :3] *= 0.1
    W[..., 3] += 1.0
    W[..., 4] += 1.0
    W[tuple(max(n - 2, 0) for n in shape) + (1,)] = 9.0
    U, V = np.asfortranarray(prim_to_cons(W)), farr(*shape, 4)
    oracle.u2v(U, V)
    nd = 2 if shape[2] == 1 else 3
    _, vm, dt = oracle.set_dt(U, V, 0.1, 0.01, nd)
    nx, ny, nz = (n - 2 for n in shape)
    s = Solver(nx, ny, 0.1, nz=nz if nd == 3 else 0, cfl=0.01)
    s.upload(U if nd == 3 else np.asfortranarray(U[:, :, 0]))
    dts, chs = s.step(1, trace=True)
    s.close()
    assert vm > 9.0 and bits_equal([chs[0], dts[0]], [vm, dt])
