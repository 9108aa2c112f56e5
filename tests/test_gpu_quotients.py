"""The shared-reciprocal quotients and short roots of u2v, HLLD and set_dt
(csrc/omhd_device.h) at the edges of the range they are used in: each kernel
takes `/` and sqrt for a wavefront with an operand outside it, and the results
are the oracle's bit for bit either way (NaN: NaN in the same places)."""
import numpy as np
import pytest

from omhd_testlib import farr, make_problem, smooth_state

pytestmark = pytest.mark.gpu

# factors on (rho, p, v, B): ordinary, out of the moderate range either way,
# tiny and denormal velocities and fields, a flow that swamps the fast speed
SCALES = [(1, 1, 1, 1), (2.0 ** -101, 2.0 ** -101, 1, 2.0 ** -60), (2.0 ** 101, 2.0 ** 101, 1, 2.0 ** 49),
          (1e-200, 1e-200, 1, 1e-110), (1, 1, 1e-300, 1), (1, 1, 1, 1e-300), (1, 1, 1e-310, 1e-310), (1, 1, 0, 0),
          (1, 1, -0.0, 1), (1, 1, 1e18, 1), (1e-120, 1, 1, 1)]


def same(a, b):
    a, b = np.asarray(a), np.asarray(b)
    nan = np.isnan(a) & np.isnan(b)
    return np.array_equal(np.where(nan, 0.0, a).view(np.int64), np.where(nan, 0.0, b).view(np.int64))


def states(seed, shape, scales):
    rng = np.random.default_rng(seed)
    ro, p = rng.uniform(0.2, 2.0, shape), rng.uniform(0.2, 2.0, shape)
    v, B, ps = (rng.standard_normal((3,) + shape) for _ in range(3))
    k = rng.integers(0, len(scales), shape)
    s = np.moveaxis(np.array(scales, dtype=np.float64)[k], -1, 0)
    W = farr(*shape, 9)
    for m in range(3):
        W[..., m] = v[m] * s[2]
        W[..., 5 + m] = B[m] * s[3]
    W[..., 3], W[..., 4], W[..., 8] = p * s[1], ro * s[0], ps[0]
    return W


@pytest.mark.parametrize("scales", [SCALES] + [[s] for s in SCALES], ids=["mixed"] + [str(i) for i in range(len(SCALES))])
@pytest.mark.parametrize("dir", (1, 2))
def test_flux(oracle, scales, dir):
    from openmhd_amd import api

    shape = (131, 7)
    VL, VR = states(1, shape, scales), states(2, shape, scales)
    VR[::3] = VL[::3]  # no jump
    VL[1, :, 3], VL[1, :, 5:8] = 0.6, 0.0  # gamma p = Bn^2 = B^2: a zero root
    VL[1, :, 4 + dir] = 1.0
    F1, F2 = farr(*shape, 9), farr(*shape, 9)
    with np.errstate(all="ignore"):
        oracle.flux_solver(F2, VL, VR, 1.3, dir, 3)
    api.flux_solver(F1, VL, VR, 1.3, *shape, dir, 3)
    assert same(F1, F2)


@pytest.mark.parametrize("scales", [SCALES] + [[s] for s in SCALES], ids=["mixed"] + [str(i) for i in range(len(SCALES))])
def test_u2v_and_set_dt(oracle, scales):
    from openmhd_amd import OMHDError, api

    shape = (131, 7)
    W = states(3, shape, scales)
    U = farr(*shape, 9)
    with np.errstate(all="ignore"):
        U[:] = W
        for m in range(3):
            U[..., m] = W[..., 4] * W[..., m]
        U[..., 3] = W[..., 3] / (2.0 / 3.0) + 0.5 * (W[..., 4] * (W[..., :3] ** 2).sum(-1) + (W[..., 5:8] ** 2).sum(-1))
    V1, V2 = farr(*shape, 4), farr(*shape, 4)
    oracle.u2v(U, V2)
    try:
        api.u2v(U, V1, *shape)
    except OMHDError as e:  # a pressure lost to rounding in the energy
        assert e.code in (1, 2) and (V2[..., 3].min() <= 0 or U[..., 4].min() <= 0)
    assert same(V1, V2)


@pytest.mark.parametrize("nx,ny", [(2, 2), (60, 9), (61, 29), (122, 57)])
@pytest.mark.parametrize("lm,tt", [(1, 0), (2, 1), (4, 0)])
def test_step_with_vanishing_fields(oracle, nx, ny, lm, tt):
    """A smooth flow whose third components are zero but for a spot of 1e-306
    that spreads and decays through the denormals, between walls."""
    from openmhd_amd import Solver

    rng = np.random.default_rng(nx)
    U = np.asfortranarray(smooth_state(rng, nx + 2, ny + 2))
    if U.ndim == 4:
        U = np.asfortranarray(U[:, :, 0])
    U[..., 2] = U[..., 7] = 0.0
    U[1 + nx // 2, 1 + ny // 2, 2] = 3e-306
    U[1 + nx // 2, 1 + ny // 2, 7] = -2e-306
    p = make_problem(nx + 2, ny + 2, dx=0.1, cfl=0.4, lm_type=lm, time_type=tt, bc=("periodic", "wall", "periodic"))
    oracle.bc_u(U, p)
    s = Solver(nx, ny, 0.1, cfl=0.4, lm_type=lm, time_type=tt, bc=("periodic", "wall"))
    s.upload(U)
    s.step(12)
    G = s.download()
    s.close()
    O = U.copy(order="F")
    assert oracle.run(p, O, 12)[0] == 0
    assert same(G, O)


@pytest.mark.parametrize("dir", (1, 2))
def test_flux_of_infinite_states(oracle, dir):
    """Infinite velocities and pressures: where an infinite fast speed takes the
    fan's edge to NaN, so is the flux."""
    from openmhd_amd import api

    cases = [(v, p, w, q) for v in (1.0, np.inf, -np.inf) for p in (1.0, np.inf) for w in (1.0, np.inf, -np.inf)
             for q in (1.0, np.inf)]
    shape = (len(cases) + 2, 5) if dir == 1 else (5, len(cases) + 2)
    VL, VR = states(4, shape, SCALES[:1]), states(5, shape, SCALES[:1])
    for i, (v, p, w, q) in enumerate(cases):
        at = (i + 1, slice(None)) if dir == 1 else (slice(None), i + 1)
        VL[at + (dir - 1,)], VL[at + (3,)] = v, p
        VR[at + (dir - 1,)], VR[at + (3,)] = w, q
    F1, F2 = farr(*shape, 9), farr(*shape, 9)
    with np.errstate(all="ignore"):
        oracle.flux_solver(F2, VL, VR, 1.3, dir, 3)
    api.flux_solver(F1, VL, VR, 1.3, *shape, dir, 3)
    assert same(F1, F2)


def conserved(W):
    U = W.copy(order="F")
    with np.errstate(all="ignore"):
        for m in range(3):
            U[..., m] = W[..., 4] * W[..., m]
        U[..., 3] = W[..., 3] / (2.0 / 3.0) + 0.5 * (W[..., 4] * (W[..., :3] ** 2).sum(-1) + (W[..., 5:8] ** 2).sum(-1))
    return U


@pytest.mark.parametrize("scales", [SCALES] + [[s] for s in SCALES], ids=["mixed"] + [str(i) for i in range(len(SCALES))])
def test_u2v_reports_every_bad_state(oracle, scales):
    """u2v raises exactly where the oracle's does, with its code and cell."""
    from openmhd_amd import OMHDError, api

    shape = (131, 7)
    U = conserved(states(3, shape, scales))
    V1, V2 = farr(*shape, 4), farr(*shape, 4)
    rc, bad = oracle.u2v(U, V2)
    code, cell = 0, None
    try:
        api.u2v(U, V1, *shape)
    except OMHDError as e:
        code, cell = e.code, e.cell[:2]
    assert code == rc and same(V1, V2)
    assert rc == 0 or cell == (bad % shape[0] + 1, bad // shape[0] + 1)


# states whose energy holds their pressure and whose jumps a step keeps positive
MIXED, ALONE = [(0, 1, 4, 5, 6, 7, 8), (0, 2, 4, 5, 6, 7, 8)], (0, 1, 2, 3, 4, 5, 6, 7, 8, 10)


@pytest.mark.parametrize("nz", (0, 5))
@pytest.mark.parametrize("which", MIXED + [(i,) for i in ALONE],
                         ids=["mixed low", "mixed high"] + [str(i) for i in ALONE])
def test_speeds_of_a_run(oracle, which, nz):
    """The CFL speed after an upload and after a step (first-order faces and a
    tiny step, so that the states stay what they are): dt and ch of the first
    two steps."""
    from openmhd_amd import Solver

    shape = (133, 9) + ((nz + 2,) if nz else ())
    scales = [SCALES[i] for i in which]
    W = states(6, shape, scales)
    W[..., 8] = 0.0
    ro, p = scales[0][:2]
    b = 32 * 2.0 ** round(0.5 * np.log2(p))
    W[5, 5] = 0.0  # gamma p = Bx^2 = B^2 in one column, the fastest: a zero inner root
    W[5, 5, ..., 3], W[5, 5, ..., 4], W[5, 5, ..., 5] = 0.6 * b * b, ro, b
    U = conserved(W)
    V = farr(*shape, 4)
    assert oracle.u2v(U, V)[0] == 0 and np.all(5 / 3 * V[5, 5, ..., 3] == b * b)
    kw = dict(cfl=1e-9 if len(which) == 1 else 1e-40, lm_type=0, time_type=1)
    dx = 4e-7 / kw["cfl"] * oracle.set_dt(U, V, 1.0, 1.0, ndim=3 if nz else 2)[1]
    p = make_problem(*shape, dx=dx, **kw)
    oracle.bc_u(U, p)
    rc, dts, chs = oracle.run(p, U.copy(order="F"), 2)
    assert rc == 0 and np.isfinite(chs).all()
    s = Solver(shape[0] - 2, shape[1] - 2, dx, nz=nz, bc=("periodic",) * (3 if nz else 2), **kw)
    s.upload(U)
    got = s.step(2, trace=True)
    s.close()
    assert same(got[0], dts) and same(got[1], chs)
