"""Face states that are not between their cells: MC and Koren slopes may take a
cell's whole difference to its neighbour, and w0 - (w0 - wm) is zero where wm
is below half an ulp of w0.  The oracle's flux of a face of zero density is NaN
(its fast speed is infinite), and the step has to stop on it, not go on with a
finite flux of the other side's."""
import numpy as np
import pytest

from omhd_testlib import farr, make_problem, prim_to_cons

pytestmark = pytest.mark.gpu

LOW = 2.0 ** -60  # below half an ulp of the 1 beside it


def contrast(nd, axis, flip):
    """rho 10, 10, .., 1, LOW, 1, 1 along `axis`, every cell in the range of the
    shared reciprocals: the face between the 1 and the LOW has a density of zero
    on the side of the 1, while the gas of the LOW runs towards it."""
    n = [24, 10, 10][:nd]
    n[0], n[axis] = n[axis], n[0]
    W = np.zeros([e + 2 for e in n] + [9])
    line = np.full(26, 10.0)
    line[12:] = 1.0
    line[13] = LOW
    speed = np.full(26, -0.3)
    speed[13] = -0.5 / np.sqrt(LOW)
    if flip:
        line, speed = line[::-1], -speed[::-1]
    shape = [1] * nd
    shape[axis] = 26
    W[..., 4] = line.reshape(shape)
    W[..., axis] = speed.reshape(shape)
    W[..., 3] = 1.0
    W[..., 5 + axis], W[..., 5 + (axis + 1) % 3] = 0.1, 0.05
    return n, np.asfortranarray(prim_to_cons(W))


@pytest.mark.parametrize("lm", (2, 4))
@pytest.mark.parametrize("flip", (False, True))
@pytest.mark.parametrize("nd,axis", [(2, 0), (2, 1), (3, 0), (3, 1), (3, 2)])
def test_zero_face_density_stops_the_step(oracle, nd, axis, flip, lm):
    from openmhd_amd import OMHDError, Solver

    n, U = contrast(nd, axis, flip)
    kw = dict(cfl=1e-3, lm_type=lm, time_type=0)
    p = make_problem(*U.shape[:-1], dx=1e6, **kw)
    oracle.bc_u(U, p)
    s = Solver(n[0], n[1], 1e6, nz=n[2] if nd == 3 else 0, bc=("periodic",) * nd, **kw)
    s.upload(U)
    O = U.copy(order="F")
    oracle.run(p, O, 1)
    assert np.isnan(O).any()  # the oracle's u2v does not stop on a NaN
    with pytest.raises(OMHDError) as e:
        s.step(1)
    s.close()
    assert e.value.code == 1 and e.value.steps_done == 0
