"""The adjoint kernels where their paths part: extents down to two cells
(periodic neighbours wrap onto the same cell, every cell of a walled axis is at
a wall), rows that share wavefronts, and a state whose faces take every HLLD
branch.  Against the CPU build of the same reverse forms, with the bounds of the
larger cases."""
import numpy as np
import pytest

import test_gpu_adjoint3d as base
from omhd_testlib import prim_to_cons
from test_gpu_adjoint3d import ac  # noqa: F401

pytestmark = pytest.mark.gpu
P, W = "periodic", "wall"


@pytest.mark.parametrize("nx,ny,nz,bc,lm,res", [
    (2, 3, 2, (P, P, P), 2, 1), (3, 2, 5, (W, P, W), 1, 1), (5, 4, 3, (P, W, P), 4, 1), (2, 2, 0, (P, P, P), 3, 0),
    (67, 5, 4, (P, P, P), 3, 1), (130, 3, 0, (P, W, P), 4, 0)])
def test_small_extents(ac, oracle, nx, ny, nz, bc, lm, res):  # noqa: F811
    base.test_adjoint_matches_cpu_reverse(ac, oracle, nx, ny, nz, bc, lm, 0, res, 2, 1, None)


def blocks(rng, ix, jx, kx=1):
    """Constant blocks of 4 cells a side under small noise: calm and supersonic
    flow either way, strong and vanishing fields."""
    def spread(choices):
        c = rng.choice(choices, [(n + 3) // 4 for n in (ix, jx, kx)])
        for a, n in enumerate((ix, jx, kx)):
            c = np.take(np.repeat(c, 4, axis=a), range(n), axis=a)
        return c

    V = 1e-3 * rng.standard_normal((ix, jx, kx, 9))
    for m in range(3):
        V[..., m] += spread([0.0, 0.1, 2.5, -2.5])
        V[..., 5 + m] += spread([0.0, 0.0, 0.6, -1.0])
    V[..., 3] += spread([0.3, 1.0, 2.0])
    V[..., 4] += spread([1.0, 2.0])
    U = prim_to_cons(V)
    return np.asfortranarray(U if kx > 1 else U[:, :, 0])


@pytest.mark.parametrize("nx,ny,nz", [(90, 71, 0), (36, 25, 22)])
@pytest.mark.parametrize("lm", (1, 2))
def test_every_branch(ac, oracle, monkeypatch, nx, ny, nz, lm):  # noqa: F811
    monkeypatch.setattr(base, "smooth_state", blocks)
    base.test_adjoint_matches_cpu_reverse(ac, oracle, nx, ny, nz, (P, W, P), lm, 0, 0, 1, 1, None)
