"""The step of small grids (three sweeps in one launch, then the update) against
the oracle and against the separate kernels: the smallest extents, both sides
of the size up to which it is taken, batches, sources and a potential."""
import numpy as np
import pytest

import binary_supernova_amd as bsn
from binary_supernova_amd import problems as P
from oracle import oracle as O

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 1), (3, 5, 4), (65, 3, 3), (3, 3, 65), (16, 17, 15), (56, 56, 56), (60, 58, 59), (64, 64, 64)]


def state(shape, seed):
    rng = np.random.default_rng(seed)
    U = P.empty_state(*shape)
    s = U.shape[:-1]
    rho, p = rng.uniform(0.2, 2.0, s), rng.uniform(0.1, 2.0, s)
    v = rng.normal(0.0, 1.0, s + (3,))
    U[..., 0], U[..., 1:4] = rho, rho[..., None] * v
    U[..., 4] = p / 0.4 + 0.5 * rho * (v * v).sum(-1)
    return U


@pytest.mark.parametrize("shape", SHAPES[:5])
def test_small_step_bitwise(shape):
    print(f"small {shape}", flush=True)
    U, d = state(shape, sum(shape)), (0.1, 0.07, 0.13)
    Uo = U.copy()
    dt = O.cfl_dt_3d(U, *d, 1.4, 0.3)
    assert bsn.cfl_dt_3d(U, *shape, *d, 1.4, 0.3) == dt
    O.euler3d_step(Uo, *d, dt, 1.4, "outflow", 1e-3, 1e-3)
    bsn.euler3d_step_(U, *shape, *d, dt, 1.4, bc="outflow", rho_floor=1e-3, P_floor=1e-3)
    np.testing.assert_array_equal(U, Uo)


@pytest.mark.parametrize("prec", ["split", "fp64"])
@pytest.mark.parametrize("shapes", [[s] for s in SHAPES] + [SHAPES[:5]], ids=str)
def test_small_run_agrees_with_separate_kernels(shapes, prec):
    print(f"small run {shapes} {prec}", flush=True)
    out = []
    for separate in (False, True):
        grids = [bsn.Grid(*s, prec).set_state(state(s, k)) for k, s in enumerate(shapes)]
        for g, s in zip(grids, shapes):
            g.set_params(0.1, 0.07, 0.13, 1.4, "outflow", 1e-3, 1e-3)
            g.set_phi(0.05 * np.random.default_rng(3).normal(size=s[::-1]))
        bh = bsn.BlackHole(pos=[0.1, 0.2, 0.1], vel=[0.0, 0.0, 0.0], mass=0.1, eps=0.1, c_code=1e3, r_floor=0.2)
        bsn.set_point_masses(grids[0], [bh], 0.0, 0.0, 0.0)
        b = bsn.Batch(grids)
        if separate:
            b.set_shapes(0, 7, 7)
        b.run(0.3, 3, graph=True)
        out.append([g.get_state() for g in grids] + [np.array(b.times())])
    for a, c in zip(*out):
        np.testing.assert_array_equal(a, c)
