"""GPU parity of the flat tiles (rows that leave lanes of a 64 x 4 tile idle run as
consecutive columns, or x interfaces, wrapping from row to row): the smallest x
and y extents they take, rows of just over and far over 64, waves that wrap
into the next plane, lists that end inside a tile."""
import numpy as np
import pytest

import binary_supernova_amd as bsn
from binary_supernova_amd import problems as P
from oracle import oracle as O

pytestmark = pytest.mark.gpu

SHAPES = [(8, 8, 8), (9, 8, 5), (7, 9, 8), (31, 8, 7), (65, 8, 3), (100, 11, 3), (200, 9, 3), (48, 13, 12)]


def state(shape, seed):
    nx, ny, nz = shape
    rng = np.random.default_rng(seed)
    U = P.empty_state(nx, ny, nz)
    s = U.shape[:-1]
    rho, p = rng.uniform(0.2, 2.0, s), rng.uniform(0.1, 2.0, s)
    v = rng.normal(0.0, 1.0, s + (3,))
    U[..., 0], U[..., 1:4] = rho, rho[..., None] * v
    U[..., 4] = p / 0.4 + 0.5 * rho * (v * v).sum(-1)
    return U


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("bc", ["outflow", "periodic"])
def test_flat_tiles_bitwise(shape, bc):
    print(f"flat tiles {shape} {bc}", flush=True)
    nx, ny, nz = shape
    U, d = state(shape, sum(shape)), (0.1, 0.07, 0.13)
    Ug, Us, Uo = U.copy(), U.copy(), U.copy()
    dU, Fx, Fy, Fz = O.euler3d_rhs(U, *d, 1.4, bc, 1e-3, 1e-3)
    outs = [np.empty(U.shape)] + [np.empty(s) for s in bsn.flux_shapes(nx, ny, nz)]
    bsn.euler3d_rhs_(*outs, Ug, nx, ny, nz, *d, 1.4, bc=bc, rho_floor=1e-3, P_floor=1e-3)
    for a, b in zip(outs, (dU, Fx, Fy, Fz)):
        np.testing.assert_array_equal(a, b)
    O.euler3d_step(Uo, *d, 1e-3, 1.4, bc, 1e-3, 1e-3)
    bsn.euler3d_step_(Us, nx, ny, nz, *d, 1e-3, 1.4, bc=bc, rho_floor=1e-3, P_floor=1e-3)
    np.testing.assert_array_equal(Us, Uo)


@pytest.mark.parametrize("prec", ["split", "fp64"])
def test_mixed_batch_agrees_with_blocked_tiles(prec):
    # flat and 64 x 4 grids in one list against the 32 x 8 x tiles, the tiled y
    # sweep and the in-place update, none of which has flat tiles
    print(f"mixed batch {prec}", flush=True)
    shapes = SHAPES + [(64, 8, 8), (128, 9, 4)]
    out = []
    for blocked in (False, True):
        grids = [bsn.Grid(*s, prec).set_state(state(s, k)) for k, s in enumerate(shapes)]
        for g in grids:
            g.set_params(0.1, 0.07, 0.13, 1.4, "outflow", 1e-3, 1e-3)
        b = bsn.Batch(grids)
        if blocked:
            b.set_shapes(1, 0, 0)
            b.set_mode(True)
        else:
            b.set_shapes(0, 7, 7)
        for _ in range(2):
            b.step([1e-3] * len(grids))
        out.append([g.get_state() for g in grids])
    for a, c in zip(*out):
        np.testing.assert_array_equal(a, c)
