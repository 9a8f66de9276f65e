"""GPU: the kernels that steps of large grids take, one per sweep and the z sweep
fused with the update, where small grids take the merged form: the FP64 flux
where its shared reciprocals change path (the states of test_gpu_flux_range) in
every kernel shape, and levels of a hierarchy that are too large for the merged
form, whose fused kernel stores the z faces that the flux registers read."""
import numpy as np
import pytest

import binary_supernova_amd as bsn
from binary_supernova_amd import problems as P
from oracle import oracle as O
from test_gpu_flux_range import CASES, same, state as range_state

pytestmark = pytest.mark.gpu

D = (0.1, 0.07, 0.13)


@pytest.mark.parametrize("kind,g", CASES)
@pytest.mark.parametrize("shape", [(70, 9, 7), (7, 12, 70)])
def test_fp64_flux_range_in_every_kernel_shape(kind, g, shape):
    U = range_state(kind, shape, g)
    want = U.copy()
    O.euler3d_step(want, *D, 1e-3, g, "outflow")
    forms = [(0, 7, 7, u, False) for u in range(12)]
    forms += [(x, 7, 7, 11, False) for x in range(6)]
    forms += [(0, y, y, 11, inplace) for y in range(8) for inplace in (False, True)]
    for form in forms:
        print(f"flux range {kind} gamma {g} {shape} {form}", flush=True)
        sx, sy, sz, su, inplace = form
        grid = bsn.Grid(*shape).set_state(U)
        grid.set_params(*D, g, "outflow", 0.0, 0.0)
        b = bsn.Batch([grid])
        b.set_shapes(sx, sy, sz)
        b.set_update_shape(su)
        b.set_mode(inplace)
        b.step([1e-3])
        same(grid.get_state(), want)


BOX = (18, 49, 17, 47, 16, 48)
DIMS = [(66, 60, 62), (64, 62, 66), (60, 66, 64)]
BOX2 = (17, 46, 15, 47, 18, 49)


def level_state(n, seed):
    rng = np.random.default_rng(seed)
    U = P.empty_state(*n)
    s = U.shape[:-1]
    rho, p = rng.uniform(0.5, 2.0, s), rng.uniform(0.5, 2.0, s)
    v = rng.normal(0.0, 0.3, s + (3,))
    U[..., 0], U[..., 1:4] = rho, rho[..., None] * v
    U[..., 4] = p / 0.4 + 0.5 * rho * (v * v).sum(-1)
    return U


@pytest.mark.parametrize("prec", ["fp64", "split"])
@pytest.mark.parametrize("levels", [2, 3])
def test_large_levels_fused(levels, prec):
    print(f"large levels {levels} {prec}", flush=True)
    dims, boxes = DIMS[:levels], [BOX, BOX2][:levels - 1]
    ds = [(0.1 / 2 ** l,) * 3 for l in range(levels)]
    Us = [level_state(n, 20 + l) for l, n in enumerate(dims)]
    phis = None
    if levels == 2:
        phis = [0.05 * np.random.default_rng(l).normal(size=n[::-1]) for l, n in enumerate(dims)]
    out = []
    for inplace in (False, True):
        H = bsn.FMRHierarchy(dims, ds, boxes, [2] * len(boxes), 1.4, "outflow", 1e-3, 1e-3, precision=prec)
        H.set_mode(inplace)
        for lev, U in zip(H.levels, Us):
            lev.set_state(U)
            # no merged form for a grid of this size
            assert bsn.Batch([lev]).get_shapes() == [0, 7, 7, 11]
        if phis:
            H.set_phis(phis)
        H.step(1e-3)
        out.append([lev.get_state() for lev in H.levels])
    for a, b in zip(*out):
        np.testing.assert_array_equal(a, b)
    if prec == "fp64":
        O.fmr_multilevel_step(Us, ds, boxes, [2] * len(boxes), 1.4, 1e-3, "outflow", 1e-3, 1e-3,
                              phis=phis)
        for a, U in zip(out[0], Us):
            np.testing.assert_array_equal(a, U)
