"""GPU parity of the FMR transfers at every refinement ratio, on boxes of odd
and of smallest size and off the parent's centre: the prolongation takes fine
cells in groups that share a coarse centre, cut by the box and the slabs."""
import numpy as np
import pytest

import binary_supernova_amd as bsn
from binary_supernova_amd import problems as P
from oracle import oracle as O

pytestmark = pytest.mark.gpu

BOXES = [(5, 7, 4, 8, 5, 6), (6, 6, 4, 9, 5, 9)]


def state(n, seed):
    rng = np.random.default_rng(seed)
    U = P.empty_state(*n)
    s = U.shape[:-1]
    rho, p = rng.uniform(0.5, 2.0, s), rng.uniform(0.5, 2.0, s)
    v = rng.normal(0.0, 0.3, s + (3,))
    U[..., 0], U[..., 1:4] = rho, rho[..., None] * v
    U[..., 4] = p / 0.4 + 0.5 * rho * (v * v).sum(-1)
    return U


@pytest.mark.parametrize("box", BOXES)
@pytest.mark.parametrize("ratio", [1, 2, 3, 4])
def test_transfers_bitwise(ratio, box):
    print(f"fmr transfers r={ratio} {box}", flush=True)
    n, d = (11, 12, 13), 0.1
    nf = tuple((box[2 * a + 1] - box[2 * a] + 1) * ratio for a in range(3))
    Uc, Uf = state(n, ratio), state(nf, 10 + ratio)
    O.fill_ghost(Uc, "outflow")
    H = bsn.FMRHierarchy([n, nf], [(d,) * 3, (d / ratio,) * 3], [box], [ratio], 1.4, "outflow", 1e-3, 1e-3)
    H.levels[0].set_state(Uc)
    want = Uf.copy()
    O.prolong_all(want, Uc, box, ratio)
    H.prolong_all(1)
    np.testing.assert_array_equal(H.levels[1].get_state(), want)
    H.levels[1].set_state(Uf)
    O.prolong_fine_ghosts(Uf, Uc, box, ratio)
    H.prolong_fine_ghosts(1)
    np.testing.assert_array_equal(H.levels[1].get_state(), Uf)
    for _ in range(2):
        O.fmr_multilevel_step([Uc, Uf], [(d,) * 3, (d / ratio,) * 3], [box], [ratio], 1.4, 2e-3, "outflow",
                              1e-3, 1e-3)
        H.step(2e-3)
    for lev, U in zip(H.levels, (Uc, Uf)):
        np.testing.assert_array_equal(lev.get_state(), U)
