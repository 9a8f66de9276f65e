"""GPU parity of cfl_dt_3d on both sides of the number of tiles up to which small
grids take one cell per thread, with the fastest cell in the last tile."""
import numpy as np
import pytest

import binary_supernova_amd as bsn
from binary_supernova_amd import problems as P
from oracle import oracle as O

pytestmark = pytest.mark.gpu


# 600 and 615 tiles, a wide grid of 600, and 2310 of a narrow one
@pytest.mark.parametrize("shape", [(17, 60, 40), (17, 60, 41), (65, 40, 30), (17, 130, 70)])
@pytest.mark.parametrize("prec", ["fp64", "split"])
def test_cfl_dt_bitwise(shape, prec):
    print(f"cfl tiles {shape} {prec}", flush=True)
    rng = np.random.default_rng(sum(shape))
    U = P.empty_state(*shape)
    s = U.shape[:-1]
    U[..., 0], U[..., 4] = rng.uniform(0.5, 2.0, s), rng.uniform(3.0, 4.0, s)
    U[..., 1:4] = rng.normal(0.0, 0.3, s + (3,))
    U[-4, -4, -4, 1:4] = 2.0, -1.5, 1.0
    d = (0.1, 0.07, 0.13)
    g = bsn.Grid(*shape, prec).set_state(U)
    assert bsn.cfl_dt_3d(g, *shape, *d, 1.4, 0.3) == O.cfl_dt_3d(U, *d, 1.4, 0.3)
