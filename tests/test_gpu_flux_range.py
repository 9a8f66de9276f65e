"""GPU parity of the FP64 flux where its shared reciprocals change path: face
momenta from denormal to ordinary (full divisions below 2^-900), zero and tiny
pressures, densities and momenta past the 2^96 and 2^180 bounds, infinities and
NaN, and gamma next to 1 and very large.  Bit for bit against the CPU oracle,
signs of zero included, through the sweeps (euler3d_rhs_) and the fused step."""
import numpy as np
import pytest

import binary_supernova_amd as bsn
from binary_supernova_amd import problems as P
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def state(kind, shape, g):
    nx, ny, nz = shape
    rng = np.random.default_rng(sum(map(ord, kind)) + nx)
    U = P.empty_state(nx, ny, nz)
    s = U.shape[:-1]
    rho = rng.uniform(0.5, 2.0, s)
    m = rng.normal(0.0, 1.0, s + (3,))
    p = rng.uniform(0.1, 2.0, s)
    some = rng.random(s) < 0.15
    if kind == "tiny_momenta":
        # all magnitudes down to the smallest denormal, zeros of both signs
        m = np.ldexp(m, rng.integers(-1080, -150, s + (3,)))
        m[rng.random(m.shape) < 0.1] = -0.0
        m[:, : ny // 2][some[:, : ny // 2]] = 1.0
    elif kind == "cold":
        # zero and tiny pressures beside momenta of every size
        m = np.ldexp(m, rng.integers(-500, 0, s + (3,)))
        p = np.where(some, np.ldexp(p, rng.integers(-900, -500, s)), p)
        p[:, :, : nx // 2] = 0.0
    elif kind == "large":
        m = np.where(some[..., None], np.ldexp(m, rng.integers(150, 500, s + (3,))), m)
        rho = np.where(rng.random(s) < 0.05, np.ldexp(rho, rng.integers(90, 400, s)), rho)
    elif kind == "not_finite":
        v = np.array([np.inf, -np.inf, np.nan])
        m[some, 1] = v[rng.integers(0, 3, int(some.sum()))]
        rho[rng.random(s) < 0.01] = np.nan
    with np.errstate(all="ignore"):
        ke = 0.5 * (m * m).sum(-1) / rho
        U[..., 0], U[..., 1:4], U[..., 4] = rho, m, p / (g - 1) + ke
    return U


CASES = [("tiny_momenta", 1.4), ("cold", 5 / 3), ("large", 1.4), ("not_finite", 1.4),
         ("ordinary", 1 + 2.0 ** -41), ("ordinary", 2.0 ** 41)]


def same(a, b):
    np.testing.assert_array_equal(a, b)
    ok = ~np.isnan(b)
    np.testing.assert_array_equal(np.signbit(a[ok]), np.signbit(b[ok]))


@pytest.mark.parametrize("kind,g", CASES)
@pytest.mark.parametrize("shape", [(70, 9, 7), (7, 12, 70)])
def test_fp64_flux_range_bitwise(kind, g, shape):
    print(f"flux range {kind} gamma {g} {shape}", flush=True)
    nx, ny, nz = shape
    U = state(kind, shape, g)
    d = (0.1, 0.07, 0.13)
    Ug, Us, Uo = U.copy(), U.copy(), U.copy()
    dU, Fx, Fy, Fz = O.euler3d_rhs(U, *d, g, "outflow", 0.0, 0.0)
    sx, sy, sz = bsn.flux_shapes(nx, ny, nz)
    gd, gx, gy, gz = np.empty(U.shape), np.empty(sx), np.empty(sy), np.empty(sz)
    bsn.euler3d_rhs_(gd, gx, gy, gz, Ug, nx, ny, nz, *d, g, bc="outflow")
    for a, b in ((gx, Fx), (gy, Fy), (gz, Fz)):
        same(a, b)
    np.testing.assert_array_equal(gd, dU)
    O.euler3d_step(Uo, *d, 1e-3, g, "outflow")
    bsn.euler3d_step_(Us, nx, ny, nz, *d, 1e-3, g, bc="outflow")
    np.testing.assert_array_equal(Us, Uo)
