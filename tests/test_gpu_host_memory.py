"""GPU: calls on host arrays, page-locked ones, which the library copies directly,
and ordinary ones of sizes around which its copies change: what a call was given
has been read, and what it returns has arrived, when it returns.  The oracle
sees the values each call was given."""
import ctypes as C

import numpy as np
import pytest

import binary_supernova_amd as bsn
from binary_supernova_amd import problems as P
from binary_supernova_amd._lib import BSN_HOST, call
from oracle import oracle as O

pytestmark = pytest.mark.gpu

D = (0.1, 0.07, 0.13)


def hip():
    # the HIP runtime libbsn_hip.so itself links
    bsn.load()
    L = C.CDLL("/opt/rocm/lib/libamdhip64.so")
    L.hipHostMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t, C.c_uint]
    L.hipHostFree.argtypes = [C.c_void_p]
    return L


@pytest.fixture
def pinned():
    """pinned(shape): a float64 array in page-locked memory."""
    L, held = hip(), []

    def make(shape):
        p = C.c_void_p()
        assert L.hipHostMalloc(C.byref(p), 8 * int(np.prod(shape)), 0) == 0
        held.append(p)
        return np.ctypeslib.as_array(C.cast(p, C.POINTER(C.c_double)), shape=tuple(shape))
    yield make
    for p in held:
        assert L.hipHostFree(p) == 0


def state(shape, seed):
    rng = np.random.default_rng(seed)
    U = P.empty_state(*shape)
    s = U.shape[:-1]
    rho, p = rng.uniform(0.5, 2.0, s), rng.uniform(0.5, 2.0, s)
    v = rng.normal(0.0, 0.3, s + (3,))
    U[..., 0], U[..., 1:4] = rho, rho[..., None] * v
    U[..., 4] = p / 0.4 + 0.5 * rho * (v * v).sum(-1)
    return U


def sg_force(g, dU):
    call("bsn_apply_sg_force", g.handle, C.c_void_p(dU.ctypes.data), BSN_HOST, *D)


# a potential of 480 bytes, and one of 9.4 MB
SHAPES = [(3, 5, 4), (128, 96, 96)]


@pytest.mark.parametrize("shape", SHAPES)
def test_phi_from_a_refilled_pinned_array(pinned, shape):
    print(f"pinned phi {shape}", flush=True)
    nx, ny, nz = shape
    phis = [0.1 * np.random.default_rng(k).normal(size=(nz, ny, nx)) for k in range(2)]
    buf = pinned((nz, ny, nx))
    U = state(shape, 1)
    grids = [bsn.Grid(*shape).set_state(U) for _ in phis]
    for g, phi in zip(grids, phis):
        buf[...] = phi
        g.set_phi(buf)
        buf[...] = 7.0
    for g, phi in zip(grids, phis):
        dU, want = np.zeros(U.shape), np.zeros(U.shape)
        sg_force(g, dU)
        O.apply_sg_force(want, U, phi, *D)
        np.testing.assert_array_equal(dU, want)


@pytest.mark.parametrize("shape", SHAPES)
def test_states_through_pinned_arrays(pinned, shape):
    # up, one step, down; then dU up and down in place
    print(f"pinned state {shape}", flush=True)
    nx, ny, nz = shape
    U = state(shape, 2)
    buf, out = pinned(U.shape), pinned(U.shape)
    buf[...] = U
    g = bsn.Grid(*shape).set_state(buf)
    buf[...] = 7.0
    dt = bsn.cfl_dt_3d(g, *shape, *D, 1.4, 0.3)
    bsn.euler3d_step_(g, *shape, *D, dt, 1.4, bc="outflow")
    g.get_state(out)
    assert dt == O.cfl_dt_3d(U, *D, 1.4, 0.3)
    O.euler3d_step(U, *D, dt, 1.4, "outflow")
    np.testing.assert_array_equal(out, U)
    phi = 0.1 * np.random.default_rng(3).normal(size=(nz, ny, nx))
    g.set_phi(phi)
    dU, want = pinned(U.shape), np.zeros(U.shape)
    dU[...] = 0.0
    sg_force(g, dU)
    O.apply_sg_force(want, U, phi, *D)
    np.testing.assert_array_equal(dU, want)


# bytes of a state around 16 kB (a small slot without an event), 1 MB (one part
# or several) and 8 MB (parts of 1 or 2 MB)
@pytest.mark.parametrize("nx", [1, 2, 3, 528, 529, 4273, 4274])
def test_states_of_every_transfer_size(nx):
    print(f"state transfers {nx}", flush=True)
    U = np.random.default_rng(nx).normal(size=(7, 7, nx + 6, 5))
    g = bsn.Grid(nx, 1, 1)
    for k in range(3):
        g.set_state(U + k)
        np.testing.assert_array_equal(g.get_state(), U + k)


# up to 3 MB posted through slots, more of them than there are, or straight
@pytest.mark.parametrize("nz", [96, 97])
def test_phis_posted_one_after_the_other(nz):
    print(f"posted phis {nz}", flush=True)
    shape = (64, 64, nz)
    U = state(shape, 5)
    grids = [bsn.Grid(*shape).set_state(U) for _ in range(3)]
    phi = np.empty(shape[::-1])
    for k, g in enumerate(grids):
        phi[...] = 0.1 * np.random.default_rng(k).normal(size=phi.shape)
        g.set_phi(phi)
        phi[...] = 7.0
    for k, g in enumerate(grids):
        dU, want = np.zeros(U.shape), np.zeros(U.shape)
        sg_force(g, dU)
        O.apply_sg_force(want, U, 0.1 * np.random.default_rng(k).normal(size=phi.shape), *D)
        np.testing.assert_array_equal(dU, want)
