"""GPU: the library's stream against the null stream, on which callers prepare
device memory (torch's default stream is it): the null stream is given some
milliseconds of copies first, so that an ordering that is missing shows."""
import ctypes as C

import numpy as np
import pytest

import binary_supernova_amd as bsn
from binary_supernova_amd import problems as P
from binary_supernova_amd._lib import BSN_DEVICE, call
from oracle import oracle as O

pytestmark = pytest.mark.gpu

D = (0.1, 0.07, 0.13)
D2D, H2D = 3, 1


class Hip:
    """The HIP runtime that libbsn_hip.so itself links."""

    def __init__(self):
        bsn.load()
        L = self.L = C.CDLL("/opt/rocm/lib/libamdhip64.so")
        p, n = C.c_void_p, C.c_size_t
        L.hipMalloc.argtypes, L.hipFree.argtypes = [C.POINTER(p), n], [p]
        L.hipMemcpy.argtypes, L.hipMemcpyAsync.argtypes = [p, p, n, C.c_int], [p, p, n, C.c_int, p]
        L.hipStreamCreateWithFlags.argtypes = [C.POINTER(p), C.c_uint]
        L.hipStreamDestroy.argtypes = L.hipStreamSynchronize.argtypes = [p]
        self.held = []

    def __getattr__(self, name):
        def run(*a):
            assert getattr(self.L, name)(*a) == 0, name
        return run

    def buffer(self, n, values=None):
        p = C.c_void_p()
        self.hipMalloc(C.byref(p), n)
        self.held.append(p)
        if values is not None:
            self.hipMemcpy(p, values.ctypes.data, values.nbytes, H2D)
        return p

    def keep_null_stream_busy(self):
        n = 512 << 20
        a, b = self.buffer(n), self.buffer(n)
        for _ in range(60):
            self.hipMemcpyAsync(a, b, n, D2D, None)

    def close(self):
        self.L.hipDeviceSynchronize()
        for p in self.held:
            self.L.hipFree(p)


@pytest.fixture
def hip():
    h = Hip()
    yield h
    h.close()


def state(shape, seed):
    rng = np.random.default_rng(seed)
    U = P.empty_state(*shape)
    s = U.shape[:-1]
    rho, p = rng.uniform(0.5, 2.0, s), rng.uniform(0.5, 2.0, s)
    v = rng.normal(0.0, 0.3, s + (3,))
    U[..., 0], U[..., 1:4] = rho, rho[..., None] * v
    U[..., 4] = p / 0.4 + 0.5 * rho * (v * v).sum(-1)
    return U


def test_phi_from_device_memory(hip):
    # phi reaches the caller's buffer late, in the null stream's order, and the
    # buffer is written again on a stream of its own once the call is back
    print("device phi", flush=True)
    shape = (24, 18, 20)
    U, phi = state(shape, 1), 0.1 * np.random.default_rng(2).normal(size=shape[::-1])
    src, buf = hip.buffer(phi.nbytes, phi), hip.buffer(phi.nbytes, np.full_like(phi, 5.0))
    other = hip.buffer(phi.nbytes, np.full_like(phi, 7.0))
    g = bsn.Grid(*shape).set_state(U)
    g.set_params(*D, 1.4)
    s = C.c_void_p()
    hip.hipStreamCreateWithFlags(C.byref(s), 1)
    hip.keep_null_stream_busy()
    hip.hipMemcpyAsync(buf, src, phi.nbytes, D2D, None)
    call("bsn_grid_set_phi", g.handle, buf, BSN_DEVICE)
    hip.hipMemcpyAsync(buf, other, phi.nbytes, D2D, s)
    bsn.euler3d_step_(g, *shape, *D, 2e-3, 1.4)
    O.euler3d_step(U, *D, 2e-3, 1.4, "outflow", phi=phi)
    np.testing.assert_array_equal(g.get_state(), U)
    hip.hipStreamSynchronize(s)
    hip.hipStreamDestroy(s)


def test_work_buffers_made_beside_a_busy_null_stream(hip):
    # the right-hand side's scratch and the levels' second work buffer are made,
    # and cleared, by the first call that needs them
    print("work buffers", flush=True)
    d, n, box, r = 0.1, (20, 18, 16), (6, 13, 5, 12, 5, 10), 2
    nf = tuple((box[2 * a + 1] - box[2 * a] + 1) * r for a in range(3))
    U, Uf = state(n, 3), state(nf, 4)
    g = bsn.Grid(*n).set_state(U)
    bsn.cfl_dt_3d(g, *n, d, d, d, 1.4, 0.3)
    H = bsn.FMRHierarchy([n, nf], [(d,) * 3, (d / r,) * 3], [box], [r], 1.4, "outflow", 1e-3, 1e-3)
    for lev, A in zip(H.levels, (U, Uf)):
        lev.set_state(A)
    dU = np.empty(U.shape)
    hip.keep_null_stream_busy()
    bsn.euler3d_rhs_(dU, None, None, None, g, *n, d, d, d, 1.4, bc="outflow")
    H.step(2e-3)
    np.testing.assert_array_equal(dU, O.euler3d_rhs(U.copy(), d, d, d, 1.4, "outflow", 0.0, 0.0)[0])
    O.fmr_multilevel_step([U, Uf], [(d,) * 3, (d / r,) * 3], [box], [r], 1.4, 2e-3, "outflow", 1e-3, 1e-3)
    for lev, A in zip(H.levels, (U, Uf)):
        np.testing.assert_array_equal(lev.get_state(), A)


def device_state(g):
    p, fs = C.c_void_p(), C.c_int64()
    call("bsn_grid_device_state", g.handle, C.byref(p), C.byref(fs), None)
    return p, 5 * fs.value * 8


@pytest.mark.parametrize("graph", [False, True])
def test_states_written_on_the_null_stream(hip, graph):
    # a new state reaches the grid's own buffer late, in the null stream's order,
    # before each call on the batch and on the hierarchy
    print(f"device states graph {graph}", flush=True)
    n, nf, box, d = (18, 16, 20), (16, 16, 12), (6, 13, 5, 12, 8, 13), 0.1
    news = [bsn.Grid(*s).set_state(state(s, 5 + k)) for k, s in enumerate((n, nf))]

    def make():
        g = bsn.Grid(*n).set_state(state(n, 7))
        g.set_params(d, d, d, 1.4)
        H = bsn.FMRHierarchy([n, nf], [(d,) * 3, (d / 2,) * 3], [box], [2], 1.4, "outflow", 1e-3, 1e-3)
        for lev, s in zip(H.levels, (n, nf)):
            lev.set_state(state(s, 8))
        return g, bsn.Batch([g]), H

    g, b, H = make()
    for what, grids in ((b, [g]), (H, H.levels)):
        for _ in range(2):                  # the first call, and one on kept tables
            hip.keep_null_stream_busy()
            for to, new in zip(grids, news):
                (p, size), (q, _) = device_state(to), device_state(new)
                hip.hipMemcpyAsync(p, q, size, D2D, None)
            what.run(0.3, 2, graph=graph)
    g2, b2, H2 = make()
    for what, grids in ((b2, [g2]), (H2, H2.levels)):
        for to, new in zip(grids, news):
            to.set_state(new.get_state())
        what.run(0.3, 2, graph=graph)
    for x, y in zip([g] + H.levels, [g2] + H2.levels):
        np.testing.assert_array_equal(x.get_state(), y.get_state())
