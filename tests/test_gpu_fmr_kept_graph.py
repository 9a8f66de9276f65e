"""GPU: the graph of a root step that a hierarchy keeps between calls: everything
that callers may change in between reaches it.  Each call is compared bit for
bit with the same call, launched step by step, on a second hierarchy."""
import numpy as np
import pytest

import binary_supernova_amd as bsn
from binary_supernova_amd import problems as P

pytestmark = pytest.mark.gpu

DIMS = [(18, 16, 20), (16, 16, 12), (12, 16, 16)]
BOXES = [(6, 13, 5, 12, 8, 13), (6, 11, 5, 12, 3, 10)]
DS = [(0.1 / 2 ** l,) * 3 for l in range(3)]


def state(n, seed):
    rng = np.random.default_rng(seed)
    U = P.empty_state(*n)
    s = U.shape[:-1]
    rho, p = rng.uniform(0.5, 2.0, s), rng.uniform(0.5, 2.0, s)
    v = rng.normal(0.0, 0.3, s + (3,))
    U[..., 0], U[..., 1:4] = rho, rho[..., None] * v
    U[..., 4] = p / 0.4 + 0.5 * rho * (v * v).sum(-1)
    return U


def states(H, seed):
    for l, lev in enumerate(H.levels):
        lev.set_state(state(DIMS[l], seed + l))


def phis(H, seed):
    H.set_phis([0.05 * np.random.default_rng(seed + l).normal(size=DIMS[l][::-1]) for l in range(len(H.levels))])


def params(H, g, bc, floor):
    for lev, d in zip(H.levels, DS):
        lev.set_params(*d, g, bc, floor, floor)


def bodies(H):
    b = bsn.BlackHole(pos=[0.9, 0.8, 1.0], vel=[0.0, 0.0, 0.0], mass=0.1, eps=0.1, c_code=1e3, r_floor=0.2)
    bsn.set_point_masses(H.levels[0], [b], 0.0, 0.0, 0.0)


def gravity(H, on):
    H.set_self_gravity(on, 0.02)


# (what changes before the call, cfl, steps, t_end)
CALLS = [
    (None, 0.3, 3, 0.0),
    (None, 0.3, 2, 0.0),
    (lambda H: states(H, 30), 0.3, 1, 0.0),
    (lambda H: phis(H, 40), 0.3, 2, 0.0),
    (lambda H: phis(H, 50), 0.3, 1, 0.0),
    (lambda H: H.levels[1].set_phi(None), 0.3, 2, 0.0),
    (lambda H: params(H, 5 / 3, "outflow", 1e-4), 0.3, 2, 0.0),
    (lambda H: params(H, 5 / 3, ("periodic", "outflow", "periodic"), 1e-3), 0.3, 2, 0.0),
    (None, 0.2, 2, 0.0),
    (None, 0.2, 3, 0.004),
    (None, 0.2, 2, 0.003),
    (None, 0.2, 2, 0.0),
    (bodies, 0.2, 2, 0.0),
    (lambda H: H.step(1e-3), 0.2, 2, 0.0),
    (lambda H: H.set_mode(True), 0.2, 2, 0.0),
    (lambda H: H.set_mode(False), 0.2, 2, 0.0),
    (lambda H: gravity(H, True), 0.2, 2, 0.0),
    (lambda H: gravity(H, False), 0.2, 2, 0.0),
    (lambda H: H.set_phis([None] * len(H.levels)), 0.2, 2, 0.0),
    (lambda H: H.autotune(), 0.2, 2, 0.0),
    (lambda H: H.prolong_all(1), 0.2, 0, 0.0),
    (None, 0.2, 2, 0.0),
]


@pytest.mark.parametrize("prec", ["fp64", "split"])
@pytest.mark.parametrize("levels", [2, 3])
def test_kept_graph_follows_every_change(levels, prec):
    H = [bsn.FMRHierarchy(DIMS[:levels], DS[:levels], BOXES[:levels - 1], [2] * (levels - 1), 1.4, "outflow",
                          1e-3, 1e-3, precision=prec) for _ in range(2)]
    for h in H:
        states(h, 10)
    for n, (change, cfl, steps, t_end) in enumerate(CALLS):
        print(f"kept graph {levels} {prec} call {n}", flush=True)
        for h, graph in zip(H, (True, False)):
            if change:
                change(h)
            h.run(cfl, steps, t_end=t_end, graph=graph)
        assert H[0].time() == H[1].time()
        for a, b in zip(*(h.levels for h in H)):
            a, b = a.get_state(), b.get_state()
            assert np.isfinite(P.active(a)).all()
            np.testing.assert_array_equal(a, b)
