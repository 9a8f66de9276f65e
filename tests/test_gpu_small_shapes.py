"""GPU: the shape ids of batches of small grids, whose steps take the merged form
(id 12 in the fused kernel's place): what is in use is what get_shapes says and
what the tuner timed, setting it again changes nothing, and every choice gives
the same bits."""
import numpy as np
import pytest

import binary_supernova_amd as bsn
from binary_supernova_amd import problems as P

pytestmark = pytest.mark.gpu

MERGED = 12


def state(shape, seed):
    rng = np.random.default_rng(seed)
    U = P.empty_state(*shape)
    s = U.shape[:-1]
    rho, p = rng.uniform(0.5, 2.0, s), rng.uniform(0.5, 2.0, s)
    v = rng.normal(0.0, 0.3, s + (3,))
    U[..., 0], U[..., 1:4] = rho, rho[..., None] * v
    U[..., 4] = p / 0.4 + 0.5 * rho * (v * v).sum(-1)
    return U


def batch(shape, prec="fp64"):
    g = bsn.Grid(*shape, prec).set_state(state(shape, 1))
    g.set_params(0.1, 0.07, 0.13, 1.4, "outflow", 1e-3, 1e-3)
    return g, bsn.Batch([g])


@pytest.mark.parametrize("prec", ["split", "fp64"])
def test_small_batch_ids_round_trip(prec):
    print(f"small ids {prec}", flush=True)
    out = []
    for how in ("as made", "set again", "separate", "separate, then merged", "tuned", "tuned, set again"):
        g, b = batch((24, 20, 17), prec)
        if how.startswith("separate"):
            b.set_shapes(0, 7, 7)
            assert b.get_shapes() == [0, 7, 7, 11]
        if how.endswith("merged"):
            b.set_update_shape(MERGED)
        if how.startswith("tuned"):
            rep = b.autotune()["zupdate"]
            assert rep["merged"] == (rep["merged_stage"] < rep["stage"])
            assert (b.get_shapes()[3] == MERGED) == rep["merged"]
        ids = b.get_shapes()
        if how in ("as made", "separate, then merged"):
            assert ids == [0, 7, 7, MERGED]
        if how.endswith("again"):
            b.set_shapes(*ids[:3])
            b.set_update_shape(ids[3])
            assert b.get_shapes() == ids
        b.run(0.3, 3, graph=True)
        out.append(g.get_state())
    for a in out[1:]:
        np.testing.assert_array_equal(a, out[0])


def test_merged_form_is_refused_for_large_grids():
    print("merged refused", flush=True)
    g, b = batch((96, 96, 96))
    assert b.get_shapes() == [0, 7, 7, 11]
    with pytest.raises(bsn.BsnError):
        b.set_update_shape(MERGED)
    with pytest.raises(bsn.BsnError):
        batch((24, 20, 17))[1].set_update_shape(MERGED + 1)
    assert b.get_shapes() == [0, 7, 7, 11]
