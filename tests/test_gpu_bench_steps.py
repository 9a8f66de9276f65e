"""GPU: the steps that bench.py times are CFL-limited steps of the workload's own
state, with and without warm-up: the state they end in is the one Batch.run
reaches from there."""
import os
import sys

import numpy as np
import pytest

import binary_supernova_amd as bsn

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
import bench  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("warmup", [0, 2])
@pytest.mark.parametrize("prec", ["split", "fp64"])
def test_timed_steps_are_steps_of_the_workload(prec, warmup):
    print(f"bench steps {prec} warm-up {warmup}", flush=True)
    U, dims, d = bsn.problems.turbulent_box(24, seed=1)
    args = (5.0 / 3.0, "periodic", (0.0, 0.0))
    r = bench.run_uniform(bsn, U, dims, d, *args, prec, 3, warmup)
    g = bsn.Grid(*dims, prec).set_state(U)
    g.set_params(*d, args[0], args[1], *args[2])
    bsn.Batch([g]).run(0.4, 3)
    want = g.get_state()
    assert np.isfinite(want).all()
    np.testing.assert_array_equal(r["state"], want)
