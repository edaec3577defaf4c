"""The streamed plain step, which gives each bead a second thread for its random
force and LJ sum: partly filled and several blocks, fixed beads, open and
periodic, against the FP32 oracle under the engine's own random streams.
Tolerance: 1e-3 nm and rad, the suite's bound for FP32 trajectories of this
length; the states of the streams are exact."""
import numpy as np
import pytest

from mt_amd.engine import Engine, MODE_STREAMED
from oracle.oracle import Oracle, generate_seeds
from tests.helpers import branch_params, uneven_batch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("block", [64, 128, 256])
@pytest.mark.parametrize("side", [0.0, 400.0])
@pytest.mark.parametrize("lengths,n_free", [((1,), (0,)), ((1, 1), (19, 20)), ((2, 4), (6, 70))])
def test_streamed_step(lengths, n_free, side, block):
    print(f"case streamed step, rows {lengths}, free dimers {n_free}, side {side}, block {block}", flush=True)
    p = branch_params()
    p.is_wall = 0 if side else p.is_wall   # the walls know no images
    b = uneven_batch(lengths=lengths, n_free=n_free)
    b.box = np.full(len(lengths), side, np.float32)
    eng = Engine(p, b.copy(), max_lj=64, mode=MODE_STREAMED, rseed=5)
    seeds = generate_seeds(5, 2 * b.nb)
    eng.set_tuning(stream_block=block)
    ref = Oracle(p, b.copy(), max_lj=64, precision="f32")
    eng.run(60)
    assert ref.run(0, 60, seeds=seeds) == 0
    got, rng = eng.get_state(), eng.get_rng()
    eng.close()
    assert np.abs(got[:, :6] - ref.b.coords[:, :6]).max() < 1e-3
    np.testing.assert_array_equal(rng, seeds)
