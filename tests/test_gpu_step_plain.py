"""The streamed plain step and the forces gathered from global memory, which give
each bead a second thread for its random force and LJ sum: partly filled and several blocks, fixed beads, open and
periodic, against the FP32 oracle under the engine's own random streams.
Tolerance: 1e-3 nm and rad, the suite's bound for FP32 trajectories of this
length; the states of the streams are exact.  Forces: 1e-5 of the largest
component of the FP64 oracle's, the suite's bound."""
import numpy as np
import pytest

from mt_amd import params as P
from mt_amd.engine import Engine, FORCES_GLOBAL, MODE_STREAMED
from oracle.oracle import Oracle, generate_seeds
from tests.helpers import ANG, BRANCH, XYZ, branch_params, rel_err, uneven_batch

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


@pytest.mark.parametrize("block", [64, 128, 256])
@pytest.mark.parametrize("lengths,n_free", [((1,), (0,)), ((1, 1), (19, 20)), ((2, 4), (6, 70))])
def test_forces_from_global_memory(lengths, n_free, block):
    print(f"case forces from global memory, rows {lengths}, free dimers {n_free}, block {block}", flush=True)
    p = P.derive(dict(P.TEA, **BRANCH))
    b = uneven_batch(lengths=lengths, n_free=n_free)
    eng = Engine(p, b.copy(), max_lj=64)
    eng.set_tuning(forces=FORCES_GLOBAL, stream_block=block)
    ref = Oracle(p, b.copy(), max_lj=64)
    assert ref.rebuild() == 0
    f, want = eng.forces(), ref.forces()
    eng.close()
    assert rel_err(f, want, XYZ) < 1e-5 and rel_err(f, want, ANG) < 1e-5
