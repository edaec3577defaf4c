"""Plain steps of a batch that mixes open and periodic trajectories.

One periodic trajectory takes the whole batch to the kernels with the minimum
image; an open one's separations must come out unchanged.  Every plan of the
resident kernel (one, two and three beads per thread) and the streamed kernel
run the same injected noise as the FP32 oracle, with every branch of the force
field on.  Tolerance: 1e-3 nm and rad after 120 steps, the suite's bound for
this many steps from the same start in FP32 (single-step differences of 1e-6
growing with the stiff springs).
"""
import numpy as np
import pytest

from mt_amd.engine import Engine, MODE_RESIDENT, MODE_STREAMED
from oracle.oracle import Oracle
from tests.helpers import branch_batch, branch_params, noise

pytestmark = pytest.mark.gpu
NSTEPS = 120
SIDE = 150.0   # more than a list cutoff beyond the tube (96 nm long)


def _batch(boxes):
    """Trajectories of one tube each; in a periodic one every third dimer is
    moved to a neighbouring image."""
    b = branch_batch(ntraj=len(boxes), jitter=0.2)
    b.box = np.array(boxes, np.float32)
    for t, side in enumerate(boxes):
        if side:
            lo, hi = int(b.off[t]), int(b.off[t + 1])
            b.coords[lo:hi, 0] += np.where((np.arange(hi - lo) // 2) % 3 == 0, np.float32(side), np.float32(0))
    return b


@pytest.mark.parametrize("boxes", [(0.0, SIDE), (SIDE, SIDE)])
@pytest.mark.parametrize("plan", [0, 1, 2, 3])
def test_open_and_periodic_trajectories_match_oracle(plan, boxes):
    print(f"case plain steps, boxes {boxes}, beads per thread {plan} (0: streamed)", flush=True)
    p = branch_params()
    p.is_wall = 0   # the walls know no images
    b = _batch(boxes)
    eng = Engine(p, b.copy(), max_lj=64, mode=MODE_RESIDENT if plan else MODE_STREAMED)
    if plan:
        eng.set_tuning(resident_per_thread=plan)
    orc = Oracle(p, b.copy(), max_lj=64, precision="f32")
    nz = noise(np.random.default_rng(7), NSTEPS, b.nb)
    eng.set_noise(nz)
    eng.run(NSTEPS)
    assert orc.run(0, NSTEPS, noise=nz) == 0
    d = np.abs(eng.get_state()[:, :6] - orc.b.coords[:, :6]).max()
    eng.close()
    assert d < 1e-3
