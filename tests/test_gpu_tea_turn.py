"""TEA steps whose end and next forces share a launch (trajectories of up to
640 beads) against the same steps with separate force and update kernels, which
add the same terms in the same order: the same random streams, and states that
differ by at most one rounding at 150 nm (1.5e-5) per step.  Sizes at the edges: one
dimer row, the largest trajectory with a helper thread per bead (494) and the
first without (520), the largest of the fused kernel (624) and the first
beyond it; batches of several lengths, open, periodic and mixed, drawn
and injected noise, across a tensor refresh."""
import numpy as np
import pytest

from mt_amd import params as P
from mt_amd.engine import Engine, FORCES_GLOBAL, FORCES_LDS
from tests.helpers import noise, uneven_batch

pytestmark = pytest.mark.gpu


def _run(b, forces, nz, steps):
    eng = Engine(P.derive(dict(P.TEA, tea_epsilon_freq=20)), b.copy(), max_lj=64)
    eng.set_tuning(forces=forces)
    assert eng.tuning()["forces"] == forces
    if nz is not None:
        eng.set_noise(nz)
    eng.run(steps)
    out = eng.get_state(), eng.get_rng().copy()
    eng.close()
    return out


@pytest.mark.parametrize("lengths,boxes", [
    ((1,), (0.0,)), ((19, 2), (0.0, 0.0)), ((20,), (0.0,)), ((24,), (0.0,)), ((25, 3), (0.0, 0.0)), ((12, 1, 24), (0.0, 0.0, 0.0)),
    ((12, 5), (150.0, 0.0)), ((5, 12, 1, 2, 3, 4, 6, 7, 8), (150.0,) * 9)])
@pytest.mark.parametrize("injected", [False, True])
def test_fused_turn_equals_separate_kernels(lengths, boxes, injected):
    print(f"case fused end and forces, lengths {lengths}, boxes {boxes}, injected {injected}", flush=True)
    b = uneven_batch(lengths=lengths, n_free=(0,) * len(lengths))
    b.box = np.array(boxes, np.float32)
    steps = 33
    nz = noise(np.random.default_rng(4), steps, b.nb) if injected else None
    # forces from LDS (the fused kernel where it fits), forces gathered from memory (never fused)
    got, want = _run(b, FORCES_LDS, nz, steps), _run(b, FORCES_GLOBAL, nz, steps)
    np.testing.assert_array_equal(got[1], want[1])
    assert np.abs(got[0] - want[0]).max() <= steps * 1.5e-5
