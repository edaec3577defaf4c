"""The resident kernel with a second thread for every bead (at most 512 mobile
beads per trajectory) against two beads per thread, bit for bit: the helper
only sums and draws what the owner would, and the sums are added in the same
order.  At the edges: one dimer row, a workgroup of whole and of partly filled
waves, the last size with helpers and the first without (494 and 520 mobile
beads), several lengths in a batch, open and periodic; drawn noise (the same
final streams), and injected noise with a bead thrown out of its skin in the
middle and at the last step, so that the lists are refilled."""
import numpy as np
import pytest

from mt_amd.engine import Engine, MODE_RESIDENT
from tests.helpers import base_params, noise, uneven_batch

pytestmark = pytest.mark.gpu
NSTEPS = 60


def _run(b, pt, nz):
    eng = Engine(base_params(), b.copy(), max_lj=64, mode=MODE_RESIDENT)
    eng.set_tuning(resident_per_thread=pt)
    if nz is not None:
        eng.set_noise(nz)
    eng.run(NSTEPS)
    out = eng.get_state(), eng.get_rng().copy()
    eng.close()
    return out


@pytest.mark.parametrize("lengths,side", [((1,), 0.0), ((12,), 0.0), ((20,), 0.0), ((21,), 0.0),
                                          ((19, 2, 7), 0.0), ((12, 5), 200.0)])
@pytest.mark.parametrize("kick", [None, 30, NSTEPS - 1])
def test_helped_equals_two_per_thread(lengths, side, kick):
    print(f"case helped resident steps, lengths {lengths}, side {side}, kick {kick}", flush=True)
    b = uneven_batch(lengths=lengths, n_free=(0,) * len(lengths))
    b.box = np.full(len(lengths), side, np.float32)
    nz = None
    if kick is not None:
        nz = noise(np.random.default_rng(9), NSTEPS, b.nb)
        nz[kick, b.nb // 2, 0] += 70.0   # about 1 nm (varR is 0.0149 nm)
    got, want = _run(b, 1, nz), _run(b, 2, nz)
    np.testing.assert_array_equal(got[1], want[1])
    np.testing.assert_array_equal(got[0], want[0])


@pytest.mark.parametrize("length", [35, 36, 48])
def test_one_per_thread_when_the_helpers_find_no_room(length):
    """Long trajectories, mostly immobile: 500 mobile beads of 910 (the last
    such tube whose LDS holds the helpers' buffer), of 936 (the first without)
    and of 1248 (the longest that one bead per thread takes)."""
    print(f"case one bead per thread, 500 mobile beads, length {length}", flush=True)
    b = uneven_batch(lengths=(length,), n_free=(0,))
    b.fixed[500:] = 1
    got, want = _run(b, 1, None), _run(b, 2, None)
    np.testing.assert_array_equal(got[1], want[1])
    np.testing.assert_array_equal(got[0], want[0])


@pytest.mark.parametrize("length,out,leaves", [(12, 4.0, 4), (12, 3.5, 5), (20, 4.0, 5), (20, 3.5, 6)])
def test_drawn_noise_goes_on_across_a_refill(length, out, leaves):
    """A bead set `out` nm off its place springs back and leaves its skin
    (0.75 nm from where the launch began) at step `leaves`, even or odd, in the
    middle of the launch: the lists are refilled and the helper's normals,
    drawn a step ahead, are used from there on, none twice and none skipped."""
    print(f"case helped resident steps, refill at step {leaves} of {length}", flush=True)
    b = uneven_batch(lengths=(length,), n_free=(0,))
    k = b.nb // 2
    r = b.coords[k, :2].copy()
    b.coords[k, :2] += out * r / np.hypot(*r)
    eng = Engine(base_params(), b.copy(), max_lj=64, mode=MODE_RESIDENT)
    eng.set_tuning(resident_per_thread=2)
    moved = []
    for _ in range(leaves + 1):
        eng.run(1)
        moved.append(np.linalg.norm(eng.get_state()[:, :3] - b.coords[:, :3], axis=1).max())
    eng.close()
    assert moved[-1] > 0.76 > 0.74 > max(moved[:-1])   # well clear of 0.75 either way
    got, want = _run(b, 1, None), _run(b, 2, None)
    np.testing.assert_array_equal(got[1], want[1])
    np.testing.assert_array_equal(got[0], want[0])
