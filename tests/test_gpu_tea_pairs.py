"""The symmetric TEA pair kernel at the edges of its chunks, I pairs, J runs
and step splits, open and periodic, against the FP64 drift, and its wrapped
integer coordinates for beads many boxes away from the origin."""
import numpy as np
import pytest

from mt_amd import lattice, params as P, topology
from mt_amd.engine import Engine, MODE_STREAMED, TEA_SYMMETRIC
from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu


def _dimers(sizes, box, seed):
    """Trajectories of free dimers (beads: 2 x dimers) in periodic boxes, or
    far apart on open boundaries (box 0)."""
    rng = np.random.default_rng(seed)
    atoms = [lattice.free_dimers(s, box if box else 260.0, rng, min_sep=8.0) for s in sizes]
    b = topology.make_batch(atoms, [lattice.coords7(a, 0.2, rng) for a in atoms],
                            box=[box] * len(sizes) if box else None)
    return b


def _drift(p, b, F, shift=0.0):
    """F + sum_j D_hat_ij F_j in FP64 per trajectory (minimum image)."""
    out = np.zeros((b.nb, 3))
    for t in range(b.ntraj):
        s, e = int(b.off[t]), int(b.off[t + 1])
        x = b.coords[s:e, :3].astype(np.float64)
        f = F[s:e]
        d = x[None] - x[:, None]
        L = float(b.box[t]) if b.box.size else 0.0
        if L > 0:
            d -= L * np.rint(d / L)
        r = np.sqrt((d * d).sum(2))
        np.fill_diagonal(r, 1.0)
        u = p.tea_a / r
        near = r <= 2 * p.tea_a
        cii = np.where(near, 1 - 9 / 32 / u, 0.75 * u * (1 + 2 / 3 * u * u))
        crr = np.where(near, 3 / 32 / u, 0.75 * u * (1 - 2 * u * u))
        np.fill_diagonal(cii, 0.0)
        np.fill_diagonal(crr, 0.0)
        e3 = d / r[:, :, None]
        out[s:e] = f + cii @ f + np.einsum("ij,ija,ijb,jb->ia", crr, e3, e3, f, optimize=True)
    return out


# beads: below one chunk, one chunk, an I pair, a pair and a bead, odd chunk
# counts, several J runs; the batch sizes reach eight, four and one wave per
# unit and J runs of several chunks
@pytest.mark.parametrize("box", [0.0, 300.0])
@pytest.mark.parametrize("sizes", [(1,), (31, 32, 33), (64, 65), (97, 160), (500, 333, 129), (1100,) * 30])
def test_pair_sums_at_chunk_edges(sizes, box):
    print(f"case TEA pairs, dimers={sizes[:4]}x{len(sizes)}, box={box}", flush=True)
    p = P.derive(dict(P.TEA, tea_epsilon_freq=1, dt=1000.0, LJPairsCutoff=8.0))
    b = _dimers(sizes, box, 7)
    # a zero-noise step of dt = 1000 ps moves beads by dt / gammaR times the
    # hydrodynamic force: fractions of a nm, against positions' 2^-23 x 300 nm
    eng = Engine(p, b.copy(), mode=MODE_STREAMED)
    eng.set_tuning(tea_chunk=TEA_SYMMETRIC)
    F = eng.forces()[:, :3].astype(np.float64)
    eng.set_noise(np.zeros((1, b.nb, 6), np.float32))
    eng.run(1)
    moved = eng.get_state()[:, :3].astype(np.float64) - b.coords[:, :3].astype(np.float64)
    want = p.dt / p.gammaR * _drift(p, b, F)
    # the sums' FP32 rounding (1e-5 of the largest move) and the state's own
    tol = 1e-5 * np.abs(want).max() + 2 * 2.0 ** -24 * np.abs(b.coords[:, :3]).max()
    assert np.abs(moved - want).max() <= tol
    eng.close()


def test_periodic_pairs_of_beads_many_boxes_away():
    """Unwrapped positions: whole boxes added to a bead change nothing beyond
    the rounding of its larger float coordinates."""
    print("case TEA pairs, beads moved by whole boxes", flush=True)
    p = P.derive(dict(P.TEA, tea_epsilon_freq=1, dt=1000.0))
    b = _dimers((150,), 256.0, 3)
    moved = []
    for k in (0, 5):
        c = b.copy()
        shift = 256.0 * k * (np.arange(b.nb) // 2 % 3 - 1)[:, None]   # whole dimers, either way
        c.coords[:, :3] += shift.astype(np.float32)
        eng = Engine(p, c.copy(), mode=MODE_STREAMED)
        eng.set_tuning(tea_chunk=TEA_SYMMETRIC)
        eng.set_noise(np.zeros((1, b.nb, 6), np.float32))
        eng.run(1)
        moved.append(eng.get_state()[:, :3].astype(np.float64) - c.coords[:, :3])
        eng.close()
    # positions of up to 1600 nm: coordinates and bond gaps round at 2^-24 x
    # 1600 nm; the spring (C dt / gammaR = 62 per step) carries a gap's error
    tol = 4 * 2.0 ** -24 * 1600 * (1 + 300.0 * p.dt / p.gammaR)
    assert np.abs(moved[1] - moved[0]).max() <= tol
