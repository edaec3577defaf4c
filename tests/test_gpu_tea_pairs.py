"""The symmetric TEA pair kernel at the edges of its chunks, I pairs, J runs
and step splits, open and periodic, against the FP64 drift, and its wrapped
integer coordinates for beads many boxes away from the origin."""
import numpy as np
import pytest

from mt_amd import lattice, params as P, topology
from mt_amd.engine import Engine, MODE_STREAMED, TEA_EPS_ONEPASS, TEA_EPS_TWOSIDED, TEA_SYMMETRIC
from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu


def _dimers(sizes, box, seed):
    """Trajectories of free dimers (beads: 2 x dimers) in periodic boxes, or
    far apart on open boundaries (box 0)."""
    rng = np.random.default_rng(seed)
    # chain Y: mobile beads (chain X marks extra ones)
    atoms = [lattice.free_dimers(s, box if box else 260.0, rng, min_sep=8.0, chain="Y") for s in sizes]
    b = topology.make_batch(atoms, [lattice.coords7(a, 0.2, rng) for a in atoms],
                            box=[box] * len(sizes) if box else None)
    return b


def _drift(p, b, F):
    """F + sum_j D_hat_ij F_j in FP64 per trajectory (minimum image); NaN for
    a bead exactly half a box from another along an axis, where the two
    images are equally near and the sum is not defined."""
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
        if L > 0:
            out[s:e][(np.abs(d) == L / 2).any((1, 2))] = np.nan
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
    ok = np.isfinite(want[:, 0])
    assert ok.mean() > 0.99
    tol = 1e-5 * np.abs(want[ok]).max() + 2 * 2.0 ** -24 * np.abs(b.coords[:, :3]).max()
    assert np.abs(moved - want)[ok].max() <= tol
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


def _eps_ci(p, b):
    """Epsilon per trajectory and ci per bead in FP64 (minimum image), extra
    beads left out."""
    eps, ci = np.zeros(b.ntraj), np.zeros((b.nb, 3))
    for t in range(b.ntraj):
        s, e = int(b.off[t]), int(b.off[t + 1])
        on = (b.extra[s:e] == 0).astype(np.float64)
        x = b.coords[s:e, :3].astype(np.float64)
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
        w = on[:, None] * on[None]
        np.fill_diagonal(w, 0.0)
        e3 = d / r[:, :, None]
        ci[s:e] = ((w * cii ** 2)[:, :, None] + (w * crr * (2 * cii + crr))[:, :, None] * e3 ** 2).sum(1)
        m = on.sum()
        eps[t] = (w * (3 * cii + crr * e3.sum(2) ** 2)).sum() / max(3 * m * (3 * m - 3), 1e-300)
    return eps, ci


# 1025 trajectories fill the chip with 1024-bead groups (four chunks per
# wave), 9 of them take 256-bead groups (one): sizes from one dimer over the
# chunk and group edges to several groups
@pytest.mark.parametrize("ntraj", [9, 1025])
@pytest.mark.parametrize("box", [0.0, 300.0])
@pytest.mark.parametrize("extra", [False, True])
def test_eps_sums_at_group_edges(ntraj, box, extra):
    print(f"case TEA eps groups, {ntraj} trajectories, box={box}, extra={extra}", flush=True)
    p = P.derive(dict(P.TEA, tea_epsilon_freq=1, tea_capricious=False))
    edges = (2, 32, 33, 64, 127, 128, 129, 513, 1100)
    b = _dimers(edges + tuple(2 + k % 5 for k in range(ntraj - len(edges))), box, 5)
    if extra:
        b.extra[np.random.default_rng(2).random(b.nb) < 0.2] = 1
        b.extra[b.off[:-1]] = 0
        b.extra[b.off[:-1] + 1] = 0
    eng = Engine(p, b.copy(), mode=MODE_STREAMED)
    eng.set_noise(np.zeros((1, b.nb, 6), np.float32))
    eng.run(1)
    eps, _ = eng.tea_stats()
    ci = eng.tea_ci().astype(np.float64)
    want_eps, want_ci = _eps_ci(p, b)
    # FP32 sums of up to 2200 positive terms
    np.testing.assert_allclose(eps, np.minimum(want_eps, 1.0), rtol=1e-5)
    keep = b.extra == 0
    np.testing.assert_allclose(ci[keep], want_ci[keep], rtol=1e-5, atol=1e-6)
    eng.close()


# a from none (free draining) over radii below the clamp of coincident beads
# (1e-6 nm) to the usual one
RADII = [0.0, 1e-8, 1e-4, 0.02, 2.0]


@pytest.mark.parametrize("a", RADII)
@pytest.mark.parametrize("box", [0.0, 300.0])
def test_eps_sums_of_any_radius(a, box):
    """Epsilon and ci hold no trace of the bead itself, however small the
    other beads' terms are."""
    print(f"case TEA eps, a={a}, box={box}", flush=True)
    p = P.derive(dict(P.TEA, tea_epsilon_freq=1, tea_capricious=False))
    p.tea_a = a
    b = _dimers((97, 20), box, 7)
    eng = Engine(p, b.copy(), mode=MODE_STREAMED)
    eng.set_tuning(tea_chunk=TEA_SYMMETRIC)
    eng.set_noise(np.zeros((1, b.nb, 6), np.float32))
    eng.run(1)
    eps, beta = eng.tea_stats()
    ci = eng.tea_ci().astype(np.float64)
    eng.close()
    p.tea_a = max(a, 1e-30)   # (the FP64 sums divide by it; a^2 is below any float)
    want_eps, want_ci = _eps_ci(p, b)
    # FP32 sums of up to 200 positive terms
    np.testing.assert_allclose(eps, want_eps, rtol=1e-5, atol=1e-25)
    np.testing.assert_allclose(ci, want_ci, rtol=1e-5, atol=1e-37)
    if a <= 1e-8:
        np.testing.assert_array_equal(beta, 0.5)   # |a_TEA| < 1e-7


@pytest.mark.parametrize("a", RADII)
@pytest.mark.parametrize("box", [0.0, 300.0])
@pytest.mark.parametrize("chunk", [64, 128, 256, TEA_SYMMETRIC])
def test_pair_sums_of_any_radius(a, box, chunk):
    """The one-sided kernels meet the bead itself, at distance 0, and take it
    out: for every radius."""
    print(f"case TEA pairs, a={a}, box={box}, chunk={chunk}", flush=True)
    p = P.derive(dict(P.TEA, tea_epsilon_freq=1, tea_capricious=False, dt=1000.0, LJPairsCutoff=8.0))
    p.tea_a = a
    b = _dimers((97, 20), box, 7)
    eng = Engine(p, b.copy(), mode=MODE_STREAMED)
    eng.set_tuning(tea_chunk=chunk)
    F = eng.forces()[:, :3].astype(np.float64)
    eng.set_noise(np.zeros((1, b.nb, 6), np.float32))
    eng.run(1)
    moved = eng.get_state()[:, :3].astype(np.float64) - b.coords[:, :3].astype(np.float64)
    eng.close()
    p.tea_a = max(a, 1e-30)
    want = p.dt / p.gammaR * _drift(p, b, F)
    ok = np.isfinite(want[:, 0])
    assert ok.mean() > 0.99
    # the sums' FP32 rounding (1e-5 of the largest move) and the state's own
    tol = 1e-5 * np.abs(want[ok]).max() + 2 * 2.0 ** -24 * np.abs(b.coords[:, :3]).max()
    assert np.abs(moved - want)[ok].max() <= tol


# the largest box of the integer coordinates, the next float, and boxes whose
# 2^-32 is no longer below the rounding of a pair's distance
@pytest.mark.parametrize("box", [1000.0, 4096.0, float(np.nextafter(np.float32(4096), np.float32(1e9))), 1e6, 1e7])
@pytest.mark.parametrize("chunk", [128, TEA_SYMMETRIC])
def test_tube_at_the_origin_of_a_large_box(box, chunk):
    """Beads that are near one another and near the origin keep the precision
    of their float differences however large the box."""
    print(f"case TEA tube in a box of {box}, chunk={chunk}", flush=True)
    p = P.derive(dict(P.TEA, tea_epsilon_freq=1, dt=1000.0))
    at = lattice.microtubule(12)
    b = topology.make_batch([at, at], [lattice.coords7(at, 0.2, np.random.default_rng(k)) for k in (3, 4)],
                            box=[box, 0.0])
    eng = Engine(p, b.copy(), mode=MODE_STREAMED)
    eng.set_tuning(tea_chunk=chunk)
    F = eng.forces()[:, :3].astype(np.float64)
    eng.set_noise(np.zeros((1, b.nb, 6), np.float32))
    eng.run(1)
    moved = eng.get_state()[:, :3].astype(np.float64) - b.coords[:, :3].astype(np.float64)
    eps, _ = eng.tea_stats()
    ci = eng.tea_ci().astype(np.float64)
    eng.close()
    want = p.dt / p.gammaR * _drift(p, b, F)
    want_eps, want_ci = _eps_ci(p, b)
    free = b.fixed == 0
    # the sums' FP32 rounding (1e-5 of the largest move) and the state's own
    tol = 1e-5 * np.abs(want).max() + 2 * 2.0 ** -24 * np.abs(b.coords[:, :3]).max()
    assert np.abs(moved - want)[free].max() <= tol
    np.testing.assert_allclose(eps, want_eps, rtol=1e-5)
    np.testing.assert_allclose(ci, want_ci, rtol=1e-5, atol=1e-6)


@pytest.mark.parametrize("chunk", [128, TEA_SYMMETRIC])
def test_cluster_across_the_faces_of_a_large_box(chunk):
    """Neighbours on both sides of every face of the largest box of the
    integer coordinates."""
    print(f"case TEA cluster across the faces, chunk={chunk}", flush=True)
    box = 4096.0
    p = P.derive(dict(P.TEA, tea_epsilon_freq=1, dt=1000.0, LJPairsCutoff=8.0))
    rng = np.random.default_rng(11)
    at = lattice.free_dimers(150, 80.0, rng, min_sep=8.0, chain="Y")
    b = topology.make_batch([at], [lattice.coords7(at, 0.2, rng)], box=[box])
    x = b.coords[:, :3].astype(np.float64) - 40.0
    b.coords[:, :3] = np.where(x < 0, x + box, x).astype(np.float32)
    eng = Engine(p, b.copy(), mode=MODE_STREAMED)
    eng.set_tuning(tea_chunk=chunk)
    F = eng.forces()[:, :3].astype(np.float64)
    eng.set_noise(np.zeros((1, b.nb, 6), np.float32))
    eng.run(1)
    moved = eng.get_state()[:, :3].astype(np.float64) - b.coords[:, :3].astype(np.float64)
    eng.close()
    want = p.dt / p.gammaR * _drift(p, b, F)
    tol = 1e-5 * np.abs(want).max() + 2 * 2.0 ** -24 * box
    assert np.abs(moved - want).max() <= tol


@pytest.mark.parametrize("box", [0.0, 60.0])
@pytest.mark.parametrize("eps", [TEA_EPS_ONEPASS, TEA_EPS_TWOSIDED])
@pytest.mark.parametrize("capricious", [False, True])
def test_a_bead_alone_in_its_trajectory_drains_freely(box, eps, capricious):
    """Dimers of which one bead, or both, are extra, beside whole ones: a
    bead with no other to meet has beta 0.5, ci 0 and moves by its own force
    and noise."""
    print(f"case TEA bead alone, box={box}, eps={eps}, capricious={capricious}", flush=True)
    p = P.derive(dict(P.TEA, tea_epsilon_freq=1, tea_capricious=capricious))
    b = _dimers((1,) * 40 + (20,), box, 9)
    one, none = np.arange(1, 40, 4), np.arange(2, 40, 4)   # trajectories with one bead left, with none
    b.extra[b.off[one]] = 1
    for k in (0, 1):
        b.extra[b.off[none] + k] = 1
    eng = Engine(p, b.copy(), mode=MODE_STREAMED)
    eng.set_tuning(tea_chunk=TEA_SYMMETRIC, tea_eps=eps)
    F = eng.forces()[:, :3].astype(np.float64)
    nz = np.random.default_rng(1).standard_normal((1, b.nb, 6)).astype(np.float32)
    eng.set_noise(nz)
    eng.run(1)
    e, beta = eng.tea_stats()
    got = eng.get_state()
    assert np.isfinite(got).all() and np.isfinite(e).all() and np.isfinite(beta).all()
    np.testing.assert_array_equal(e[np.r_[one, none]], 0.0)
    np.testing.assert_array_equal(beta[np.r_[one, none]], 0.5)
    i = b.off[one] + 1
    np.testing.assert_allclose(eng.tea_ci()[i], 0.0, atol=1e-6)
    moved = got[i, :3].astype(np.float64) - b.coords[i, :3]
    want = p.dt / p.gammaR * F[i] + p.varR * nz[0, i, :3]
    assert np.abs(moved - want).max() <= 1e-5 * np.abs(want).max() + 2 * 2.0 ** -24 * np.abs(b.coords[:, :3]).max()
    eng.close()
