"""Lists from the cell tables against the all-pairs rebuild, entry for entry:
tables of 64 buckets, where the 27 (or 125) cells about a bead collide in the
hash and beads are met more than once; trajectories that share a span of the
slot kernel and ones that cross its edge; more candidates than the sorting
network holds; open and periodic, both stencils."""
import numpy as np
import pytest

from mt_amd import lattice, topology
from mt_amd.engine import Engine, LISTS_CELLS, LISTS_ALLPAIRS, MODE_STREAMED
from tests.helpers import base_params, uneven_batch

pytestmark = pytest.mark.gpu


def _tubes(lengths, side):
    b = uneven_batch(lengths=lengths, n_free=(0,) * len(lengths))
    b.box = np.full(len(lengths), side, np.float32)
    return b


def _cloud(ndimers):
    """Free dimers in a 20 nm cube and a tube: 150 of them leave a bead in its
    middle some 75 others within 8 nm."""
    rng = np.random.default_rng(11)
    atoms = [lattice.free_dimers(ndimers, 20.0, rng, min_sep=1.5, chain="B"), lattice.microtubule(12)]
    return topology.make_batch(atoms, [lattice.coords7(a, 0.1, rng) for a in atoms], is_assembly=True)


@pytest.mark.parametrize("make,arg", [
    (_tubes, ((1,), 0.0)), (_tubes, ((1, 2, 1), 0.0)), (_tubes, ((1,) * 70 + (20, 1, 1), 0.0)),
    (_tubes, ((12, 1, 40), 0.0)), (_tubes, ((1, 12), 150.0)), (_cloud, (150,))])
@pytest.mark.parametrize("stencil", [1, 2])
def test_cell_lists_equal_all_pairs(make, arg, stencil):
    print("case cell lists", make.__name__, str(arg)[:40], "stencil", stencil, flush=True)
    b = make(*arg)
    p = base_params(is_assembly=True)
    out = []
    for method in (LISTS_CELLS, LISTS_ALLPAIRS):
        eng = Engine(p, b.copy(), max_lj=200, mode=MODE_STREAMED, list_method=method)
        if method == LISTS_CELLS:
            eng.set_tuning(cell_stencil=stencil)
        eng.rebuild()
        out.append(eng.lists())
        eng.close()
    cells, pairs = out
    if make is _cloud:
        assert pairs["lj_count"].max() > 32
    for name in ("lon", "lat", "lj"):
        n = pairs[name + "_count"]
        np.testing.assert_array_equal(cells[name + "_count"], n)
        used = np.arange(pairs[name].shape[1])[None, :] < n[:, None]
        np.testing.assert_array_equal(np.where(used, cells[name], 0), np.where(used, pairs[name], 0))
