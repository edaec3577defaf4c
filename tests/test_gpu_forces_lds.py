"""Forces from LDS with a helper thread per bead (trajectories of up to 2496
beads) and without (2497 to 2560), against the FP64 oracle (1e-5 of the largest
component, the suite's bound for forces): sizes at the edges of a tile of 256
beads and of the LDS, extra beads, walls, every branch of the force field."""
import numpy as np
import pytest

from mt_amd import params as P
from mt_amd.engine import Engine, FORCES_LDS
from oracle.oracle import Oracle
from tests.helpers import ANG, BRANCH, XYZ, rel_err, uneven_batch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lengths,n_free", [((1,), (0,)), ((9,), (11,)), ((10, 30), (0, 6)), ((96,), (0,)), ((98,), (0,))])
def test_forces_from_lds(lengths, n_free):
    print("case forces from LDS, rows", lengths, "free dimers", n_free, flush=True)
    p = P.derive(dict(P.TEA, **BRANCH))
    b = uneven_batch(lengths=lengths, n_free=n_free)
    eng = Engine(p, b.copy(), max_lj=64)
    assert eng.tuning()["forces"] == FORCES_LDS   # its default wherever a trajectory fits
    orc = Oracle(p, b.copy(), max_lj=64)
    assert orc.rebuild() == 0
    f, want = eng.forces(), orc.forces()
    eng.close()
    assert rel_err(f, want, XYZ) < 1e-5 and rel_err(f, want, ANG) < 1e-5
