"""Extra flags changed between runs of a TEA engine whose steps have been
captured: the next refresh takes the epsilon kernel of the new flags."""
import numpy as np
import pytest

from mt_amd import lattice, params as P, topology
from mt_amd.engine import Engine, MODE_STREAMED, TEA_SYMMETRIC

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("first", [False, True])
def test_refresh_after_a_change_of_the_extra_flags(first):
    """Ten drawn steps (captured, with their refresh), the flags set or taken
    back, ten more: epsilon, beta, ci and the states of an engine that had
    those flags from the start, bit for bit."""
    print(f"case TEA refresh after set_flags, extra beads before: {first}", flush=True)
    p = P.derive(dict(P.TEA, tea_epsilon_freq=10, LJPairsUpdateFreq=10, tea_capricious=False))
    rng = np.random.default_rng(5)
    at = lattice.free_dimers(520, 260.0, rng, min_sep=8.0, chain="Y")
    b = topology.make_batch([at], [lattice.coords7(at, 0.2, rng)])
    on = (np.random.default_rng(2).random(b.nb) < 0.2).astype(np.uint8)
    flags = [on, np.zeros_like(on)] if first else [np.zeros_like(on), on]
    b.extra[:] = flags[0]
    eng = Engine(p, b.copy(), mode=MODE_STREAMED)
    eng.set_tuning(tea_chunk=TEA_SYMMETRIC)
    eng.run(10)
    state, words = eng.get_state(), eng.get_rng()
    eng.set_flags(extra=flags[1])
    eng.run(10)
    b.extra[:] = flags[1]
    b.coords = state
    new = Engine(p, b.copy(), mode=MODE_STREAMED)
    new.set_tuning(tea_chunk=TEA_SYMMETRIC)
    new.set_rng(words)
    new.step = 10
    new.run(10)
    for got, want in zip(eng.tea_stats(), new.tea_stats()):
        np.testing.assert_array_equal(got, want)
    np.testing.assert_array_equal(eng.tea_ci(), new.tea_ci())
    np.testing.assert_array_equal(eng.get_state(), new.get_state())
    eng.close()
    new.close()
