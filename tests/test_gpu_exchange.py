"""The exchange calls through pinned slots of 512 KB: every byte arrives,
below one slot, over a slot boundary that no record straddles, and beyond the
eight slots of a buffer (slots reused within the call); from two threads at
once too, each with an engine of its own."""
import threading

import numpy as np
import pytest

from mt_amd.engine import Engine
from tests.helpers import base_params, c1_batch

pytestmark = pytest.mark.gpu


def _state(nb, seed):
    c = np.random.default_rng(seed).normal(0.0, 50.0, (nb, 7)).astype(np.float32)
    c[:, 6] = 0.0
    return c


@pytest.mark.parametrize("ntraj", [1, 60, 61, 500])   # 312 beads each: 8.7, 524, 533 KB and 4.4 MB
def test_state_round_trip(ntraj):
    print("case state round trip,", ntraj, "tubes of 312 beads", flush=True)
    b = c1_batch(ntraj=ntraj)
    eng = Engine(base_params(), b, max_lj=64)
    for seed in (1, 2):
        c = _state(b.nb, seed)
        eng.set_state(c)
        np.testing.assert_array_equal(eng.get_state(), c)
    eng.close()


def test_state_from_two_threads():
    print("case state round trips from two threads", flush=True)
    b = c1_batch(ntraj=61)
    bad = []

    def work(seed):
        eng = Engine(base_params(), b.copy(), max_lj=64)
        for k in range(5):
            c = _state(b.nb, 10 * seed + k)
            eng.set_state(c)
            if not np.array_equal(eng.get_state(), c):
                bad.append((seed, k))
        eng.close()

    threads = [threading.Thread(target=work, args=(s,)) for s in (1, 2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
