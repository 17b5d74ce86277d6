"""Many uniform draws at once: the generator's own values and state, across the blocks
they are drawn in."""
import random

import numpy as np
import pytest

from quict_amd.simulation import uniforms as U


@pytest.mark.parametrize("count", [0, 1, 7, 8, 9, 16, 31])
def test_blocks_give_the_generators_values(count, monkeypatch):
    monkeypatch.setattr(U, "BLOCK", 8)
    random.seed(11)
    got, after = U.uniforms(count), random.getstate()
    random.seed(11)
    want = np.array([random.random() for _ in range(count)], dtype=np.float64)
    assert np.array_equal(got, want) and got.dtype == np.float64
    assert random.getstate() == after


def test_more_draws_than_one_call_of_the_generator_gives():
    """getrandbits takes a C int: 2^25 draws of 64 bits are one more than it can."""
    count = 2 ** 25 + 3
    random.seed(12)
    got = U.uniforms(count)
    random.seed(12)
    assert len(got) == count and got[0] == random.random() and got[1] == random.random()
    assert 0.49 < float(got.mean()) < 0.51
