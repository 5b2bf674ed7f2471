"""Which kernels a build runs, and the results of those that short molecules do not
reach by themselves."""
import numpy as np
import pytest

from pkfock.engine import FockEngine
from pkfock.host import Molecule
from pkfock.molecules import alkane

pytestmark = pytest.mark.gpu


def _density(n, seed):
    A = np.random.default_rng(seed).normal(size=(n, n)) * 0.2
    return A + A.T


def test_first_build_of_many_quartets_in_few_waves():
    """n-C16H34 / STO-3G: above the quartets from which a build spreads its lists
    over the side queues, below the waves up to which it goes out in one launch.
    The first build must not time lists that no build runs."""
    eng = FockEngine(Molecule(*alkane(16), "sto-3g").shells(), "os", 1e-12)
    P = _density(eng.nbasis, 1)
    first = eng.jk(P)
    launches = eng.stats()["kernel_launches"]
    lists = eng.class_stats()
    assert eng.stats()["quartets"] >= 1 << 20 and sum(c["waves"] for c in lists) <= 32768
    assert launches < len(lists)
    again = eng.jk(P)
    assert eng.stats()["kernel_launches"] == launches
    for x, y in zip(first, again):
        assert np.abs(x - y).max() <= 1e-12 * max(1.0, np.abs(y).max())
