"""The autotuner's choices: kept for lists of the kind they were measured on,
alternative kernels only where a list has one, and the tuned shapes run by builds
too long for one launch.  Sums in another order: 1e-12 of the largest element."""
import numpy as np
import pytest

from pkfock.engine import FockEngine, PREC_MIXED
from pkfock.host import Molecule
from pkfock.molecules import water, water_cluster

pytestmark = pytest.mark.gpu


def _density(n, seed):
    A = np.random.default_rng(seed).normal(size=(n, n)) * 0.2
    return A + A.T


def _same(a, b):
    return all(np.abs(x - y).max() <= 1e-12 * max(1.0, np.abs(y).max()) for x, y in zip(a, b))


def test_alternative_kernels_only_where_a_list_has_one():
    """One water in cc-pVTZ: every list but the Obara-Saika ones and those with
    (ss) kets runs in its row kernel and has no alternative.  With every quartet in
    FP64 lists of the mixed precision the same classes are per-lane Rys lists, for
    which nothing has been measured."""
    eng = FockEngine(Molecule(*water(), "cc-pvtz").shells(), "os", 1e-12)
    P = _density(eng.nbasis, 1)
    ref = eng.jk(P)
    eng.autotune(reps=1)
    rows = [c for c in eng.class_stats() if c["kind"] != 0 and c["lc"] >= 1]
    assert len(rows) > 20 and not any(c["alt"] for c in rows)
    assert not any(c["alt"] for c in eng.class_stats() if c["kind"] == 0)
    eng.set("os", 1e-12, precision=PREC_MIXED, fp32_cutoff=0.0)
    got = eng.jk(P)
    lists = [c for c in eng.class_stats() if c["lc"] >= 1]
    assert any(c["kind"] == 1 for c in lists) and not any(c["alt"] for c in lists)
    assert _same(got, ref)


def test_tuned_shapes_of_a_long_build():
    """Five waters in cc-pVDZ (some 48 thousand waves: list by list, tuned or not)."""
    Z, X = water_cluster(5, n=5)
    eng = FockEngine(Molecule(Z, X, "cc-pvdz").shells(), "os", 1e-12)
    P = _density(eng.nbasis, 2)
    ref = eng.jk(P)
    eng.autotune(reps=1)
    got = eng.jk(P)
    assert eng.stats()["kernel_launches"] >= len(eng.class_stats())
    eng.set_graph(True)
    for _ in range(3):
        assert _same(eng.jk(P), ref)
    assert _same(got, ref)


def _in_one_launch(eng):
    # prepare, s/p/d lists, f lists, finalize, and at most five classes outside
    return eng.stats()["kernel_launches"] <= 9 < len(eng.class_stats())


@pytest.mark.parametrize("basis", ["6-31g*", "cc-pvtz"])
def test_short_build_after_autotuning(basis):
    """The tuner takes the one launch of a short build or its tuned lists; the choice
    holds before and after the lists are built again, and both give the same."""
    eng = FockEngine(Molecule(*water(), basis).shells(), "os", 1e-12)
    P = _density(eng.nbasis, 3)
    ref = eng.jk(P)
    assert _in_one_launch(eng)
    eng.autotune(reps=3)
    assert _same(eng.jk(P), ref)
    one = _in_one_launch(eng)
    eng.profile(True)  # the lists, as tuned
    assert _same(eng.jk(P), ref) and not _in_one_launch(eng)
    eng.profile(False)
    eng.set("os", 0.99e-12)
    got = eng.jk(P)
    assert _in_one_launch(eng) == one
    eng.set("os", 1e-12)
    assert _same(eng.jk(P), ref) and _in_one_launch(eng) == one
    assert all(np.abs(x - y).max() < 1e-9 for x, y in zip(got, ref))
