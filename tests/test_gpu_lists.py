"""Which kernels a build runs, and the results of those that short molecules do not
reach by themselves: their builds go out in one launch, and their per-lane Rys classes
run in row kernels.  With per-class timing on the lists run in their own kernels; in
mixed precision with cutoff 0 (every quartet in FP64) the Rys classes of kets below
nine components run per lane."""
import numpy as np
import pytest

from pkfock.engine import FockEngine, PREC_MIXED, Shells
from pkfock.host import Molecule
from pkfock.molecules import ANGSTROM_TO_BOHR, alkane, water, water_cluster
from refcpu import Ref

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


MOLS = {"water": water, "water2": lambda: water_cluster(5, n=2), "ethane": lambda: alkane(2)}
_REF = {}


def _engine(mol, basis, kernels):
    """Oracle and an engine whose builds run the lists, or also the per-lane Rys kernels."""
    if (mol, basis) not in _REF:
        Z, X = MOLS[mol]()
        _REF[mol, basis] = Ref(basis, np.asarray(Z), np.asarray(X) * ANGSTROM_TO_BOHR, engine="os", tol_eri=1e-12)
    ref = _REF[mol, basis]
    eng = FockEngine(Shells(*ref.shells()), "os", 1e-12)
    if kernels == "lanes":
        eng.set("os", 1e-12, precision=PREC_MIXED, fp32_cutoff=0.0)
    else:
        eng.profile(True)
    return ref, eng


def _check_kernels(eng, kernels):
    cls = eng.class_stats()
    assert eng.stats()["kernel_launches"] >= len(cls) and not any(c["precision"] for c in cls)
    # the Rys classes of (ps) and (ds) kets: per lane, or in rows
    rys = [c["kind"] for c in cls if (c["lc"], c["ld"]) in ((1, 0), (2, 0)) and c["la"] == 2 and c["kind"] != 0]
    assert rys and set(rys) == {1 if kernels == "lanes" else 2}


@pytest.mark.parametrize("kernels", ["lists", "lanes"])
@pytest.mark.parametrize("rows", ["1", "0"])
@pytest.mark.parametrize("mol,basis", [("water", "cc-pvtz"), ("water2", "cc-pvdz"), ("ethane", "cc-pvdz")])
def test_list_kernels_match_oracle(mol, basis, rows, kernels, monkeypatch):
    """J and K, with and without exchange rows in LDS, one and two densities: 1e-9, the
    Fock bar."""
    monkeypatch.setenv("PK_EXCHANGE_ROWS", rows)
    ref, eng = _engine(mol, basis, kernels)
    Pa, Pb = _density(eng.nbasis, 2), _density(eng.nbasis, 3)
    Ja, Ka = ref.jk(Pa)
    Jb, Kb = ref.jk(Pb)
    J, K = eng.jk(Pa)
    _check_kernels(eng, kernels)
    Jt, K1, K2 = eng.jk_uhf(Pa, Pb)
    d = [np.abs(x).max() for x in (J - Ja, K - Ka, Jt - Ja - Jb, K1 - Ka, K2 - Kb)]
    print("%s/%s %s, exchange rows %s: max|dJ| %.1e |dK| %.1e, UHF %.1e %.1e %.1e" % ((mol, basis, kernels, rows) + tuple(d)))
    assert max(d) < 1e-9


@pytest.mark.parametrize("kernels", ["lists", "lanes"])
@pytest.mark.parametrize("mol,basis", [("water", "cc-pvtz"), ("ethane", "cc-pvdz")])
def test_list_eris_match_oracle(mol, basis, kernels):
    """Columns (.. | kl) of the ERI tensor from unit pair densities, as the class kernels
    of the lists compute them: 1e-11, the ERI bar."""
    ref, eng = _engine(mol, basis, kernels)
    n = eng.nbasis
    T = ref.eri_full()
    P = np.zeros((n, n))
    worst = 0.0
    for k in range(n):
        for l in range(k, n):
            P[k, l] = P[l, k] = 1.0
            J, _ = eng.jk(P)
            P[k, l] = P[l, k] = 0.0
            worst = max(worst, np.abs((J if k == l else 0.5 * J) - T[:, :, k, l]).max())
    _check_kernels(eng, kernels)
    print("%s/%s %s: max|dERI| %.2e" % (mol, basis, kernels, worst))
    assert worst < 1e-11


def test_class_statistics_of_a_short_build():
    """Every class reports its kernels and their shape, also where it shares a launch."""
    for basis in ("sto-3g", "cc-pvtz"):
        eng = FockEngine(Molecule(*water(), basis).shells(), "os", 1e-10)
        eng.jk(_density(eng.nbasis, 4))
        cls = eng.class_stats()
        assert eng.stats()["kernel_launches"] < len(cls)
        assert all(c["kernels"] >= 1 and c["block"] in (64, 128, 256) for c in cls)
