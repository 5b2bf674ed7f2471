"""J and K of the row kernels (csrc/engine/eri_rows.h) against the CPU oracle
where their work items have edges: kets fewer than a wave's quartet slots
(one water), several runs of first ket shells per item and remainders of the
slots (ethylene, two waters), every class up to (ff|ff) (cc-pVTZ), with the LDS
exchange rows and with direct global adds (PK_EXCHANGE_ROWS=0, the path of
molecules whose rows do not fit the LDS), one and two exchange densities.
Bar: 1e-9, the Fock bar (J and K of order 10; FP64 sums of at most 1e5 terms
differ by about 1e-13 relative between summation orders)."""
import numpy as np
import pytest

from pkfock.engine import FockEngine, Shells
from pkfock.molecules import ANGSTROM_TO_BOHR, alkane, water, water_cluster
from refcpu import Ref

pytestmark = pytest.mark.gpu

TOL = 1e-9
MOLS = {"water": water, "water2": lambda: water_cluster(5, n=2), "ethane": lambda: alkane(2)}


@pytest.mark.parametrize("rows", ["1", "0"])
@pytest.mark.parametrize("mol,basis", [("water", "cc-pvtz"), ("water2", "cc-pvdz"), ("ethane", "cc-pvdz")])
def test_row_kernels_match_oracle(mol, basis, rows, monkeypatch):
    monkeypatch.setenv("PK_EXCHANGE_ROWS", rows)
    Z, X = MOLS[mol]()
    ref = Ref(basis, np.asarray(Z), np.asarray(X) * ANGSTROM_TO_BOHR, engine="os", tol_eri=1e-11)
    eng = FockEngine(Shells(*ref.shells()), "os", 1e-11)
    rng = np.random.default_rng(21)
    A, B = rng.normal(size=(2, eng.nbasis, eng.nbasis)) * 0.2
    Pa, Pb = A + A.T, B + B.T
    Ja, Ka = ref.jk(Pa)
    Jb, Kb = ref.jk(Pb)
    J, K = eng.jk(Pa)
    Jt, K1, K2 = eng.jk_uhf(Pa, Pb)
    d = [np.abs(x).max() for x in (J - Ja, K - Ka, Jt - Ja - Jb, K1 - Ka, K2 - Kb)]
    print("%s/%s exchange rows %s: max|dJ| %.1e |dK| %.1e, UHF %.1e %.1e %.1e" % ((mol, basis, rows) + tuple(d)))
    assert max(d) < TOL


@pytest.mark.parametrize("mol,basis", [("water", "sto-3g"), ("water2", "cc-pvdz"), ("ethane", "3-21g")])
def test_gradient_items_match_oracle(mol, basis):
    """Work items of the gradient: contractions cut along the bra's primitives
    (nine s primitives in cc-pVDZ), slots left over, one and two exchange
    densities.  Bar: 1e-9 Eh/Bohr, as for the other gradients."""
    Z, X = MOLS[mol]()
    Xb = np.asarray(X) * ANGSTROM_TO_BOHR
    ref = Ref(basis, np.asarray(Z), Xb, engine="os", tol_eri=1e-11)
    eng = FockEngine(Shells(*ref.shells()), "os", 1e-11)
    rng = np.random.default_rng(22)
    A, B = rng.normal(size=(2, eng.nbasis, eng.nbasis)) * 0.1
    Pa, Pb = A + A.T, B + B.T
    for args in ((Pa, Pa, None, 1.0), (Pa + Pb, Pa, Pb, 2.0)):
        d = np.abs(eng.eri_gradient_atoms(Xb, *args) - ref.eri_gradient(*args)).max()
        print("%s/%s: max|dg| %.1e" % (mol, basis, d))
        assert d < TOL


@pytest.mark.parametrize("mol,basis", [("water", "sto-3g"), ("water", "cc-pvtz"), ("water2", "cc-pvdz"), ("ethane", "6-31g*")])
def test_short_build_in_one_launch_equals_its_lists(mol, basis):
    """A short build goes out in one launch; with per-class timing on, its lists
    run one by one in their own kernels.  Both must agree to the rounding of
    another summation order (1e-12), with a density that changes in between and
    on repeated calls, and replayed from a graph."""
    Z, X = MOLS[mol]()
    ref = Ref(basis, np.asarray(Z), np.asarray(X) * ANGSTROM_TO_BOHR, engine="os", tol_eri=1e-11)
    eng = FockEngine(Shells(*ref.shells()), "os", 1e-11)
    rng = np.random.default_rng(23)
    for rep in range(3):
        A = rng.normal(size=(eng.nbasis, eng.nbasis)) * 0.2
        P = A + A.T
        eng.profile(True)
        J0, K0 = eng.jk(P)
        eng.profile(False)
        J1, K1 = eng.jk(P)
        eng.set_graph(True)
        J2, K2 = eng.jk(P)
        eng.set_graph(False)
        d = [np.abs(x).max() for x in (J1 - J0, K1 - K0, J2 - J0, K2 - K0)]
        print("%s/%s: |dJ| %.1e |dK| %.1e, graph %.1e %.1e" % ((mol, basis) + tuple(d)))
        assert max(d) < 1e-12 * max(1.0, np.abs(J0).max())
        # prepare, s/p/d lists, f lists, finalize, and the five classes outside the
        # launch: (fd|ss), (ff|ss), (fd|fd), (ff|fd), (ff|ff)
        assert eng.stats()["kernel_launches"] <= 9


@pytest.mark.parametrize("engine", ["os", "rys"])
@pytest.mark.parametrize("alt", ["0", "1000"])
def test_segments_equal_plain_lists(engine, alt, monkeypatch):
    """Lists of more than 256 segments (n-C8H18 / cc-pVDZ, its waves too many for
    a short build): segments cut by steps and run most expensive first, workgroups
    of the row kernels by residency, against the same lists without exchange rows.
    Same integrals, another order of at most 1e6 FP64 sums: 1e-11 of the largest
    element."""
    Z, X = alkane(8)
    from pkfock.host import Molecule

    shells = Molecule(Z, X, "cc-pvdz").shells()
    out = []
    for rows in ("1", "0"):
        monkeypatch.setenv("PK_EXCHANGE_ROWS", rows)
        monkeypatch.setenv("PK_SEG_ALT_PRIM", alt)
        eng = FockEngine(shells, engine, 1e-11)
        rng = np.random.default_rng(24)
        A, B = rng.normal(size=(2, eng.nbasis, eng.nbasis)) * 0.2
        out.append(eng.jk(A + A.T) + eng.jk_uhf(A + A.T, B + B.T))
        eng.close()
    for x, y in zip(*out):
        assert np.abs(x - y).max() < 1e-11 * np.abs(y).max()
