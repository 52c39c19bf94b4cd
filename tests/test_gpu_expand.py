"""GPU parity of the embedding stage's two evaluations: the nets expanded in
one variable (one, two and four groups of 64 terms, four centres to a block of
four waves and, above 2,048 centres, to one wave), and slot by slot (nets too
steep to expand), on counts that leave the waves' centres incomplete; and slots
closer than the expansion's range, which evaluate the net itself. With atom
outputs and without: the backward has a form for each."""
import numpy as np
import pytest

from cases import model_bytes
from test_expand_host import scaled
from test_gpu_mixed import _check as mixed_check, _volume

pytestmark = pytest.mark.gpu

E_TOL, F_TOL, V_TOL = 1e-10, 1e-8, 1e-8


def check(dp, orc, system, m, mixed, label, atomic=True):
    coord, atype, box = system
    mb = model_bytes(m)
    ref = orc.Oracle(mb).compute(coord, atype, box)
    pot = dp.DeepPot(file_content=mb, precision=dp.PREC_MIXED if mixed else dp.PREC_FP64)
    got = pot.compute(coord, atype, box, atomic=atomic)
    if mixed:
        mixed_check(len(atype), _volume(box), got, ref, label)
        return
    e, f, v = got[:3]
    # the bars of the other parity tests, and their share of large values (a
    # close pair's forces): 1e-12 is four thousand roundings
    def tol(bar, a):
        return max(bar, 1e-12 * np.abs(a).max())
    assert abs(e - ref["energy"]) / len(atype) <= tol(E_TOL, ref["atom_energy"])
    assert np.abs(f - ref["force"]).max() <= tol(F_TOL, ref["force"])
    assert np.abs(v - ref["virial"]).max() <= tol(V_TOL, ref["virial"])
    if atomic:
        ae, av = got[3:]
        assert np.abs(ae - ref["atom_energy"]).max() <= tol(E_TOL, ref["atom_energy"])
        assert np.abs(av - ref["atom_virial"]).max() <= tol(V_TOL, ref["atom_virial"])


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("kind,scale,drop", [
    ("water", 0.25, 1),   # one group of terms
    ("water", 1.0, 2),    # two
    ("water", 2.5, 3),    # four
    ("water", 30.0, 5),   # none: slot by slot
    ("cu", 1.0, 3), ("cu", 2.5, 1), ("cu", 30.0, 2), ("hea", 1.0, 7)])
def test_both_evaluations(dp, orc, kind, scale, drop, mixed):
    build = {"water": lambda: dp.systems.water(4, 12.42, seed=51),
             "cu": lambda: dp.systems.fcc(5, 3.615, seed=52),
             "hea": lambda: dp.systems.bcc_hea(5, 3.2, seed=53)}[kind]
    coord, atype, box = build()
    keep = np.setdiff1d(np.arange(len(atype)), (np.arange(drop) * 37 + 11) % len(atype))
    check(dp, orc, (coord[keep], atype[keep], box), scaled(dp, kind, scale), mixed,
          f"{kind} x{scale}")


@pytest.mark.parametrize("atomic", [False, True])
@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("kind,cells,drop", [("water", 4, 3), ("water", 9, 10), ("hea", 11, 7)])
def test_four_groups_of_terms(dp, orc, kind, cells, drop, mixed, atomic):
    """Models 2.5 times as steep (more than 128 terms), in blocks of four waves
    (the 4-cell system) and of one, with incomplete groups of centres."""
    if kind == "water":
        coord, atype, box = dp.systems.water(cells, 3.105 * cells, seed=56)
    else:
        coord, atype, box = dp.systems.bcc_hea(cells, 3.2, seed=57)
    keep = np.setdiff1d(np.arange(len(atype)), (np.arange(drop) * 37 + 11) % len(atype))
    check(dp, orc, (coord[keep], atype[keep], box), scaled(dp, kind, 2.5), mixed,
          f"{kind} x2.5", atomic)


@pytest.mark.parametrize("atomic", [False, True])
@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("kind,cells", [("water", 4), ("hea", 4), ("water", 9), ("hea", 11)])
def test_pairs_closer_than_the_expansion(dp, orc, kind, cells, mixed, atomic):
    """Pairs on both sides of the range's end (0.6 A), several of one centre
    and of neighbouring centres, with four centres to a block of waves and (the
    larger systems) to a wave."""
    if kind == "water":
        coord, atype, box = dp.systems.water(cells, 3.105 * cells, seed=54)
    else:
        coord, atype, box = dp.systems.bcc_hea(cells, 3.2, seed=55)
    coord = coord.copy()
    n = len(atype)
    for k, (a, b, r) in enumerate([(0, n - 1, 0.59), (0, n // 2, 0.45), (1, n - 2, 0.61), (5, 6, 0.5)]):
        u = np.array([np.cos(k), np.sin(k), 0.3 * k])
        coord[b] = coord[a] + r * u / np.linalg.norm(u)
    check(dp, orc, (coord, atype, box), scaled(dp, kind, 1.0), mixed, f"{kind} close", atomic)
