"""The fitting's fp64 products at the edges of their tiles and rules, on the plain
and the fused input gradient: rows that are no multiple of 64, K split and not,
48- and 80-column tiles (the line lies at 10,880 rows for 240 columns), several
types. Against the oracle at the fp64 parity bars."""
import numpy as np
import pytest

from cases import CASES, model_bytes
from test_gpu_parity import E_TOL, F_TOL, V_TOL, assert_form

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fused", [False, True], ids=["plain_dD", "fused_dDdT"])
@pytest.mark.parametrize("case,cells,drop", [("cu864", 7, 3), ("cu864", 14, 0), ("cu864", 14, 97),
                                             ("water192", 9, 1)])
def test_products(dp, orc, case, cells, drop, fused):
    _, m = CASES[case]()
    if case == "cu864":
        coord, atype, box = dp.systems.fcc(cells, 3.615, seed=81)
    else:
        coord, atype, box = dp.systems.water(cells, cells * 3.105, seed=82)
    n = len(atype) - drop
    coord = np.ascontiguousarray(np.asarray(coord).reshape(-1, 3)[:n])
    atype = np.ascontiguousarray(atype[:n])
    mb = model_bytes(m)
    ref = orc.Oracle(mb).compute(coord, atype, box)
    pot = dp.DeepPot(file_content=mb)
    if fused:
        pot.set_fused_rows(0)
    e, f, v, ae, av = pot.compute(coord, atype, box, atomic=True)
    assert_form(dp, pot, "fused_dDdT" if fused else "plain_dD")
    assert abs(e - ref["energy"]) / n <= E_TOL
    assert np.abs(ae - ref["atom_energy"]).max() <= E_TOL
    assert np.abs(f - ref["force"]).max() <= F_TOL
    # (a sum over all atoms: the bar per atom's share)
    assert np.abs(v - ref["virial"]).max() <= V_TOL * max(1.0, n / 1000)
    assert np.abs(av - ref["atom_virial"]).max() <= V_TOL


@pytest.mark.parametrize("fused", [False, True], ids=["plain_dD", "fused_dDdT"])
def test_uneven_types(dp, orc, fused):
    """A type too large for its K loop to be split before one that is split
    (11,000 and 664 atoms): only the latter has slices in the workspace."""
    _, m = CASES["hea1024"]()
    coord, atype, box = dp.systems.bcc_hea(18, 3.2, seed=83)
    n = len(atype)
    atype = (np.arange(n) >= 11000).astype(np.int32)
    mb = model_bytes(m)
    ref = orc.Oracle(mb).compute(coord, atype, box)
    pot = dp.DeepPot(file_content=mb)
    if fused:
        pot.set_fused_rows(0)
    e, f, v, ae, av = pot.compute(coord, atype, box, atomic=True)
    assert_form(dp, pot, "fused_dDdT" if fused else "plain_dD")
    assert abs(e - ref["energy"]) / n <= E_TOL
    assert np.abs(ae - ref["atom_energy"]).max() <= E_TOL
    assert np.abs(f - ref["force"]).max() <= F_TOL
    assert np.abs(v - ref["virial"]).max() <= V_TOL * max(1.0, n / 1000)
    assert np.abs(av - ref["atom_virial"]).max() <= V_TOL
