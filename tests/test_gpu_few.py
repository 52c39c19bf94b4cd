"""GPU parity of the fitting stage's few-atoms kernels (csrc/fit_few.hip) and
of the general chains on the same small systems (the plain product dE/dD and,
where the first layer has its 240 outputs, the fused input gradient), at the
edges of the row tiles: one row of a type, an absent type, 16 and 32 rows and
one more, both sides of the tile-height switch (384 atoms) and of the 64 KB of
LDS (256 outputs in fp64 fit with 16 rows a tile, not with 32), layers that are
not square."""
import numpy as np
import pytest

from cases import model_bytes
from test_gpu_expand import E_TOL, F_TOL, V_TOL
from test_gpu_parity import FORMS, assert_form, select_form
from test_gpu_mixed import _check as mixed_check, _volume

pytestmark = pytest.mark.gpu


def subset(system, counts):
    """The first counts[t] atoms of each type t."""
    coord, atype, box = system
    keep = np.sort(np.concatenate([np.nonzero(atype == t)[0][:k] for t, k in enumerate(counts)]))
    return coord[keep], atype[keep], box


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("kind,counts,fit", [
    ("water", (1, 32), None), ("water", (0, 33), None), ("water", (16, 17), (240, 240, 80)),
    ("water", (128, 256), None), ("water", (128, 257), (240, 160, 160)),
    ("hea", (5, 0, 31, 70), None), ("cu", (384,), (256, 256, 256)),
    ("cu", (385,), (256, 256, 256))])
def test_few_atoms(dp, orc, kind, counts, fit, mixed, form):
    system = {"water": lambda: dp.systems.water(6, 18.63, seed=61),
              "hea": lambda: dp.systems.bcc_hea(6, 3.2, seed=62),
              "cu": lambda: dp.systems.fcc(5, 3.615, seed=63)}[kind]()
    coord, atype, box = subset(system, counts)
    over = {} if fit is None else dict(fit=list(fit))
    mb = model_bytes(dp.model.random_model(kind, seed=1030, **over))
    ref = orc.Oracle(mb).compute(coord, atype, box)
    pot = dp.DeepPot(file_content=mb, precision=dp.PREC_MIXED if mixed else dp.PREC_FP64)
    if form == "fused_dDdT" and fit is not None and fit[0] != 240:
        pytest.skip("no fused kernel for this first layer")
    if form == "plain_dD" and mixed and (fit is None or fit[0] == 240):
        pytest.skip("mixed precision always takes the fused kernel for this first layer")
    if form != "few":  # (these systems run the few-atoms kernels by default)
        select_form(pot, form)
    got = pot.compute(coord, atype, box, atomic=True)
    if form == "few" and kind == "cu" and counts == (385,) and not mixed:
        form = "plain_dD"  # 32 rows of 256 doubles do not fit
    assert_form(dp, pot, form)
    if mixed:
        mixed_check(len(atype), _volume(box), got, ref, f"{kind} {counts}")
        return
    e, f, v, ae, av = got
    assert abs(e - ref["energy"]) / len(atype) <= E_TOL
    assert np.abs(ae - ref["atom_energy"]).max() <= E_TOL
    assert np.abs(f - ref["force"]).max() <= F_TOL
    assert np.abs(v - ref["virial"]).max() <= V_TOL
    assert np.abs(av - ref["atom_virial"]).max() <= V_TOL
