"""Ghosts, cells and the neighbour list on both sides of the sizes at which the
kernels take the prefix sums over themselves: 4,096 ghost counts (26 images of a
tile of 256 atoms) and 8,192 cells. The extended atoms are the oracle's bit for
bit, every centre's neighbour set is the strict-cutoff set."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cells", [(1, 1, 1), (2, 2, 2),
                                   (8, 8, 157), (8, 8, 158),       # 4,082 and 4,108 counts
                                   (2, 2, 1530), (2, 2, 1540)])    # 8,181 and 8,235 cells
def test_geometry(dp, orc, cells):
    coord, atype, box = dp.systems.fcc_alloy(cells, 3.56, seed=71)
    m = dp.dpa4c.random_model("cuni", seed=345)
    rc = m["rcut"]
    pot = dp.DeepPot(file_content=dp.dpa4c.to_bytes(m))
    pot.compute(coord, atype, box)
    ext, et, mp = orc.Oracle.ghosts(coord, atype, box, rc)
    n, nall = len(atype), len(et)
    assert pot.stage(dp.STAGE_EXT_COORD, np.float64, (nall, 3)).tobytes() == ext.tobytes()
    assert np.array_equal(pot.stage(dp.STAGE_MAPPING, np.int32, (nall,)), mp)
    assert np.array_equal(pot.stage(dp.STAGE_EXT_TYPE, np.int32, (nall,)), et)
    nl = pot.stage(dp.STAGE_NLIST, np.int32, (n, pot.nnei))
    for i in range(0, n, max(1, n // 150)):
        d = ext - ext[i]
        r2 = d[:, 0] * d[:, 0] + d[:, 1] * d[:, 1] + d[:, 2] * d[:, 2]
        want = np.nonzero((r2 < rc * rc) & (np.arange(nall) != i))[0]
        assert sorted(nl[i][nl[i] >= 0].tolist()) == want.tolist(), i
