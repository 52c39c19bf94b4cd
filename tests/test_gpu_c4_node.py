"""The DPA4C readout and fitting kernel at the edges of its waves: 16 nodes a
wave up to 32,768 nodes, 64 past them, hidden widths that are no multiple of
16, both activations, the square residual layer.

A graph of unconnected copies of one small system: the first copy against the
fp64 oracle, at the acceptance limits of the reference's mixed precision
(data/numeric-tolerances.json:3-9); every other copy holds the same edge
vectors in the same order, so its energies and forces are the first one's bit
for bit wherever its nodes lie in a wave, and for both kernels."""
import numpy as np
import pytest

from test_gpu_dpa4c import E_TOL, F_MAX, _canonical, _run_canonical, C4

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fit,act,resnet", [(96, 0, 0), (1, 0, 0), (17, 1, 0), (70, 0, 1),
                                            (1024, 1, 1)])
def test_waves(dp, fit, act, resnet):
    coord, atype, box = dp.systems.water(2, 6.21, seed=61)
    n = len(atype)
    m = dp.dpa4c.random_model("water", seed=340, fit=[fit], act=act, resnet=resnet)
    mb = dp.dpa4c.to_bytes(m)
    O = C4.Dpa4cOracle(mb)
    base = O.compute(coord, atype, box)
    src, dst = np.asarray(base["mapping"])[base["src"]], base["dst"]
    pot = dp.DeepPot(file_content=mb)
    first = None
    # copies, then nodes of their own without edges, the last of a type that
    # the model does not have
    for copies, extra in [(1, 1), (1, 9), (3, 0), (32768 // n, 32768 % n), (32768 // n + 1, 41)]:
        shift = n * np.repeat(np.arange(copies), len(src))
        types = np.concatenate([np.tile(atype, copies), np.zeros(extra, int)])
        if extra:
            types[-1] = -1
        nn = len(types)
        g = _canonical(np.zeros((nn, 3)), types, np.tile(src, copies) + shift,
                       np.tile(dst, copies) + shift, np.tile(base["edge_vec"], (copies, 1)), nn)
        ae, f, av = _run_canonical(dp, pot, g, nn)
        if first is None:
            assert np.abs(ae[:n] - base["atom_energy"]).max() <= E_TOL
            assert np.abs(f[:n] - base["force"]).max() <= F_MAX
            first = ae[:n], f[:n], av[:n]
        for a, b in zip((ae, f, av), first):
            a = a[:n * copies].reshape(copies, n, -1)
            assert np.array_equal(a, np.broadcast_to(b.reshape(1, n, -1), a.shape)), (copies, extra)
        if extra:
            assert ae[-1] == 0.0 and not f[-extra:].any() and not av[-extra:].any()
        if extra > 1:
            assert np.ptp(ae[n * copies:-1]) == 0.0 and ae[-2] != 0.0
