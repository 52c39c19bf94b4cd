"""The embedding nets' expansion as the host builds it (csrc/expand.cpp),
without a GPU: accuracy of the values and slopes over the whole range, both
operand layouts, and the nets that have none."""
import os
import shutil
import subprocess

import numpy as np
import pytest

from _pkg import PKG_DIR, ROOT

HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


def scaled(dp, kind, scale):
    """A seeded model whose first-layer weights are scaled: the nets vary
    `scale` times as fast with the distance."""
    m = dp.model.random_model(kind, seed=1000)
    m["emb_params"] = m["emb_params"].copy()
    m["emb_params"][:, :m["emb"][0]] *= scale
    return m


def build(tmp_path, name):
    """tests/native/<name>.cpp with the expansion's host side."""
    exe = str(tmp_path / name)
    csrc = os.path.join(PKG_DIR, "csrc")
    subprocess.run([HIPCC, "-O2", "-std=c++17", "--offload-arch=gfx950", "-w",
                    os.path.join(ROOT, "tests", "native", name + ".cpp"),
                    os.path.join(csrc, "expand.cpp"), os.path.join(csrc, "model.cpp"), "-o", exe],
                   check=True)
    return exe


needs_hipcc = pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not found")


@needs_hipcc
def test_expansion_accuracy(dp, tmp_path):
    exe = build(tmp_path, "expand_check")
    def poisoned(at, value):
        m = dp.model.random_model("cu", seed=1000)
        m["emb_params"] = m["emb_params"].copy()
        m["emb_params"][0, at] = value
        return m

    # a first-layer weight (every feature), one feature's last-layer bias (not
    # the last feature) and weight
    bad = [(poisoned(at, value), None, 0)
           for at in (3, -7, -150) for value in (np.nan, np.inf, -np.inf)]
    # features of 1e-6 at most: accuracy relative to them, not to one
    small = dp.model.random_model("cu", seed=1000)
    small["emb_params"] = small["emb_params"] * 1e-6
    bad.append((small, None, 1))
    cases = [("water", 0.25, 1), ("cu", 1.0, 1), ("water", 1.0, 2), ("hea", 1.0, 2),
             ("water", 2.5, 4), ("hea", 2.5, 4), ("water", 30.0, 0)] + bad
    paths = []
    for k, (kind, scale, _) in enumerate(cases):
        m = kind if scale is None else scaled(dp, kind, scale)
        paths.append(dp.model.write_model(str(tmp_path / f"m{k}.bin"), m))
    out = subprocess.run([exe] + paths, check=True, capture_output=True, text=True).stdout
    lines = out.strip().splitlines()
    assert len(lines) == len(cases), out
    for (kind, scale, groups), line in zip(cases, lines):
        f = line.split()
        if groups == 0:
            assert f == ["none"], (kind, scale, line)
            continue
        assert f[0] == "ok" and int(f[1]) == groups, (kind, scale, line)
        eg, ed, en, gm, dm = (float(v) for v in f[2:7])
        # values: a few dozen roundings of 2^-53 of the largest value
        assert eg <= 32 * 2.0 ** -53 * gm, line
        # slopes near the cutoff, where most neighbours are, the same of the
        # largest slope (with the range's end there, so without the margin of
        # expand.h, the seeded water and HEA nets err by 236 and 142 times 2^-53 of
        # it); towards 0.6 A the ends' loss of digits
        assert en <= 32 * 2.0 ** -53 * dm, line
        assert ed <= 256 * 2.0 ** -53 * dm, line
        assert f[7] == "0", line


@needs_hipcc
def test_expansion_out_of_memory(dp, tmp_path):
    """An allocation that fails in any of the build's threads, or while they
    are made, reaches the caller as an exception."""
    exe = build(tmp_path, "expand_memory_check")
    path = dp.model.write_model(str(tmp_path / "m.bin"), dp.model.random_model("cu", seed=1000))
    r = subprocess.run([exe, path], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stderr
    assert r.stdout.split()[0] == "ok" and int(r.stdout.split()[1]) > 10, r.stdout


@needs_hipcc
def test_steep_nets_are_found_early(dp, tmp_path):
    """A model whose nets have no expansion is known as such sooner than one
    that has is built (it took four times as long when every net was tried with
    every number of nodes); half as long again allows for a busy machine."""
    exe = build(tmp_path, "expand_check")
    paths = [dp.model.write_model(str(tmp_path / f"m{s}.bin"), scaled(dp, "hea", s)) for s in (1.0, 30.0)]
    r = subprocess.run([exe] + paths, check=True, capture_output=True, text=True)
    assert r.stdout.splitlines()[1] == "none"
    flat, steep = (float(t) for t in r.stderr.split())
    assert steep <= 1.5 * flat, (flat, steep)
