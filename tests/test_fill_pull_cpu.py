"""The ghost fill looked up by destination (fill_pull.hpp) against the program the
sequential compile makes of the same tree, element by element, along whole runs
of the oracle: both tile forms, periodic and mirror boundaries, every tree a
run meets."""
import numpy as np
import pytest

import oracle as O


def _check(NT, ng, lp, ic, lf):
    from amr2d_mhd_amd._lib import lib

    lp, ic, lf = (np.ascontiguousarray(x, np.int32) for x in (lp, ic, lf))
    counts = np.zeros(4, np.int64)
    r = lib().amr_debug_pull_fill(NT, ng, lp.shape[0], lp.ctypes.data, ic.ctypes.data, lf.ctypes.data, counts.ctypes.data)
    return r, counts


@pytest.mark.parametrize("cfg,tiles,steps", [
    (dict(ic="BWx", limiter="MC", flux="RUSA", cfl=0.4, maxlevs=4), [(20, 2), (12, 2), (24, 4)], 300),
    (dict(ic="rotor", limiter="MC", flux="HLLD", cfl=0.5, maxlevs=5), [(20, 2), (24, 4)], 80),
    (dict(ic="rotor", limiter="MC", flux="HLLD", cfl=0.4, maxlevs=4, periodic=True), [(20, 2), (12, 2), (24, 4)], 60),
    (dict(ic="OT", limiter="MC", flux="HLLD", cfl=0.4, maxlevs=5, periodic=True), [(24, 4)], 20),
], ids=["tube", "rotor", "periodic rotor", "vortex"])
def test_every_tree_of_a_run(cfg, tiles, steps):
    dom = O.Domain(**cfg)
    assert dom.init() == 0
    last, trees, kinds = None, 0, np.zeros(4, np.int64)
    for s in range(steps):
        lp, ic, lf = dom.get_tree()
        key = (lp.tobytes(), lf.tobytes())
        if key != last:
            for NT, ng in tiles:
                r, counts = _check(NT, ng, lp, ic, lf)
                assert r == 0, f"step {s}, tile {NT}: {r}"
                kinds += counts
            last, trees = key, trees + 1
        if dom.done() or dom.step() != 0:
            break
    assert trees > 3 and kinds[0] > 0
    print(trees, kinds)
