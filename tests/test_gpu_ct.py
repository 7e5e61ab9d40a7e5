"""Constrained transport with its ghost fills (CT2D.cpp:11-124, boundaryec.cpp,
boundaryfc.cpp) against the oracle, bitwise: the phase by itself (a launch a
kernel and a fill), and within steps, on trees whose levels step by one (two
launches a stage with the flux fills) and on a tree with a jump of two levels,
whose fills read blocks that are no leaves (the separate launches)."""
import numpy as np
import pytest

import oracle as O
from gpu_util import FIELD_MAP, compare_states, gpu_state, oracle_state

pytestmark = pytest.mark.gpu

SON, STRIDE = (1, 0, 2, 0), (2, 2, 1, 1)  # finer neighbours' first adjacent son and the step to the second, by side


def _two_level_jumps(lp, lf):
    jumps = 0
    for nb in np.flatnonzero(lf):
        for s in range(4):
            n = lp[nb, 4 + s]
            if n >= 0 and not lf[n] and lp[n, 0] >= lp[nb, 0]:
                f = lp[n, 2] + SON[s]
                jumps += not (lf[f] and lf[f + STRIDE[s]])
    return jumps


def _merge_next_to_finer(st):
    """Makes a leaf of the first father whose sons are leaves and that has finer
    leaves than those beside it."""
    lp, lf = st["lp"], st["leafs"]
    for dad in np.flatnonzero((lf == 0) & (lp[:, 2] > 0)):
        s0 = lp[dad, 2]
        sons = np.arange(s0, s0 + 4)
        if not lf[sons].all():
            continue
        lp2, lf2 = lp.copy(), lf.copy()
        lf2[dad], lf2[sons] = 1, 0
        outside = np.ones(len(lp), bool)
        outside[sons] = False
        links = lp2[outside, 4:8]
        links[np.isin(links, sons)] = dad
        lp2[outside, 4:8] = links
        if _two_level_jumps(lp2, lf2):
            return dict(st, lp=lp2, leafs=lf2)
    raise AssertionError("no such father")


CONFIGS = pytest.mark.parametrize("cfg", [
    dict(ic="rotor", limiter="MC", flux="HLLD", cfl=0.5, nx=16, nghosts=2, maxlevs=5),
    dict(ic="rotor", limiter="MC", flux="HLLC", cfl=0.5, nx=8, nghosts=2, maxlevs=4, ct_type=2),
    dict(ic="rotor", limiter="WENO5", flux="HLLD", cfl=0.4, nx=16, nghosts=4, maxlevs=4, rk_stages=3),
    dict(ic="rotor", limiter="MC", flux="HLLD", cfl=0.4, nx=16, nghosts=2, maxlevs=4, periodic=True, rk_stages=3,
         ct_type=2),
], ids=["RK2", "8 cells, type 2", "4 ghosts, RK3", "periodic, RK3, type 2"])


def _pair(cfg, jump, scale):
    """GPU and oracle in the same state: six steps of the run, with `jump` on the
    changed tree, every field scaled cell by cell within 1 +- `scale`."""
    import amr2d_mhd_amd as A

    dom = O.Domain(**cfg)
    assert dom.init() == 0
    for _ in range(6):
        assert dom.step() == 0
    st = oracle_state(dom)
    assert _two_level_jumps(st["lp"], st["leafs"]) == 0
    if jump:
        st = _merge_next_to_finer(st)
    rng = np.random.default_rng(7)
    for f in ("ff", "gg", "Us", "Bis", "Bi", "U"):
        st[f] = st[f] * rng.uniform(1 - scale, 1 + scale, st[f].shape)
    sim = A.Simulation(cfg)
    sim.init()
    sim.load_state(st)
    dom.set_tree(st["lp"], st["icoord"], st["leafs"])
    for name, f in FIELD_MAP.items():
        dom.set_field(f, st[name])
    inf = dom.info()
    sim.set_time(inf["t"], inf["dt"], inf["dt_next"], inf["count"])
    return sim, dom


@pytest.mark.parametrize("jump", [False, True], ids=["one level", "two levels"])
@CONFIGS
def test_ct_bitwise(cfg, jump):
    sim, dom = _pair(cfg, jump, 0.02)
    dom.locate_bounds()
    for step in range(1, cfg.get("rk_stages", 2) + 1):
        sim.ct(step)
        assert dom.ct(step) == 0
        d = compare_states(gpu_state(sim), oracle_state(dom))
        assert not d, f"after stage {step}: " + "; ".join(d[:4])
    sim.close()


@pytest.mark.parametrize("jump", [False, True], ids=["one level", "two levels"])
@CONFIGS
def test_steps_bitwise(cfg, jump):
    """The first step fills from unfilled ghosts, the second (without a change of
    the tree) runs its first fill on the programs' tails."""
    sim, dom = _pair(cfg, jump, 1e-4)
    for step in range(2):
        assert dom.step() == 0
        sim.step()
        d = compare_states(gpu_state(sim), oracle_state(dom))
        assert not d, f"after step {step}: " + "; ".join(d[:4])
    sim.close()
