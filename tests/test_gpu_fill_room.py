"""The device compile of fill programs (fillprog.hip) and the tables of the fused
constrained transport out of room: the host compiles, the separate launches run
instead, with the same results, bitwise against the oracle."""
import numpy as np
import pytest

import oracle as O
from gpu_util import compare_states, gpu_state, oracle_state

pytestmark = pytest.mark.gpu

BIG = 2 ** 31 - 1
CFG = dict(ic="rotor", limiter="MC", flux="HLLD", cfl=0.5, nx=8, nghosts=2, maxlevs=6)


def _compiled(sim):
    from amr2d_mhd_amd._lib import lib

    out = np.zeros(3, np.int64)
    assert lib().amr_debug_compiled(sim.h, out.ctypes.data) == 0
    return out


def _run(room, cfg=CFG, steps=27, tables=True):
    """Steps in lockstep with the oracle; the programs compiled on the device, on
    the host, and on the host after the device."""
    import amr2d_mhd_amd as A
    from amr2d_mhd_amd._lib import lib

    sim, dom = A.Simulation(cfg), O.Domain(**cfg)
    sim.init()
    assert dom.init() == 0
    sim.set_fill_cache(0)
    assert lib().amr_debug_pull_room(sim.h, *(room + (BIG,))[:5]) == 0
    if not tables:
        assert lib().amr_debug_drop_ct_tables(sim.h) == 1
        assert lib().amr_debug_drop_ct_tables(sim.h) == 0
    before = _compiled(sim)
    for step in range(steps):
        sim.step()
        assert dom.step() == 0
        if step % 5 == 4 or step == steps - 1:
            d = compare_states(gpu_state(sim), oracle_state(dom))
            assert not d, f"after step {step}: " + "; ".join(d[:4])
    n = _compiled(sim) - before
    sim.close()
    return n


def test_group_larger_than_allowed():
    """Groups of linked ops beyond the size the device places (several workgroups
    find one at once)."""
    device, host, again = _run((BIG, BIG, BIG, 1))
    assert device == 0 and again > 1 and host >= again


@pytest.mark.parametrize("room", [(BIG, 0, BIG, 256), (BIG, 100, BIG, 256), (BIG, BIG, 0, 256), (BIG, BIG, 256, 256)],
                         ids=["no pairs", "few pairs", "no tail", "one chunk of tail"])
def test_out_of_room(room):
    """No room for pairs of ops or linked ops, or for the first of them only.  (The
    trees of these runs need no explicit operands.)"""
    device, host, again = _run(room)
    assert 0 < again <= host


@pytest.mark.parametrize("cfg,steps", [
    (dict(ic="rotor", limiter="minmod", flux="HLLC", cfl=0.5, nx=16, nghosts=2, maxlevs=5), 18),
    (CFG, 27),
    (dict(ic="OT", limiter="WENO5", flux="HLLD", cfl=0.4, nx=16, nghosts=4, maxlevs=5, periodic=True, rk_stages=3), 6),
], ids=["20x20", "12x12", "24x24 periodic"])
def test_every_large_tree_on_the_device(cfg, steps):
    """With its own room the device compiles every changed tree of 8192 ring
    elements or more, and the host every smaller one."""
    import amr2d_mhd_amd as A

    nt = cfg["nx"] + 2 * cfg["nghosts"]
    ring = nt * nt - cfg["nx"] ** 2
    sim = A.Simulation(cfg)
    sim.init()
    sim.set_fill_cache(0)
    want = np.zeros(2, np.int64)
    tree = sim.get_tree()[2].tobytes()
    sim.step()  # (the initial tree's program)
    before = _compiled(sim)
    for _ in range(steps):
        now = sim.get_tree()[2].tobytes()
        if now != tree:  # compiled by the step that follows
            want[0 if sim.info()["nleaf"] * ring >= 8192 else 1] += 1
        tree = now
        sim.step()
    got = _compiled(sim) - before
    sim.close()
    assert want[0] > 1
    assert got[2] == 0 and (got[:2] == want).all(), (got, want)


@pytest.mark.parametrize("words", [0, 20000])
def test_no_scratch(words):
    """Memory without room for the device compile's scratch, for that of any tree
    or of the larger ones."""
    device, host, again = _run((BIG, BIG, BIG, 256, words))
    assert again == 0 and host > 1 and (words or device == 0)


@pytest.mark.parametrize("extra", [dict(), dict(ct_type=2, flux="HLLC"), dict(rk_stages=3)], ids=["RK2", "type 2", "RK3"])
def test_no_tables(extra):
    """A context whose memory had no room for the fused CT's tables."""
    _run((BIG, BIG, BIG, 256), cfg=dict(CFG, maxlevs=5, **extra), steps=12, tables=False)
