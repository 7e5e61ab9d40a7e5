"""The device compile of fill programs (fillprog.hip) out of room: the host
compiles instead, with the same results, bitwise against the oracle."""
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


def _run(room, cfg=CFG, steps=27):
    """Steps in lockstep with the oracle; the programs compiled on the device, on
    the host, and on the host after the device."""
    import amr2d_mhd_amd as A
    from amr2d_mhd_amd._lib import lib

    sim, dom = A.Simulation(cfg), O.Domain(**cfg)
    sim.init()
    assert dom.init() == 0
    sim.set_fill_cache(0)
    assert lib().amr_debug_pull_room(sim.h, *room) == 0
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
