"""Fill programs compiled on the device: runs whose trees change, large enough for
that path (engine.cpp, kPullElements), in lockstep with the oracle, bitwise, on
every tile form, at mirror and periodic boundaries, and several instances of
different trees in one context."""
import numpy as np
import pytest

import oracle as O
from gpu_util import FIELD_MAP, compare_states, gpu_state, oracle_state

pytestmark = pytest.mark.gpu

ELEMENTS = 8192  # ring elements from which the device compiles


def _ring(cfg):
    nx, ng = cfg["nx"], cfg["nghosts"]
    return (nx + 2 * ng) ** 2 - nx ** 2


@pytest.mark.parametrize("steps,cfgs", [
    (18, [dict(ic="rotor", limiter="minmod", flux="HLLC", cfl=0.5, nx=16, nghosts=2, maxlevs=5)]),
    (27, [dict(ic="rotor", limiter="MC", flux="HLLD", cfl=0.5, nx=8, nghosts=2, maxlevs=6)]),
    (6, [dict(ic="OT", limiter="WENO5", flux="HLLD", cfl=0.4, nx=16, nghosts=4, maxlevs=5, periodic=True, rk_stages=3)]),
    (18, [dict(ic="rotor", limiter="MC", flux="HLLD", cfl=0.5, nx=16, nghosts=2, maxlevs=4, periodic=True),
          dict(ic="rotor", limiter="minmod", flux="HLLC", cfl=0.5, nx=16, nghosts=2, maxlevs=5),
          dict(ic="BWx", limiter="MC", flux="HLLE", cfl=0.4, nx=16, nghosts=2, maxlevs=3)]),
], ids=["20x20", "12x12", "24x24 periodic", "three instances"])
def test_runs_bitwise(steps, cfgs):
    import amr2d_mhd_amd as A

    sim = A.Simulation(cfgs)
    sim.init()
    doms = [O.Domain(**c) for c in cfgs]
    for d in doms:
        assert d.init() == 0
    changed = 0
    before = [d.get_tree()[2].tobytes() for d in doms]
    for step in range(steps):
        sim.step()
        for d in doms:
            assert d.step() == 0
        after = [d.get_tree()[2].tobytes() for d in doms]
        now = [q for q in range(len(doms)) if after[q] != before[q]]
        changed += sum(doms[q].info()["nleaf"] * _ring(cfgs[q]) for q in now) >= ELEMENTS
        before = after
        if step % 4 == 1 or step == steps - 1:
            for q, d in enumerate(doms):
                diff = compare_states(gpu_state(sim, q), oracle_state(d))
                assert not diff, f"instance {q} after step {step}: " + "; ".join(diff[:4])
    assert changed > 1
    sim.close()


@pytest.mark.parametrize("cfg,steps", [
    (dict(ic="BWx", limiter="MC", flux="HLLE", cfl=0.4, nx=16, nghosts=2, maxlevs=2), 1),
    (dict(ic="rotor", limiter="MC", flux="HLLD", cfl=0.5, nx=8, nghosts=2, maxlevs=6), 6),
    (dict(ic="OT", limiter="MC", flux="HLLD", cfl=0.4, nx=16, nghosts=2, maxlevs=5, periodic=True), 4),
    (dict(ic="OT", limiter="WENO5", flux="HLLD", cfl=0.4, nx=16, nghosts=4, maxlevs=4, periodic=True), 2),
], ids=["16 leaves", "12x12", "over 320 chunks", "24x24"])
def test_cell_fill_bitwise(cfg, steps):
    """The fill of U by itself, random values in every element: programs below and
    above the chunk count to which a chunk's components go to several workgroups,
    restrictions, copies and linked (stale-read) ops."""
    import amr2d_mhd_amd as A

    dom = O.Domain(**cfg)
    assert dom.init() == 0
    for _ in range(steps):
        assert dom.step() == 0
    st = oracle_state(dom)
    rng = np.random.default_rng(3)
    st["U"] = rng.standard_normal(st["U"].shape)
    sim = A.Simulation(cfg)
    sim.init()
    sim.load_state(st)
    for name, f in FIELD_MAP.items():
        dom.set_field(f, st[name])
    dom.locate_bounds()
    for _ in range(2):
        sim.fill("U", "cell")
        assert dom.fill(O.U, O.FILL_CC) == 0
        d = compare_states(gpu_state(sim), oracle_state(dom), ("U",))
        assert not d, "; ".join(d[:4])
    sim.close()
