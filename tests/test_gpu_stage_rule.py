"""Which stage kernel a launch takes: the rule goes by the launch's own leaf
blocks, also where a stage is one launch a class of instances, and the times that
stage_tuning reports are those of the launches timed."""
import pytest

pytestmark = pytest.mark.gpu

STRIPS, WIDE, NARROW = 7, 2, 3


def _rotor(**k):
    return dict(dict(ic="rotor", limiter="MC", flux="HLLD", cfl=0.5, nx=16, nghosts=2, maxlevs=5), **k)


def _rule(n):
    return STRIPS if n < 128 else WIDE if n < 512 else NARROW


def _bucket(n):
    return n.bit_length() - 1


@pytest.mark.parametrize("cfgs", [
    [_rotor()],
    [_rotor(), _rotor(), _rotor(), _rotor(), _rotor(flux="HLLC", maxlevs=3)],
    [_rotor(), _rotor(), _rotor(flux="HLLC", maxlevs=3), _rotor(flux="HLLE", maxlevs=4)],
], ids=["one class", "two classes", "three classes"])
def test_rule_by_launch(cfgs):
    import amr2d_mhd_amd as A

    sim = A.Simulation(cfgs)
    sim.init()
    sim.run(3)
    sim.profile(("stage",))
    used, launched = set(sim.stage_tuning()), set()
    for _ in range(12):
        # the trees a step runs on
        counts = {}
        for q, c in enumerate(cfgs):
            counts[c["flux"]] = counts.get(c["flux"], 0) + sim.info(q)["nleaf"]
        launched |= set(counts.values())
        sim.step()
    sim.profile_read()
    got = sim.stage_tuning()
    assert set(got) - used <= {_bucket(n) for n in launched} <= set(got)
    for n in launched:
        variant, us = got[_bucket(n)]
        assert variant == _rule(n)
        assert us[variant] > 0 and all(t == 0 for v, t in enumerate(us) if v != variant), (n, us)
    sim.close()


def test_times_of_fixed_variants():
    import amr2d_mhd_amd as A

    sim = A.Simulation([_rotor(maxlevs=3)])
    sim.init()
    for v in (STRIPS, WIDE, NARROW):
        sim.set_stage_variant(v)
        sim.profile(("stage",))
        sim.run(2)
        sim.profile_read()
    seen = [v for v, t in enumerate(next(iter(sim.stage_tuning().values()))[1]) if t > 0]
    assert seen == sorted((STRIPS, WIDE, NARROW))
    sim.close()
