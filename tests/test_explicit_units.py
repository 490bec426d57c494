"""Work units per compute unit that a caller names are kept also where the default would share few
large systems' units among several blocks, and the tuner still finds that default."""
import numpy as np
import pytest

from stormm_amd import synthetic
from stormm_amd import synthesis as S


# One large system among 100 small ones on 256 compute units: a unit to each with any target, fewer
# by default.
@pytest.mark.parametrize("target", [1, 2, 4])
def test_named_units_are_kept(target):
    large, _ = synthetic.uniform_batch(1, 480, 480, seed=5, gb=True)
    small, _ = synthetic.uniform_batch(1, 17, 17, seed=6, gb=True)
    topos = list(large) + list(small) * 100
    assert S.plan_synthesis(topos, {"target_wu_per_cu": target}).work_unit_count == 101
    assert S.plan_synthesis(topos).work_unit_count < 101


@pytest.mark.gpu
@pytest.mark.parametrize("prec", ["single", "double"])
def test_results_and_tuning(prec):
    topos, coords = synthetic.generate([400] * 6, list(range(600, 606)), gb=True, perturb=0.05,
                                       workers=1)
    bits = (32, 23, 26) if prec == "single" else (32, 40, 32)

    def run(shape):
        ag = S.AtomGraphSynthesis(topos, shape)
        ps = S.PhaseSpaceSynthesis(ag, bits[0], bits[1])
        sc = S.ScoreCard(ag.system_count, bits[2])
        ps.upload(coords)
        ps.initialize_forces()
        sc.initialize()
        S.launch_mm_evaluation(prec, ag, None, ps, sc, True, True)
        return ag.part_count, np.concatenate(ps.fixed()[1]), sc.accumulators()

    parts, forces, energies = run(None)
    assert parts > len(topos)
    named, f, e = run({"target_wu_per_cu": 2})
    assert named == 0
    assert np.array_equal(f, forces) and np.array_equal(e, energies)
    shape, _ = S.autotune(topos, prec, coords)
    assert S.AtomGraphSynthesis(topos, shape).part_count > 0
