"""Work units of batches that two units to a compute unit cannot hold: a multiple of the compute
units of them unless they would be nearly full, and the same results in any units."""
import numpy as np
import pytest

from stormm_amd import synthetic
from stormm_amd import synthesis as S


# (systems, atoms each, capacity, units) on 256 compute units, systems that pack two to a unit
# unless noted: three and four units to a compute unit, exactly and nearly full ones (then packed
# to the capacity), one to a unit, by the limit of 32 systems to a unit, two to a compute unit.
@pytest.mark.parametrize("count,natom,cap,units", [(1400, 32, 64, 768), (1600, 32, 64, 1024),
                                                   (1536, 32, 64, 768), (1520, 32, 64, 760),
                                                   (600, 30, 32, 600), (16400, 16, 512, 768),
                                                   (512, 48, 64, 512)])
def test_unit_count(count, natom, cap, units):
    topos, _ = synthetic.uniform_batch(1, natom, natom, seed=3, gb=True)
    info = S.plan_synthesis(list(topos) * count, {"wu_atom_capacity": cap})
    assert info.max_wu_atoms <= cap
    assert info.work_unit_count == units


@pytest.mark.gpu
@pytest.mark.parametrize("prec", ["single", "double"])
def test_results_in_any_units(prec):
    topos, coords = synthetic.uniform_batch(1400, 17, 32, seed=4, gb=True)
    bits = (32, 23, 26) if prec == "single" else (32, 40, 32)

    def run(shape):
        ag = S.AtomGraphSynthesis(topos, shape)
        ps = S.PhaseSpaceSynthesis(ag, bits[0], bits[1])
        sc = S.ScoreCard(ag.system_count, bits[2])
        ps.upload(coords)
        ps.initialize_forces()
        sc.initialize()
        S.launch_mm_evaluation(prec, ag, None, ps, sc, True, True)
        return np.concatenate(ps.fixed()[1]), sc.accumulators()

    forces, energies = run(None)
    for shape in ({"wu_atom_capacity": 64}, {"wu_atom_capacity": 64, "target_wu_per_cu": 5}):
        f, e = run(shape)
        assert np.array_equal(f, forces) and np.array_equal(e, energies)
