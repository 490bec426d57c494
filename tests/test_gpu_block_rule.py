"""Default block sizes of the evaluation (by precision and by units per compute unit) against the
explicitly chosen ones: results do not depend on the block, bit for bit."""
import numpy as np
import pytest

from stormm_amd import synthetic
from stormm_amd import synthesis as S

pytestmark = pytest.mark.gpu


def evaluate(topos, coords, prec, shape):
    bits = (32, 23, 26) if prec == "single" else (32, 40, 32)
    ag = S.AtomGraphSynthesis(topos, shape)
    ps = S.PhaseSpaceSynthesis(ag, bits[0], bits[1])
    sc = S.ScoreCard(ag.system_count, bits[2])
    ps.upload(coords)
    ps.initialize_forces()
    sc.initialize()
    S.launch_mm_evaluation(prec, ag, None, ps, sc, True, True)
    return np.concatenate(ps.fixed()[1]), sc.accumulators()


# One tile and one tile and an atom, the largest system, and more units than compute units.
@pytest.mark.parametrize("count,lo,hi", [(1, 16, 16), (3, 17, 17), (2, 511, 512), (300, 20, 40)])
@pytest.mark.parametrize("prec", ["single", "double"])
def test_default_block_equals_explicit_blocks(count, lo, hi, prec):
    topos, coords = synthetic.uniform_batch(count, lo, hi, seed=77, gb=True)
    forces, energies = evaluate(topos, coords, prec, None)
    for threads in (256, 512, 1024):
        f, e = evaluate(topos, coords, prec, {"block_threads": threads})
        assert np.array_equal(f, forces) and np.array_equal(e, energies), threads


# Units at the sizes where the double-precision block changes, alone on a compute unit (112 and
# 144 atoms) and in greater number (336 and 352 atoms), plain and clash-damped.
@pytest.mark.parametrize("count,natom", [(3, 112), (3, 129), (260, 336), (260, 337)])
@pytest.mark.parametrize("clash", [0.0, 1.5])
def test_double_block_by_unit_size(count, natom, clash):
    topos, coords = synthetic.uniform_batch(count, natom, natom, seed=78, gb=True)

    def run(shape):
        ag = S.AtomGraphSynthesis(topos, shape)
        ps = S.PhaseSpaceSynthesis(ag, 32, 40)
        sc = S.ScoreCard(ag.system_count, 32)
        ps.upload(coords)
        ps.initialize_forces()
        sc.initialize()
        S.launch_nonbonded("double", ag, None, ps, sc, True, True, clash_distance=clash,
                           clash_ratio=0.7 if clash else 0.0)
        return np.concatenate(ps.fixed()[1]), sc.accumulators()

    forces, energies = run(None)
    f, e = run({"block_threads": 256})
    assert np.array_equal(f, forces) and np.array_equal(e, energies)


# Units of more than 336 atoms are packed anew for double precision: as evaluated in them and as
# evaluated in the units of an explicit capacity, in and out of a minimization.
@pytest.mark.parametrize("cycles", [0, 3])
def test_double_units(cycles):
    topos, coords = synthetic.uniform_batch(1300, 17, 240, seed=79, gb=True)
    shape = {"wu_atom_capacity": 512}
    assert S.plan_synthesis(topos, shape).max_wu_atoms > 336
    if cycles == 0:
        forces, energies = evaluate(topos, coords, "double", None)
        f, e = evaluate(topos, coords, "double", shape)
        assert np.array_equal(f, forces) and np.array_equal(e, energies)
        return

    def minimize(shape):
        ag = S.AtomGraphSynthesis(topos, shape)
        ps = S.PhaseSpaceSynthesis(ag, 32, 40)
        sc = S.ScoreCard(ag.system_count, 32)
        ps.upload(coords)
        controls = S.minimize_controls(cycles, sd_cycles=1)
        line = S.LineMinimization(ag.system_count, 0.01)
        S.launch_minimization("double", ag, ps, controls, sc, line)
        return np.concatenate(ps.fixed()[0]), sc.accumulators()

    xyz, energies = minimize(None)
    x, e = minimize(shape)
    assert np.array_equal(x, xyz) and np.array_equal(e, energies)
