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
