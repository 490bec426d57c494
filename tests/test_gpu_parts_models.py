"""Evaluations and minimizations in parts against one block per unit (the entry points on
caller-owned arrays) for the solvent models and coordinate widths: the HCT model, whose derivative
chain has no factor of its own, Debye screening, and coordinates split over two words."""
import ctypes

import numpy as np
import pytest

from stormm_amd import _lib, synthetic
from stormm_amd import synthesis as S

pytestmark = pytest.mark.gpu

# (generalized Born model, salt concentration, coordinate bits)
MODELS = [(1, 0.0, 32), (1, 0.15, 32), (5, 0.15, 32), (2, 0.0, 45), (1, 0.2, 45)]


def objects(model, prec):
    igb, salt, gpos_bits = model
    sizes = [497, 17, 385, 33]
    topos, coords = synthetic.generate(sizes, [500 + i for i in range(len(sizes))], gb=True,
                                       perturb=0.05, workers=1)
    for t in topos:
        t.igb, t.salt = igb, salt
    ag = S.AtomGraphSynthesis(topos)
    assert ag.part_count > len(sizes)
    ps = S.PhaseSpaceSynthesis(ag, gpos_bits, 23 if prec == "single" else 40)
    sc = S.ScoreCard(ag.system_count, 26 if prec == "single" else 32)
    ps.upload(coords)
    ps.initialize_forces()
    sc.initialize()
    w = _lib.ScoreCardWriter()
    _lib.check(_lib.load().stormm_scorecard_data(sc.handle, ctypes.byref(w)))
    return ag, ps, sc, w


@pytest.mark.parametrize("prec", ["single", "double"])
@pytest.mark.parametrize("model", MODELS)
def test_evaluation(model, prec):
    got = []
    for parts in (True, False):
        ag, ps, sc, scw = objects(model, prec)
        if parts:
            S.launch_mm_evaluation(prec, ag, None, ps, sc, True, True)
        else:
            w = ps.writer()
            _lib.check(_lib.load().stormm_launch_mm_evaluation_kit(
                S.precision_code(prec), ag.handle, None, ctypes.byref(w), ctypes.byref(scw), 1, 1,
                0.0, 0.0, None))
        got.append((np.concatenate(ps.fixed()[1]), sc.accumulators()))
    assert np.array_equal(got[0][0], got[1][0])
    assert np.array_equal(got[0][1], got[1][1])


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("prec", ["single", "double"])
@pytest.mark.parametrize("model", MODELS)
def test_minimization(model, prec, mode):
    if mode == 1 and model[2] > 38:
        pytest.skip("the fused modes take at most 38 coordinate bits")
    mc = S.minimize_controls(5, 2, 0.01, 0.0, clash_cycles=2)
    got = []
    for parts in (True, False):
        ag, ps, sc, scw = objects(model, prec)
        lm = S.LineMinimization(ag.system_count, 0.01)
        if parts:
            S.launch_minimization(prec, ag, ps, mc, sc, lm, persistent=mode)
        else:
            w, lw = ps.writer(), _lib.LinMinWriter()
            L = _lib.load()
            _lib.check(L.stormm_line_min_data(lm.handle, ctypes.byref(lw)))
            _lib.check(L.stormm_launch_minimization_kit(
                S.precision_code(prec), ag.handle, ctypes.byref(w), ctypes.byref(mc),
                ctypes.byref(scw), ctypes.byref(lw), mode, None))
        S.synchronize()
        got.append(ps.fixed() + (sc.accumulators(),))
    for a, b in zip(got[0][:2], got[1][:2]):
        assert np.array_equal(np.concatenate(a), np.concatenate(b))
    assert np.array_equal(got[0][2], got[1][2])
