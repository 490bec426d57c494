"""Evaluations in parts (several blocks to a work unit, where few large systems leave compute units
idle) against one block per unit, which the entry points on caller-owned arrays take: forces,
energies and whole minimizations equal bit for bit."""
import ctypes

import numpy as np
import pytest

from stormm_amd import _lib, restraints, synthetic
from stormm_amd import synthesis as S

pytestmark = pytest.mark.gpu


def molecule_set(case):
    """(topologies, coordinates, restraints): sizes at tile edges, one large system among small
    ones, stored Lennard-Jones tables (no combining rule), vacuum, and restrained atoms."""
    held = None
    if case == "tile_edges":
        sizes, gb = [496, 497, 511, 512], True
    elif case == "one_among_small":
        sizes, gb = [512] + [17] * 12, True
    elif case == "vacuum":
        sizes, gb = [400, 385], False
    else:
        sizes, gb = [330, 449, 401], True
    topos, coords = synthetic.generate(sizes, [900 + i for i in range(len(sizes))], gb=gb,
                                       perturb=0.05, workers=1)
    if case == "tables":
        for t in topos:
            a, b, a14, b14 = (np.array(x) for x in t.lj_tables())
            a = a.reshape(t.n_lj_types, -1)
            a[0, -1] = a[-1, 0] = 1.05 * a[0, -1]
            t.lja, t.ljb, t.lja14, t.ljb14 = a.reshape(-1), b, a.reshape(-1).copy(), b14
            t.lj_sigma = t.lj_epsilon = None
    if case == "restrained":
        held = [restraints.apply_positional_restraints(x, range(0, t.natom, 5), 10.0)
                for t, x in zip(topos, coords)]
    return topos, coords, held


def objects(topos, coords, held, prec):
    bits = (32, 23, 26) if prec == "single" else (32, 40, 32)
    ag = S.AtomGraphSynthesis(topos, restraints=held)
    ps = S.PhaseSpaceSynthesis(ag, bits[0], bits[1])
    sc = S.ScoreCard(ag.system_count, bits[2])
    ps.upload(coords)
    ps.initialize_forces()
    sc.initialize()
    return ag, ps, sc


def kit(sc):
    w = _lib.ScoreCardWriter()
    _lib.check(_lib.load().stormm_scorecard_data(sc.handle, ctypes.byref(w)))
    return w


CASES = ["tile_edges", "one_among_small", "vacuum", "tables", "restrained"]


@pytest.mark.parametrize("prec", ["single", "double"])
@pytest.mark.parametrize("clash", [0.0, 0.4])
@pytest.mark.parametrize("case", CASES)
def test_evaluation_in_parts_equals_one_block(case, clash, prec):
    topos, coords, held = molecule_set(case)
    code = S.precision_code(prec)
    got = []
    for parts in (True, False):
        ag, ps, sc = objects(topos, coords, held, prec)
        # Twice: sums are added to what the arrays hold.
        for _ in range(2):
            if parts:
                S.launch_mm_evaluation(prec, ag, None, ps, sc, True, True, clash_distance=clash,
                                       clash_ratio=clash)
            else:
                w, s = ps.writer(), kit(sc)
                _lib.check(_lib.load().stormm_launch_mm_evaluation_kit(
                    code, ag.handle, None, ctypes.byref(w), ctypes.byref(s), 1, 1, clash, clash,
                    None))
        got.append((np.concatenate(ps.fixed()[1]), sc.accumulators()))
    assert np.array_equal(got[0][0], got[1][0])
    assert np.array_equal(got[0][1], got[1][1])


@pytest.mark.parametrize("mode", [0, 1, 2, 3, 4])
@pytest.mark.parametrize("case", ["one_among_small", "vacuum", "restrained"])
def test_minimization_in_parts_equals_one_block(case, mode):
    topos, coords, held = molecule_set(case)
    if held is not None and mode not in (0, 2):
        pytest.skip("the fused modes take no restraints")
    mc = S.minimize_controls(6, 3, 0.01, 0.0, clash_cycles=2)
    got = []
    for parts in (True, False):
        ag, ps, sc = objects(topos, coords, held, "single")
        lm = S.LineMinimization(ag.system_count, 0.01)
        # Twice in a row, so that the second run starts from what the first left behind.
        for _ in range(2):
            if parts:
                S.launch_minimization("single", ag, ps, mc, sc, lm, persistent=mode)
            else:
                w, s, lw = ps.writer(), kit(sc), _lib.LinMinWriter()
                L = _lib.load()
                _lib.check(L.stormm_line_min_data(lm.handle, ctypes.byref(lw)))
                _lib.check(L.stormm_launch_minimization_kit(
                    S.PREC_SINGLE, ag.handle, ctypes.byref(w), ctypes.byref(mc), ctypes.byref(s),
                    ctypes.byref(lw), mode, None))
        S.launch_mm_evaluation("single", ag, None, ps, sc, True, True)
        got.append(ps.fixed() + (sc.accumulators(), lm.values()))
    a, b = got
    assert np.array_equal(np.concatenate(a[0]), np.concatenate(b[0]))
    assert np.array_equal(np.concatenate(a[1]), np.concatenate(b[1]))
    assert np.array_equal(a[2], b[2])
    for k in a[3]:
        assert np.array_equal(a[3][k], b[3][k]), k
