"""Minimizations in parts that an RMS force stops: the same state as with one block per unit (the
entry point on caller-owned arrays), and evaluations of stopped units that cost next to nothing."""
import ctypes
import time

import numpy as np
import pytest

from stormm_amd import _lib, synthetic
from stormm_amd import synthesis as S

pytestmark = pytest.mark.gpu


def objects(topos, coords, prec):
    bits = (32, 23, 26) if prec == "single" else (32, 40, 32)
    ag = S.AtomGraphSynthesis(topos)
    ps = S.PhaseSpaceSynthesis(ag, bits[0], bits[1])
    sc = S.ScoreCard(ag.system_count, bits[2])
    ps.upload(coords)
    return ag, ps, sc, S.LineMinimization(ag.system_count, 0.01)


def minimize_one_block(prec, ag, ps, sc, lm, mc, mode):
    L = _lib.load()
    w, s, lw = ps.writer(), _lib.ScoreCardWriter(), _lib.LinMinWriter()
    _lib.check(L.stormm_scorecard_data(sc.handle, ctypes.byref(s)))
    _lib.check(L.stormm_line_min_data(lm.handle, ctypes.byref(lw)))
    _lib.check(L.stormm_launch_minimization_kit(S.precision_code(prec), ag.handle, ctypes.byref(w),
                                                ctypes.byref(mc), ctypes.byref(s),
                                                ctypes.byref(lw), mode, None))


# One large system among small ones that share units, stopping at different cycles: in damped
# cycles, after them, and not at all.
@pytest.mark.parametrize("mode", [1, 3, 4])
@pytest.mark.parametrize("prec", ["single", "double"])
def test_stopped_state_equals_one_block(prec, mode):
    sizes = [480, 401] + [17 + k for k in range(12)]
    topos, coords = synthetic.generate(sizes, [700 + i for i in range(len(sizes))], gb=True,
                                       perturb=0.05, workers=1)
    got = []
    for parts in (True, False):
        ag, ps, sc, lm = objects(topos, coords, prec)
        mc = S.minimize_controls(40, 10, 0.01, 9.0, clash_cycles=6)
        if parts:
            S.launch_minimization(prec, ag, ps, mc, sc, lm, persistent=mode)
        else:
            minimize_one_block(prec, ag, ps, sc, lm, mc, mode)
        S.synchronize()
        cycles, rms = ag.minimization_status()
        got.append(ps.fixed() + (sc.accumulators(), lm.values(), cycles, rms))
    a, b = got
    assert len(set(a[4].tolist())) > 2 and a[4].min() < 40
    assert np.array_equal(np.concatenate(a[0]), np.concatenate(b[0]))
    assert np.array_equal(np.concatenate(a[1]), np.concatenate(b[1]))
    assert np.array_equal(a[2], b[2])
    for k in a[3]:
        assert np.array_equal(a[3][k], b[3][k]), k
    assert np.array_equal(a[4], b[4]) and np.array_equal(a[5], b[5])


def test_stopped_units_cost_next_to_nothing():
    topos, coords = synthetic.generate([400] * 24, list(range(800, 824)), gb=True, perturb=0.05,
                                       workers=1)
    ag, ps, sc, lm = objects(topos, coords, "single")

    def seconds(rms):
        best = 1.0e9
        for _ in range(3):
            ps.upload(coords)
            mc = S.minimize_controls(200, 50, 0.01, rms, clash_cycles=0)
            S.synchronize()
            t0 = time.perf_counter()
            S.launch_minimization("single", ag, ps, mc, sc, lm, persistent=1)
            S.synchronize()
            best = min(best, time.perf_counter() - t0)
        return best

    running = seconds(0.0)
    stopped = seconds(1.0e6)
    cycles, _ = ag.minimization_status()
    print(f"200 cycles: running {running * 1e3:.2f} ms, stopped {stopped * 1e3:.2f} ms")
    assert cycles.max() == 0
    # Empty launches in place of evaluations of some ten microseconds each.
    assert stopped < 0.5 * running


# Runs that stop early against the same units with one block each, which the caller gets by naming
# their number: in every fused mode the cycles after the stop cost less than they do there.
@pytest.mark.parametrize("mode", [1, 3, 4])
def test_early_stop_is_no_slower_than_one_block(mode):
    topos, coords = synthetic.generate([400] * 24, list(range(800, 824)), gb=True, perturb=0.05,
                                       workers=1)

    def run(shape):
        ag = S.AtomGraphSynthesis(topos, shape)
        ps = S.PhaseSpaceSynthesis(ag, 32, 23)
        sc = S.ScoreCard(ag.system_count, 26)
        lm = S.LineMinimization(ag.system_count, 0.01)
        mc = S.minimize_controls(400, 50, 0.01, 6.0, clash_cycles=0, ntpr=7)
        best = 1.0e9
        for _ in range(3):
            ps.upload(coords)
            S.synchronize()
            t0 = time.perf_counter()
            S.launch_minimization("single", ag, ps, mc, sc, lm, persistent=mode)
            S.synchronize()
            best = min(best, time.perf_counter() - t0)
        state = [sc.accumulators()] + [np.asarray(h) for h in sc.history()] + list(sc.series())
        return ag.part_count, best, ps.fixed(), state, ag.minimization_status()

    parts, t_parts, x, e, status = run(None)
    none, t_one, x1, e1, status1 = run({"target_wu_per_cu": 2})
    print(f"mode {mode}: {t_parts * 1e3:.2f} ms in parts, {t_one * 1e3:.2f} ms in one block")
    assert parts > 0 and none == 0
    assert status[0].max() < 100 and np.array_equal(status[0], status1[0])
    assert np.array_equal(np.concatenate(x[0]), np.concatenate(x1[0]))
    assert np.array_equal(np.concatenate(x[1]), np.concatenate(x1[1]))
    for a, b in zip(e, e1):
        assert np.array_equal(a, b)
    assert t_parts < t_one
