"""A serving pool whose few large systems are evaluated in parts (several blocks to a work unit)."""
import ctypes
import time

import numpy as np
import pytest

from stormm_amd import _lib, serving, synthetic
from stormm_amd import synthesis as S

pytestmark = pytest.mark.gpu


def test_a_call_does_not_cost_with_the_budget():
    topo, x = synthetic.branched_molecule(400, seed=90, gb=True)
    confs = [x + 0.01 * k for k in range(8)]

    def seconds(budget):
        pool = serving.MinimizationPool(budget_bytes=budget, max_systems=64, total_cycles=1000,
                                        conv_rms=0.0, clash_cycles=0)
        pool.admit_conformers(topo, confs)
        best = 1.0e9
        for _ in range(30):
            S.synchronize()
            t0 = time.perf_counter()
            pool.minimize(1)
            S.synchronize()
            best = min(best, time.perf_counter() - t0)
        return best

    small, large = seconds(64 << 20), seconds(64 << 30)
    print(f"one cycle: {small * 1e6:.0f} us in a pool of 64 MiB, {large * 1e6:.0f} us in 64 GiB")
    assert large < 1.5 * small


# Ticks with and without a large system among small ones, so that the planner goes into parts and
# out of them: every trajectory is its molecule's in the batch minimizer on caller-owned arrays, one
# block to a unit.  The first cycles are clash-damped; some ticks end inside them.
@pytest.mark.parametrize("prec", ["single", "double"])
def test_trajectories_in_and_out_of_parts(prec):
    cycles = 12
    bits = (32, 23, 26) if prec == "single" else (32, 40, 32)
    sizes = [511, 33, 400, 17, 60]
    molecules = [synthetic.branched_molecule(n, seed=95 + k, gb=True) for k, n in enumerate(sizes)]
    rng = np.random.default_rng(96)
    molecules = [(t, x + rng.normal(0.0, 0.1, x.shape)) for t, x in molecules]
    topos, coords = [m[0] for m in molecules], [m[1] for m in molecules]
    assert S.AtomGraphSynthesis(topos).part_count > len(topos)
    assert S.AtomGraphSynthesis([topos[1], topos[3]]).part_count == 0

    ag = S.AtomGraphSynthesis(topos)
    ps = S.PhaseSpaceSynthesis(ag, bits[0], bits[1])
    sc = S.ScoreCard(ag.system_count, bits[2])
    lm = S.LineMinimization(ag.system_count, 0.01)
    ps.upload(coords)
    mc = S.minimize_controls(cycles, 4, 0.01, 0.0, clash_cycles=5)
    L = _lib.load()
    w, s, lw = ps.writer(), _lib.ScoreCardWriter(), _lib.LinMinWriter()
    _lib.check(L.stormm_scorecard_data(sc.handle, ctypes.byref(s)))
    _lib.check(L.stormm_line_min_data(lm.handle, ctypes.byref(lw)))
    _lib.check(L.stormm_launch_minimization_kit(S.precision_code(prec), ag.handle, ctypes.byref(w),
                                                ctypes.byref(mc), ctypes.byref(s),
                                                ctypes.byref(lw), 0, None))
    want = ps.fixed()[0]
    energies = sc.potential_energies()

    pool = serving.MinimizationPool(precision=prec, total_cycles=cycles, sd_cycles=4, conv_rms=0.0,
                                    clash_cycles=5)
    slot = {}

    def admit(*ks):
        for k in ks:
            slot[k] = pool.admit([topos[k]], [coords[k]])[0]

    def finished(k):
        steps, done, _, energy = pool.status([slot[k]])
        assert done[0] and steps[0] == cycles
        assert np.array_equal(pool.coordinates(slot[k], sizes[k], fixed=True), want[k]), sizes[k]
        assert energy[0] == energies[k], sizes[k]

    admit(1, 3)
    pool.minimize(3)          # one block to a unit
    admit(0)
    pool.minimize(4)          # in parts
    admit(4, 2)
    pool.minimize(8)          # the small ones end
    for k in (0, 1, 3):
        finished(k)
    pool.release([slot[0], slot[1]])
    admit(1)                  # takes the place of a system that was evaluated in parts
    pool.minimize(cycles)
    for k in (1, 2, 4):
        finished(k)
    pool.release([slot[2]])
    admit(0, 2)
    pool.minimize(cycles)
    for k in (0, 2):
        finished(k)
