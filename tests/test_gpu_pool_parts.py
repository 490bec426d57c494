"""A serving pool whose few large systems are evaluated in parts (several blocks to a work unit)."""
import time

import numpy as np
import pytest

from stormm_amd import serving, synthetic
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
