"""Launch shapes of a serving pool outside the documented sizes: the block size that a launch uses
(tests/capi/launch_host.cpp, on the host), and the same trajectories as with the default shape."""
import os
import subprocess

import numpy as np
import pytest

from stormm_amd import build, serving, synthetic


def test_block_sizes():
    exe = os.path.join(build.CAPI_BIN, "launch_host")
    if not os.path.exists(exe):
        build.build_capi_programs()
    out = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    print(out.stdout)
    assert out.returncode == 0
    assert "launch ok" in out.stdout


# A unit of more than 256 atoms with fewer threads than two atoms to each need, sizes that are no
# whole wavefronts, and capacities beyond a unit's 512 atoms (three molecules would share one).
@pytest.mark.gpu
@pytest.mark.parametrize("shape", [{"block_threads": 128}, {"block_threads": 300},
                                   {"block_threads": 4096}, {"wu_atom_capacity": 2048},
                                   {"block_threads": 64, "wu_atom_capacity": 1024}])
@pytest.mark.parametrize("prec", ["single", "double"])
def test_trajectories_do_not_depend_on_the_shape(shape, prec):
    sizes = [410, 33] + [96] * 300
    topos, coords = [], []
    for k, n in enumerate([410, 33, 96]):
        topo, x = synthetic.branched_molecule(n, seed=60 + k, gb=True)
        topos.append(topo)
        coords.append(x)
    rng = np.random.default_rng(61)
    sets = [[coords[0]], [coords[1]],
            [coords[2] + rng.normal(0.0, 0.05, coords[2].shape) for _ in range(len(sizes) - 2)]]

    def run(shape):
        pool = serving.MinimizationPool(precision=prec, total_cycles=20, shape=shape)
        slots = [pool.admit_conformers(t, c) for t, c in zip(topos, sets)]
        pool.minimize(2)
        return [pool.coordinates(s, t.natom, fixed=True)
                for t, held in zip(topos, slots) for s in held[:4]]

    for got, want in zip(run(shape), run(None)):
        assert np.array_equal(got, want)
