"""Coordinates of a serving pool's systems, in and out, at the sizes where the transfer kernels'
blocks end: exactly the fixed-point values of what was admitted."""
import numpy as np
import pytest

from stormm_amd import serving, synthetic

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("natoms", [(16,), (255, 256, 257), (512, 511, 31, 33)])
def test_coordinates_of_admitted_systems(natoms):
    pool = serving.MinimizationPool(precision="single", total_cycles=10)
    held = []
    for k, n in enumerate(natoms):
        topo, x = synthetic.branched_molecule(n, seed=40 + k, gb=True)
        confs = [x + 0.125 * c for c in range(3)]
        held.append((topo, confs, pool.admit_conformers(topo, confs)))
    # A released range is taken again.
    topo, confs, slots = held[0]
    pool.release(slots)
    confs = [-c for c in confs]
    held[0] = (topo, confs, pool.admit_conformers(topo, confs))
    bits = 2.0 ** pool.config.gpos_bits
    for topo, confs, slots in held:
        for x, slot in zip(confs, slots):
            scaled = np.asarray(x) * bits
            want = (np.sign(scaled) * np.floor(np.abs(scaled) + 0.5)).astype(np.int64)
            got = pool.coordinates(slot, topo.natom, fixed=True)
            assert np.array_equal(got, want)
            assert np.array_equal(pool.coordinates(slot, topo.natom), want / bits)


# More atoms than one staged copy takes (32768), with a remainder: first, last and the systems
# on either side of the seam.
def test_admission_in_several_copies():
    pool = serving.MinimizationPool(precision="single", total_cycles=10)
    topo, x = synthetic.branched_molecule(31, seed=50, gb=True)
    rng = np.random.default_rng(50)
    confs = [x + rng.normal(0.0, 0.25, x.shape) for _ in range(1030)]
    slots = pool.admit_conformers(topo, confs)
    bits = 2.0 ** pool.config.gpos_bits
    for k in (0, 1, 1022, 1023, 1024, 1025, 1029):
        scaled = confs[k] * bits
        want = (np.sign(scaled) * np.floor(np.abs(scaled) + 0.5)).astype(np.int64)
        assert np.array_equal(pool.coordinates(slots[k], topo.natom, fixed=True), want)
    alone = serving.MinimizationPool(precision="single", total_cycles=10)
    some = [0, 1023, 1024, 1029]
    few = alone.admit_conformers(topo, [confs[k] for k in some])
    pool.minimize(3)
    alone.minimize(3)
    for k, slot in zip(some, few):
        assert np.array_equal(pool.coordinates(slots[k], topo.natom, fixed=True),
                              alone.coordinates(slot, topo.natom, fixed=True))
