"""The incremental sort's placement (one launch that reorders the state, the
phase list, the positions in phase order and the cell table from counted
moves) against the radix path, which forms each of them in its own pass: the
same permutation, keys, cellStart and neighbour sums, bit for bit, at counts
around a wave, a block and a 2048-slot tile, with one phase empty, and with
speeds from at rest to a cell's width per step (every particle a newcomer,
long chains in the edge cells the hash clamps into)."""
import numpy as np
import pytest

from sph_seepage_flows_amd import SFSystem, scenes

pytestmark = pytest.mark.gpu

DT = 1e-4
FIELDS = ("sort_perm", "sorted_keys", "cell_start", "label", "pos", "vel", "col", "max_saturation", "density",
          "voidage", "saturation", "acc")


@pytest.mark.parametrize("speed", [0.0, 5.0, 400.0])
@pytest.mark.parametrize("n_water,n_sand", [(1, 0), (0, 1), (64, 1), (255, 1), (256, 0), (0, 257), (1024, 1023),
                                            (1024, 1024), (1025, 1024), (1440, 1152)])
def test_placement_equals_radix_path(n_water, n_sand, speed):
    sc = scenes.mixed(n_water=n_water, n_sand=n_sand, collider=False, vel_sigma=speed, sf_type=n_sand % 2)
    a, b = SFSystem.from_scene(sc), SFSystem.from_scene(sc)
    a.set_sort_strategy(False)
    b.set_sort_strategy(True)
    for step in range(4):
        a.step(DT)
        b.step(DT)
        for f in FIELDS:
            np.testing.assert_array_equal(a.get(f), b.get(f), err_msg=f"step {step} {f}")


def test_placement_between_strategies_and_handouts():
    # counted moves that a radix build, a handed-out position buffer or a
    # second build without an advect leave unused must not reach a later sort
    sc = scenes.mixed(vel_sigma=3.0)
    a, b = SFSystem.from_scene(sc), SFSystem.from_scene(sc)
    a.set_sort_strategy(False)
    a.step(DT, 9)
    b.step(DT, 3)
    b.set_sort_strategy(False)
    b.step(DT, 2)
    b.set_sort_strategy(True)
    b.step(DT, 2)
    b.device_buffer("pos")
    b.step(DT, 2)
    for f in FIELDS:
        np.testing.assert_array_equal(a.get(f), b.get(f), err_msg=f)
