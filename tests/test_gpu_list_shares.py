"""The interface passes' capped grid: above 16384 blocks' worth of listed
particles each block takes several shares, with the same LDS lists and stage.
With 64 threads and four lanes a block holds 16 particles, so 300k listed ones
take two shares in some blocks; with 256 threads one share holds them all.  A
particle's sums are its own lanes' work in candidate order either way: the same
bits."""
import numpy as np
import pytest

from sph_seepage_flows_amd import Physics, SFSystem
from sph_seepage_flows_amd.scenes import lattice

from _scene_util import make_scene

pytestmark = pytest.mark.gpu

FIELDS = ("voidage", "saturation", "avg_flow_vel", "adhesion_force", "avg_adhesion_force", "avg_drag_force", "acc",
          "pos", "vel")


@pytest.mark.parametrize("lanes", [4, 1])
def test_second_shares_change_nothing(lanes):
    r, side = 0.005, 54
    n = side * side * 52 * (4 // lanes)  # of each phase: lanes 1 put 64 particles in a block
    layers = n // (side * side)
    hi = (2 * r * (side + 2), 2 * r * (layers + 2), 2 * r * (side + 2))
    ph = Physics(hi=tuple(4 * r * np.ceil(x / (4 * r)) for x in hi), r_water=r, r_sand=r)
    counts = (side, layers, side)
    pos = np.concatenate([lattice((2 * r,) * 3, 2 * r, counts, n, jitter=0.1 * r, seed=3, stream=0),
                          lattice((r,) * 3, 2 * r, counts, n, jitter=0.1 * r, seed=3, stream=1)])
    label = (np.arange(2 * n) >= n).astype(np.uint64)
    vel = np.random.default_rng(3).normal(0.0, 0.05, (2 * n, 3)).astype(np.float32)
    sc = make_scene(pos, label, vel=vel, ph=ph)
    many, one = SFSystem.from_scene(sc), SFSystem.from_scene(sc)
    for g, nb in ((many, 64), (one, 256)):
        g.set_interface_lanes(lanes)
        for name in ("avg_flow", "voidage_adhesion"):
            g.set_launch_config(name, nb)
        g.step(1e-5, 2)
    water = one.get("label") == 0  # at least those with sums of their own are listed
    listed = int(np.where(water, one.get("voidage") < 1, one.get("saturation") > 0).sum())
    assert listed > 16384 * 64 // lanes
    print(f"{listed} listed", flush=True)
    for name in FIELDS:
        np.testing.assert_array_equal(many.get(name), one.get(name), err_msg=name)
