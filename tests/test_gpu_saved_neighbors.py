"""The neighbours the avg-flow pass saves for the passes after it.

A particle's lanes save up to 80 neighbours of the other phase between them; a
particle with more on one lane is walked again.  h is 4 r, so a lattice of
spacing 2 r s puts 33 / s^3 of them within reach: all saved at s = 1, some
walked at s = 0.8 (65), nearly all inside at s = 0.7 (98).  Masses scaled by
s^3 keep density and voidage as they are at s = 1.  Tolerances: the
single-step ones.  At s = 0.8 the lattice has pairs at r = h / 2, where the
adhesion's quarter power starts from zero and rounding of r alone moves it by
up to 1.5e-4 in any FP32 evaluation (the oracle's own at 32 bits); there the
adhesion is compared between one lane and four instead, whose pairs round alike
and of which the one saves what the other walks again: sums of 65 terms in
another order, 1e-5 of the largest.

And the water momentum pass's layouts for a caller that holds the mass buffer:
built and solved in one call (the mass beside the records) or in two (the
slots as they are by then) the same terms in the same order, so the same bits
as without it."""
import numpy as np
import pytest

from sph_seepage_flows_amd import SFSystem, scenes

from _compare import norm_err
from test_gpu_records import FIELDS, _assert_same
from test_gpu_step import _compare

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("s", [1.0, 0.8, 0.7])
@pytest.mark.parametrize("lanes", [1, 2, 4])
def test_saved_and_walked_again(oracle_mod, lanes, s):
    sc = scenes.mixed(collider=False)
    lo = sc.pos.min(0)
    sc.pos = (lo + (sc.pos - lo) * np.float32(s)).astype(np.float32)
    sc.mass = (sc.mass * np.float32(s ** 3)).astype(np.float32)
    g = SFSystem.from_scene(sc)
    g.set_interface_lanes(lanes)
    o, o32 = (oracle_mod.OracleSystem(sc, bits) for bits in (64, 32))
    for x in (g, o, o32):
        x.step(1e-5)
    adhesion = ("adhesion_force", "avg_adhesion_force")
    _compare(g, o, f"lanes {lanes} spacing {s}", skip=adhesion if s == 0.8 else (), o32=o32)
    if s == 0.8:
        one = SFSystem.from_scene(sc)
        one.set_interface_lanes(1)
        one.step(1e-5)
        water = o.get("label") == 0
        for q in adhesion:
            assert norm_err(g.get(q), one.get(q), water) < 1e-5, q


@pytest.mark.parametrize("hand_out", [None, "mass"])
def test_build_and_solve_in_two_calls(hand_out):
    sc = scenes.mixed()
    a, b = SFSystem.from_scene(sc), SFSystem.from_scene(sc)
    for x in (a, b):
        if hand_out:
            x.device_buffer(hand_out)
    for q in range(3):
        a.UpdateSystem(1.0 / 30.0)
        b.BuildGNSearcher()
        b.UpdateSolver(1.0 / 30.0)
        _assert_same(a, b, f"step {q}", FIELDS[:-1])
