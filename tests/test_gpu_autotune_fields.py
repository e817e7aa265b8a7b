"""sf_autotune builds the neighbours, solves, and then launches every pass
again and again on that solve's inputs.  Each pass rewrites its outputs from
values that no later launch of it changes, so the fields it leaves are those of
one build and solve: bit for bit (the launch shape does not change a sum's
order) what a step of an untuned handle leaves, whose advect, with the DEM
damping at zero, keeps the accelerations as the solve wrote them."""
import dataclasses

import numpy as np
import pytest

from sph_seepage_flows_amd import BatchSystem, SFSystem, scenes

pytestmark = pytest.mark.gpu

FIELDS = ("density", "pressure", "voidage", "saturation", "avg_flow_vel", "avg_drag_force", "adhesion_force",
          "avg_adhesion_force", "acc", "max_saturation", "col")


def _undamped(sc):
    sc.physics = dataclasses.replace(sc.physics, damping=0.0)
    return sc


@pytest.mark.parametrize("kind", ["single", "multi", "batch", "shared"])
def test_fields_after_autotune_are_the_solve_s(kind):
    sc = _undamped(scenes.mixed(sf_type=1 if kind == "multi" else 0))
    make = (lambda: BatchSystem.from_scenes([sc, sc])) if kind == "batch" else (lambda: SFSystem.from_scene(sc))
    a, b = make(), make()
    if kind == "shared":
        for x in (a, b):
            x.device_buffer("mass")
    a.autotune(reps=2)
    b.step(1e-4)
    assert np.abs(b.get("avg_adhesion_force")).max() > 0 and np.abs(b.get("avg_drag_force")).max() > 0
    for name in FIELDS:
        np.testing.assert_array_equal(a.get(name), b.get(name), err_msg=f"{kind} {name}")


@pytest.mark.parametrize("scene", ["block", "mixed"])
def test_default_is_the_shape_an_untuned_handle_launches(scene):
    """A pass that keeps the shape it launches anyway (64 threads in the momentum
    passes at these sizes, 256 in the others) gains nothing: the two times are
    one measurement."""
    g = SFSystem.from_scene(scenes.small_block() if scene == "block" else scenes.mixed())
    kept = 0
    for _ in range(4):
        for name, (nb, cap, best, dflt) in g.autotune(reps=20).items():
            assert 0 < best <= dflt
            if (nb, cap) == (64 if name.endswith("momentum") else 256, 16):
                assert best == dflt, name
                kept += 1
    print(f"{kept} of 20 kept their shape", flush=True)
