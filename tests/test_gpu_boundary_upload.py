"""Boundary uploads: what they hold on the device, and what an upload that
fails leaves behind."""
import ctypes as C

import numpy as np
import pytest

from sph_seepage_flows_amd import SFSystem, scenes

from _hip import runtime

pytestmark = pytest.mark.gpu


def _free_bytes() -> int:
    free, total = C.c_size_t(), C.c_size_t()
    assert runtime().hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def test_boundary_does_not_size_the_particle_arrays():
    """1M boundary particles in a handle for 2,592 particles: 16 bytes of state
    and 20 + 1 of sort arrays each, and the column ranges of the cells near them;
    none of the several hundred bytes a particle takes."""
    sc = scenes.mixed(collider=False)
    g = SFSystem.from_scene(sc)
    n = 1_000_000
    rng = np.random.default_rng(1)
    bpos = rng.uniform(0.0, sc.physics.hi[0], (n, 3)).astype(np.float32)
    before = _free_bytes()
    g.upload_boundary(bpos)
    took = before - _free_bytes()
    print(f"{took / n:.1f} bytes per boundary particle", flush=True)
    assert took < 64 * n
    g.step(1e-6)
    assert g.sizes()[:2] == (sc.n, n)
