"""Boundary uploads: what they hold on the device, and what an upload that
fails leaves behind."""
import ctypes as C
import subprocess
import sys
from pathlib import Path

import numpy as np
import pytest

from sph_seepage_flows_amd import Physics, SFSystem, scenes

from _hip import runtime
from _scene_util import make_scene

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


def test_more_than_2_29_column_ranges():
    """Boundary particles three cells apart along z in every column of a 400^3
    grid: each cell has nine columns that hold one, 5.7e8 ranges in all, past
    what a 32-bit byte offset reaches.  (Along x they come in pairs 5/8 h apart,
    which gives them their volumes.)  A water particle near the even one of a
    pair has the same density and acceleration in every interior cell, those of
    the same surroundings in a grid of 12^3: all positions are multiples of
    2^-10, so the differences, and with them every sum, are the same bits."""
    r = 0.0625
    h = 4 * r
    off = np.float32([0.05078125, 0.03125, 0.015625])

    def handle(cells, at):
        ph = Physics(hi=(cells * h,) * 3, r_water=r, r_sand=r)
        pos = ((np.float32(at) + np.float32(0.5)) * np.float32(h) + off).astype(np.float32)
        g = SFSystem.from_scene(make_scene(pos, np.zeros(len(pos), np.uint64), ph=ph))
        c = (np.arange(cells, dtype=np.float32) + np.float32(0.5)) * np.float32(h)
        z = c[1::3]
        b = np.empty((cells, cells, len(z), 3), np.float32)
        x = c - np.where(np.arange(cells) % 2 == 1, np.float32(0.09375), np.float32(0.0))
        b[..., 0], b[..., 1], b[..., 2] = x[:, None, None], c[None, :, None], z
        g.upload_boundary(b.reshape(-1, 3))
        g.step(1e-6)
        return g

    small = handle(12, [(6, 6, 4)])
    ref = {k: small.get(k)[0] for k in ("density", "pressure", "acc")}
    assert 1e3 < ref["density"] < 1e5 and np.isfinite(ref["acc"]).all()
    at = [(6, 6, 4), (100, 50, 199), (250, 300, 100), (374, 10, 394), (386, 200, 10), (394, 390, 304)]
    big = handle(400, at)
    print(f"{big.sizes()} density {ref['density']}", flush=True)
    for k, v in ref.items():
        np.testing.assert_array_equal(big.get(k), np.broadcast_to(v, (len(at),) + v.shape), err_msg=k)


SHIM = """
#include <dlfcn.h>
#include <stddef.h>
static long left = -1;
static int refused;
void refuse_malloc(long k) { left = k; refused = 0; }
int malloc_refused(void) { return refused; }
int hipMalloc(void** p, size_t n) {
    static int (*real)(void**, size_t);
    if (!real) real = (int (*)(void**, size_t))dlsym(dlopen("libamdhip64.so.7", RTLD_NOW | RTLD_NOLOAD), "hipMalloc");
    if (left == 0) {
        left = -1;
        refused = 1;
        *p = NULL;
        return 2; /* hipErrorOutOfMemory */
    }
    if (left > 0) --left;
    return real(p, n);
}
"""
CHILD = """
import ctypes, sys
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)  # before the library: its hipMalloc is this one
shim.refuse_malloc.argtypes = [ctypes.c_long]
sys.path.insert(0, sys.argv[2])
import numpy as np
from sph_seepage_flows_amd import SFError, SFSystem, scenes
sc = scenes.mixed()
a, b = SFSystem.from_scene(sc), SFSystem.from_scene(sc)
names = ("pos", "vel", "acc", "density", "col", "sort_perm", "b_pos", "b_volume", "b_label", "b_cell_start")
def same(n):
    a.step(1e-4, n)
    b.step(1e-4, n)
    for name in names:
        np.testing.assert_array_equal(a.get(name), b.get(name), err_msg=name)
same(3)
copies = lambda n, d: (np.concatenate([sc.bpos + np.float32(d * q) for q in range(n)]), np.tile(sc.blabel, n))
# no more than the handle's particles; more than the sort has room for; as many again
for other, label in (copies(1, 0.003), copies(5, 0.002), copies(5, 0.0015)):
    failed = 0
    while True:
        shim.refuse_malloc(failed)
        try:
            a.upload_boundary(other, label)
        except SFError:
            assert shim.malloc_refused() == 1
        else:
            break
        failed += 1
        assert a.sizes() == b.sizes()
        same(2)
    assert shim.malloc_refused() == 0
    shim.refuse_malloc(-1)
    b.upload_boundary(other, label)
    same(2)
    print(len(other), "boundary particles, failed uploads", failed)
"""


def test_failed_upload_leaves_the_old_boundary(tmp_path):
    """Each allocation of an upload in turn reports that there is no memory (a
    hipMalloc in front of the runtime's, in a process of its own): the handle
    steps on with its old boundary, bit for bit like one that was never asked."""
    src, lib_ = tmp_path / "shim.c", tmp_path / "shim.so"
    src.write_text(SHIM)
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", str(src), "-o", str(lib_), "-ldl"], check=True)
    root = str(Path(__file__).resolve().parents[1])
    r = subprocess.run([sys.executable, "-c", CHILD, str(lib_), root], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stdout + r.stderr
    print(r.stdout, flush=True)
    counts = [int(line.split()[-1]) for line in r.stdout.splitlines()]
    # the state and the cells' bytes; the six arrays of the sort; those two, the
    # particles as given and, of the larger boundary's, the ranges
    assert len(counts) == 3 and counts[0] >= 2 and counts[1] >= 6 and counts[2] >= 3
