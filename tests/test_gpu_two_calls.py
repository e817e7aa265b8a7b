"""Positions and masses written between BuildGNSearcher and UpdateSolver
(CudaGNBaseSearcher::BuildGNSearcher, CudaWCSphSFSolver::UpdateSolver called
one after the other, cuda_base_system.cu:29-56), by a caller that holds them.

The solve runs on the build's cells.  The interface passes take a particle's own
position and mass as they are now and its neighbours' as they were at the build,
the same ones for the range test and for every weight; the water momentum pass
takes both as they are now.  The reference below restates that in float64 over
the build's cells, from the density, pressure and drag the solve left.  A
neighbour's own sums exist only if it has the other phase in the 27 cells around
where it is now; particles with a neighbour for which that fails are left out.

Tolerances, of the largest value: saturation and voidage of water 1e-5 (at most
a few hundred positive terms, a few 6e-8 each).  A grain's voidage is a mean of
its neighbours' with weights (h^2 - r^2)^3; where they add up to 1e-3 of the
largest or more, one has 1 - (r/h)^2 above 0.05 and an FP32 error below
3 x 2e-7 / 0.05: 5e-5.  Adhesion: its quarter power starts from zero at r = h/2,
where an error of 1e-7 in r / h at a distance of 1e-5 (the nearest of 1e4 pairs)
moves it by 1.4e-4: 1e-3.  Acceleration: 1e-4 (sums of up to 70 terms, some
ten times the net)."""
import numpy as np
import pytest

from sph_seepage_flows_amd import SFSystem, scenes

from _compare import norm_err
from _hip import d2h, h2d

pytestmark = pytest.mark.gpu

EPS = 1e-6


def _bezier(s, py0, py1, px1, py2):
    b = -(px1 + 1.0) / 2.0
    t = s / px1
    low = (1 - t) ** 2 * py0 + 2 * t * (1 - t) * py1 + t * t * py1
    t = (b + np.sqrt(np.maximum(b * b - 4.0 * (1.0 + b - px1) * (px1 - s), 0.0))) / (2.0 * (1.0 + b - px1))
    high = (1 - t) ** 2 * py1 + 2 * t * (1 - t) * py1 + t * t * py2
    return np.where(s >= 1, py2, np.where(s < 0, py0, np.where(s <= px1, low, high)))


def _cells(pos, ph, h32):
    q = (np.asarray(pos, np.float32) - np.float32(ph.lo)) / h32
    g = ((np.float32(ph.hi) - np.float32(ph.lo)) / h32).astype(np.int64)
    return np.clip(np.floor(q).astype(np.int64), 0, g - 1)


class _Reference:
    """Float64 sums of one solve: P, m0 at the build, Q, m1 at the solve."""

    def __init__(self, sc, water, P, m0, Q, m1):
        self.ph, self.prm = sc.physics, sc.params()[0]
        h32 = np.float32(self.prm.sph_kernel_radius)
        self.h = float(h32)
        self.water, self.m0, self.m1 = water, m0.astype(np.float64), m1.astype(np.float64)
        ci, cj = _cells(Q, self.ph, h32), _cells(P, self.ph, h32)
        self.near = (np.abs(ci[:, None] - cj[None]) <= 1).all(2)
        self.P, self.Q = P.astype(np.float64), Q.astype(np.float64)

    def pairs(self, i, j, pos_j):
        d = self.Q[i][:, None] - pos_j[j][None]
        r2 = (d * d).sum(2)
        return d, r2, self.near[np.ix_(i, j)] & (r2 < self.h ** 2)

    def W(self, r2, ok):
        return np.where(ok, 315.0 / (64.0 * np.pi * self.h ** 9) * np.maximum(self.h ** 2 - r2, 0.0) ** 3, 0.0)

    def interface(self, rho):
        w, s = np.nonzero(self.water)[0], np.nonzero(~self.water)[0]
        rho_s, p = float(self.prm.dem_density), self.prm
        d, r2, ok = self.pairs(w, s, self.P)
        vs = (self.m0[s] / rho_s * self.W(r2, ok)).sum(1)
        _, q2, kk = self.pairs(s, w, self.P)
        V = self.m0[w] / rho[w] * self.W(q2, kk)
        sat = V.sum(1)
        eps = 1.0 - vs
        mean = (V * eps).sum(1) / np.where(sat != 0, sat, 1.0)
        r = np.sqrt(r2)
        A = 0.007 / self.h ** 3.25 * np.maximum(2.0 / self.h * (2 * r - self.h) * (self.h - r), 0.0) ** 0.25
        A = np.where(ok & (2 * r > self.h), A, 0.0)
        G = _bezier(sat, p.sf_a0, p.sf_amc, p.sf_amc_p, p.sf_asat)
        F = (d * (G * self.m0[s] * A / np.maximum(r, EPS))[..., None]).sum(1) * self.m1[w, None]
        # particles all of whose neighbours have sums of their own
        listed = lambda i, j: self.near[np.ix_(i, j)].any(1)
        s_ok = (~(kk & ~listed(w, s)[None])).all(1)
        w_ok = (~(ok & ~(listed(s, w) & s_ok)[None])).all(1)  # its adhesion takes their saturations
        return w, s, vs, eps, sat, mean, F, w_ok, s_ok

    def water_acc(self, rho, pres, eps, vel, drag, F):
        """Without boundary particles."""
        w, s = np.nonzero(self.water)[0], np.nonzero(~self.water)[0]
        p = self.prm
        rt = rho[w] / np.maximum(EPS, eps)
        pt = pres[w] / np.maximum(EPS, rt * rt)

        def grad(r2, ok):
            r = np.sqrt(r2)
            return np.where(ok & (r >= EPS), -45.0 / (np.pi * self.h ** 6) * (self.h - r) ** 2 / np.maximum(r, EPS), 0.0)

        d, r2, ok = self.pairs(w, w, self.Q)
        dv = vel[w][:, None] - vel[w][None]
        dd = (dv * d).sum(2)
        visc = np.where(dd < 0, -float(p.sph_nu) / (rt[:, None] + rt[None]) * dd / (r2 + EPS), 0.0)
        c = -self.m1[w][None] * (pt[:, None] + pt[None] + visc) * grad(r2, ok)
        a = (d * c[..., None]).sum(1)
        d, r2, ok = self.pairs(w, s, self.Q)
        c = -self.m1[s][None] * (pres[w] / np.maximum(EPS, rt * float(p.dem_density)))[:, None] * grad(r2, ok)
        a += (d * c[..., None]).sum(1)
        a -= (self.W(r2, ok) @ drag[s]) / rt[:, None]
        return a - F / self.m1[w, None] + np.float64(self.ph.gravity)


def _write_between(hand_out, masses):
    """(scene, handle after the solve, reference)"""
    sc = scenes.mixed(collider=False)
    sc.bpos = sc.blabel = None
    rng = np.random.default_rng(11)
    if masses == "unequal":
        sc.mass = (sc.mass * rng.uniform(0.9, 1.1, sc.n)).astype(np.float32)
    g = SFSystem.from_scene(sc)
    g.BuildGNSearcher()
    P, m0, water = g.get("pos"), g.get("mass"), g.get("label") == 0
    h = float(sc.params()[0].sph_kernel_radius)
    Q = (P + rng.uniform(-0.3 * h, 0.3 * h, P.shape)).astype(np.float32)
    m1 = m0 if masses == "kept" else (m0 * rng.uniform(0.95, 1.05, sc.n)).astype(np.float32)
    if hand_out == "view":
        h2d(g.view("pos"), Q)
        h2d(g.view("mass"), m1)
    else:
        addr, stride = g.device_buffer("pos")
        assert stride == 16
        raw = d2h(addr, (sc.n, 4), np.float32)
        h2d(addr, np.column_stack([Q, np.where(water, m1, -m1)]).astype(np.float32))
        np.testing.assert_array_equal(raw[:, :3], P)
    vel = g.get("vel").astype(np.float64)
    g.UpdateSolver(1e-5)
    return sc, g, _Reference(sc, water, P, m0, Q, m1), vel


CASES = [("view", "kept"), ("device_buffer", "kept"), ("view", "unequal"), ("device_buffer", "unequal")]


@pytest.mark.parametrize("hand_out,masses", CASES)
def test_interface_sums_on_written_positions(hand_out, masses):
    sc, g, ref, _ = _write_between(hand_out, masses)
    rho = g.get("density").astype(np.float64)
    w, s, vs, eps, sat, mean, F, w_ok, s_ok = ref.interface(rho)
    voidage, saturation = g.get("voidage"), g.get("saturation")
    assert norm_err(voidage[w], eps) < 1e-5
    assert norm_err(saturation[s], sat, s_ok) < 1e-5
    wet = s_ok & (sat > 1e-3 * sat.max())
    assert wet.sum() > 100
    assert norm_err(voidage[s], mean, wet) < 5e-5
    assert norm_err(g.get("adhesion_force")[w], F, w_ok) < 1e-3
    inside = w_ok & (vs > 1e-3 * vs.max())
    assert inside.sum() > 100
    avg = F / np.where(vs != 0, vs, 1.0)[:, None]
    assert norm_err(g.get("avg_adhesion_force")[w], avg, inside) < 1e-3


@pytest.mark.parametrize("hand_out,masses", CASES)
def test_water_momentum_on_written_positions(hand_out, masses):
    sc, g, ref, vel = _write_between(hand_out, masses)
    rho, pres = g.get("density").astype(np.float64), g.get("pressure").astype(np.float64)
    w = np.nonzero(ref.water)[0]
    _, s, *_, w_ok, s_ok = ref.interface(rho)
    drag = g.get("avg_drag_force").astype(np.float64)
    bad = s[~s_ok]  # grains without a defined drag, and the water they reach
    drag[bad] = 0.0
    w_ok &= ~ref.pairs(w, bad, ref.Q)[2].any(1)
    assert w_ok.sum() > 1000
    acc = ref.water_acc(rho, pres, g.get("voidage").astype(np.float64)[w], vel, drag,
                        np.where(w_ok[:, None], g.get("adhesion_force")[w].astype(np.float64), 0.0))
    assert norm_err(g.get("acc")[w], acc, w_ok) < 1e-4


def test_labels_written_between():
    """A water particle the caller turned into a grain after the build counts as
    one in the others' seepage term (with no drag of its own where it had no
    grain near), and is no longer moved as water."""
    sc = scenes.mixed(n_sand=1, collider=False)  # the grain touches no water's 27 cells
    sc.pos[sc.label == 1] = np.float32(0.45)
    sc.bpos = sc.blabel = None
    g = SFSystem.from_scene(sc)
    g.BuildGNSearcher()
    P, m0, label = g.get("pos"), g.get("mass"), g.get("label")
    water = label == 0
    flip = np.nonzero(water)[0][::7]
    lab = label.copy()
    lab[flip] = 1
    h2d(g.view("label"), lab)
    vel = g.get("vel").astype(np.float64)
    g.UpdateSolver(1e-5)
    now = lab == 0
    ref = _Reference(sc, now, P, m0, P, m0)
    rho, pres = g.get("density").astype(np.float64), g.get("pressure").astype(np.float64)
    w = np.nonzero(now)[0]
    acc = ref.water_acc(rho, pres, np.ones(len(w)), vel, np.zeros_like(vel), np.zeros((len(w), 3)))
    assert norm_err(g.get("acc")[w], acc) < 1e-4
    assert np.abs(g.get("acc")[flip]).max() == 0.0
