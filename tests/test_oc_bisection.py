"""The density update's bisection, three steps a pass for exponents from a quarter
to one and a step a pass outside, against the same bisection in numpy (a trial's
densities in FP32, its volume summed in FP64): the same multiplier and number of
trials, and the densities to 2e-6, FP32 powers of a few units in the last place
(where the sensitivity over the multiplier is a normal number). Sensitivities over
many decades (with a small exponent those far below the largest still weigh), exact
zeros, positive ones (taken as zero), scales far from one, goals that every trial
misses from below and above, and shell elements."""
import numpy as np
import pytest

import robtop_amd as rt
from robtop_amd.workloads import cube_bits, cube_side

pytestmark = pytest.mark.gpu


def reference(rho, g, shell, vgoal, step, damp, rho_min):
    gg = np.abs(np.minimum(g, 0)).astype(np.float32)
    lo, up = np.float32(0), np.float32(np.abs(g).max())
    it = n = 0
    step, damp, rho_min = np.float32(step), np.float32(damp), np.float32(rho_min)
    while True:
        thr = (lo + up) / np.float32(2)
        rn = rho * (gg / thr) ** damp
        rn = np.minimum(np.maximum(rn, rho - step), rho + step)
        rn = np.minimum(np.maximum(rn, rho_min), np.float32(1))
        rn[shell] = 1
        V = np.float32(rn.sum(dtype=np.float64) / rn.size)
        n += 1
        if V > np.float32(vgoal):
            lo = thr
        elif V < np.float32(vgoal):
            up = thr
        go = abs(V - np.float32(vgoal)) > 1e-4 and it < 30
        it += 1
        if not go:
            return thr, n, rn


@pytest.mark.parametrize("vgoal,step,damp,scale,spread", [
    (0.4, 0.03, 0.5, 1.0, 1), (0.38, 0.2, 0.5, 1e-9, 3), (0.45, 0.05, 1.0, 1e12, 2), (0.42, 0.1, 0.3, 1.0, 8),
    (0.9, 0.03, 0.5, 1.0, 1), (0.05, 0.03, 0.5, 1.0, 1), (0.42, 0.1, 1.5, 1e-3, 2),
    (0.24, 0.5, 0.01, 1e25, 60), (0.25, 0.5, 0.25, 1e25, 60), (0.4, 0.2, 0.2, 1.0, 4)])
def test_bisection_matches_numpy(vgoal, step, damp, scale, spread):
    print(f"[oc] goal {vgoal} step {step} damp {damp} scale {scale}", flush=True)
    ex, ey, ez = 57, 19, 23
    a = np.zeros((cube_side(ex, ey, ez),) * 3, bool)
    a[:ex, :ey, :ez] = True
    a[20:26, 5:, :9] = False
    hg = rt.HierarchyGrid.genFromMesh(cube_bits(a), a.shape[0])
    hg.set_material(1e6, 0.4, 3.0)
    eact, _ = hg[0].masks()
    rng = np.random.default_rng(int(100 * vgoal) + spread)
    n = eact.size
    rho = (rng.uniform(0.2, 0.6, n) * eact).astype(np.float32)
    g = (-scale * 10.0 ** rng.uniform(-spread, 0, n) * eact).astype(np.float32)
    g[rng.random(n) < 0.02] = 0
    g[rng.random(n) < 0.02] *= -0.5
    shell = eact & (rng.random(n) < 0.05)
    hg.set_density(rho)
    hg.set_shell(shell)
    hg.set_sensitivity(g)
    thr, ntr = hg.update_densities(vgoal, step, damp, 1e-3)
    want, nwant, rn = reference(rho[eact], g[eact], shell[eact], vgoal, step, damp, 1e-3)
    assert ntr == nwant and thr == want
    got = hg.get_density()[eact]
    gg = np.abs(np.minimum(g[eact], 0))
    ok = (gg == 0) | (gg / thr >= np.finfo(np.float32).tiny)
    assert np.max(np.abs(got - rn)[ok] / rn[ok]) < 2e-6
    hg.close()
