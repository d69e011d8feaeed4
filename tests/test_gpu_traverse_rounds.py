"""GPU traversal at the limits of the quantised nodes and of the LDS stack.

Closest and any hit against the FP64 oracle's brute force over every triangle,
in scenes that reach what ordinary ones do not: stacks past the ten LDS slots
(large overlapping triangles enter every child), nodes flat along an axis (a
zero extent still needs a grid spacing), very small and very large scales, a
scene far from the origin, rays with zero direction components in every
pattern, and a lone triangle (empty child slots).

Tolerance: the FP32 error of the watertight test, |dt| <= 1e-5 t + 4e-7 C with
C the largest coordinate magnitude, and ids equal outside ties (another
triangle within 1e-5 of t, or the hit within barycentric 1e-5 of an edge)."""
import numpy as np
import pytest

import oracle
import wurstrenderer_amd as wr
from wurstrenderer_amd import scenes

pytestmark = pytest.mark.gpu
INV = 0xFFFFFFFF


def _mesh(verts, tris):
    b = scenes.SceneBuilder()
    b.mesh(verts, tris, material=b.material(scenes.LAMBERT, rho_d=(0.5, 0.5, 0.5)))
    return b.build(dict(pos=(0, 0, 8), lookat=(0, 0, 0), fovy=45.0, resolution=(8, 8)), name="mesh")


def _soup(n, size, seed, flat=None, scale=1.0, shift=0.0):
    rng = np.random.default_rng(seed)
    v = rng.uniform(-1, 1, (n, 1, 3)) + size * rng.normal(size=(n, 3, 3))
    if flat is not None:
        v[:, :, flat] = 0.25
    return _mesh(v.reshape(-1, 3) * scale + shift, np.arange(3 * n).reshape(-1, 3))


CASES = {
    "overlapping": lambda: _soup(1500, 1.5, 1),       # deep stacks: most boxes are entered
    "flat_y": lambda: _soup(300, 0.2, 2, flat=1),     # every node flat along y
    "tiny": lambda: _soup(600, 0.1, 3, scale=1e-3),
    "huge": lambda: _soup(600, 0.1, 4, scale=1e6),
    "far": lambda: _soup(600, 0.1, 5, shift=1e3),
    "one": lambda: _soup(1, 0.5, 6),
    "six": lambda: _soup(6, 0.4, 7),
}


def _rays(sc, n, seed):
    """Random rays through the scene and rays with one or two zero direction components."""
    rays = [scenes.random_rays(sc, n, seed=seed), scenes.random_rays(sc, n, seed=seed + 1, inside=True)]
    lo, hi = sc.verts.min(0).astype(np.float64), sc.verts.max(0).astype(np.float64)
    rng = np.random.default_rng(seed)
    ext = float((hi - lo).max())
    for zero in ([0], [1], [2], [0, 1], [0, 2], [1, 2]):
        d = rng.normal(size=(n // 4, 3))
        d[:, zero] = 0.0
        d /= np.linalg.norm(d, axis=1, keepdims=True)
        r = np.zeros((n // 4, 8), np.float32)
        r[:, 0:3] = rng.uniform(lo, hi, (n // 4, 3)) - 2 * ext * d
        r[:, 3], r[:, 4:7], r[:, 7] = 1e-4, d, np.inf
        rays.append(r)
    return np.concatenate(rays)


@pytest.mark.parametrize("name", sorted(CASES))
def test_rounds_against_brute_force(gpu_device, name):
    sc = CASES[name]()
    gs, osc = wr.GpuScene(gpu_device, sc), oracle.OracleScene(sc)
    gs.bvh_check(sc)  # the quantised planes contain every box
    rays = _rays(sc, 2000, 11)
    print(f"rounds: {name} rays={len(rays)} stack={gs.info()['max_stack']}", flush=True)
    g, p, t = gs.trace_closest(rays)
    og, op, ot, sec, mar = osc.trace_closest(rays, brute=True)
    C = float(np.abs(sc.verts).max())
    near = np.where(np.isfinite(ot), ot * (1 + 1e-5) + 4e-7 * C, np.inf)
    tie = (np.isfinite(sec) & (sec <= near)) | ((og != INV) & (mar < 1e-5))
    ok = ~tie
    bad = ok & ((g != og) | (p != op))
    assert bad.sum() == 0, (np.nonzero(bad)[0][:5], g[bad][:5], og[bad][:5])
    hit = ok & (og != INV)
    assert (np.abs(t[hit] - ot[hit]) <= 1e-5 * ot[hit] + 4e-7 * C).all()
    assert np.isinf(t[ok & (og == INV)]).all()
    # any hit: occluded exactly where the closest hit lies before tmax, away from it
    rng = np.random.default_rng(3)
    seg = rays.copy()
    seg[:, 7] = (np.where(np.isfinite(ot), ot, 1.0) * rng.uniform(0.3, 1.7, len(rays))).astype(np.float32)
    occ = gs.trace_any(seg).astype(bool)
    clear = ok & (np.abs(seg[:, 7] - ot) > 1e-4 * ot + 4e-6 * C)
    assert (occ[clear] == (ot[clear] < seg[clear, 7])).all()
