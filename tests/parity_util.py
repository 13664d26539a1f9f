"""Shared helpers of the parity tests: seeded ray batches and comparisons."""
import numpy as np

from crisoptix_amd import scenes


def small_grid_scene():
    """A reduced object grid: 3x3 objects (icosphere subdivision 2 or boxes) on a 20x20 ground,
    under a tent of 4 traced light triangles."""
    return scenes.object_grid(grid=3, seed=5, ground_quads=20, ico_subdiv=2, num_lights=4)


def tent_grid_scene():
    """The Conditional ReSTIR workload's scene reduced: 3x3 objects on a 20x20 ground under the
    tent of 16 traced light triangles of the full scene, a closed scene in which about a third
    of the pixels hold a valid suffix."""
    return scenes.object_grid(grid=3, seed=5, ground_quads=20, ico_subdiv=2, num_lights=16)


def random_rays(scene, n, seed, kind="mixed"):
    """Rays [n][8] (origin, dir, tmin, tmax).  A third aim exactly at triangle vertices and edge
    midpoints, where a non-watertight test would leak or double-hit."""
    rng = np.random.default_rng(seed)
    pos = scene.positions.astype(np.float64)
    lo, hi = pos.min(0), pos.max(0)
    ext = hi - lo
    o = lo + rng.random((n, 3)) * ext
    o[:, 1] = lo[1] + 0.05 * ext[1] + rng.random(n) * 0.9 * ext[1]
    d = rng.normal(size=(n, 3))
    m = n // 3
    tri = scene.indices[rng.integers(0, scene.indices.shape[0], m)]
    w = rng.integers(0, 3, m)
    tgt = pos[tri[np.arange(m), w]]
    e2 = pos[tri[np.arange(m), (w + 1) % 3]]
    half = rng.random(m) < 0.5
    tgt[half] = 0.5 * (tgt[half] + e2[half])
    d[:m] = tgt - o[:m]
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    rays = np.zeros((n, 8), np.float32)
    rays[:, 0:3] = o
    rays[:, 3:6] = d
    rays[:, 6] = 1e-3
    rays[:, 7] = 1e16
    return rays


def shadow_rays(scene, n, seed):
    rng = np.random.default_rng(seed)
    pos = scene.positions.astype(np.float64)
    lo, hi = pos.min(0), pos.max(0)
    a = lo + rng.random((n, 3)) * (hi - lo)
    b = lo + rng.random((n, 3)) * (hi - lo)
    v = b - a
    L = np.linalg.norm(v, axis=1)
    rays = np.zeros((n, 8), np.float32)
    rays[:, 0:3] = a
    rays[:, 3:6] = v / L[:, None]
    rays[:, 6] = 1e-3
    rays[:, 7] = L
    return rays


def float_rays(sc, n, seed):
    """{name: rays}: the same n rays with one thing about them at the ends of the float range."""
    base = random_rays(sc, n, seed=seed)
    size = np.float32(sc.scene_size())
    with np.errstate(over="ignore", under="ignore", invalid="ignore"):
        def d(axis, v):
            r = base.copy()
            r[:, 3 + axis] = v
            return r

        def o(axis, v, back=False):
            r = base.copy()
            r[:, axis] = v
            if back:   # still through the scene
                r[:, 3:6] = 0.0
                r[:, 3 + axis] = -np.sign(v)
            return r

        def scale(v, zero=None):
            r = base.copy()
            r[:, 3:6] *= np.float32(v)
            r[:, 6] = 0.0
            r[:, 7] = np.inf if v > 1e-36 else 3.4e38   # below, the t of a hit may be infinite itself
            if zero is not None:
                r[:, 3 + zero] = 0.0
            return r

        out = {"as they are": base, "x 1e-40": d(0, 1e-40), "y 1e-40": d(1, 1e-40), "z -1e-42": d(2, -1e-42),
               "x 1e-26": d(0, 1e-26), "x 0": d(0, 0.0), "x inf": d(0, np.inf), "x nan": d(0, np.nan),
               "1e-20": scale(1e-20), "1e-30": scale(1e-30), "1e-37": scale(1e-37), "1e-39": scale(1e-39),
               "1e30": scale(1e30), "1e-6, z 0": scale(1e-6, 2), "1e-30, y 0": scale(1e-30, 1),
               "1e-37, x 0": scale(1e-37, 0), "1e30, x 0": scale(1e30, 0)}
        for v in (1e5, 1e10, -1e15, 1e30, 3e38, np.inf, -np.inf, np.nan):
            out[f"origin x {v}"] = o(0, v)
            out[f"origin z {v}, back"] = o(2, v, True)
        far = d(2, 0.0)
        far[:, 2] += np.float32(1e10)
        out["z 0, origin z 1e10"] = far
        behind = base.copy()
        behind[:, 6] = -10.0 * size
        out["from behind the origin"] = behind
        anywhere = base.copy()
        anywhere[:, 6:8] = -np.inf, np.inf
        out["the whole line"] = anywhere
    return out


def bits(a):
    return np.ascontiguousarray(a).view(np.uint32)


def rel_mismatch(a, b, rtol=1e-4, atol=1e-6):
    a = np.asarray(a, np.float64)
    b = np.asarray(b, np.float64)
    bad = np.abs(a - b) > rtol * np.maximum(np.abs(a), np.abs(b)) + atol
    bad |= np.isnan(a) != np.isnan(b)
    return bad


def random_soup(seed):
    """A random triangle soup with degenerate triangles mixed in: zero-area (repeated vertex),
    collinear, exact duplicates, and clusters at very different scales."""
    import dataclasses
    rng = np.random.default_rng(seed)
    base = scenes.cornell_box(1, 8)
    n = int(rng.integers(1, 600))
    c = rng.normal(size=(n, 1, 3)) * rng.choice([1e-3, 1.0, 50.0], size=(n, 1, 1))
    tri = c + rng.normal(size=(n, 3, 3)) * rng.choice([1e-4, 0.05, 2.0], size=(n, 1, 1))
    k = n // 8
    tri[:k, 2] = tri[:k, 1]                                          # zero area
    tri[k:2 * k, 2] = 2.0 * tri[k:2 * k, 1] - tri[k:2 * k, 0]        # collinear
    if n > 4 * k:
        tri[2 * k:3 * k] = tri[3 * k:4 * k]                          # duplicates
    pos = tri.reshape(-1, 3).astype(np.float32)
    return dataclasses.replace(
        base, positions=pos, normals=np.tile(np.float32([[0, 0, 1]]), (pos.shape[0], 1)),
        indices=np.arange(pos.shape[0], dtype=np.uint32).reshape(-1, 3),
        tri_material=np.zeros(n, np.uint32), uvs=None, material_tex=None, textures=[])
