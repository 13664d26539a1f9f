"""The wide (4- and 8-child) BVH collapse and its traversal, checked on the CPU: the device
traversal code compiled for the host (cx_bvh_host_trace) over binary, 4-wide and 8-wide node
arrays gives the oracle's closest hits (primitive, t, barycentrics) and occlusion bit for bit.
Results are a function of the ray and the triangle set alone, so every BVH shape must agree."""
import numpy as np
import pytest

from crisoptix_amd import runtime, scenes
from parity_util import bits, float_rays, random_rays, random_soup, shadow_rays, small_grid_scene

pytestmark = pytest.mark.skipif(not __import__("os").path.exists(runtime.LIB_PATH), reason="HIP library not built")


@pytest.mark.parametrize("name", ["cornell", "grid3"])
@pytest.mark.parametrize("width,max_leaf", [(2, 4), (4, 4), (8, 4), (4, 1), (8, 8)])
def test_host_traversal_matches_oracle(name, width, max_leaf, orc):
    sc = scenes.cornell_box(1, 8) if name == "cornell" else small_grid_scene()
    rays = random_rays(sc, 6000, seed=21)
    po, to, uo, vo = orc.OracleScene(sc).trace_closest(rays)
    pg, tg, ug, vg, used = runtime.host_trace(sc, rays, width=width, max_leaf=max_leaf)
    assert used == width
    assert np.array_equal(po, pg)
    assert np.array_equal(bits(to), bits(tg))
    assert np.array_equal(bits(uo), bits(ug))
    assert np.array_equal(bits(vo), bits(vg))
    srays = shadow_rays(sc, 6000, seed=22)
    oo = orc.OracleScene(sc).trace_occluded(srays)
    og, _ = runtime.host_trace(sc, srays, any_hit=True, width=width, max_leaf=max_leaf)
    assert np.array_equal(oo.astype(np.uint32), og)


def axis_rays(sc, n, seed):
    """Rays at the edges of the slab test's arithmetic: one or two direction components exactly
    zero or far below the others (1e-9, 1e-20, 1e-40), of either sign, origins on vertex
    coordinates (so on box faces, the ground plane y = 0 among them) or up to 1000 scene sizes
    away along the ray's main axis, directions scaled by 1e-6 .. 1e6, tmax infinite or limited,
    tmin 0 or 1e-3 over the scale (an origin on a surface has a rounding error of about 1e-8 in
    space, which a tmin below it in space would let through as a hit at a point that the box of
    its triangle does not hold)."""
    rng = np.random.default_rng(seed)
    pos = sc.positions.astype(np.float32)
    size = np.float32(sc.scene_size())
    rays = np.zeros((n, 8), np.float32)
    for a in range(3):   # each coordinate that of a random vertex
        rays[:, a] = pos[rng.integers(0, len(pos), n), a]
    main = rng.integers(0, 3, n)
    d = rng.choice([0.0, -0.0, 1e-9, -1e-9, 1e-20, -1e-20, 1e-40, -0.3, 0.4], size=(n, 3)).astype(np.float32)
    sign = rng.choice([-1.0, 1.0], n).astype(np.float32)
    d[np.arange(n), main] = sign
    far = rng.random(n) < 0.4
    away = (size * 10.0 ** rng.uniform(0, 3, n)).astype(np.float32)
    straight = np.abs(d).sum(1) < 1.1          # a tilted far ray would pass the scene by
    pick = far & straight
    rays[pick, main[pick]] = -sign[pick] * away[pick]
    rays[:, 3:6] = d * (10.0 ** rng.uniform(-6, 6, n)).astype(np.float32)[:, None]
    rays[:, 6] = np.where(rng.random(n) < 0.5, 0.0, 1e-3 / np.abs(rays[:, 3:6]).max(1))
    rays[:, 7] = np.where(rng.random(n) < 0.7, np.inf, size / np.abs(rays[:, 3:6]).max(1))
    return rays


@pytest.mark.parametrize("name", ["cornell", "grid3"])
def test_axis_parallel_and_far_rays_match_brute_force(name, orc):
    """The slab test's interval arithmetic loses no hit: closest hits and occlusion of every width
    equal the oracle's loop over all triangles, bit for bit."""
    sc = scenes.cornell_box(1, 8) if name == "cornell" else small_grid_scene()
    rays = axis_rays(sc, 6000, seed=23)
    brute = orc.OracleScene(sc, brute_force=True)
    ref = brute.trace_closest(rays)
    occ = brute.trace_occluded(rays).astype(np.uint32)
    assert 0.2 < np.mean(ref[0] != 0xFFFFFFFF) < 0.98
    for width in (2, 4, 8):
        *got, _ = runtime.host_trace(sc, rays, width=width)
        for x, y in zip(ref, got):
            assert np.array_equal(bits(x), bits(y)), width
        og, _ = runtime.host_trace(sc, rays, any_hit=True, width=width)
        assert np.array_equal(occ, og), width


@pytest.mark.parametrize("name", ["cornell", "grid3"])
def test_rays_of_any_floats_match_brute_force(name, orc):
    """Directions, origins and intervals at the ends of the float range: closest hits and occlusion of
    every width equal the oracle's loop over all triangles, bit for bit."""
    sc = scenes.cornell_box(1, 8) if name == "cornell" else small_grid_scene()
    brute = orc.OracleScene(sc, brute_force=True)
    hits = 0
    for what, rays in float_rays(sc, 300, seed=29).items():
        ref, occ = brute.trace_closest(rays), brute.trace_occluded(rays).astype(np.uint32)
        hits += int(np.sum(ref[0] != 0xFFFFFFFF))
        for width in (2, 4, 8):
            *got, _ = runtime.host_trace(sc, rays, width=width)
            for x, y in zip(ref, got):
                assert np.array_equal(bits(x), bits(y)), (what, width)
            og, _ = runtime.host_trace(sc, rays, any_hit=True, width=width)
            assert np.array_equal(occ, og), (what, width)
    assert hits > 1500


def test_rays_of_any_floats_visit_few_nodes():
    """Such rays do not visit most of the tree.  A call's processor time beyond the tree's build stands for
    its visits: on 70 k triangles 30000 plain rays take 0.05 s, and 2 s (one component of 1e-40) to many
    minutes (directions of 1e-39) where an interval of the box test overflowed and constrained nothing."""
    import time
    sc = scenes.object_grid(4, 2, ground_quads=40)

    def best(rays):
        t = []
        for _ in range(2):
            t0 = time.process_time()
            runtime.host_trace(sc, rays, width=4)
            t.append(time.process_time() - t0)
        return min(t)

    kinds = float_rays(sc, 30_000, seed=31)
    # a direction of 1e-39 reaches less than one unit before its t overflows, and a box test of such times
    # is that much blurred
    kinds["1e-39"] = kinds["1e-39"][:1000]
    build = best(kinds["as they are"][:8])
    took = {what: best(rays) - build for what, rays in kinds.items()}
    print({k: round(v, 3) for k, v in took.items()})
    assert max(took.values()) < 5 * max(took["as they are"], 0.1) + 0.5, took


def test_wide8_collapse_falls_back_to_greedy_on_large_scene():
    """The 1.06 M-triangle object grid of the 1080p benchmark: the least-area collapse at width 8
    needs more than 64 traversal-stack entries, so the collapse takes the greedy rule, which fits;
    width 8 is kept (not the binary fallback) and its answers equal the 4-wide tree's.  (With its
    16 light panels traced as well, the greedy tree does not fit either and width 8 falls back
    to the binary tree, which test_traced_emitters_* cover.)"""
    sc = scenes.object_grid(16, 2, trace_emitters=False)
    rays = random_rays(sc, 3000, seed=31)
    *a8, used8 = runtime.host_trace(sc, rays, width=8)
    *a4, used4 = runtime.host_trace(sc, rays, width=4)
    assert (used8, used4) == (8, 4)
    assert np.mean(a4[0] != 0xFFFFFFFF) > 0.3
    for x, y in zip(a8, a4):
        assert np.array_equal(bits(x), bits(y))


def test_empty_geometry_misses():
    """A scene with no triangles (explicit emitters only): every query misses, at every width."""
    import dataclasses
    sc = scenes.cornell_box(1, 8)
    rays = random_rays(sc, 200, seed=32)
    sc = dataclasses.replace(sc, indices=np.zeros((0, 3), np.uint32), tri_material=np.zeros(0, np.uint32))
    for width in (2, 4, 8):
        prim, t, u, v, _ = runtime.host_trace(sc, rays, width=width)
        assert (prim == 0xFFFFFFFF).all() and (t == 0).all()
        occ, _ = runtime.host_trace(sc, rays, any_hit=True, width=width)
        assert not occ.any()


@pytest.mark.parametrize("seed", range(6))
def test_random_soups_match_oracle(seed, orc):
    """Random soups with degenerate triangles: every width and leaf size gives the oracle's
    closest hits and occlusion bit for bit (the builds and both collapses on odd trees)."""
    sc = random_soup(seed)
    rays = random_rays(sc, 3000, seed=40 + seed)
    srays = shadow_rays(sc, 2000, seed=50 + seed)
    oscene = orc.OracleScene(sc)
    ref = oscene.trace_closest(rays)
    assert np.mean(ref[0] != 0xFFFFFFFF) > 0.1   # about a quarter of the rays hit
    occ = oscene.trace_occluded(srays).astype(np.uint32)
    for width in (2, 4, 8):
        for max_leaf in (1, 2, 4, 15):
            *got, _ = runtime.host_trace(sc, rays, width=width, max_leaf=max_leaf)
            for x, y in zip(ref, got):
                assert np.array_equal(bits(x), bits(y)), (width, max_leaf)
            og, _ = runtime.host_trace(sc, srays, any_hit=True, width=width, max_leaf=max_leaf)
            assert np.array_equal(occ, og), (width, max_leaf)


@pytest.mark.parametrize("width", [2, 4, 8])
def test_traced_emitters_are_invisible_to_occlusion(width, orc):
    """C9': the same scene with and without its light panels as geometry.  Occlusion rays pass
    over triangles that lack CX_VIS_OCCLUSION, so every occlusion answer is the same for both
    scenes; closest-hit rays see the panels, so a closest hit changes only where the traced
    scene's hit is a panel triangle no farther than the untraced scene's hit.  Host traversal
    and oracle agree bit for bit on the traced scene."""
    traced = scenes.object_grid(grid=3, seed=5, ground_quads=20, ico_subdiv=2, num_lights=4)
    plain = scenes.object_grid(grid=3, seed=5, ground_quads=20, ico_subdiv=2, num_lights=4, trace_emitters=False)
    nplain = plain.num_triangles
    assert traced.num_triangles == nplain + 4
    assert (traced.tri_mask[:nplain] == 3).all() and (traced.tri_mask[nplain:] == 1).all()
    # shadow rays from random ground / object points to random points of the lights
    rng = np.random.default_rng(61)
    n = 4000
    tri = plain.indices[rng.integers(0, nplain, n)]
    bary = rng.dirichlet((1, 1, 1), n)
    src = np.einsum("nk,nkd->nd", bary, plain.positions[tri].astype(np.float64))
    faces = traced.emitter_faces.astype(np.float64)
    fb = rng.dirichlet((1, 1, 1), n)
    dst = np.einsum("nk,nkd->nd", fb, faces[rng.integers(0, faces.shape[0], n)])
    v = dst - src
    dist = np.linalg.norm(v, axis=1)
    rays = np.zeros((n, 8), np.float32)
    rays[:, 0:3] = src
    rays[:, 3:6] = v / dist[:, None]
    rays[:, 6] = 1e-3
    rays[:, 7] = dist
    occ_t, _ = runtime.host_trace(traced, rays, any_hit=True, width=width)
    occ_p, _ = runtime.host_trace(plain, rays, any_hit=True, width=width)
    assert np.array_equal(occ_t, occ_p)
    assert 0.05 < occ_t.mean() < 0.95
    assert np.array_equal(orc.OracleScene(traced).trace_occluded(rays).astype(np.uint32), occ_t)
    # the same rays as closest-hit queries without the length limit: the unoccluded ones end on
    # the light they aim at
    rays[:, 7] = 1e16
    pt, tt, ut, vt, _ = runtime.host_trace(traced, rays, width=width)
    pp, tp, _, _, _ = runtime.host_trace(plain, rays, width=width)
    ref = orc.OracleScene(traced).trace_closest(rays)
    for x, y in zip(ref, (pt, tt, ut, vt)):
        assert np.array_equal(bits(x), bits(y))
    panel = pt >= nplain
    assert panel[occ_t == 0].mean() > 0.99
    same = pt == pp
    assert (same | panel).all()
    assert (tt[panel & (pp != 0xFFFFFFFF)] <= tp[panel & (pp != 0xFFFFFFFF)]).all()


@pytest.mark.parametrize("width", [2, 4, 8])
def test_overflowing_box_areas_and_non_finite_positions(width, orc):
    """Box areas that overflow to +inf leave no collapse cost below +inf (the least-area collapse
    then has no split to follow): the collapse must still produce a tree, or fall back, whose
    answers are the oracle's.  Two scenes: an object grid scaled by 3e18 (every area is +inf; the
    triangle test overflows as well, in the oracle too, so every ray misses), and the unscaled
    grid with two small triangles 1e19 away on either side (the upper levels' areas are +inf,
    rays through the grid hit).  A NaN or infinite vertex coordinate is refused."""
    import dataclasses
    base = scenes.object_grid(4, 1)
    huge = dataclasses.replace(base, positions=(base.positions.astype(np.float64) * 3e18).astype(np.float32))
    far = np.asarray([[1e19, 0, 0], [1e19, 1, 0], [1e19, 0, 1], [-1e19, 0, 0], [-1e19, 1, 0], [-1e19, 0, 1]],
                     np.float32)
    nv = len(base.positions)
    spread = dataclasses.replace(
        base, positions=np.concatenate([base.positions, far]),
        normals=np.concatenate([base.normals, np.tile([[1, 0, 0]], (6, 1)).astype(np.float32)]),
        indices=np.concatenate([base.indices, np.asarray([[nv, nv + 1, nv + 2], [nv + 3, nv + 4, nv + 5]],
                                                         np.uint32)]),
        tri_material=np.concatenate([base.tri_material, base.tri_material[:2]]),
        tri_mask=None if base.tri_mask is None else np.concatenate([base.tri_mask, [3, 3]]).astype(np.uint8))
    for sc, rays, hit_frac in ((huge, random_rays(huge, 2000, seed=33), 0.0),
                               (spread, random_rays(base, 2000, seed=34), 0.3)):
        rays[:, 7] = 1e30
        po, to, uo, vo = orc.OracleScene(sc).trace_closest(rays)
        pg, tg, ug, vg, used = runtime.host_trace(sc, rays, width=width)
        assert used in (2, width)
        assert np.mean(po != 0xFFFFFFFF) >= hit_frac
        assert np.array_equal(po, pg)
        for a, b in ((to, tg), (uo, ug), (vo, vg)):
            assert np.array_equal(bits(a), bits(b))
    for bad in (np.nan, np.inf, -np.inf):
        pos = base.positions.copy()
        pos[5, 1] = bad
        with pytest.raises(runtime.CxError):
            runtime.host_trace(dataclasses.replace(base, positions=pos), random_rays(base, 10, seed=1), width=width)
