"""Closest-hit and occlusion parity of the HIP BVH traversal against the oracle (bit-exact
primitive index, t and barycentrics), replacing optixTrace (include/graph/trace.h:25-88)."""
import numpy as np
import pytest

from crisoptix_amd import scenes
from parity_util import bits, float_rays, random_rays, random_soup, shadow_rays, small_grid_scene

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name", ["cornell", "grid3"])
def test_closest_hit_bit_exact(name, orc, cx_runtime, cx_ctx):
    sc = scenes.cornell_box(1, 8) if name == "cornell" else small_grid_scene()
    rays = random_rays(sc, 60000, seed=11)
    oscene = orc.OracleScene(sc)
    gscene = cx_runtime.Scene(cx_ctx, sc)
    po, to, uo, vo = oscene.trace_closest(rays)
    pg, tg, ug, vg = gscene.trace_closest(rays)
    print(f"{name}: hits {np.mean(po != 0xFFFFFFFF):.3f}, prim mismatches {(po != pg).sum()}")
    assert np.array_equal(po, pg)
    assert np.array_equal(bits(to), bits(tg))
    assert np.array_equal(bits(uo), bits(ug))
    assert np.array_equal(bits(vo), bits(vg))


@pytest.mark.parametrize("name", ["cornell", "grid3"])
def test_occlusion_bit_exact(name, orc, cx_runtime, cx_ctx):
    sc = scenes.cornell_box(1, 8) if name == "cornell" else small_grid_scene()
    rays = shadow_rays(sc, 60000, seed=12)
    oscene = orc.OracleScene(sc)
    gscene = cx_runtime.Scene(cx_ctx, sc)
    oo = oscene.trace_occluded(rays)
    og = gscene.trace_occluded(rays)
    print(f"{name}: occluded fraction {oo.mean():.3f}")
    assert np.array_equal(oo, og)


def test_leaf_size_independence(orc, cx_runtime, cx_ctx):
    """Different BVHs (leaf sizes 1 and 8) give identical hits: results do not depend on the tree."""
    sc = small_grid_scene()
    rays = random_rays(sc, 20000, seed=13)
    a = cx_runtime.Scene(cx_ctx, sc, max_leaf=1).trace_closest(rays)
    b = cx_runtime.Scene(cx_ctx, sc, max_leaf=8).trace_closest(rays)
    for x, y in zip(a, b):
        assert np.array_equal(bits(x), bits(y))


@pytest.mark.parametrize("name", ["cornell", "grid3"])
def test_bvh_width_independence(name, orc, cx_runtime, cx_ctx):
    """Binary, 4-wide and 8-wide node arrays give the oracle's hits and occlusion bit for bit."""
    sc = scenes.cornell_box(1, 8) if name == "cornell" else small_grid_scene()
    rays = random_rays(sc, 30000, seed=14)
    srays = shadow_rays(sc, 30000, seed=15)
    oscene = orc.OracleScene(sc)
    ref = oscene.trace_closest(rays)
    occ = oscene.trace_occluded(srays)
    for width in (2, 4, 8):
        gscene = cx_runtime.Scene(cx_ctx, sc, width=width)
        assert gscene.info.bvhWidth == width
        got = gscene.trace_closest(rays)
        for x, y in zip(ref, got):
            assert np.array_equal(bits(x), bits(y)), width
        assert np.array_equal(occ, gscene.trace_occluded(srays)), width


def centroid_rays(scene, seed):
    """One ray per triangle, from a seeded point of the scene's box towards the triangle's
    centroid: a triangle missing from a tree (or a box that does not cover it) changes an answer."""
    rng = np.random.default_rng(seed)
    pos = scene.positions.astype(np.float64)
    lo, hi = pos.min(0), pos.max(0)
    c = pos[scene.indices].mean(axis=1)
    o = lo + rng.random(c.shape) * (hi - lo)
    d = c - o
    d /= np.maximum(np.linalg.norm(d, axis=1, keepdims=True), 1e-12)
    rays = np.zeros((c.shape[0], 8), np.float32)
    rays[:, 0:3] = o
    rays[:, 3:6] = d
    rays[:, 6] = 0.0
    rays[:, 7] = 1e16
    return rays


def _check_against_oracle(sc, gscene, oscene, rays, srays):
    ref = oscene.trace_closest(rays)
    got = gscene.trace_closest(rays)
    for x, y in zip(ref, got):
        assert np.array_equal(bits(x), bits(y))
    assert np.array_equal(oscene.trace_occluded(srays), gscene.trace_occluded(srays))


@pytest.mark.parametrize("name", ["cornell", "grid3", "grid8"])
@pytest.mark.parametrize("width", [2, 4, 8])
def test_device_build_bit_exact(name, width, orc, cx_runtime, cx_ctx):
    """BVH built on the GPU (Morton sort, PLOC clustering, SAH leaves, wide collapse): closest-hit
    and occlusion answers equal the oracle's bit for bit, also for one ray per triangle."""
    if name == "cornell":
        sc = scenes.cornell_box(1, 8)
    elif name == "grid3":
        sc = small_grid_scene()
    else:
        sc = scenes.object_grid(grid=8, seed=9, ground_quads=40, ico_subdiv=3, num_lights=4)
    rays = np.concatenate([random_rays(sc, 30000, seed=16), centroid_rays(sc, seed=17)])
    srays = shadow_rays(sc, 30000, seed=18)
    gscene = cx_runtime.Scene(cx_ctx, sc, width=width, builder="device")
    info = gscene.info
    print(f"{name} width {width}: {sc.indices.shape[0]} triangles, {info.numNodes} binary nodes, depth "
          f"{info.maxDepth}, {info.numWideNodes} wide nodes, stack bound {info.stackBound}, {info.buildMs:.2f} ms")
    assert info.bvhBuilder == 1 and info.bvhWidth == width
    assert 0 < info.numNodes < sc.indices.shape[0]
    assert info.stackBound + 1 <= 64
    _check_against_oracle(sc, gscene, orc.OracleScene(sc), rays, srays)


def _subset(sc, k):
    import dataclasses
    return dataclasses.replace(sc, indices=sc.indices[:k].copy(), tri_material=sc.tri_material[:k].copy())


@pytest.mark.parametrize("k", [0, 1, 2, 3, 5, 17])
def test_device_build_tiny_scenes(k, orc, cx_runtime, cx_ctx):
    """0 to 17 triangles: no geometry, a single leaf holding every triangle (k <= max leaf) and
    small trees."""
    full = scenes.cornell_box(1, 8)
    sc = _subset(full, k)
    rays = random_rays(full, 3000, seed=19)   # aimed at the full box (its vertices stay in the scene)
    if k:
        rays = np.concatenate([rays, centroid_rays(sc, seed=20)])
    srays = shadow_rays(sc, 3000, seed=21)
    oscene = orc.OracleScene(sc)
    for width in (2, 4, 8):
        for max_leaf in (1, 4, 8):
            gscene = cx_runtime.Scene(cx_ctx, sc, width=width, max_leaf=max_leaf, builder="device")
            if k <= 1:
                assert gscene.info.numNodes == 0
            _check_against_oracle(sc, gscene, oscene, rays, srays)


def test_device_build_coincident_triangles(orc, cx_runtime, cx_ctx):
    """64 copies of one triangle (one Morton key, equal areas) among the Cornell box: the copies
    tie on every comparison of the clustering; the lowest primitive index must still win."""
    import dataclasses
    sc = scenes.cornell_box(1, 8)
    dup = np.repeat(sc.indices[5:6], 64, axis=0)
    sc = dataclasses.replace(sc, indices=np.concatenate([sc.indices, dup]).astype(np.uint32),
                             tri_material=np.concatenate([sc.tri_material, np.repeat(sc.tri_material[5:6], 64)])
                             .astype(np.uint32))
    rays = np.concatenate([random_rays(sc, 20000, seed=22), centroid_rays(sc, seed=23)])
    srays = shadow_rays(sc, 20000, seed=24)
    oscene = orc.OracleScene(sc)
    for width in (2, 4, 8):
        gscene = cx_runtime.Scene(cx_ctx, sc, width=width, builder="device")
        assert gscene.info.bvhBuilder == 1   # the copies merge pairwise: no chain, no fallback
        _check_against_oracle(sc, gscene, oscene, rays, srays)


def test_device_build_falls_back_when_too_deep(orc, cx_runtime, cx_ctx):
    """100 nested triangles around one centre (each contains the smaller ones): every merge
    candidate of a triangle costs its own box, so the clustering can only peel one triangle per
    iteration and the tree would be a chain deeper than the traversal stack.  The scene build
    then takes the host build (bvhBuilder reports it) and answers stay exact."""
    import dataclasses
    sc = scenes.cornell_box(1, 8)
    shape = np.array([[-1.0, -0.6, 0.0], [1.0, -0.6, 0.0], [0.0, 1.2, 0.0]])
    centre = sc.positions.astype(np.float64).mean(axis=0)
    tri = np.concatenate([centre + 0.002 * 1.05 ** k * shape for k in range(100)]).astype(np.float32)
    nv = sc.positions.shape[0]
    nrm = np.tile(np.array([[0.0, 0.0, 1.0]], np.float32), (tri.shape[0], 1))
    sc = dataclasses.replace(
        sc, positions=np.concatenate([sc.positions, tri]), normals=np.concatenate([sc.normals, nrm]),
        indices=np.concatenate([sc.indices, nv + np.arange(tri.shape[0], dtype=np.uint32).reshape(-1, 3)]),
        tri_material=np.concatenate([sc.tri_material, np.zeros(100, np.uint32)]))
    if sc.uvs is not None:
        sc = dataclasses.replace(sc, uvs=np.concatenate([sc.uvs, np.zeros((tri.shape[0], 2), np.float32)]))
    rays = np.concatenate([random_rays(sc, 20000, seed=26), centroid_rays(sc, seed=27)])
    srays = shadow_rays(sc, 20000, seed=28)
    gscene = cx_runtime.Scene(cx_ctx, sc, width=4, builder="device")
    assert gscene.info.bvhBuilder == 0
    _check_against_oracle(sc, gscene, orc.OracleScene(sc), rays, srays)


def test_device_build_deterministic(cx_runtime, cx_ctx):
    """Two device builds of one scene give the same tree shape (the build orders by scans, not
    by atomics) and the same answers as the host-built tree."""
    sc = small_grid_scene()
    a = cx_runtime.Scene(cx_ctx, sc, builder="device")
    b = cx_runtime.Scene(cx_ctx, sc, builder="device")
    for f in ("numNodes", "maxDepth", "numWideNodes", "stackBound", "deviceBytes"):
        assert getattr(a.info, f) == getattr(b.info, f), f
    rays = random_rays(sc, 20000, seed=25)
    h = cx_runtime.Scene(cx_ctx, sc, builder="host").trace_closest(rays)
    for x, y, z in zip(h, a.trace_closest(rays), b.trace_closest(rays)):
        assert np.array_equal(bits(x), bits(y)) and np.array_equal(bits(y), bits(z))


@pytest.mark.parametrize("seed", range(4))
def test_device_build_random_soups(seed, orc, cx_runtime, cx_ctx):
    """Random soups with zero-area, collinear and duplicated triangles at mixed scales: the device
    build's answers equal the oracle's at every width."""
    sc = random_soup(seed)
    rays = np.concatenate([random_rays(sc, 3000, seed=60 + seed), centroid_rays(sc, seed=70 + seed)])
    srays = shadow_rays(sc, 2000, seed=80 + seed)
    oscene = orc.OracleScene(sc)
    for width in (2, 4, 8):
        gscene = cx_runtime.Scene(cx_ctx, sc, width=width, builder="device")
        _check_against_oracle(sc, gscene, oscene, rays, srays)


@pytest.mark.parametrize("width", [2, 4, 8])
def test_ray_counts_and_alignment(width, orc, cx_runtime, cx_ctx):
    """Every split of the rays over the device gives the oracle's bits: counts at the edges of a
    wavefront and a block, of one ray per quad, of the device's capacity (width 8: 164 k rays,
    width 2: four times that) and beyond, with the rays at addresses that are aligned to 16 bytes
    and to 4 bytes only."""
    from crisoptix_amd.runtime import DeviceArray, lib, synchronize
    sc = small_grid_scene()
    gscene = cx_runtime.Scene(cx_ctx, sc, width=width)
    assert gscene.info.bvhWidth == width
    part = np.concatenate([random_rays(sc, 9000, seed=91), shadow_rays(sc, 2000, seed=92)])
    part[5, 3:6] = 0.0        # no direction
    part[6, 0] = np.nan
    part[7, 3:5] = 0.0        # along an axis
    part[8, 6] = -5.0         # from behind the origin
    part[9, 6:8] = np.nan
    part[10, 7] = -1.0        # an empty interval
    part[11, 7] = np.inf
    oscene = orc.OracleScene(sc)
    ref, occ = oscene.trace_closest(part), oscene.trace_occluded(part)
    most = 700_001
    rays = np.resize(part, (most, 8))
    for shift in (0, 1, 3):
        dev = DeviceArray.from_numpy(np.concatenate([np.zeros(shift, np.float32), rays.ravel()]))
        for n in (1, 2, 63, 65, 129, 4096, 114_688, 114_689, 163_841, most):
            outs = [DeviceArray((n,), dt) for dt in (np.uint32, np.float32, np.float32, np.float32)]
            flags = DeviceArray((n,), np.uint32)
            cx_ctx.check(lib().cx_trace_closest(cx_ctx.h, gscene.h, dev.ptr + 4 * shift, n, *[o.ptr for o in outs], None),
                         "cx_trace_closest")
            cx_ctx.check(lib().cx_trace_occluded(cx_ctx.h, gscene.h, dev.ptr + 4 * shift, n, flags.ptr, None),
                         "cx_trace_occluded")
            synchronize()
            for x, y in zip(ref, outs):
                assert np.array_equal(np.resize(bits(x), n), bits(y.numpy())), (n, shift)
            assert np.array_equal(np.resize(occ, n), flags.numpy()), (n, shift)


@pytest.mark.parametrize("width,most", [(2, 700_001), (4, 130_001), (8, 200_001)])
@pytest.mark.parametrize("name", ["cornell", "grid3"])
def test_rays_of_any_floats(name, width, most, orc, cx_runtime, cx_ctx):
    """Directions, origins and intervals at the ends of the float range, few and many (the kernels of
    short and long arrays): the bits of the oracle's loop over all triangles."""
    sc = scenes.cornell_box(1, 8) if name == "cornell" else small_grid_scene()
    gscene = cx_runtime.Scene(cx_ctx, sc, width=width)
    assert gscene.info.bvhWidth == width
    rays = np.concatenate(list(float_rays(sc, 150, seed=37).values()))
    brute = orc.OracleScene(sc, brute_force=True)
    ref, occ = brute.trace_closest(rays), brute.trace_occluded(rays)
    for n in (len(rays), most):
        print(f"{name} width {width} rays {n}", flush=True)
        got = gscene.trace_closest(np.resize(rays, (n, 8)))
        flags = gscene.trace_occluded(np.resize(rays, (n, 8)))
        for x, y in zip(ref, got):
            assert np.array_equal(np.resize(bits(x), n), bits(y)), n
        assert np.array_equal(np.resize(occ, n), flags), n


@pytest.mark.parametrize("k", [1023, 1024, 1025, 1100, 2304])
def test_device_build_at_the_tail_of_the_clustering(k, orc, cx_runtime, cx_ctx):
    """Triangle counts around the one that a single block clusters to the root (1024), and coincident
    and zero-area triangles among them (areas that tie): the answers stay the oracle's."""
    sc = _subset(scenes.cornell_box(1, 8), k)
    sc.indices[k // 2:k // 2 + 40] = sc.indices[3]        # coincident
    sc.indices[k // 3:k // 3 + 40, 1] = sc.indices[k // 3:k // 3 + 40, 0]   # zero area
    rays = np.concatenate([random_rays(sc, 4000, seed=93), centroid_rays(sc, seed=94)])
    srays = shadow_rays(sc, 4000, seed=95)
    oscene = orc.OracleScene(sc)
    for width in (2, 4, 8):
        gscene = cx_runtime.Scene(cx_ctx, sc, width=width, builder="device")
        assert gscene.info.bvhBuilder == 1
        _check_against_oracle(sc, gscene, oscene, rays, srays)


@pytest.mark.parametrize("fault,message", [("index", "vertex index out of range"), ("material", "material id out of range"),
                                           ("nan", "non-finite vertex position"), ("inf", "non-finite vertex position"),
                                           ("index and width", "vertex index out of range")])
@pytest.mark.parametrize("builder", ["host", "device"])
def test_faulty_geometry_is_refused(fault, message, builder, cx_runtime, cx_ctx):
    """One wrong element at the end of an array is refused by name with either builder (the device
    builder checks the uploaded arrays on the device, before anything reads through them), and the
    same bounds and scene size are reported for the sound scene."""
    sc = small_grid_scene()
    a, b = (cx_runtime.Scene(cx_ctx, sc, builder=k).info for k in ("host", builder))
    assert a.sceneSize == b.sceneSize and list(a.boundsMin) == list(b.boundsMin) and list(a.boundsMax) == list(b.boundsMax)
    import copy
    bad = copy.deepcopy(sc)
    if "index" in fault:
        bad.indices[-1, 2] = len(bad.positions)
    if fault == "material":
        bad.tri_material[-1] = 10**6
    if fault in ("nan", "inf"):
        bad.positions[-1, 1] = np.nan if fault == "nan" else -np.inf
    with pytest.raises(Exception, match=message):
        cx_runtime.Scene(cx_ctx, bad, width=3 if "width" in fault else 4, builder=builder)
