"""Frame-level parity: the HIP frame loop against the oracle's restatement of the reference
shader logic (shader/*.cu, include/graph/restir/*.h) on identical seeded inputs.

Per-pixel radiance must agree within 1e-4 relative after every frame; reservoir records,
RNG states and neighbour sets are compared bit for bit.  Both execution modes of the HIP
library (wavefront state machines and one megakernel per pass) are checked; the wavefront mode
with its default rounds (by machine and image size, then the in-place tail kernel), with every round as
traversal + step (rounds0) and with the tail after one round (rounds1)."""
import numpy as np
import pytest

from crisoptix_amd import abi, scenes
from parity_util import rel_mismatch, small_grid_scene, tent_grid_scene

pytestmark = pytest.mark.gpu

CASES = {
    "pt_cornell": dict(scene="cornell", mode="path_tracer", W=64, H=48, frames=3),
    "restir_pt_cornell": dict(scene="cornell", mode="restir_pt_cornell", W=64, H=48, frames=6),
    "restir_pt_temporal": dict(scene="cornell", mode="restir_pt_cornell", W=40, H=40, frames=5,
                               over=dict(prefixEnableSpatial=0)),
    "cond_cornell": dict(scene="cornell", mode="conditional_restir", W=48, H=40, frames=4,
                         over=dict(gatherRadius=0.08)),
    "cond_cornell_gatherN2": dict(scene="cornell", mode="conditional_restir", W=32, H=24, frames=3,
                                  over=dict(gatherRadius=0.08, gatherN=2, suffixSpatialCount=2, windowRadius=6)),
    "cond_grid_orbit": dict(scene="grid3", mode="conditional_restir", W=48, H=32, frames=4, orbit=True,
                            over=dict(gatherRadius=0.3)),
    # the same with the BVH built on the GPU (PLOC): same images as with the host-built tree
    "cond_grid_orbit_devbvh": dict(scene="grid3", mode="conditional_restir", W=48, H=32, frames=4, orbit=True,
                                   over=dict(gatherRadius=0.3), builder="device"),
    # textured materials (diffuse, roughness and OccRoughMetal specular textures, wrapped uvs)
    "pt_grid_tex": dict(scene="grid3_tex", mode="path_tracer", W=48, H=32, frames=3),
    "restir_pt_grid_tex": dict(scene="grid3_tex", mode="restir_pt_cornell", W=48, H=32, frames=4),
    "cond_grid_tex_orbit": dict(scene="grid3_tex", mode="conditional_restir", W=48, H=32, frames=4, orbit=True,
                                over=dict(gatherRadius=0.3)),
    # the Conditional ReSTIR workload reduced (tent of 16 traced lights, k = 8): the final gather
    # sees every neighbour count from 1 to 8, and at least 250 pixels gather all 8 neighbours
    "cond_tent_orbit": dict(scene="tent16", mode="conditional_restir", W=48, H=32, frames=4, orbit=True,
                            over=dict(gatherRadius=0.6), full_k=250, every_count=True),
    # the ends of the neighbour count the reference accepts (gatherM in [1, 32], Renderer.cpp:462):
    # no neighbours at all, one, and 31 (the wide query kernel), at least 200 pixels gathering 31
    "cond_cornell_gatherM1": dict(scene="cornell", mode="conditional_restir", W=40, H=32, frames=3,
                                  over=dict(gatherRadius=0.08, gatherM=1)),
    "cond_tent_gatherM2": dict(scene="tent16", mode="conditional_restir", W=40, H=32, frames=3, orbit=True,
                               over=dict(gatherRadius=0.6, gatherM=2), full_k=300),
    "cond_tent_gatherM32": dict(scene="tent16", mode="conditional_restir", W=40, H=32, frames=3, orbit=True,
                                over=dict(gatherRadius=1.2, gatherM=32), full_k=200),
    # the closed Cornell box with its light traced as geometry (C9')
    "cond_cornell_traced_light": dict(scene="cornell_tl", mode="conditional_restir", W=40, H=32, frames=3,
                                      over=dict(gatherRadius=0.08)),
}


def _scene(name):
    if name == "cornell":
        return scenes.cornell_box(1, 8)
    if name == "cornell_tl":
        return scenes.cornell_box(1, 8, trace_emitters=True)
    if name == "tent16":
        return tent_grid_scene()
    sc = small_grid_scene()
    return scenes.with_textures(sc) if name.endswith("_tex") else sc


def _setup(case, orc, rt, ctx, exec_mode="wavefront"):
    c = CASES[case]
    sc = _scene(c["scene"])
    W, H = c["W"], c["H"]
    gscene = rt.Scene(ctx, sc, builder=c.get("builder", "host"))
    oscene = orc.OracleScene(sc)
    assert abs(gscene.size - oscene.size) == 0.0
    p = abi.workload_params(c["mode"], W, H, gscene.size)
    for k, v in c.get("over", {}).items():
        setattr(p, k, v)
    cam = scenes.cornell_camera(W, H) if c["scene"].startswith("cornell") else scenes.orbit_camera(sc, W, H)
    ren = rt.Renderer(W, H, ctx, cam, gscene, params=p, seed=1234)
    if exec_mode.startswith("rounds"):   # wavefront rounds (0: all), then the in-place tail kernel
        ren.set_exec_mode("wavefront")
        ren.set_wave_rounds(int(exec_mode[6:]))
    else:
        ren.set_exec_mode(exec_mode)
    oren = orc.OracleRenderer(oscene, W, H, p, seed=1234)
    return c, cam, ren, oren


def _compare_prefix(g, o, which_valid):
    valid = (o["flags"] >> 16) & 1
    assert np.array_equal(g["flags"], o["flags"])
    v = valid.astype(bool) & which_valid
    assert np.array_equal(g["rngState"][v], o["rngState"][v])
    for name in ("f", "postReconF", "p", "wSum", "confidence", "pathLen", "reconOutDir"):
        gv = np.asarray(g[name])[v]
        ov = np.asarray(o[name])[v]
        assert not rel_mismatch(gv, ov).any(), name
    assert np.array_equal(g["primary_prim"][v], o["primaryInt"]["prim"][v])
    assert np.array_equal(g["last_prim"][v], o["lastInt"]["prim"][v])


@pytest.mark.parametrize("exec_mode", ["wavefront", "megakernel", "rounds0", "rounds1"])
@pytest.mark.parametrize("case", list(CASES))
def test_frames_match_oracle(case, exec_mode, orc, cx_runtime, cx_ctx):
    print(f"case {case} exec {exec_mode}", flush=True)
    c, cam, ren, oren = _setup(case, orc, cx_runtime, cx_ctx, exec_mode)
    P = c["W"] * c["H"]
    worst = 0
    for f in range(c["frames"]):
        if c.get("orbit") and f > 0:
            cam.rotate_around_origin([0, 1, 0], 2 * np.pi / 64)
        cd = abi.CameraData.from_dict(cam.data())
        changed = f == 0 or bool(c.get("orbit"))
        out_o = oren.frame(cd, changed).copy()
        out_g = ren.launch_frame(cd, changed).numpy()
        bad = rel_mismatch(out_g, out_o).any(axis=-1)
        exact = np.array_equal(out_g.view(np.uint32), out_o.view(np.uint32))
        print(f"{case} frame {f}: mismatching pixels {bad.sum()}/{P}, bit-exact {exact}, "
              f"mean {out_o.mean():.5f} vs {out_g.mean():.5f}")
        worst = max(worst, int(bad.sum()))
        if bad.any():
            idx = np.argwhere(bad)[:5]
            for y, x in idx:
                print("   px", x, y, out_o[y, x], out_g[y, x])
    assert worst == 0
    assert ren.stats().queueOverflow == 0
    front, back, _, _ = oren.buffers()
    st = ren.state()
    assert (st.frontBufferIdx, st.backBufferIdx) == (front, back)
    if c["mode"] != "path_tracer":
        go = ren.gbuffer()
        oo = oren.gbuffer()
        assert np.array_equal(go["primaryIntValid"], oo[:, 2])
        assert np.array_equal(go["canonFlags"], oo[:, 3])
        assert np.array_equal(go["rngState"], oo[:, 0].astype(np.uint64) | (oo[:, 1].astype(np.uint64) << np.uint64(32)))
        for which in (front, back):
            _compare_prefix(ren.prefix(which), {n: oren.prefix(which)[n] for n in orc.PREFIX_DT.names},
                            np.ones(P, bool))
    if c["mode"] == "conditional_restir":
        gs = ren.suffix(front)
        os_ = oren.suffix(front)
        assert np.array_equal(gs["flags"], os_["flags"])
        v = ((os_["flags"] >> 16) & 1).astype(bool)
        for name in ("f", "postReconF", "p", "wSum", "confidence"):
            assert not rel_mismatch(np.asarray(gs[name])[v], np.asarray(os_[name])[v]).any(), name
        gi, gd, gc = ren.neighbors()
        oi, od, oc = oren.neighbors()
        assert np.array_equal(gc, oc)
        for p in range(P):
            n = oc[p]
            assert np.array_equal(gi[p, :n], oi[p, :n])
            assert np.array_equal(gd[p, :n].view(np.uint32), od[p, :n].view(np.uint32))
        k = int(c.get("over", {}).get("gatherM", 9)) - 1
        hist = np.bincount(oc, minlength=k + 1)
        print(f"{case}: mean neighbours {oc.mean():.2f}, histogram {hist.tolist()}, "
              f"valid suffixes {v.mean():.2f}")
        if c.get("every_count"):
            assert (hist[1:] > 0).all(), hist
        if "full_k" in c:
            assert hist[k] >= c["full_k"], hist


@pytest.mark.parametrize("rounds", [0, 1, 2, 6])
@pytest.mark.parametrize("mode", ["path_tracer", "restir_pt_cornell", "conditional_restir"])
def test_final_shadow_rays_in_queue_and_tail_match_megakernel(mode, rounds, cx_runtime, cx_ctx):
    """A walk or shift whose last ray is a shadow ray stores its result ahead of the ray, and the
    kernel that answers the ray takes it back if it is occluded: in the traversal of a queue, or in
    the tail after `rounds` rounds (0: no tail), with accumulation, eagerly and replayed from a
    frame graph.  Every frame equals the one-kernel-per-pass mode, which traces first, bit for
    bit, and so do the reservoirs."""
    W, H = 40, 24
    sc = tent_grid_scene()
    gs = cx_runtime.Scene(cx_ctx, sc)
    p = abi.workload_params(mode, W, H, gs.size)
    p.enableAccum = 0 if mode == "conditional_restir" else 1
    cam = scenes.orbit_camera(sc, W, H)
    cd = abi.CameraData.from_dict(cam.data())
    rens = [cx_runtime.Renderer(W, H, cx_ctx, cam, gs, params=p, seed=9) for _ in range(3)]
    rens[0].set_exec_mode("megakernel")
    for ren in rens[1:]:
        ren.set_wave_rounds(rounds)
    rens[2].set_graph_mode(True)
    for f in range(4):
        imgs = [ren.launch_frame(cd, f == 0).numpy() for ren in rens]
        for img in imgs[1:]:
            assert np.array_equal(imgs[0].view(np.uint32), img.view(np.uint32)), f
    if mode != "path_tracer":
        ref = rens[0].prefix(rens[0].state().frontBufferIdx)
        for ren in rens[1:]:
            got = ren.prefix(ren.state().frontBufferIdx)
            for k in ref:
                assert np.array_equal(ref[k].view(np.uint32), got[k].view(np.uint32)), k
    assert all(ren.stats().queueOverflow == 0 for ren in rens[1:])


# Pixels: above the most jobs that a tail holds at four lanes each (65536); above them and the most
# possible jobs (two per pixel and neighbour) of a prefix shift that goes to the tail at once.
@pytest.mark.parametrize("W,H", [(401, 301), (1701, 1063)])
@pytest.mark.parametrize("mode", ["path_tracer", "restir_pt_cornell", "conditional_restir"])
def test_rounds_that_leave_the_rest_to_the_tail_match_megakernel(mode, W, H, cx_runtime, cx_ctx):
    """At the default rounds an image of more pixels than the tail holds starts with queue rounds, and
    the round that finds few enough jobs left, known on the device only, hands them to the tail: with
    accumulation, on a closed scene (long paths, whose jobs thin out over the rounds), every frame and
    the reservoirs equal the one-kernel-per-pass mode bit for bit."""
    print(f"rounds and tail {mode} {W}x{H}", flush=True)
    sc = scenes.cornell_box(1, 8)
    gs = cx_runtime.Scene(cx_ctx, sc)
    assert gs.info.bvhWidth == 4
    p = abi.workload_params(mode, W, H, gs.size)
    p.enableAccum = 0 if mode == "conditional_restir" else 1
    cam = scenes.cornell_camera(W, H)
    cd = abi.CameraData.from_dict(cam.data())
    ref, ren = (cx_runtime.Renderer(W, H, cx_ctx, cam, gs, params=p, seed=15) for _ in range(2))
    ref.set_exec_mode("megakernel")
    for f in range(3):
        a, b = (r.launch_frame(cd, f == 0).numpy() for r in (ref, ren))
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), f
    st, sr = ren.stats(), ref.stats()
    assert st.queueOverflow == 0
    # wavefront mode leaves out the shadow rays whose answer changes nothing, and a prefix vertex's
    # second closest-hit ray
    assert 0 < st.shadowRays <= sr.shadowRays
    assert st.closestRays == sr.closestRays if mode == "path_tracer" else 0 < st.closestRays <= sr.closestRays
    assert 0 < st.tailClosestRays + st.tailShadowRays < st.closestRays + st.shadowRays
    if mode != "path_tracer":
        front = ref.state().frontBufferIdx
        x, y = ref.prefix(front), ren.prefix(front)
        for k in x:
            assert np.array_equal(x[k].view(np.uint32), y[k].view(np.uint32)), k


@pytest.mark.parametrize("W,H,neighbours,launches", [(500, 400, 10, 4), (500, 400, 3, 2), (1280, 720, 1, 2),
                                                     (1920, 1080, 1, 6)])
def test_prefix_shift_rounds_follow_the_jobs(W, H, neighbours, launches, cx_runtime, cx_ctx):
    """A prefix shift starts with the tail up to 3.5 M possible jobs, two per pixel and neighbour
    (spatial) or two per pixel (temporal), else it takes two queue rounds, as the prefix walk does:
    the traversal launches of a ReSTIR PT frame say which.  The image is that of two rounds throughout,
    bit for bit."""
    sc = scenes.cornell_box(1, 8)
    gs = cx_runtime.Scene(cx_ctx, sc)
    p = abi.workload_params("restir_pt_cornell", W, H, gs.size)
    p.prefixSpatialCount = neighbours
    cam = scenes.cornell_camera(W, H)
    cd = abi.CameraData.from_dict(cam.data())
    two, ren = (cx_runtime.Renderer(W, H, cx_ctx, cam, gs, params=p, seed=19) for _ in range(2))
    two.set_wave_rounds(2)
    ren.enable_timing(True)
    for f in range(2):
        a, b = (r.launch_frame(cd, f == 0).numpy() for r in (two, ren))
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), f
    st = ren.stats()
    assert st.queueOverflow == 0 and two.stats().queueOverflow == 0
    assert st.traceLaunches == launches


@pytest.mark.parametrize("width", [2, 4, 8])
@pytest.mark.parametrize("queue_grid", [1, 3, 8192])
@pytest.mark.parametrize("mode", ["path_tracer", "conditional_restir"])
def test_queue_paths_match_megakernel(mode, queue_grid, width, cx_runtime, cx_ctx):
    """The traversal of a queue takes one lane per ray when there are more rays than its grid holds
    at four lanes each, or when the tree is not 4-wide; the tail likewise.  A grid of one or three
    blocks over a small image takes the long-queue path, the default grid the four-lane one; both
    with every round in the queue and with the default rounds.  All equal the one-kernel-per-pass
    mode bit for bit."""
    W, H = 61, 37
    sc = tent_grid_scene()
    gs = cx_runtime.Scene(cx_ctx, sc, width=width)
    assert gs.info.bvhWidth == width
    p = abi.workload_params(mode, W, H, gs.size)
    cam = scenes.orbit_camera(sc, W, H)
    cd = abi.CameraData.from_dict(cam.data())
    rens = [cx_runtime.Renderer(W, H, cx_ctx, cam, gs, params=p, seed=31) for _ in range(3)]
    rens[0].set_exec_mode("megakernel")
    for ren in rens[1:]:
        ren.set_queue_grid(queue_grid)
    rens[1].set_wave_rounds(0)
    for f in range(2):
        imgs = [ren.launch_frame(cd, f == 0).numpy() for ren in rens]
        for img in imgs[1:]:
            assert np.array_equal(imgs[0].view(np.uint32), img.view(np.uint32)), f
    assert all(ren.stats().queueOverflow == 0 for ren in rens[1:])
