"""Passes launched one by one (cx_renderer_begin_frame + cx_pass_launch), eagerly and recorded into
the caller's graph, beside whole frames and graph replays on the same renderer.  What a pass
enqueues does not depend on what the host saw before it: every image and reservoir equals that of
the one-kernel-per-pass mode, which has no queues, bit for bit."""
import ctypes as C

import numpy as np
import pytest

from crisoptix_amd import abi, scenes
from parity_util import tent_grid_scene

pytestmark = pytest.mark.gpu

(PREFIX_GEN_TEMP, PREFIX_SPATIAL, SUFFIX_GEN_TEMP, SUFFIX_SPATIAL, STORE_ENTRIES, ENTRIES_BUILD,
 FINAL_GATHER) = range(7)
W, H = 40, 24


def _params(name, size):
    """The settings whose frames take the most machines: two gathers, prefix spatial reuse; eight gathers
    take more than there are sets of counters (16)."""
    mode = "conditional_restir" if name in ("gather2", "gather8", "prefix_spatial") else name
    p = abi.workload_params(mode, W, H, size)
    if mode == "conditional_restir":
        p.gatherRadius = 0.6
        p.gatherN = {"gather2": 2, "gather8": 8}.get(name, 1)
        p.prefixEnableSpatial = 1 if name == "prefix_spatial" else 0
        p.prefixSpatialRounds = 2
    if mode == "path_tracer":
        p.enableAccum = 1
    return p


def _passes(p):
    """The passes of one frame in order, with the spatial round of each."""
    out = [(PREFIX_GEN_TEMP, 0)]
    restir = p.rendererType != abi.CX_PATH_TRACER
    cond = p.rendererType == abi.CX_CONDITIONAL_RESTIR
    if restir and p.prefixEnableSpatial:
        out += [(PREFIX_SPATIAL, i) for i in range(p.prefixSpatialRounds)]
    if cond:
        out.append((SUFFIX_GEN_TEMP, 0))
        if p.suffixEnableSpatial and p.suffixSpatialCount > 0:
            out += [(SUFFIX_SPATIAL, i) for i in range(p.suffixSpatialRounds)]
        out += [(STORE_ENTRIES, 0), (ENTRIES_BUILD, 0), (FINAL_GATHER, 0)]
    return out


def _begin(rt, ren, cd, changed, out):
    ren.ctx.check(rt.lib().cx_renderer_begin_frame(ren.h, C.byref(cd), 1 if changed else 0, out.ptr), "begin_frame")


def _launch_passes(rt, ren, stream=None):
    lp = ren.params()
    for which, rnd in _passes(lp):
        lp.spatialRoundIdx = rnd
        ren.ctx.check(rt.lib().cx_pass_launch(ren.h, which, C.byref(lp), stream), "cx_pass_launch")


def _hand_frame(rt, ren, cd, changed):
    _begin(rt, ren, cd, changed, ren.output)
    _launch_passes(rt, ren)
    return ren.output


def _equal(a, b, tag):
    assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), tag


def _same_records(ref, ren, tag):
    for which in (0, 1):
        a, b = ref.prefix(which), ren.prefix(which)
        for k in a:
            _equal(np.ascontiguousarray(a[k]), np.ascontiguousarray(b[k]), (tag, which, k))


@pytest.mark.parametrize("rounds", [abi.CX_WAVE_ROUNDS_DEFAULT, 1])
@pytest.mark.parametrize("name", ["path_tracer", "restir_pt_cornell", "gather2", "gather8", "prefix_spatial"])
def test_recorded_passes_replay(name, rounds, cx_runtime, cx_ctx):
    """One frame's passes recorded into a caller's graph and replayed four times, with eager work and
    synchronisations between, against the same passes launched eagerly as often."""
    import torch
    print(f"recorded passes {name} rounds {rounds}", flush=True)
    sc = tent_grid_scene()
    gs = cx_runtime.Scene(cx_ctx, sc)
    p = _params(name, gs.size)
    cam = scenes.orbit_camera(sc, W, H)
    cd = abi.CameraData.from_dict(cam.data())
    ref = cx_runtime.Renderer(W, H, cx_ctx, cam, gs, params=p, seed=5)
    rec = cx_runtime.Renderer(W, H, cx_ctx, cam, gs, params=p, seed=5)
    ref.set_exec_mode("megakernel")
    rec.set_wave_rounds(rounds)
    for f in range(2):
        _equal(ref.launch_frame(cd, f == 0).numpy(), rec.launch_frame(cd, f == 0).numpy(), ("eager", f))
    stream = torch.cuda.Stream()
    _begin(cx_runtime, ref, cd, False, ref.output)
    _begin(cx_runtime, rec, cd, False, rec.output)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        _launch_passes(cx_runtime, rec, stream.cuda_stream)
    side = torch.ones(1024, device="cuda")
    for f in range(4):
        graph.replay()
        stream.synchronize()
        _launch_passes(cx_runtime, ref)
        cx_runtime.synchronize()
        _equal(ref.output.numpy(), rec.output.numpy(), ("replay", f))
        if p.rendererType != abi.CX_PATH_TRACER:
            _same_records(ref, rec, f)
        side.mul_(1.0001)
        torch.cuda.synchronize()
    assert rec.stats().queueOverflow == 0
    # whole frames and passes after the replays
    for f in range(3):
        go = _hand_frame if f == 1 else (lambda rt, r, c, ch: r.launch_frame(c, ch))
        _equal(go(cx_runtime, ref, cd, False).numpy(), go(cx_runtime, rec, cd, False).numpy(), ("after", f))
    assert rec.stats().queueOverflow == 0


@pytest.mark.parametrize("rounds", [abi.CX_WAVE_ROUNDS_DEFAULT, 1])
@pytest.mark.parametrize("name", ["gather2", "gather8", "prefix_spatial"])
def test_hand_driven_frames_between_graph_replays(name, rounds, cx_runtime, cx_ctx):
    """Graph-mode frames, frames driven pass by pass and frames of another renderer type, which
    takes fewer machines, in turn on one renderer."""
    print(f"mixed frames {name} rounds {rounds}", flush=True)
    sc = tent_grid_scene()
    gs = cx_runtime.Scene(cx_ctx, sc)
    p = _params(name, gs.size)
    other = abi.LaunchParams.from_buffer_copy(p)
    other.rendererType = abi.CX_PATH_TRACER
    cam = scenes.orbit_camera(sc, W, H)
    cd = abi.CameraData.from_dict(cam.data())
    ref = cx_runtime.Renderer(W, H, cx_ctx, cam, gs, params=p, seed=7)
    ren = cx_runtime.Renderer(W, H, cx_ctx, cam, gs, params=p, seed=7)
    ref.set_exec_mode("megakernel")
    ren.set_wave_rounds(rounds)
    ren.set_graph_mode(True)
    # f: a whole frame (captured or replayed), p: the frame pass by pass, t: a whole path-traced
    # frame, e: a whole frame enqueued without graph mode
    for f, kind in enumerate("ffffpfpffptfpfepfppfff"):
        for r in (ref, ren):
            r.set_params(other if kind == "t" else p)
        ren.set_graph_mode(kind != "e")
        if kind == "p":
            a, b = (_hand_frame(cx_runtime, r, cd, f == 0) for r in (ref, ren))
        else:
            a, b = (r.launch_frame(cd, f == 0) for r in (ref, ren))
        _equal(a.numpy(), b.numpy(), (f, kind))
        _same_records(ref, ren, (f, kind))
    assert ren.stats().queueOverflow == 0
