"""Who zeroes a list's working counters (ocr_internal.h, make_lists and
WorkState): a render leaves them zero, so the next one need not; after one that
was not enqueued to its end, and in a recorded one, which runs later, the
render zeroes them itself.  The no-allocation render's list belongs to the GPU,
not to a context.  Host code over the stand-in for the HIP runtime."""
import numpy as np
import pytest

import host_hip

GROUND = """
ctxs = [runtime.Context(0), runtime.Context(0)]
sc, view = scenes.random_scene(3)
gs = [runtime.GpuScene(c, sc) for c in ctxs]
buf = np.zeros(64 * 48, np.uint64)
st = stream()
def noalloc(g):
    v = np.ascontiguousarray(view, dtype=abi.VIEW)
    runtime.check(g.lib.ocr_render_noalloc(g.h, v.ctypes.data, *[buf.ctypes.data] * 4, st))
def zeroed(call):
    H.host_clear()
    call()
    ks = kernels(log())
    assert any("k_shade" in k for k in ks) or not ks
    return int("k_zero_work" in (ks or [""])[0])
def failing(call, n):
    H.host_fail_launch(n)
    try:
        call()
        raise SystemExit("no error")
    except runtime.OcrError:
        pass
"""


def test_noalloc_after_a_failed_call(tmp_path):
    out = host_hip.run(tmp_path, GROUND + """
r = [zeroed(lambda: noalloc(gs[0])), zeroed(lambda: noalloc(gs[1]))]
for n in (1, 2, 3):
    failing(lambda: noalloc(gs[0]), n)     # depth, ids, shading not enqueued
    r += [zeroed(lambda: noalloc(gs[1])), zeroed(lambda: noalloc(gs[0]))]
print(*r)
""")
    assert out.split() == ["0", "0"] + ["1", "0"] * 3, out


def test_recorded_renders_zero_their_own(tmp_path):
    """Recorded: always, without a word about the present state."""
    out = host_hip.run(tmp_path, GROUND + """
fr, fb = runtime.Frame(ctxs[0], 64, 48), runtime.Frame(ctxs[0], 64, 48)
b = runtime.Batch(ctxs[0], 1)
b.set_views([gs[0]], [view], [fb])
for call, n in ((lambda: noalloc(gs[0]), 1), (lambda: b.render(st), 1)):
    r = [zeroed(call)]
    H.host_capture(st, 1); r.append(zeroed(call)); H.host_capture(st, 0)
    r.append(zeroed(call))
    failing(call, n)
    H.host_capture(st, 1); r.append(zeroed(call)); H.host_capture(st, 0)
    r += [zeroed(call), zeroed(call)]      # the recorded one has not run
    print(*r)
fr.close()
""")
    assert [l.split() for l in out.split("\n") if l] == [["0", "1", "0", "1", "1", "0"]] * 2, out


def test_renders_and_batches_after_a_failed_one(tmp_path):
    out = host_hip.run(tmp_path, GROUND + """
fr, fb = runtime.Frame(ctxs[0], 64, 48), runtime.Frame(ctxs[0], 64, 48)
b = runtime.Batch(ctxs[0], 1)
b.set_views([gs[0]], [view], [fb])
r = [zeroed(lambda: b.render(st))]
failing(lambda: b.render(st), 2)
r += [zeroed(lambda: b.render(st)), zeroed(lambda: b.render(st))]
for _ in range(3): fr.render(gs[0], view, st)
failing(lambda: fr.render(gs[0], view, st), 2)
r += [zeroed(lambda: fr.render(gs[0], view, st)) for _ in range(6)]
print(*r)
""")
    got = out.split()
    assert got[:3] == ["0", "1", "0"], out
    assert got[3:].count("1") == 1, out    # the set of the failed one, when its turn comes


@pytest.mark.gpu
def test_recorded_noalloc_replays(gpu_ctx):
    """A recorded no-allocation render, replayed between eager ones of another
    view and size, draws its view each time."""
    import ctypes as C

    from openclrenderer_amd import abi, runtime, scenes
    hip = C.CDLL("libamdhip64.so")
    vp = C.c_void_p

    def ok(name, *args):
        rc = getattr(hip, name)(*args)
        assert rc == 0, (name, rc)

    sc, view = scenes.config1()
    g, fr = runtime.GpuScene(gpu_ctx, sc), runtime.Frame(gpu_ctx, 800, 600)
    ref = fr.render_read(g, view)
    small = np.ascontiguousarray(scenes.make_view(96, 64, (30.0, 0.0, -900.0)), dtype=abi.VIEW)
    big = np.ascontiguousarray(view, dtype=abi.VIEW)
    n, sizes = 800 * 600, (4, 8, 4, 4)
    out, other = [vp() for _ in sizes], [vp() for _ in sizes]
    for p, s in zip(out + other, sizes * 2):
        ok("hipMalloc", C.byref(p), C.c_size_t(s * n))
    st, graph, ex = vp(), vp(), vp()
    ok("hipStreamCreateWithFlags", C.byref(st), C.c_uint(1))

    def render(v, to):
        runtime.check(g.lib.ocr_render_noalloc(g.h, v.ctypes.data, *to, st))

    render(small, other)
    ok("hipStreamSynchronize", st)
    ok("hipStreamBeginCapture", st, C.c_int(1))
    render(big, out)
    ok("hipStreamEndCapture", st, C.byref(graph))
    ok("hipGraphInstantiate", C.byref(ex), graph, None, None, C.c_size_t(0))
    for i in range(4):
        for p, s in zip(out, sizes):
            ok("hipMemset", p, C.c_int(i), C.c_size_t(s * n))
        ok("hipDeviceSynchronize")
        ok("hipGraphLaunch", ex, st)
        ok("hipStreamSynchronize", st)
        for k, name in ((0, "depth"), (2, "rgba"), (3, "normals")):
            got = np.empty(n, np.uint32)
            ok("hipMemcpy", got.ctypes.data_as(vp), out[k], C.c_size_t(4 * n), C.c_int(2))
            assert np.array_equal(got, np.ascontiguousarray(ref[name]).reshape(-1).view(np.uint32)), (i, name)
        render(small, other)
        ok("hipStreamSynchronize", st)
    ok("hipGraphExecDestroy", ex)
    ok("hipGraphDestroy", graph)
    fr.close()
    g.close()
    ok("hipStreamDestroy", st)
    for p in out + other:
        ok("hipFree", p)
