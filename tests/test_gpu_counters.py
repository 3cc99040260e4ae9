"""A render finds its working counters zeroed by the render before it
(ocr_internal.h, make_lists) and clears its buffers in the prearrange launch:
renders in a row, through overflows, changes of the raster path and empty
scenes, give the same frames and statistics as a fresh frame's first."""
import ctypes as C

import numpy as np
import pytest

from openclrenderer_amd import abi, runtime, scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h", [(4, 4), (63, 37), (333, 129), (1024, 768)])
def test_renders_in_a_row(gpu_ctx, w, h):
    views = [scenes.make_view(w, h, (0.0, 0.0, -10.0), c_rot=(0.05 * k, 0.1 * k, 0.0), hfov=70.0) for k in range(2)]
    scs = [scenes.random_scene(40 + k, n_tris=50 + 200 * k)[0] for k in range(2)]
    gs = [runtime.GpuScene(gpu_ctx, s) for s in scs]
    first = []
    for g in gs:
        for v in views:
            f = runtime.Frame(gpu_ctx, w, h)
            out = f.render_read(g, v)
            first.append((out, f.stats()))
            f.close()
    fr = runtime.Frame(gpu_ctx, w, h)
    for k in range(14):
        i, j = k % 2, (k // 2) % 2
        if k == 6:
            fr.set_raster(runtime.RASTER_TILES, 4, 4)
        if k == 9:
            fr.set_raster(runtime.RASTER_SAMPLES)
        if k == 11:
            fr.reserve(1)      # overflows, and grows when read
        out, st = fr.render_read(gs[i], views[j]), fr.stats()
        ref, rst = first[2 * i + j]
        for n in ("depth", "tri_id", "rgba", "normals"):
            assert np.array_equal(out[n], ref[n]), (k, n)
        assert (st["n_cut"], st["n_frag"]) == (rst["n_cut"], rst["n_frag"]), k
    for x in [fr] + gs:
        x.close()


@pytest.mark.parametrize("shift", [0, 4, 8])
def test_noalloc_into_unaligned_buffers(gpu_ctx, shift):
    """Caller buffers at any element boundary: the depth buffer `shift`
    bytes, the id buffer twice that into an allocation."""
    hip = C.CDLL("libamdhip64.so")
    hip.hipMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t]
    hip.hipMemcpy.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_int]
    hip.hipFree.argtypes = [C.c_void_p]
    w, h = 61, 35
    n = w * h
    sc, view = scenes.random_scene(8, n_tris=90, width=w, height=h)
    g, fr = runtime.GpuScene(gpu_ctx, sc), runtime.Frame(gpu_ctx, w, h)
    ref = fr.render_read(g, view)
    base, sizes = [C.c_void_p() for _ in range(4)], (4, 8, 4, 4)
    for b, s in zip(base, sizes):
        assert hip.hipMalloc(C.byref(b), s * n + 64) == 0
    ptr = [b.value + (2 * shift if s == 8 else shift) for b, s in zip(base, sizes)]
    v = np.ascontiguousarray(view, dtype=abi.VIEW)
    for _ in range(3):
        runtime.check(g.lib.ocr_render_noalloc(g.h, v.ctypes.data, *[C.c_void_p(p) for p in ptr], None))
        got = []
        for p, s, dt in zip(ptr, sizes, (np.uint32, np.uint64, np.uint32, np.uint32)):
            a = np.empty(n, dt)
            assert hip.hipMemcpy(a.ctypes.data, p, s * n, 2) == 0
            got.append(a)
        assert np.array_equal(got[0], ref["depth"].ravel())
        assert np.array_equal(runtime.id_keys_to_tri(got[1], got[0]), ref["tri_id"].ravel())
        assert np.array_equal(got[2].view(np.uint8), ref["rgba"].ravel())
        assert np.array_equal(got[3].view(np.uint16), ref["normals"].ravel())
    for b in base:
        hip.hipFree(b)
    for x in (fr, g):
        x.close()


@pytest.mark.parametrize("tiles", [0, 1])
def test_empty_scenes_in_a_row(gpu_ctx, tiles):
    """Scenes without triangles and with none in view, between others."""
    w, h = 161, 97
    view = scenes.make_view(w, h, (0.0, 0.0, -10.0), hfov=70.0)
    away = scenes.make_view(w, h, (0.0, 0.0, -4.0e5), c_rot=(0.0, np.pi, 0.0), hfov=70.0)
    full, _ = scenes.random_scene(44, n_tris=300)
    none, _ = scenes.random_scene(45, n_tris=30)
    none.tris = none.tris[:0]
    gs = [runtime.GpuScene(gpu_ctx, s) for s in (full, none)]
    fr = runtime.Frame(gpu_ctx, w, h)
    if tiles:
        fr.set_raster(runtime.RASTER_TILES, 4, 4)
    ref, st = fr.render_read(gs[0], view), fr.stats()
    assert st["n_cut"] > 0 and np.count_nonzero(ref["tri_id"] != 0xFFFFFFFF) > 0
    for k in range(9):
        for g, v in ((gs[1], view), (gs[0], away))[: 1 + k % 2]:
            out, e = fr.render_read(g, v), fr.stats()
            assert (e["n_cut"], e["n_frag"]) == (0, 0), k
            assert (out["tri_id"] == 0xFFFFFFFF).all() and (out["depth"] == 0xFFFFFFFF).all(), k
        out, e = fr.render_read(gs[0], view), fr.stats()
        for n in ("depth", "tri_id", "rgba", "normals"):
            assert np.array_equal(out[n], ref[n]), (k, n)
        assert (e["n_cut"], e["n_frag"]) == (st["n_cut"], st["n_frag"]), k
    for x in [fr] + gs:
        x.close()
