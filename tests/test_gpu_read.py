"""ocr_frame_read's triangle ids, formed on the device: the ids of the raw
keys and depth, at frame sizes around a block, for sample-space, tiled and
batched frames, with any subset of outputs asked for."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h", [(4, 4), (16, 16), (257, 1 + 4), (321, 199)])
@pytest.mark.parametrize("how", ["samples", "tiles", "batch"])
def test_ids_from_keys(gpu_ctx, w, h, how):
    from openclrenderer_amd import runtime, scenes
    sc, _ = scenes.random_scene(61, n_tris=70, width=w, height=h)
    view = scenes.make_view(w, h, (0.0, 0.0, -10.0), hfov=70.0)
    g, fr = runtime.GpuScene(gpu_ctx, sc), runtime.Frame(gpu_ctx, w, h)
    if how == "batch":
        b = runtime.Batch(gpu_ctx, 1)
        b.set_views([g], [view], [fr])
        b.render_checked()
        out = fr.read()
    else:
        if how == "tiles":
            fr.set_raster(runtime.RASTER_TILES, 4, 4)
        out = fr.render_read(g, view)
    hip = C.CDLL("libamdhip64.so")
    hip.hipMemcpy.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_int]
    keys = np.empty((h, w), np.uint64)
    assert hip.hipMemcpy(keys.ctypes.data, fr.device_buffers()[1], 8 * w * h, 2) == 0
    assert np.array_equal(runtime.id_keys_to_tri(keys, out["depth"]), out["tri_id"])
    only = fr.read(depth=False, rgba=False, normals=False)
    assert np.array_equal(only["tri_id"], out["tri_id"]) and only["depth"] is None
    # the frame renders on as before
    if how != "batch":
        again = fr.render_read(g, view)
        for k in ("depth", "tri_id", "rgba", "normals"):
            assert np.array_equal(again[k], out[k]), k
    else:
        b.close()
    fr.close()
    g.close()
