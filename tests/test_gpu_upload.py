"""Scene and texture uploads in pieces: texture groups split by count and by
staging size give the oracle's atlas, and triangles staged in more than one
chunk arrive whole."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [[(16, 16)] * 65, [(2048, 2048)] * 5 + [(33, 17)],
                                   [(1, 16), (100, 60), (256, 256), (2047, 3)] * 17])
def test_texture_groups(gpu_ctx, oracle, sizes):
    from openclrenderer_amd import runtime, scenes
    rng = np.random.default_rng(len(sizes))
    texs = [scenes.Texture(w, h, rng.integers(0, 256, (h, w, 4), dtype=np.uint8)) for w, h in sizes]
    sc, _ = scenes.random_scene(5)
    sc.textures = texs
    g = runtime.GpuScene(gpu_ctx, sc)
    pages, nums, sz, ms = g.read_atlas()
    op, on, osz, oms = oracle.atlas(texs)
    assert ms == oms and np.array_equal(nums, on) and np.array_equal(sz, osz[:sz.shape[0]])
    assert np.array_equal(pages, op.reshape(pages.shape))
    g.close()


@pytest.mark.parametrize("n", [1, 255, 257, 400000, 400001])
def test_triangle_chunks(gpu_ctx, oracle, n):
    """The first and last triangles of a scene of n are drawn (the rest lies
    behind the camera) with the attributes they were given."""
    from openclrenderer_amd import runtime, scenes
    base, view = scenes.random_scene(12, n_tris=max(8, min(n, 40)), width=96, height=64)
    k = min(n, 20)
    sc = scenes.Scene(np.zeros(n, base.tris.dtype), base.objs, base.lights, base.textures, base.light_buffer_dim, "chunks")
    sc.tris["v"]["pos"][:, :, 2] = -5000.0
    sc.tris[:k] = base.tris[:k]
    sc.tris[n - k:] = base.tris[-k:] if n > 2 * k else base.tris[:k]
    g, fr = runtime.GpuScene(gpu_ctx, sc), runtime.Frame(gpu_ctx, 96, 64)
    out, ref = fr.render_read(g, view), oracle.render(sc, view)
    for name in ("depth", "tri_id", "rgba", "normals"):
        assert np.array_equal(out[name], ref[name]), name
    fr.close()
    g.close()
