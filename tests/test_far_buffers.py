"""Buffers above 4 GiB that shading gathers from (shade.hip, ocr_internal.h
needs_far): cut lists of more than 2^27 records, whose last partitions begin
beyond 4 GiB however little is visible, atlases of more than 256 pages, cube
maps of more than 2^30 texels.  The kernels with 32-bit byte offsets run up to
4 GiB and no further."""
import numpy as np
import pytest

import host_hip

GROUND = """
ctx = runtime.Context(0)
def shading(call):
    H.host_clear()
    call()
    return [k for k in kernels(log()) if "k_shade" in k]
"""


def test_cut_list_variant(tmp_path):
    """Views of one scene of 2^20 triangles: 64 of them have 2^26 triangle
    slots and a list of 2^27 records and one block per partition."""
    out = host_hip.run(tmp_path, GROUND + """
sc, view = scenes.random_scene(3)
sc.tris = np.repeat(sc.tris[:1], 1 << 20)
g = runtime.GpuScene(ctx, sc)
frames = [runtime.Frame(ctx, 64, 48) for _ in range(64)]
for n in (63, 64):
    b = runtime.Batch(ctx, n)
    b.set_views([g] * n, [view] * n, frames[:n])
    print(n, *shading(b.render))
    b.close()
b = runtime.Batch(ctx, 64)
b.set_views([g] * 63, [view] * 63, frames[:63])
H.host_clear(); b.launch_graph(); print("graph", *[k for k in kernels(log()) if "k_shade" in k])
b.set_views([g] * 64, [view] * 64, frames)
H.host_clear(); b.launch_graph(); print("graph", *[k for k in kernels(log()) if "k_shade" in k])
""")
    lines = out.split("\n")
    assert "k_shade_batch_unshadowed" in lines[0] and "k_shade_batch_far" in lines[1], out
    assert "k_shade_batch_unshadowed" in lines[2] and "k_shade_batch_far" in lines[3], out


def test_small_views_in_a_large_list(tmp_path):
    """A list that grew beyond 4 GiB serves small renders from its front."""
    out = host_hip.run(tmp_path, GROUND + """
sc, view = scenes.random_scene(3)
sc.tris = np.repeat(sc.tris[:1], 1 << 20)
g = runtime.GpuScene(ctx, sc)
frames = [runtime.Frame(ctx, 64, 48) for _ in range(64)]
b = runtime.Batch(ctx, 64)
for n in (64, 63, 1):
    b.set_views([g] * n, [view] * n, frames[:n])
    print(n, *shading(b.render), *[k for k in shading(b.launch_graph) if "shade" in k])
""")
    lines = out.split("\n")
    assert lines[0].count("k_shade_batch_far") == 2, out
    assert lines[1].count("k_shade_batch_unshadowed") == lines[2].count("k_shade_batch_unshadowed") == 2, out


def test_atlas_and_map_variants(tmp_path):
    out = host_hip.run(tmp_path, GROUND + """
rgba = np.zeros((2048, 2048, 4), np.uint8)
sc, view = scenes.random_scene(3)
fr = runtime.Frame(ctx, 64, 48)
for n in (150, 200):
    sc.textures = [scenes.Texture(2048, 2048, rgba)] * n
    g = runtime.GpuScene(ctx, sc)
    pages = C.c_uint32()
    runtime.check(g.lib.ocr_scene_atlas_info(g.h, C.byref(pages), None, None, None))
    print(pages.value, *shading(lambda: fr.render(g, view)))
    g.close()
sc.textures = sc.textures[:1]
g = runtime.GpuScene(ctx, sc)
for static in (0, 1):
    for n in (11, 12):
        g.upload_lights(np.concatenate([scenes.make_light((0.0, 0.0, 0.0), shadow=1, is_static=static)] * n), 4000)
        print(static, n, *shading(lambda: fr.render(g, view)))
""")
    rows = [l.split() for l in out.split("\n") if l]
    assert int(rows[0][0]) <= 256 < int(rows[1][0]), out
    for r in rows:
        far = int(r[0]) > 256 or r[1] == "12"
        assert ("k_shade_far" in r[-1]) == far, r


@pytest.mark.gpu
def test_batch_list_above_4_gib(gpu_ctx):
    """66 views of 2^20 triangles each, a few thousand of them visible from
    each camera (the list's last partition begins beyond record 2^27): every
    view is what the scene's own render is."""
    from openclrenderer_amd import runtime, scenes
    n = 1 << 20
    base = scenes.small_scene(5, 16, 6000, box_units=8.0)
    base.objs["scale"] *= 2.0
    sc = scenes.Scene(np.zeros(n, base.tris.dtype), base.objs, base.lights, base.textures, base.light_buffer_dim, "far")
    sc.tris["v"]["pos"][:, :, :3] = 1.0        # no area: culled
    # in every block of 256, so that every partition holds visible records
    sc.tris[np.linspace(0, n - 1, len(base.tris)).astype(np.int64)] = base.tris
    rng = np.random.default_rng(1)
    views = [scenes.orbit_view(rng, 160, 120, 6.0) for _ in range(4)]
    g, fr = runtime.GpuScene(gpu_ctx, sc), runtime.Frame(gpu_ctx, 160, 120)
    refs = [fr.render_read(g, v) for v in views]
    frames = [runtime.Frame(gpu_ctx, 160, 120) for _ in range(66)]
    b = runtime.Batch(gpu_ctx, 66)
    b.set_views([g] * 66, [views[i % 4] for i in range(66)], frames)
    for launch in (b.render, b.launch_graph):
        launch()
        b.stats()
        for i in (0, 1, 2, 31, 63, 64, 65):
            out = frames[i].read()
            for k in ("depth", "tri_id", "normals", "rgba"):
                assert np.array_equal(out[k], refs[i % 4][k]), (i, k)
    assert all(np.count_nonzero(r["depth"] != 0xFFFFFFFF) > 500 for r in refs)
    for x in [b, *frames, fr, g]:
        x.close()


@pytest.mark.gpu
def test_atlas_above_4_gib(gpu_ctx):
    """200 textures of 2048^2 (268 pages): an object's frame with the first or
    the last of them is that of the texture alone."""
    from openclrenderer_amd import runtime, scenes
    sc, _ = scenes.config1()
    view = scenes.make_view(800, 600, (0.0, 0.0, -1.2 * scenes.UNIT))   # close: the full-size level is read
    tex = [scenes.value_noise_texture(2048, 7 + i, lattice=16) for i in range(2)]
    fr = runtime.Frame(gpu_ctx, 800, 600)
    sc.textures, ref = [tex[0]], []
    for t in tex:
        sc.textures = [t]
        g = runtime.GpuScene(gpu_ctx, sc)
        ref.append(fr.render_read(g, view))
        g.close()
    sc.textures = [tex[0]] + [tex[1]] * 199
    for tid in (0, 199):
        sc.objs["tid"] = tid
        g = runtime.GpuScene(gpu_ctx, sc)
        out = fr.render_read(g, view)
        g.close()
        assert np.array_equal(out["rgba"], ref[tid != 0]["rgba"]), tid
    assert not np.array_equal(ref[0]["rgba"], ref[1]["rgba"])
    fr.close()


@pytest.mark.gpu
def test_maps_above_4_gib(gpu_ctx):
    """The last of twelve shadow-casting lights of 4000^2 texels a face, the
    others without colour, shades as it does alone; as a static light too."""
    from openclrenderer_amd import abi, runtime, scenes
    sc, view = scenes.config1(shadow=1)
    sc.objs["feature_flag"][1::3] |= abi.FEATURE_IS_STATIC
    last = scenes.make_light((150.0, -420.0, -260.0), col=(1.0, 0.9, 0.7), shadow=1, is_static=1)
    black = [scenes.make_light((40.0 * i, -300.0, 30.0 * i), col=(0.0, 0.0, 0.0), shadow=1, is_static=1) for i in range(11)]
    fr = runtime.Frame(gpu_ctx, 800, 600)
    out = []
    for lights in ([last], black + [last]):
        sc.lights, sc.light_buffer_dim = np.concatenate(lights), 4000
        g = runtime.GpuScene(gpu_ctx, sc)
        g.shadow_pass()
        out.append(fr.render_read(g, view))
        g.close()
    # the ambient share of a light without colour is nothing
    assert np.array_equal(out[0]["rgba"], out[1]["rgba"])
    fr.close()
