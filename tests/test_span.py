"""The raster passes' row form (raster.hip: span_exact, edge_span) covers the
pixels that point_in_tri (cl2.cl:4798-4807) covers, row by row, for every
triangle it accepts, and a triangle of zero rounded area that it accepts
covers none: tests/span_check.c over triangles from below a pixel to many
times the screen, with horizontal, vertical and collinear ones among them, on
frames of 64x48 to 3840x2160 and cube faces to 4000x4000."""
import os
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.parametrize("seed", ["1", "2"])
def test_rows_equal_point_in_tri(tmp_path, seed):
    exe = str(tmp_path / "span_check")
    subprocess.run(["gcc", "-O2", "-ffp-contract=off", "-o", exe, os.path.join(HERE, "span_check.c"), "-lm"], check=True)
    r = subprocess.run([exe, "60000", seed], capture_output=True, text=True, timeout=300)
    print(r.stdout)
    assert r.returncode == 0 and " 0 mismatches" in r.stdout, r.stdout
    assert int(r.stdout.split("exact ")[1].split(",")[0]) > 500000


@pytest.mark.gpu
@pytest.mark.parametrize("size,tris,spread", [((64, 48), 3, 20.0), ((67, 33), 400, 6.0), ((640, 360), 3000, 25.0),
                                              ((1279, 719), 200, 400.0), ((3840, 2160), 60, 3000.0)])
def test_chunks_and_rows_match_oracle(gpu_ctx, oracle, size, tris, spread):
    """Frames whose sample totals take every chunk size, from a few samples
    in one chunk to more than the largest chunk's share, over triangles of
    one pixel to ones far larger than the screen (drawn sample by sample)."""
    from openclrenderer_amd import runtime, scenes
    w, h = size
    sc, _ = scenes.random_scene(900 + w, n_tris=tris, width=w, height=h)
    view = scenes.make_view(w, h, (0.0, 0.0, -10.0), hfov=70.0)
    rng = np.random.default_rng(w)
    px = 400.0 / float(view["fov_const"][0])
    centre = rng.uniform(-0.5, 0.5, (tris, 1, 2)) * [w * px, h * px]
    sc.tris["v"]["pos"][:, :, :2] = centre + rng.normal(size=(tris, 3, 2)) * spread * px
    sc.tris["v"]["pos"][:, :, 2] = rng.uniform(-50, 50, (tris, 3))
    sc.objs["world_pos"][:, :3] = (0.0, 0.0, 400.0)
    sc.objs["world_rot_quat"] = (0.0, 0.0, 0.0, 1.0)
    sc.objs["scale"] = 1.0
    g, fr = runtime.GpuScene(gpu_ctx, sc), runtime.Frame(gpu_ctx, w, h)
    out, ref = fr.render_read(g, view), oracle.render(sc, view)
    assert np.count_nonzero(ref["tri_id"] != 0xFFFFFFFF) > 0
    for k in ("depth", "tri_id", "rgba", "normals"):
        assert np.array_equal(out[k], ref[k]), k
    fr.close()
    g.close()


@pytest.mark.gpu
@pytest.mark.parametrize("n_inst,tris", [(4, 16200), (8, 33000), (40, 300000)])
def test_partitioned_lists_match_reserved(gpu_ctx, n_inst, tris):
    """Lists of 1, 2 and 32 partitions (triangle counts around 64 and 128
    blocks of 256, and far more) give the frames and statistics of a reserved
    list, which has one partition and blocks of 512."""
    from openclrenderer_amd import runtime, scenes
    sc = scenes.small_scene(77 + n_inst, n_inst, tris, box_units=8.0)
    view = scenes.make_view(401, 303, (0.0, 0.0, -1300.0))
    g = runtime.GpuScene(gpu_ctx, sc)
    a, b = runtime.Frame(gpu_ctx, 401, 303), runtime.Frame(gpu_ctx, 401, 303)
    b.reserve(2 * sc.ntri + 64)
    oa, ob = a.render_read(g, view), b.render_read(g, view)
    for k in ("depth", "tri_id", "rgba", "normals"):
        assert np.array_equal(oa[k], ob[k]), k
    sa, sb = a.stats(), b.stats()
    assert sa["n_cut"] == sb["n_cut"] > 0 and sa["n_frag"] == sb["n_frag"] > 0
    for x in (a, b, g):
        x.close()
