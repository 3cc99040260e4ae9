"""The shadow pass's list (runtime.hip, shadow_list_cap): what does not fit is
drawn by single wavefronts, so every list of a small scene holds the six pieces
a triangle can have per light, whichever partition they fall in, and a larger
one three for two triangles and a light.  Allocations over the stand-in for the
HIP runtime; and the maps of a room whose pieces all are large against the
oracle."""
import numpy as np
import pytest

import host_hip

MB = 1 << 20


@pytest.mark.parametrize("ntri,lights,least,most", [
    (1, 1, 6, 1), (12, 16, 6, 6), (48, 17, 6, 20), (768, 4, 6, 65), (12288, 4, 4, 65), (16384, 16, 3, 65),
    (200_000, 4, 1.5, 83), (300_000, 3, 1.5, 91), (1_000_000, 16, 0.8, 897)])
def test_room_for_the_pieces(tmp_path, ntri, lights, least, most):
    out = host_hip.run(tmp_path, f"""
ctx = runtime.Context(0)
sc, _ = scenes.config1(shadow=1)
sc.tris = np.repeat(sc.tris[:1], {ntri}, axis=0)
sc.lights = np.concatenate([scenes.make_light((0.0, 0.0, 100.0 * i), shadow=1) for i in range({lights})])
sc.light_buffer_dim = 16
g = runtime.GpuScene(ctx, sc)
before = H.host_device_bytes()
g.shadow_pass()
print(H.host_device_bytes() - before)
""")
    records = int(out) // 64
    blocks = -(-ntri // 256)
    assert records // 64 >= least * -(-blocks // 64) * min(ntri, 256) * min(lights, 16), records
    assert records * 64 <= most * MB


@pytest.mark.gpu
@pytest.mark.parametrize("split,lights,dim", [(1, 3, 64), (2, 16, 64), (9, 5, 256)])
def test_room_around_its_lights(gpu_ctx, oracle, split, lights, dim):
    """Six two-sided walls of split x split quads around the lights: every
    piece goes to the list, many triangles have several."""
    from openclrenderer_amd import abi, runtime, scenes
    lin = np.linspace(-1000.0, 1000.0, split + 1)
    u, v = (a.ravel() for a in np.meshgrid(np.arange(split), np.arange(split)))
    tris = []
    for axis in range(3):
        for side in (-1000.0, 1000.0):
            def corner(i, j):
                p = np.zeros((len(u), 3))
                p[:, axis], p[:, (axis + 1) % 3], p[:, (axis + 2) % 3] = side, lin[i], lin[j]
                return p
            a, b, c, d = corner(u, v), corner(u + 1, v), corner(u + 1, v + 1), corner(u, v + 1)
            tris += [np.stack([a, b, c], 1), np.stack([a, c, d], 1)]
    pos = np.concatenate(tris)
    sc, _ = scenes.config1(shadow=1)
    t = np.zeros(len(pos), sc.tris.dtype)
    t["v"] = sc.tris["v"][0]
    t["v"]["pos"][..., :3] = pos
    t["v"]["object_id"] = 0
    sc.tris, sc.objs = t, sc.objs[:1].copy()
    sc.objs["world_pos"], sc.objs["scale"] = 0.0, 1.0
    sc.objs["world_rot_quat"] = (0.0, 0.0, 0.0, 1.0)
    sc.objs["feature_flag"] = abi.FEATURE_TWO_SIDED
    rng = np.random.default_rng(split)
    sc.lights = np.concatenate([scenes.make_light(tuple(rng.uniform(-700.0, 700.0, 3)), shadow=1) for _ in range(lights)])
    sc.light_buffer_dim = dim
    g = runtime.GpuScene(gpu_ctx, sc)
    g.shadow_pass()
    got, want = g.read_shadow_maps()[0], oracle.shadow_maps(sc, 16)[0]
    assert np.count_nonzero(want != 0xFFFFFFFF) > want.size // 2
    assert np.array_equal(got, want), f"{int((got != want).sum())} texels differ"
    g.close()
