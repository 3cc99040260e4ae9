"""The shadow prearrange's wavefronts gather (triangle, face) items over lights
and clipped pieces over items until 64 wait, and draw what is left at the end:
maps against the oracle, bit for bit, for triangle counts around multiples of a
wavefront, one light to two launches' worth, faces small enough that most pieces
round to nothing and past the size up to which those are recognised early, with
two-sided and static objects and a light whose near plane cuts triangles."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ntri,lights,dim", [(1, 1, 64), (63, 2, 512), (64, 1, 32), (65, 3, 32), (257, 16, 64),
                                             (1000, 17, 128), (1000, 2, 1148), (1000, 2, 1304)])
def test_left_over_items_and_pieces(gpu_ctx, oracle, ntri, lights, dim):
    from openclrenderer_amd import abi, runtime, scenes
    rng = np.random.default_rng(ntri + lights)
    sc, _ = scenes.config1(shadow=1)
    sc.tris = sc.tris[rng.permutation(len(sc.tris))[:ntri]]
    first = sc.objs["world_pos"][int(sc.tris["v"]["object_id"][0, 0]), :3]
    sc.lights = np.concatenate([scenes.make_light(tuple(first + rng.uniform(-60.0, 60.0, 3) * (1 + 6 * i)), shadow=1,
                                                  is_static=int(i == 1)) for i in range(lights)])
    sc.light_buffer_dim = dim
    sc.objs["feature_flag"][1::5] |= abi.FEATURE_IS_STATIC
    sc.objs["feature_flag"][::3] |= abi.FEATURE_TWO_SIDED
    g = runtime.GpuScene(gpu_ctx, sc)
    g.shadow_pass()
    for got, want in zip(g.read_shadow_maps(), oracle.shadow_maps(sc, 16)):
        assert np.array_equal(got, want), f"{int((got != want).sum())} texels differ"
    g.close()
