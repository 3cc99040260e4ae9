"""Pieces and reference fragments of a render are counted in one 64-bit add
per block (raster.hip, block_alloc): a frame of so many fragments that their
sum passes 2^32 still counts its pieces right, and the fragments modulo 2^32."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIDE = 1440


def _lines(runs):
    """`n` triangles of zero area for each (n, length) of `runs`: diagonals
    `length` pixels across, two of their vertices the same."""
    from openclrenderer_amd import abi, scenes
    sc, _ = scenes.config1()
    view = scenes.make_view(SIDE, SIDE, (0.0, 0.0, 0.0))
    z = 1000.0
    tris = np.zeros(sum(n for n, _ in runs), sc.tris.dtype)
    tris["v"] = sc.tris["v"][0]
    tris["v"]["object_id"] = 0
    at = 0
    for n, length in runs:
        lo = (1 - SIDE / 2) * z / float(view["fov_const"][0])
        hi = (1 + length - SIDE / 2) * z / float(view["fov_const"][0])
        p = tris["v"]["pos"][at:at + n]
        p[:, 0, :3] = (lo, lo, z)
        p[:, 1:, :3] = (hi, hi, z)
        at += n
    sc.tris = tris
    sc.objs = sc.objs[:1].copy()
    sc.objs["world_pos"] = 0.0
    sc.objs["scale"] = 1.0
    sc.objs["world_rot_quat"] = (0.0, 0.0, 0.0, 1.0)
    sc.objs["feature_flag"] = abi.FEATURE_TWO_SIDED
    return sc, view


def _counts(ctx, runs):
    from openclrenderer_amd import runtime
    sc, view = _lines(runs)
    g, fr = runtime.GpuScene(ctx, sc), runtime.Frame(ctx, SIDE, SIDE)
    fr.render(g, view)
    st = fr.stats()
    fr.close()
    g.close()
    assert not st["overflow"]
    return st["n_cut"], st["n_frag"]


@pytest.mark.parametrize("runs", [((1_060_000, 1436),), ((300_000, 90), (700_000, 1436), (70_001, 700))])
def test_many_fragments(gpu_ctx, runs):
    total = 0
    for n, length in runs:
        one = _counts(gpu_ctx, ((1, length),))
        assert one[0] == 1 and one[1] >= length * length // 500, one
        total += n * one[1]
    assert len(runs) > 1 or total >= 2**32
    assert _counts(gpu_ctx, runs) == (sum(n for n, _ in runs), total % 2**32)
