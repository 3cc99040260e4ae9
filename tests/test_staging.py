"""Loading and map reads stage through a buffer of the context (runtime.hip,
stage_buffer).  Where the device has no room for all of it they take what there
is, in more parts: what fitted without staging still does.  Host code over the
stand-in for the HIP runtime (device memory is host memory there, kernels are
logged and not run)."""
import pytest

import host_hip

GROUND = """
ctx = runtime.Context(0)
sc, view = scenes.config1(shadow=1)
sc.light_buffer_dim = 64
def count(name):
    return sum(name in k for k in kernels(log()))
"""


@pytest.mark.parametrize("room,parts", [("1 << 40", 1), ("112 * n + 40 * n * 2 + (90 << 10) + 144 * n // 4", 6),
                                        ("112 * n + 40 * n * 2 + (90 << 10) + 147456", 20)])
def test_scene_creation(tmp_path, room, parts):
    out = host_hip.run(tmp_path, GROUND + f"""
n = 20000
sc.tris = np.repeat(sc.tris[:1], n, axis=0)
sc.objs = sc.objs[:1]
sc.tris["v"]["object_id"] = 0
H.host_limit_device({room})
tris, objs = np.ascontiguousarray(sc.tris), np.ascontiguousarray(sc.objs)
h = C.c_void_p()
H.host_clear()
rc = ctx.lib.ocr_scene_create(ctx.h, C.c_void_p(tris.ctypes.data), n, C.c_void_p(objs.ctypes.data), 1, C.byref(h))
print(rc, count("k_split"))
ctx.lib.ocr_scene_destroy(h)
""")
    rc, n = map(int, out.split())
    assert rc == 0 and (n == 1 if parts == 1 else 1 < n <= parts), out


@pytest.mark.parametrize("room,parts", [(1 << 40, 1), (3 << 20, 4), (1 << 20, 8)])
def test_textures(tmp_path, room, parts):
    """Eight textures of 512 x 512: 8 MiB of staging beside three pages."""
    out = host_hip.run(tmp_path, GROUND + f"""
import types
t = types.SimpleNamespace(width=512, height=512, rgba=np.zeros((512, 512, 4), np.uint8))
sc.textures = []
sc.tris, sc.objs = sc.tris[:1], sc.objs[:1]
g = runtime.GpuScene(ctx, sc)
pages = 5 * (16 << 20)                     # 512, 256, 128, 64 and 32 wide
H.host_limit_device({room} + pages - (16 << 20) + 4096)   # the scene's one empty page goes
H.host_clear()
g.upload_textures([t] * 8)
print(count("k_atlas_upload"))
""")
    assert int(out) == parts, out


@pytest.mark.parametrize("room,parts", [(1 << 40, 1), (5000, 64), (1024, 192)])
def test_map_read(tmp_path, room, parts):
    """Two cube maps of 64 x 64: 192 strips of four rows, 1 KiB each."""
    out = host_hip.run(tmp_path, GROUND + f"""
sc.lights = np.concatenate([scenes.make_light((0.0, 0.0, 100.0 * i), shadow=1) for i in range(2)])
sc.textures, sc.tris, sc.objs = [], sc.tris[:1], sc.objs[:1]
g = runtime.GpuScene(ctx, sc)
g.shadow_pass()
H.host_limit_device({room})
H.host_clear()
dyn = np.ones((2, 6, 64, 64), np.uint32)
runtime.check(g.lib.ocr_scene_read_shadow_maps(g.h, C.c_void_p(dyn.ctypes.data), None))
print(count("k_map_rows"))
""")
    assert int(out) == parts, out
