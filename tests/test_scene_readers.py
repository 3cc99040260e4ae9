"""A scene keeps the events of the renders that read it (ocr_internal.h,
Scene::note_read) until an update or a shadow pass has waited for them, and of
frames that are gone none: a scene that is rendered into frames made and
dropped for each picture holds no more than the last few.  Host code over the
stand-in for the HIP runtime."""
import host_hip


def test_transient_frames_leave_no_events(tmp_path):
    out = host_hip.run(tmp_path, """
ctx = runtime.Context(0)
sc, view = scenes.random_scene(3)
lit, _ = scenes.config1(shadow=1)
for scene in (sc, lit):
    g = runtime.GpuScene(ctx, scene)
    g.shadow_pass()
    n = []
    for k in range(60):
        fr = runtime.Frame(ctx, 64, 48)
        for _ in range(3): fr.render(g, view)
        fr.close()
        n.append(H.host_live_events())
    print(n[5], n[59])
    g.update_objs_async(0, scene.objs[:1])
    g.shadow_pass()
    fr = runtime.Frame(ctx, 64, 48)
    for _ in range(3): fr.render(g, view)
    H.host_clear()
    for _ in range(2): g.update_objs_async(0, scene.objs[:1])
    print(sum(l[0] == "wait" for l in log()) >= 3)   # of the live frame's renders
    fr.close()
    g.close()
print(H.host_live_events())
""")
    lines = [l.split() for l in out.split("\n")[:-1]]
    assert [int(l[1]) - int(l[0]) for l in lines[0:4:2]] == [0, 0], out
    assert lines[1] == lines[3] == ["True"] and lines[4] == ["0"], out
