"""A render runs on the stream of its output set, behind what the caller's
stream held before the render but one was issued: work of the caller's own that
is still under way there does not hold it up.  Host code over the stand-in for
the HIP runtime."""
import host_hip


def test_render_beside_the_callers_work(tmp_path):
    out = host_hip.run(tmp_path, """
ctx = runtime.Context(0)
sc, view = scenes.random_scene(3)
g, fr = runtime.GpuScene(ctx, sc), runtime.Frame(ctx, 64, 48)
st = stream()
for k in range(6):                     # each finished before the next is issued
    H.host_hold(st, int(k > 2))        # from the fourth on, the caller's work is still running
    H.host_clear()
    fr.render(g, view, st)
    l = log()
    me = str(H.host_stream_id(st))
    used = {x[2] for x in l if x[0] == "launch"}
    waited = [x for x in l if x[0] == "wait" and x[1] == me]
    print(int(me in used), len(used), len(waited))
    H.host_hold(st, 0)
fr.close()
""")
    assert out.split("\n")[:-1] == ["0 1 1"] * 6, out
