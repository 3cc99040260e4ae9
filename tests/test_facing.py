"""The shadow prearrange's early drop of triangles that face away from a light
(raster.hip: faces_away) drops only what the culling after projection drops:
tests/facing_check.c, triangles of every size and angle, most of them nearly
edge-on, against the same operations."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.parametrize("seed", ["1", "2", "3"])
def test_dropped_triangles_are_culled(tmp_path, seed):
    exe = str(tmp_path / "facing_check")
    subprocess.run(["gcc", "-O2", "-ffp-contract=off", "-o", exe, os.path.join(HERE, "facing_check.c"), "-lm"], check=True)
    r = subprocess.run([exe, "4000000", seed], capture_output=True, text=True, timeout=300)
    print(r.stdout)
    assert r.returncode == 0 and " 0 mismatches" in r.stdout, r.stdout
    assert int(r.stdout.split("dropped ")[1].split(",")[0]) > 500000
