"""The walk's launch plans (csrc/hv_plan.h, plain C++) on the host: the buckets a level's rays are
counted into, for more meshes than the buckets' limit as well (the choice of the shift has to end),
and the room for the waiting nodes of the 16-NN lists' walk."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_walk_plans(tmp_path):
    exe = str(tmp_path / "walk_plan")
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-I", os.path.join(ROOT, "highvoronoi.jl_amd", "csrc"),
                           os.path.join(ROOT, "tests", "native", "walk_plan.cpp"), "-o", exe])
    r = subprocess.run([exe], timeout=60, capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
