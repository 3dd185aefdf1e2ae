"""Host check of the regions that integration workgroups take
(marching_cube_amd/csrc/mcx_region_order.h, compiled with g++ from the same
header the kernels include): every region once, and none past the last, whose
place would be computed with a division by the extent 0 of an empty block.
The program counts the workgroups for which that would happen; the count must
stay positive, or the check no longer exercises the hazard."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_region_order(tmp_path):
    exe = str(tmp_path / "region_order_check")
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-Wall", "-I",
                           os.path.join(ROOT, "marching_cube_amd", "csrc"), "-o", exe,
                           os.path.join(ROOT, "tests", "cpp", "region_order_check.cpp")])
    out = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0, out.stdout + out.stderr
    tag, shapes, empty = out.stdout.split()
    assert tag == "ok"
    assert int(shapes) == 1000
    assert int(empty) > 0
