"""The raster's pixel box (common/pixel_box.h) of large triangles on the CPU: none of the samples
round the box and near the vertices that lies outside it may pass the edge tests."""
import os
import re
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


def test_no_covered_sample_lies_outside_a_large_box(tmp_path):
    exe = tmp_path / "pixel_box_large_check"
    subprocess.run(["g++", "-O2", "-std=c++17", "-mfma", "-ffp-contract=off", "-I",
                    os.path.join(ROOT, "ifrit-v2_amd", "csrc", "common"),
                    os.path.join(HERE, "native", "pixel_box_large_check.cpp"), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe), "20000"], capture_output=True, text=True, timeout=120)
    print(r.stdout)
    assert r.returncode == 0, r.stdout
    n, boxes, large = (int(x) for x in re.search(r"(\d+) triangles, (\d+) boxes, (\d+) of more", r.stdout).groups())
    assert boxes > n and large > n // 4  # two boxes are asked for per triangle
