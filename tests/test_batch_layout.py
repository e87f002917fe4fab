"""The work list of a batch on the CPU: laid out by job, it is item for item the
list that the rule gives tile by tile, at a fraction of the time (the scheduler
builds one for every burst, between the requests and their launch)."""
import os
import re
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_items_equal_the_list_built_tile_by_tile(tmp_path):
    exe, lib = str(tmp_path / "items_tool"), os.path.join(ROOT, "math_amd", "lib")
    subprocess.run(["g++", "-std=c++17", "-O2", os.path.join(ROOT, "tests", "cpp", "items_tool.cpp"), "-o", exe,
                    "-L" + lib, "-lmdft", "-Wl,-rpath," + lib], check=True)
    runs = []
    for _ in range(3):
        r = subprocess.run([exe], capture_output=True, text=True)
        print(r.stdout)
        assert r.returncode == 0 and r.stdout.startswith("equal 400 "), r.stdout
        runs.append([float(v) for v in re.findall(r"([\d.]+) us", r.stdout)])
    ours, per_tile = min(r[0] for r in runs), min(r[1] for r in runs)
    assert ours <= per_tile / 3, runs
