"""The single-image tile rule on the CPU: the sizes of the GPU tests reach the
tiles they are there for (a moved line fails here, where the GPU test would
quietly compare a kernel with itself)."""
import os
import re
import subprocess

import pytest

from tests import test_gpu_dispatch as G

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
GEN_SHAPE = 60  # smooth lengths: their own kernels


@pytest.fixture(scope="module")
def ask(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("tool") / "tile_tool")
    lib = os.path.join(ROOT, "math_amd", "lib")
    subprocess.run(["g++", "-std=c++17", "-O1", os.path.join(ROOT, "tests", "cpp", "tile_tool.cpp"), "-o", exe,
                    "-L" + lib, "-lmdft", "-Wl,-rpath," + lib], check=True)

    def run(query):
        r = subprocess.run([exe], input=" ".join(str(int(q) if isinstance(q, bool) else q) for q in query) + "\n",
                           capture_output=True, text=True, check=True)
        return [int(v) for v in r.stdout.split()]

    return run


def column_tile(ask, w, h, variant):
    shape = ask(("n", h, 1))[0]
    direct = h & (h - 1) == 0 or (h % 3 == 0 and (h // 3) & (h // 3 - 1) == 0)
    assert shape != GEN_SHAPE
    threads, x2 = ask((shape, not direct, True, w, variant))
    return shape, not direct, threads, bool(x2)


@pytest.mark.parametrize("w,h,threads,x2", G.IMAGE_COLUMNS + G.PLAN_COLUMNS)
def test_sizes_reach_their_tiles(ask, w, h, threads, x2):
    assert column_tile(ask, w, h, 1)[2:] == (threads, x2)


@pytest.mark.parametrize("w,h,threads,x2", G.PLAN_COLUMNS)
def test_the_tables_narrow_entry_gives_another_tile(ask, w, h, threads, x2):
    t, two = column_tile(ask, w, h, 0)[2:]
    assert not two and t < threads or (x2 and not two)


# 8192-point columns: wide tiles where they are fewer than the CUs but faster all the same, narrow ones below
@pytest.mark.parametrize("w,h,threads", [(509, 8192, 1024), (508, 8192, 256), (637, 4093, 1024), (636, 4093, 256)])
def test_8192_point_columns(ask, w, h, threads):
    assert column_tile(ask, w, h, 1)[2:] == (threads, False)


def test_image_cases_with_smooth_heights_are_named_apart(ask):
    assert ask(("n", 1080, 1)) == [GEN_SHAPE]
    assert ask(("n", 71, 1)) == [38] and ask(("n", 139, 1)) == [39]


# Two-line tiles: the library holds the ones the rule picks over all counts, and no others (the autotuner times what
# the rule picks, too)
@pytest.mark.parametrize("kernel,args", [("k_axis", r"true"), ("k_image_axis", r"true, 2")])
def test_two_line_tiles_are_the_ones_the_rule_picks(ask, kernel, args):
    names = subprocess.run(["nm", "-C", os.path.join(ROOT, "math_amd", "lib", "libmdft.so")], capture_output=True,
                           text=True, check=True).stdout
    held = {tuple(m) for m in re.findall(rf"device_stub__{kernel}<(\d+), (\d+), (true|false), {args}>", names)
            if int(m[0]) >= 64}
    picked = set()
    for shape in (10, 11, 12, 41, 42):
        for blue in (False, True):
            queries = [q for count in range(1, 20000, 61) for q in (shape, blue, True, count, 1)]
            answers = ask(queries)
            for threads, x2 in zip(answers[::2], answers[1::2]):
                if x2:
                    picked.add((str(shape + 64), str(threads), "true" if blue else "false"))
    if kernel == "k_image_axis":  # direct columns below 3072 points: 512 threads only
        picked -= {(str(s + 64), t, "false") for s in (10, 11, 41) for t in ("256", "1024")}
    assert held == picked


# one launch: all rows and all columns in 256 threads, and not two Bluestein axes of 32 points or more
@pytest.mark.parametrize("w,h,one", [(2, 2, 1), (16, 16, 1), (64, 64, 1), (65, 64, 0), (64, 65, 0), (50, 50, 1),
                                     (100, 37, 0), (9, 9, 1), (6, 10, 1), (10, 10, 0), (14, 11, 0), (22, 11, 0),
                                     (31, 31, 0), (61, 29, 0), (61, 13, 0), (20, 11, 1), (64, 11, 1), (11, 64, 1),
                                     (1, 5, 0), (5, 1, 0), (4096, 2, 0), (256, 16, 1), (257, 16, 0)])
def test_images_of_one_launch(ask, w, h, one):
    assert ask(("one", w, h)) == [one]
