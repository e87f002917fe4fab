"""Tile kernels at the edges of their dispatch: smooth lengths (direct
mixed-radix FFTs), wide column tiles with two lines per thread, images that one
workgroup runs in one launch, and loads past the end of a line."""
import numpy as np
import pytest

from tests.helpers import check_against_fp64, rand_c64

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def mdft():
    from math_amd import mdft as M

    M.init(0)
    return M


def run_exec(M, x, inverse):
    h, w = x.shape
    d = np.ascontiguousarray(x.copy())
    p = M.Plan(w, h)
    p.exec(inverse, d)
    p.close()
    return d


# every radix first, in the middle and last; two to seven passes; the shortest and the longest,
# and lengths whose passes would need more than 256 threads (3675, 4000, 4050: Bluestein)
@pytest.mark.parametrize("n", [18, 20, 21, 24, 25, 35, 49, 63, 81, 100, 105, 175, 189, 243, 245, 343, 375, 441, 625,
                               729, 945, 1000, 1125, 1323, 1575, 1715, 1920, 2025, 2187, 2401, 2560, 3000, 3125, 3375,
                               3500, 3600, 3675, 3750, 3840, 4000, 4050])
def test_smooth_lengths(mdft, n):
    rng = np.random.default_rng(n)
    print(f"smooth {n}", flush=True)
    for inv in (False, True):
        x = rand_c64(rng, (3, n))
        check_against_fp64(run_exec(mdft, x, inv), x, inv, "rows")
        xt = rand_c64(rng, (n, 5))
        check_against_fp64(run_exec(mdft, xt, inv), xt, inv, "cols")


@pytest.mark.parametrize("flags", [0, 2, 8])
def test_smooth_batch_equals_single(mdft, flags):
    import torch

    sizes = [(100, 300), (640, 480), (1080, 60), (45, 1920), (1, 90), (90, 1), (20, 18), (18, 20), (3000, 2), (37, 3600)]
    invs = [i % 2 == 1 for i in range(len(sizes))]
    rng = np.random.default_rng(5)
    xs = [rand_c64(rng, (h, w)) for w, h in sizes]
    offs = np.cumsum([0] + [w * h for w, h in sizes])[:-1].tolist()
    src = torch.from_numpy(np.concatenate([x.ravel() for x in xs])).cuda()
    dst = torch.empty_like(src)
    print(f"smooth batch flags={flags}", flush=True)
    b = mdft.Batch(sizes, invs, offs, offs, flags)
    b.exec_device(src.data_ptr(), dst.data_ptr(), torch.cuda.current_stream().cuda_stream)
    b.check()
    torch.cuda.synchronize()
    out = dst.cpu().numpy()
    b.close()
    for (w, h), inv, x, o in zip(sizes, invs, xs, offs):
        got = out[o:o + w * h].reshape(h, w)
        assert np.array_equal(got, run_exec(mdft, x, inv)), f"{w}x{h}"
        check_against_fp64(got, x, inv, "batch")


# (width, height, shape of the columns, Bluestein): enough columns for the wide tiles, the last tile short of a
# column or of a pair
@pytest.mark.parametrize("w,h,shape,blue", [(1025, 4096, 12, 0), (2049, 4096, 12, 0), (4099, 1024, 10, 0),
                                            (1027, 2047, 12, 1), (2043, 1021, 11, 1), (1022, 1201, 42, 1),
                                            (2045, 701, 41, 1), (1025, 8192, 13, 0), (515, 2999, 43, 1)])
def test_wide_column_tiles_bitwise(mdft, w, h, shape, blue):
    import torch

    g = torch.Generator(device="cuda")
    g.manual_seed(w + h)
    src = torch.randn(w * h, dtype=torch.complex64, device="cuda", generator=g)
    st = torch.cuda.current_stream().cuda_stream
    keep = mdft.tune_get(shape, blue, 1)
    outs = []
    p = mdft.Plan(w, h)
    print(f"wide tiles {w}x{h}", flush=True)
    try:
        for variant in (0, 1):
            mdft.tune_set(shape, blue, 1, variant)
            for inv in (False, True):
                dst = torch.full_like(src, float("nan"))
                p.exec_device(inv, src.data_ptr(), dst.data_ptr(), st)
                outs.append(dst)
    finally:
        mdft.tune_set(shape, blue, 1, keep)
    torch.cuda.synchronize()
    p.close()
    assert torch.equal(torch.view_as_real(outs[0]), torch.view_as_real(outs[2]))
    assert torch.equal(torch.view_as_real(outs[1]), torch.view_as_real(outs[3]))
    ref = torch.fft.fft2(src.cpu().reshape(h, w).to(torch.complex128))
    err = torch.linalg.norm(outs[2].cpu().reshape(h, w) - ref) / torch.linalg.norm(ref)
    assert err <= 2e-6 * np.log2(w * h), float(err)


# the largest images of one workgroup (256 threads hold all rows, and all columns) and the first ones past it
@pytest.mark.parametrize("w,h", [(2, 2), (16, 16), (64, 64), (65, 64), (64, 65), (17, 31), (100, 16), (512, 2),
                                 (2, 512), (4096, 2), (1000, 2), (61, 29), (256, 16), (257, 16)])
def test_one_launch_images(mdft, w, h):
    import torch

    rng = np.random.default_rng(w * 1000 + h)
    x = rand_c64(rng, (h, w))
    st = torch.cuda.current_stream().cuda_stream
    p = mdft.Plan(w, h)
    print(f"one launch {w}x{h}", flush=True)
    for inv in (False, True):
        src = torch.from_numpy(x).cuda()
        dst = torch.full_like(src, float("nan"))
        p.exec_device(inv, src.data_ptr(), dst.data_ptr(), st)
        inplace = src.clone()
        p.exec_device(inv, inplace.data_ptr(), inplace.data_ptr(), st)
        torch.cuda.synchronize()
        assert np.array_equal(dst.cpu().numpy(), inplace.cpu().numpy())
        check_against_fp64(dst.cpu().numpy(), x, inv, "one launch")
    p.close()


# an image between NaNs: nothing outside it enters the result (slots past the end of a line, lines past the last)
@pytest.mark.parametrize("w,h", [(1025, 3), (3, 1025), (2047, 2), (5, 2049), (4097, 1), (1, 8193), (300, 5), (5, 1001),
                                 (1000, 3), (7, 1080), (20000, 1), (3, 16385), (8193, 2), (1300, 1021)])
def test_nothing_outside_the_image_is_used(mdft, w, h):
    import torch

    pad = 4096
    rng = np.random.default_rng(w + 7 * h)
    x = rand_c64(rng, (h, w))
    buf = torch.full((w * h + 2 * pad,), complex("nan"), dtype=torch.complex64, device="cuda")
    buf[pad:pad + w * h] = torch.from_numpy(x.ravel()).cuda()
    clean = torch.from_numpy(x.ravel()).cuda()
    st = torch.cuda.current_stream().cuda_stream
    p = mdft.Plan(w, h)
    print(f"between NaNs {w}x{h}", flush=True)
    for inv in (False, True):
        a, b = torch.empty_like(clean), torch.empty_like(clean)
        p.exec_device(inv, buf.data_ptr() + 8 * pad, a.data_ptr(), st)
        p.exec_device(inv, clean.data_ptr(), b.data_ptr(), st)
        torch.cuda.synchronize()
        assert not torch.isnan(torch.view_as_real(a)).any()
        assert torch.equal(torch.view_as_real(a), torch.view_as_real(b))
    p.close()
