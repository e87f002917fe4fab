"""Which kernel a call reaches, by what it costs and by what it returns: the
forms that a rule on sizes picks, at the sizes where picking another one would
show.  Times are GPU times of captured launches, always of two calls of the
same process and card against each other."""
import statistics

import numpy as np
import pytest

from tests.helpers import rand_c64, tol_nl2

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def mdft():
    from math_amd import mdft as M

    M.init(0)
    return M


def captured(enqueue, reps=20):
    """A graph of `reps` calls of enqueue(stream handle)."""
    import torch

    s = torch.cuda.Stream()
    enqueue(s.cuda_stream)
    s.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        for _ in range(reps):
            enqueue(torch.cuda.current_stream().cuda_stream)
    return g


def time_ratio(a, b, rounds=15):
    """median time of graph a over that of graph b, replayed in turn"""
    import torch

    def once(g):
        t0, t1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        t0.record()
        g.replay()
        t1.record()
        t1.synchronize()
        return t0.elapsed_time(t1)

    ta, tb = [], []
    for i in range(rounds + 2):
        x, y = once(a), once(b)
        if i >= 2:
            ta.append(x)
            tb.append(y)
    return statistics.median(ta) / statistics.median(tb)


# Rows that lie whole in one thread, 2^24 points: 47 us in rows of 8 and 56 in rows of 16 when the thread reads and
# writes them in pairs (1.3 and 1.55 times rows of 64), 85 and 102 by single elements (2.0 to 2.8 times).
@pytest.mark.parametrize("n", [8, 16])
def test_short_rows_cost_what_longer_ones_cost(mdft, n):
    import torch

    src = torch.zeros(1 << 24, dtype=torch.complex64, device="cuda")
    dst = torch.empty_like(src)
    short, longer = mdft.Fft(src.numel() // n, n), mdft.Fft(src.numel() // 64, 64)
    print(f"short rows {n}", flush=True)
    r = time_ratio(captured(lambda st: short.exec_device(False, src.data_ptr(), dst.data_ptr(), st)),
                   captured(lambda st: longer.exec_device(False, src.data_ptr(), dst.data_ptr(), st)))
    short.close()
    longer.close()
    print(f"ratio {r:.3f}", flush=True)
    assert r <= 1.9, r


# the same rows at the edges of their tiles (64 to 1024 lines a workgroup), from buffers aligned to one element only
@pytest.mark.parametrize("n", [2, 4, 8, 16])
@pytest.mark.parametrize("count", [1, 63, 65, 1023, 1025, 70001])
def test_short_rows_at_tile_edges(mdft, n, count):
    import torch

    x = rand_c64(np.random.default_rng(n * count), (count, n))
    src = torch.full((count * n + 2,), complex("nan"), dtype=torch.complex64, device="cuda")
    src[1:-1] = torch.from_numpy(x.ravel()).cuda()
    dst = torch.full_like(src, -7.0)
    f = mdft.Fft(count, n)
    print(f"short rows {count} x {n}", flush=True)
    for inv in (False, True):
        f.exec_device(inv, src.data_ptr() + 8, dst.data_ptr() + 8, torch.cuda.current_stream().cuda_stream)
        got = dst.cpu().numpy()
        ref = (np.fft.ifft if inv else np.fft.fft)(x.astype(np.complex128), axis=1)
        assert got[0] == -7.0 and got[-1] == -7.0
        err = np.linalg.norm(got[1:-1].reshape(count, n) - ref) / np.linalg.norm(ref)
        assert err <= 2e-6 * max(1.0, np.log2(n)), (inv, err)
    f.close()


# The view's columns run in the plan's tiles: 16384-point columns of an image too narrow for wide tiles (8, 70 and
# 131 columns of one line each: 26, 37 and 41 us with 256 + 256 threads a line, 37, 46 and 51 in 1024-thread tiles
# that leave most CUs idle).
@pytest.mark.parametrize("w,h", [(8, 5681), (70, 6510), (131, 5715)])
def test_narrow_image_columns_cost_what_the_plan_costs(mdft, w, h):
    import torch

    pixels = torch.zeros((h, w, 4), dtype=torch.uint8, device="cuda")
    mag = torch.empty((h, w), dtype=torch.float32, device="cuda")
    src = torch.zeros(w * h, dtype=torch.complex64, device="cuda")
    dst = torch.empty_like(src)
    image, plan = mdft.Image(w, h, mdft.PIXEL_RGBA8), mdft.Plan(w, h)
    print(f"image columns {w}x{h}", flush=True)
    r = time_ratio(captured(lambda st: image.exec_device(pixels.data_ptr(), w, h, w, 0, 0, mag.data_ptr(), w, st)),
                   captured(lambda st: plan.exec_device(False, src.data_ptr(), dst.data_ptr(), st)))
    image.close()
    plan.close()
    print(f"ratio {r:.3f}", flush=True)
    assert r <= 1.15, r


# Columns with magnitudes in every tile the plan's rule picks on 256 CUs (the image path runs those of less than 256
# threads in 256), the last tile short of a column or a pair:
# (width, height, tile threads, two lines per thread)
IMAGE_COLUMNS = [(3067, 4096, 1024, True), (2049, 2048, 512, True), (1025, 2048, 256, True), (515, 4096, 256, True),
                 (3841, 1021, 512, True), (1923, 1201, 512, True), (1923, 2047, 512, True), (1283, 2047, 256, True),
                 (2561, 701, 256, True), (5121, 509, 256, True), (1027, 8192, 1024, False), (515, 2999, 512, False),
                 (513, 6007, 1024, False), (61, 6007, 512, False), (192, 71, 64, False), (60, 139, 64, False)]


# and of a smooth height (1921 x 1080: 512 threads)
@pytest.mark.parametrize("w,h", [c[:2] for c in IMAGE_COLUMNS] + [(1921, 1080), (31, 1080)])
def test_image_columns_in_every_tile(mdft, w, h):
    import torch

    g = torch.Generator(device="cuda")
    g.manual_seed(w + h)
    x, y, sw, pitch, out = 2, 1, w + 4, w + 9, w + 3
    px = torch.rand((h + 2, pitch, 4), dtype=torch.float32, device="cuda", generator=g)
    dst = torch.full((h, out), -7.0, dtype=torch.float32, device="cuda")
    image = mdft.Image(w, h, mdft.PIXEL_RGBA32F)
    print(f"image columns {w}x{h}", flush=True)
    image.exec_device(px.data_ptr(), sw, h + 2, pitch, x, y, dst.data_ptr(), out,
                      torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    image.close()
    assert bool((dst[:, w:] == -7.0).all())
    lum = px[y:y + h, x:x + w, :3].cpu().to(torch.float64) @ torch.tensor([0.2126, 0.7152, 0.0722],
                                                                          dtype=torch.float64)
    ref = torch.fft.fft2(lum).abs() / (w * h)
    err = torch.linalg.norm(dst[:, :w].cpu().to(torch.float64) - ref) / torch.linalg.norm(ref)
    assert err <= tol_nl2(w, h), float(err)


# Plan columns in every wide tile: the tile a size takes is checked against the rule in test_tile_rule.py
PLAN_COLUMNS = [(3067, 4096, 1024, True), (6131, 2048, 1024, True), (4099, 3072, 1024, True), (2049, 2048, 512, True),
                (4099, 1024, 512, True), (1025, 2048, 256, True), (515, 4096, 256, True), (1027, 1536, 256, True),
                (1923, 2047, 512, True), (3841, 1021, 512, True), (1923, 1201, 512, True), (1283, 2047, 256, True),
                (2563, 1021, 256, True), (1283, 1201, 256, True), (2561, 701, 256, True), (5121, 509, 256, True),
                (1027, 8192, 1024, False), (1029, 4093, 1024, False), (770, 8192, 1024, False),
                (770, 4093, 1024, False), (515, 2999, 512, False), (517, 6144, 512, False), (513, 6007, 1024, False)]


# A wide tile gives the bits of the narrow one (the tile table's entry 0), and FP64's values
@pytest.mark.parametrize("w,h", [c[:2] for c in PLAN_COLUMNS])
def test_plan_columns_in_every_wide_tile(mdft, w, h):
    import torch

    g = torch.Generator(device="cuda")
    g.manual_seed(w * 3 + h)
    src = torch.randn(w * h, dtype=torch.complex64, device="cuda", generator=g)
    st = torch.cuda.current_stream().cuda_stream
    direct = h & (h - 1) == 0 or (h % 3 == 0 and (h // 3) & (h // 3 - 1) == 0)
    shapes = [s for s in list(range(1, 15)) + list(range(38, 44))]
    keep = {s: mdft.tune_get(s, not direct, 1) for s in shapes}
    p = mdft.Plan(w, h)
    outs = []
    print(f"plan columns {w}x{h}", flush=True)
    try:
        for variant in (0, 1):
            for s in shapes:
                mdft.tune_set(s, not direct, 1, variant)
            for inv in (False, True):
                dst = torch.full_like(src, float("nan"))
                p.exec_device(inv, src.data_ptr(), dst.data_ptr(), st)
                outs.append(dst)
    finally:
        for s in shapes:
            mdft.tune_set(s, not direct, 1, keep[s])
    torch.cuda.synchronize()
    p.close()
    for a, b in ((0, 2), (1, 3)):
        assert torch.equal(torch.view_as_real(outs[a]), torch.view_as_real(outs[b]))
    ref = torch.fft.fft2(src.cpu().reshape(h, w).to(torch.complex128))
    err = torch.linalg.norm(outs[2].cpu().reshape(h, w) - ref) / torch.linalg.norm(ref)
    assert err <= tol_nl2(w, h), float(err)


@pytest.mark.parametrize("flags", [4, 6])
def test_smooth_lengths_in_a_dependent_batch(mdft, flags):
    import torch

    sizes = [(100, 300), (640, 480), (45, 1920), (1, 90), (90, 1), (20, 18), (3000, 2), (37, 3600), (1021, 75)]
    invs = [i % 2 == 0 for i in range(len(sizes))]
    rng = np.random.default_rng(12)
    xs = [rand_c64(rng, (h, w)) for w, h in sizes]
    offs = np.cumsum([0] + [w * h for w, h in sizes])[:-1].tolist()
    src = torch.from_numpy(np.concatenate([x.ravel() for x in xs])).cuda()
    dst = torch.empty_like(src)
    st = torch.cuda.current_stream().cuda_stream
    print(f"smooth dependent batch flags={flags}", flush=True)
    b = mdft.Batch(sizes, invs, offs, offs, flags)
    b.exec_device(src.data_ptr(), dst.data_ptr(), st)
    b.check()
    torch.cuda.synchronize()
    b.close()
    for (w, h), inv, o in zip(sizes, invs, offs):
        alone = torch.empty(w * h, dtype=torch.complex64, device="cuda")
        p = mdft.Plan(w, h)
        p.exec_device(inv, src.data_ptr() + 8 * o, alone.data_ptr(), st)
        torch.cuda.synchronize()
        p.close()
        assert torch.equal(torch.view_as_real(dst[o:o + w * h]), torch.view_as_real(alone)), (w, h)


def run_batch(mdft, sizes, flags=0):
    """(outputs of a batch on random images, outputs of plans on the same, info)"""
    import torch

    invs = [i % 2 == 1 for i in range(len(sizes))]
    offs = np.cumsum([0] + [w * h for w, h in sizes])[:-1].tolist()
    total = sum(w * h for w, h in sizes)
    g = torch.Generator(device="cuda")
    g.manual_seed(total)
    src = torch.randn(total, dtype=torch.complex64, device="cuda", generator=g)
    dst, alone = torch.full_like(src, float("nan")), torch.full_like(src, float("nan"))
    st = torch.cuda.current_stream().cuda_stream
    b = mdft.Batch(sizes, invs, offs, offs, flags)
    info = b.info()
    b.exec_device(src.data_ptr(), dst.data_ptr(), st)
    plans = {wh: mdft.Plan(*wh) for wh in set(sizes)}
    for wh, inv, o in zip(sizes, invs, offs):
        plans[wh].exec_device(inv, src.data_ptr() + 8 * o, alone.data_ptr() + 8 * o, st)
    torch.cuda.synchronize()
    b.close()
    for p in plans.values():
        p.close()
    return torch.view_as_real(dst), torch.view_as_real(alone), info


# The column phase of a batch by its number of tiles (256 CUs): 256 threads, 512 with one line per thread, with two:
# (count, width, height, threads, column tiles)
@pytest.mark.parametrize("count,w,h,threads,items", [
    (1, 65, 701, 256, 33), (1, 2049, 701, 512, 513), (2, 4095, 701, 512, 1024), (1, 129, 509, 256, 33),
    (1, 1025, 1201, 512, 513), (1, 2047, 1201, 512, 512), (1, 57, 4093, 256, 57), (1, 299, 4093, 512, 150),
    (1, 255, 4096, 512, 128), (1, 513, 4096, 512, 129), (1, 511, 3072, 512, 256), (1, 801, 3072, 512, 201)])
def test_batch_column_tiles(mdft, count, w, h, threads, items):
    import torch

    print(f"batch columns {count} x {w}x{h}", flush=True)
    got, alone, info = run_batch(mdft, [(w, h)] * count)
    assert torch.equal(got, alone)
    assert (info["threads"][1], info["items"][1]) == (threads, items)


# every FFT shape in one launch of each column kernel: one line per thread (a few images), two (eight times as many)
def test_every_shape_in_every_column_kernel(mdft):
    import torch

    heights = [2, 3, 5, 9, 17, 33, 65, 129, 257, 509, 1021, 2047, 4093, 4, 8, 16, 32, 64, 128, 256, 512, 1024, 2048,
               4096, 8192, 71, 139, 277, 701, 1201, 2999, 192, 384, 768, 1536, 3072, 6144, 18, 100, 1080, 2401, 3600]
    items = []
    for times in (1, 8):
        print(f"every shape x {times}", flush=True)
        got, alone, info = run_batch(mdft, [(35, h) for h in heights] * times)
        assert torch.equal(got, alone)
        assert info["threads"][1] == 512
        items.append(info["items"][1])
    assert items[1] < 8 * items[0]


# A batch of one image costs about what its plan costs: few column tiles take the small forms (two lines per thread
# in 512 threads 1.65 to 2.1 times, the small forms 1.0 to 1.3)
@pytest.mark.parametrize("w,h", [(128, 509), (64, 1021), (256, 1201), (128, 2047)])
def test_a_small_batch_costs_what_its_plans_cost(mdft, w, h):
    import torch

    src = torch.zeros(w * h, dtype=torch.complex64, device="cuda")
    dst = torch.empty_like(src)
    b, p = mdft.Batch([(w, h)], [False], [0], [0], 0), mdft.Plan(w, h)
    b.exec_device(src.data_ptr(), dst.data_ptr(), torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    print(f"small batch {w}x{h}", flush=True)
    r = time_ratio(captured(lambda st: b.exec_device(src.data_ptr(), dst.data_ptr(), st)),
                   captured(lambda st: p.exec_device(False, src.data_ptr(), dst.data_ptr(), st)))
    b.close()
    p.close()
    print(f"ratio {r:.3f}", flush=True)
    assert r <= 1.45, r
