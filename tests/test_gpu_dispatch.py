"""Which kernel a call reaches, by what it costs and by what it returns: the
forms that a rule on sizes picks, at the sizes where picking another one would
show.  Times are GPU times of captured launches, always of two calls of the
same process and card against each other."""
import statistics

import numpy as np
import pytest

from tests.helpers import rand_c64

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
# writes them in pairs, 85 and 102 by single elements; 42 in rows of 64.
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
    assert r <= 1.65, r


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
