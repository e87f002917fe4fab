"""The measured workloads of the 2-D DFT library, through its Python entry points.

Every case is one call (or one burst of calls) as a program that uses the
library makes it: plans, batches, handles and tables are created once by
`prepare`, `run` is the repeated part.  Sizes are the repository's own
configurations (the benchmark's single images, mixed batch, serving stream,
long lines and batched 1-D FFT, the tests' sizes) or generic image sizes.

Case kinds
  plan    one w x h complex<float> image on device memory (Plan.exec_device)
  image   the view's path: luminance of an RGBA rectangle in, |X|/(w*h) out
  fft     count power-of-two 1-D FFTs back to back (Fft.exec_device)
  batch   many independent images of mixed sizes in one call (Batch.exec_device)
  server  a burst of requests submitted to the continuous-batching server
  host    one image in host memory (ComputeVector.exec), copies included
"""
import math

import numpy as np
import torch

from math_amd import mdft as M

MIX_SEED = 0x6D696C6C  # the benchmark's seed base


def listed():
    return [
        # a thumbnail-sized patch, Bluestein on both axes: launches and latency only
        {"name": "plan_100x37", "kind": "plan", "w": 100, "h": 37, "inverse": False},
        # the camera frame of the single-image configuration
        {"name": "plan_640x480", "kind": "plan", "w": 640, "h": 480, "inverse": False},
        # the power-of-two image, inverse direction (filtering: back to the image)
        {"name": "plan_1024x1024_inv", "kind": "plan", "w": 1024, "h": 1024, "inverse": True},
        # odd prime-like sides, the reference's large single transform
        {"name": "plan_4093x2047", "kind": "plan", "w": 4093, "h": 2047, "inverse": False},
        # rows padded to the longest tile, the reference's rectangular test size, inverse
        {"name": "plan_6007x997_inv", "kind": "plan", "w": 6007, "h": 997, "inverse": True},
        # a large microscope or sky tile: bandwidth of both passes
        {"name": "plan_8192x8192", "kind": "plan", "w": 8192, "h": 8192, "inverse": False},
        # rows longer than one tile (signals side by side): the multi-step path
        {"name": "plan_16385x64", "kind": "plan", "w": 16385, "h": 64, "inverse": False},
        # the spectrum view of a full-HD frame, 8-bit pixels
        {"name": "image_1920x1080_rgba8", "kind": "image", "w": 1920, "h": 1080, "rgba8": True},
        # the batched 1-D FFT component
        {"name": "fft_4096x4096", "kind": "fft", "count": 4096, "n": 4096, "inverse": False},
        # the benchmark's mixed-size batch as one captured graph
        {"name": "batch_mixed256", "kind": "batch", "count": 256, "lo": 17, "hi": 2048, "p_pow2": 0.4,
         "mix": MIX_SEED + 3, "graph": True},
        # a burst of the serving stream: both directions, sides up to 4096
        {"name": "server_burst32", "kind": "server", "count": 32, "lo": 32, "hi": 4096, "p_pow2": 0.0,
         "mix": MIX_SEED + 4},
        # the drop-in call of a program whose image is a host vector
        {"name": "host_640x480", "kind": "host", "w": 640, "h": 480, "inverse": False},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def draw(rng):
    kind = rng.choice(["plan", "plan", "plan", "plan", "image", "fft", "batch", "batch", "server", "long", "host"])
    inverse = rng.random() < 0.5
    if kind == "plan":
        # any sides of one tile, up to 32 Mi points
        while True:
            w, h = _log_int(rng, 16, 8192), _log_int(rng, 16, 8192)
            if w * h <= 1 << 25:
                return {"kind": "plan", "w": w, "h": h, "inverse": inverse}
    if kind == "long":
        # one side longer than a tile, either axis
        while True:
            a, b = _log_int(rng, 8194, 1 << 20), _log_int(rng, 1, 64)
            if a * b <= 1 << 22:
                w, h = (a, b) if rng.random() < 0.5 else (b, a)
                return {"kind": "plan", "w": w, "h": h, "inverse": inverse}
    if kind == "image":
        return {"kind": "image", "w": _log_int(rng, 64, 4096), "h": _log_int(rng, 64, 4096),
                "rgba8": rng.random() < 0.5}
    if kind == "fft":
        n = 1 << rng.randint(4, 16)
        return {"kind": "fft", "count": _log_int(rng, 1, (1 << 24) // n), "n": n, "inverse": inverse}
    if kind == "batch":
        return {"kind": "batch", "count": _log_int(rng, 4, 256), "lo": 17, "hi": rng.choice([512, 1024, 2048]),
                "p_pow2": rng.choice([0.0, 0.4]), "mix": rng.randrange(1 << 30), "graph": rng.random() < 0.5}
    if kind == "server":
        return {"kind": "server", "count": _log_int(rng, 4, 48), "lo": 32, "hi": 4096, "p_pow2": 0.0,
                "mix": rng.randrange(1 << 30)}
    return {"kind": "host", "w": _log_int(rng, 16, 2048), "h": _log_int(rng, 16, 2048), "inverse": inverse}


def _mix(case):
    """Sizes and directions of a batch or a burst: a side is a power of two with
    probability p_pow2, else log-uniform in [lo, hi]."""
    rng = np.random.default_rng(case["mix"])
    lo, hi = case["lo"], case["hi"]
    sizes, invs = [], []
    for _ in range(case["count"]):
        dims = []
        for _ in range(2):
            if rng.random() < case["p_pow2"]:
                dims.append(1 << int(rng.integers(5, int(math.log2(hi)) + 1)))
            else:
                dims.append(int(min(hi, max(lo, math.floor(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))))
        sizes.append((dims[0], dims[1]))
        invs.append(bool(rng.random() < 0.5))
    return sizes, invs


def _offsets(sizes):
    offs, total = [], 0
    for w, h in sizes:
        offs.append(total)
        total += w * h
    return offs, total


def _image_source(case):
    """The view's window: a rectangle with a margin around it."""
    return case["w"] + 24, case["h"] + 10, 16, 7  # source width, height, rectangle x, y


def _normal(count, seed):
    """count complex values, re and im each N(0, 1)."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return torch.randn(count, dtype=torch.complex64, device="cuda", generator=g) * math.sqrt(2.0)


def _pixels(case, seed):
    sw, sh, _, _ = _image_source(case)
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    if case["rgba8"]:
        return torch.randint(0, 256, (sh, sw, 4), dtype=torch.uint8, device="cuda", generator=g)
    return torch.rand((sh, sw, 4), dtype=torch.float32, device="cuda", generator=g)


def _host_input(case, seed):
    rng = np.random.default_rng(seed)
    n = case["w"] * case["h"]
    return (rng.standard_normal(n, np.float32) + 1j * rng.standard_normal(n, np.float32)).astype(np.complex64)


class _DeviceView:
    """A server result as a tensor source (device address, complex64 values)."""

    def __init__(self, ptr, count):
        self.__cuda_array_interface__ = {"shape": (count,), "typestr": "<c8", "data": (ptr, False), "version": 2}


def prepare(case, seed):
    M.init(0)
    kind = case["kind"]
    st = {"case": case}
    if kind == "plan":
        st["plan"] = M.Plan(case["w"], case["h"])
        st["src"] = _normal(case["w"] * case["h"], seed)
        st["dst"] = torch.empty_like(st["src"])
    elif kind == "image":
        st["image"] = M.Image(case["w"], case["h"], M.PIXEL_RGBA8 if case["rgba8"] else M.PIXEL_RGBA32F)
        st["src"] = _pixels(case, seed)
        st["dst"] = torch.empty((case["h"], case["w"]), dtype=torch.float32, device="cuda")
    elif kind == "fft":
        st["fft"] = M.Fft(case["count"], case["n"])
        st["src"] = _normal(case["count"] * case["n"], seed)
        st["dst"] = torch.empty_like(st["src"])
    elif kind == "batch":
        sizes, invs = _mix(case)
        offs, total = _offsets(sizes)
        st["src"] = _normal(total, seed)
        st["dst"] = torch.empty_like(st["src"])
        st["batch"] = M.Batch(sizes, invs, offs, offs, M.MDFT_BATCH_GRAPH if case["graph"] else 0)
    elif kind == "server":
        sizes, invs = _mix(case)
        offs, total = _offsets(sizes)
        st["sizes"], st["invs"], st["offs"] = sizes, invs, offs
        st["src"] = _normal(total, seed)
        st["dst"] = torch.empty_like(st["src"])
        st["server"] = M.Server(2 << 30)
        st["server"].prepare(sorted({side for wh in sizes for side in wh}))
        torch.cuda.synchronize()  # submit() takes inputs that are complete
    else:
        st["cv"] = M.create_compute_vector()
        st["cv"].create_buffers(case["w"], case["h"])
        st["src"] = _host_input(case, seed)
    return st


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "host":
        # the call works in place on the caller's vector
        data = state["src"].copy()
        state["cv"].exec(case["inverse"], data)
        return data
    src, dst = state["src"], state["dst"]
    stream = torch.cuda.current_stream()
    if kind == "plan":
        state["plan"].exec_device(case["inverse"], src.data_ptr(), dst.data_ptr(), stream.cuda_stream)
    elif kind == "image":
        sw, sh, x, y = _image_source(case)
        state["image"].exec_device(src.data_ptr(), sw, sh, sw, x, y, dst.data_ptr(), case["w"], stream.cuda_stream)
    elif kind == "fft":
        state["fft"].exec_device(case["inverse"], src.data_ptr(), dst.data_ptr(), stream.cuda_stream)
    elif kind == "batch":
        state["batch"].exec_device(src.data_ptr(), dst.data_ptr(), stream.cuda_stream)
    else:
        srv, base = state["server"], src.data_ptr()
        tickets = [srv.submit(w, h, inv, base + 8 * off)
                   for (w, h), inv, off in zip(state["sizes"], state["invs"], state["offs"])]
        for t, (w, h), off in zip(tickets, state["sizes"], state["offs"]):
            ptr, _ = srv.wait(t)
            dst[off:off + w * h].copy_(torch.as_tensor(_DeviceView(ptr, w * h), device="cuda"))
        stream.synchronize()  # a result slot is given back once its reader is done
        for t in tickets:
            srv.release(t)
    return dst


def work(case):
    """Input read once, output written once; 5 N log2 N flops per transform."""
    kind = case["kind"]
    if kind == "fft":
        points = case["count"] * case["n"]
        return {"bytes": 16 * points, "flops": 5 * points * math.log2(case["n"])}
    sizes = _mix(case)[0] if kind in ("batch", "server") else [(case["w"], case["h"])]
    points = sum(w * h for w, h in sizes)
    per_point = (4 if case["rgba8"] else 16) + 4 if kind == "image" else 16
    return {"bytes": per_point * points, "flops": sum(5 * w * h * math.log2(w * h) for w, h in sizes if w * h > 1)}


def _dft2(x, inverse):
    """FP64 2-D DFT: forward unnormalised, inverse times 1/(w*h)."""
    return np.fft.ifft2(x) if inverse else np.fft.fft2(x)


def exact(case, seed):
    kind = case["kind"]
    if kind == "host":
        x = _host_input(case, seed).astype(np.complex128).reshape(case["h"], case["w"])
        return _dft2(x, case["inverse"]).ravel()
    if kind == "image":
        _, _, x0, y0 = _image_source(case)
        px = _pixels(case, seed)[y0:y0 + case["h"], x0:x0 + case["w"], :3].cpu().numpy().astype(np.float64)
        lum = (px / 255.0 if case["rgba8"] else px) @ np.array([0.2126, 0.7152, 0.0722])
        return torch.from_numpy(np.abs(_dft2(lum, False)) / (case["w"] * case["h"]))
    if kind == "fft":
        x = _normal(case["count"] * case["n"], seed).cpu().numpy().astype(np.complex128)
        x = x.reshape(case["count"], case["n"])
        return torch.from_numpy((np.fft.ifft(x) if case["inverse"] else np.fft.fft(x)).ravel())
    if kind == "plan":
        sizes, invs = [(case["w"], case["h"])], [case["inverse"]]
    else:
        sizes, invs = _mix(case)
    offs, total = _offsets(sizes)
    x = _normal(total, seed).cpu().numpy().astype(np.complex128)
    out = np.empty_like(x)
    for (w, h), inv, off in zip(sizes, invs, offs):
        out[off:off + w * h] = _dft2(x[off:off + w * h].reshape(h, w), inv).ravel()
    return torch.from_numpy(out)
