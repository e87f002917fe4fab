"""Builds libmdft.so (HIP kernels + host runtime + C ABI) for gfx950 in-tree.

Usage: python -m math_amd.build   (or __graft_entry__.build()).
"""
import concurrent.futures
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(HERE, "csrc")
BUILD = os.path.join(HERE, "_build")
LIB = os.path.join(HERE, "lib", "libmdft.so")

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = "gfx950"
COMMON = [
    "-O3", "-std=c++17", "-fPIC", f"--offload-arch={ARCH}",
    # packed FP32 instructions stay off on this target
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    # roundings are fixed by explicit fmas in the source (bitwise-reproducible lines)
    "-ffp-contract=off",
    "-Wall", "-Wno-unused-function",
    f"-I{os.path.join(ROOT, 'include')}",
]

# a source, or (source, object name, defines) for one compiled several times;
# the longest compilations first
SOURCES = [
    ("kernels/batch_kernels.hip", f"batch_{kind}_{t}{'_' + hold if hold != 'BATCH_ALL' else ''}",
     [f"-DMDFT_BATCH_T={t}", f"-DMDFT_BATCH_HOLD={hold}", f"-DMDFT_BATCH_PERSISTENT_TU={p}"])
    for p, kind, t, hold in ((0, "grid", 256, "BATCH_ALL"), (1, "persistent", 256, "BATCH_ALL"),
                             (0, "grid", 512, "BATCH_COLS_X2"), (0, "grid", 1024, "BATCH_COLS_X2"),
                             (0, "grid", 512, "BATCH_COLS"))
] + [
    "kernels/whole.hip",
    "kernels/axis.hip",
    "kernels/batch.hip",
    "kernels/tables.hip",
    "kernels/large.hip",
    "kernels/image.hip",
    "kernels/smooth.hip",
    "host/runtime.cpp",
    "host/capi.cpp",
    "host/fft1d.cpp",
    "host/image.cpp",
    "host/tune.cpp",
    "host/batch.cpp",
    "host/batch_builder.cpp",
    "host/server.cpp",
    "host/noalloc.cpp",
]


def _compile(entry):
    src, name, defines = entry if isinstance(entry, tuple) else (entry, entry.replace("/", "_"), [])
    out = os.path.join(BUILD, name + ".o")
    lang = ["-x", "hip"] if src.endswith(".hip") else ["-x", "hip"]
    cmd = [HIPCC] + COMMON + defines + lang + ["-c", os.path.join(CSRC, src), "-o", out]
    r = subprocess.run(cmd, capture_output=True, text=True)
    msgs = "\n".join(l for l in (r.stdout + r.stderr).splitlines() if "packed-fp32-ops" not in l)
    if r.returncode != 0:
        raise RuntimeError(f"compile failed: {src}\n{' '.join(cmd)}\n{msgs}")
    return out, msgs


def build(verbose=True):
    os.makedirs(BUILD, exist_ok=True)
    os.makedirs(os.path.dirname(LIB), exist_ok=True)
    jobs = int(os.environ.get("MAX_JOBS", str(min(8, os.cpu_count() or 4))))
    with concurrent.futures.ThreadPoolExecutor(max_workers=jobs) as ex:
        results = list(ex.map(_compile, SOURCES))
    objs = []
    for out, msgs in results:
        objs.append(out)
        if verbose and msgs.strip():
            print(msgs, file=sys.stderr)
    tmp = LIB + ".tmp"
    cmd = [HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", tmp] + objs
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed\n{' '.join(cmd)}\n{r.stdout}{r.stderr}")
    os.replace(tmp, LIB)
    if verbose:
        print(f"built {LIB}")
    return LIB


if __name__ == "__main__":
    build()
