#!/usr/bin/env python3
"""Generates lds_maps.inc: the padding of every LDS exchange of the tile kernels.

An exchange written by pass P of a line's FFT (radix R, Stockham stride NS)
and read by pass P + 1 stores line position p at word p + c * (p >> s) of the
line's slice (re and im in separate planes, lines LST words apart).  For each
FFT shape, workgroup size, axis (rows: a line's threads are consecutive;
columns: lines fastest) and pass, this script picks the (c, s) that

  * keeps the kernel's offsets linear: f(t + X) = f(t) + f(X) for the offset X
    of every slot a thread reads and f(base + r*NS) = f(base) + f(r*NS) for the
    writes, so every LDS access is a base register plus a compile-time
    immediate, and
  * minimises bank conflicts (32 banks of 4 bytes, 32 lanes per cycle) over
    every write and read instruction of the exchange, then the LDS footprint.

The thread-to-position mapping restates fft_device.hpp (FftPass).  Run it
after changing the FFT schedules; the output is committed beside it.
"""
import os

import numpy as np

F3_BASE, F3_MIN_K, F3_MAX_K, MAX_LOGM = 32, 6, 11, 14
THREADS = (64, 128, 256, 512, 1024)
CANDIDATES = [(0, 2)] + [(c, s) for c in (1, 2, 4, 8, 16) for s in range(2, 10)]


def is_f3(s): return s >= F3_BASE
def m_of(s): return (3 << (s - F3_BASE)) if is_f3(s) else (1 << s)


def tpl_of(s):
    if is_f3(s):
        return m_of(s) // (24 if s - F3_BASE == 11 else 12)
    return m_of(s) // (32 if s >= 13 else 1 << s if s < 4 else 16)


def radices(s):
    if is_f3(s):
        a = s - F3_BASE - 2
        if a == 9:
            return [8, 8, 8, 12]
        return [4] * (a // 2) + [2] * (a % 2) + [12]
    if s >= 13:
        return [32, 16, 16] if s == 13 else [32, 32, 16]
    return [16] * (s // 4) + ([1 << (s % 4)] if s % 4 else [])


def f(p, c, sh): return p + c * (p >> sh)


def line_stride(padm, TPL, LPW, cols):
    # lanes of one wave cover q consecutive positions of 32/q lines: an odd
    # multiple of q keeps their lines on distinct banks
    q = (1 if LPW >= 32 else 32 // LPW) if cols else (0 if TPL >= 32 else TPL)
    st = padm
    if q:
        while st % (2 * q) != q:
            st += 1
    return st


def exchange(s, T, cols, P, c, sh, LST):
    """(linear, worst degree, mean degree) of pass P's writes and pass P+1's reads."""
    M, TPL, rad = m_of(s), tpl_of(s), radices(s)
    LPW = T // TPL
    tid = np.arange(T)
    ll, t = (tid % LPW, tid // LPW) if cols else (tid // TPL, tid % TPL)
    insts = []
    R = rad[P]
    NS = int(np.prod(rad[:P], dtype=np.int64))
    nbf = M // R
    for b in range(-(-nbf // TPL)):
        j = t + b * TPL
        act = j < nbf
        k = j % NS
        bs = (j - k) * R + k
        for r in range(R):
            q = f(bs + r * NS, c, sh)
            if np.any((q != f(bs, c, sh) + f(r * NS, c, sh)) & act):
                return False, 99, 99.0
            insts.append((ll * LST + q, act))
    R2 = rad[P + 1]
    nbf = M // R2
    for b in range(-(-nbf // TPL)):
        act = t + b * TPL < nbf
        for r in range(R2):
            X = b * TPL + r * nbf
            q = f(t + X, c, sh)
            if np.any((q != f(t, c, sh) + f(X, c, sh)) & act):
                return False, 99, 99.0
            insts.append((ll * LST + q, act))
    worst, tot, n = 0, 0, 0
    a = np.array([np.where(act, q, -1) for q, act in insts]).reshape(len(insts) * (T // 32), 32)
    a = np.sort(a, axis=1)
    first = np.ones_like(a, dtype=bool)
    first[:, 1:] = a[:, 1:] != a[:, :-1]
    use = first & (a >= 0)
    cnt = np.zeros((a.shape[0], 32), dtype=np.int64)
    rows = np.repeat(np.arange(a.shape[0])[:, None], 32, axis=1)
    np.add.at(cnt, (rows[use], a[use] % 32), 1)
    d = cnt.max(axis=1)
    live = d > 0
    return True, int(d.max()), float(d[live].mean())


def choose(s, T, cols):
    """(c, s) per exchange and the worst degree, or None when a line does not fit T threads."""
    M, TPL = m_of(s), tpl_of(s)
    if TPL > T or T % TPL:
        return None
    LPW = T // TPL
    nx = len(radices(s)) - 1
    maps = [(1, 4)] * nx
    for _ in range(4):
        padm = max([M] + [f(M - 1, *m) + 1 for m in maps])
        LST = line_stride(padm, TPL, LPW, cols)
        new = []
        for P in range(nx):
            best = None
            for c, sh in CANDIDATES:
                if f(M - 1, c, sh) + 1 > M * 3 // 2 + 64:
                    continue
                lin, w, mean = exchange(s, T, cols, P, c, sh, LST)
                if not lin:
                    continue
                key = (w, mean, f(M - 1, c, sh), c, sh)
                if best is None or key < best[0]:
                    best = (key, (c, sh))
            new.append(best[1])
        if new == maps:
            break
        maps = new
    padm = max([M] + [f(M - 1, *m) + 1 for m in maps])
    LST = line_stride(padm, TPL, LPW, cols)
    worst = max([1] + [exchange(s, T, cols, P, *maps[P], LST)[1] for P in range(nx)])
    return maps, worst


def main():
    shapes = list(range(1, MAX_LOGM + 1))
    shapes += [F3_BASE + k for k in range(F3_MIN_K, F3_MAX_K + 1)]
    lines = ["// Generated by gen_lds_maps.py: LDS padding of every exchange of the tile",
             "// kernels, {shape, threads, cols, pass, c, s}: position p of the exchange",
             "// written by pass `pass` is stored at word p + c * (p >> s).  Worst bank",
             "// conflict degree per configuration in the trailing comment."]
    for s in shapes:
        for T in THREADS:
            for cols in (0, 1):
                r = choose(s, T, cols)
                if r is None:
                    continue
                maps, worst = r
                for P, (c, sh) in enumerate(maps):
                    lines.append(f"{{{s}, {T}, {cols}, {P}, {c}, {sh}}},  // worst {worst}")
    out = os.path.join(os.path.dirname(os.path.abspath(__file__)), "lds_maps.inc")
    with open(out, "w") as fh:
        fh.write("\n".join(lines) + "\n")
    print(f"wrote {out}: {len(lines) - 4} entries")


if __name__ == "__main__":
    main()
