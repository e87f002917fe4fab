#!/usr/bin/env python3
"""Generates lds_maps.inc: the padding of every LDS exchange of the tile kernels.

An exchange written by pass P of a line's FFT (radix R, Stockham stride NS)
and read by pass P + 1 stores line position p at word p + c * (p >> s) of the
line's slice (re and im in separate planes, lines LST words apart).  For each
FFT shape, workgroup size, axis (rows: a line's threads are consecutive;
columns: lines fastest) and pass, this script picks the (c, s) that

  * keeps the kernel's offsets linear: f(t + i*TPL) = f(t) + f(i*TPL) for the
    reads and f(base + r*NS) = f(base) + r*f(NS) for the writes, so every LDS
    access is a base register plus a compile-time immediate, and
  * minimises bank conflicts (32 banks of 4 bytes, 32 lanes per cycle) over
    every write and read instruction of the exchange, then the LDS footprint.

The thread-to-position mapping restates fft_device.hpp (FftPass).  Run it
after changing the FFT schedules; the output is committed beside it.
"""
import itertools
import os

F3_BASE, F3_MIN_K, F3_MAX_K, MAX_LOGM = 32, 6, 11, 14
THREADS = (64, 128, 256, 512, 1024)
CANDIDATES = [(0, 2)] + [(c, s) for c in (1, 2, 4, 8, 16) for s in range(2, 10)]


def is_f3(s): return s >= F3_BASE
def m_of(s): return (3 << (s - F3_BASE)) if is_f3(s) else (1 << s)
def is_wide(s): return s in (13, 14)
def ept_of(s): return 12 if is_f3(s) else 32 if is_wide(s) else (1 << s if s < 4 else 16)


def npass_of(s):
    if is_f3(s):
        a = s - F3_BASE - 2
        return a // 2 + a % 2 + 1
    return 3 if is_wide(s) else (s + 3) // 4


def radix_of(s, p):
    if p >= npass_of(s):
        return 1
    if is_f3(s):
        a = s - F3_BASE - 2
        return 4 if p < a // 2 else (12 if p == npass_of(s) - 1 else 2)
    if is_wide(s):
        return 32 if p == 0 or (s == 14 and p == 1) else 16
    return 1 << min(4, s - 4 * p)


def ns_of(s, p):
    n = 1
    for q in range(p):
        n *= radix_of(s, q)
    return n


def f(p, c, sh): return p + c * (p >> sh)


def lanes(T, TPL, LPW, cols):
    for tid in range(T):
        yield (tid % LPW if cols else tid // TPL), (tid // LPW if cols else tid % TPL)


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
    M, EPT = m_of(s), ept_of(s)
    TPL = M // EPT
    LPW = T // TPL
    R, NS = radix_of(s, P), ns_of(s, P)
    NB = EPT // R
    insts = []
    for b in range(NB):
        for r in range(R):
            a = []
            for ll, t in lanes(T, TPL, LPW, cols):
                j = t + b * TPL
                k = j & (NS - 1)
                base = (j - k) * R + k
                q = f(base + r * NS, c, sh)
                if q != f(base, c, sh) + r * f(NS, c, sh):
                    return False, 99, 99.0
                a.append(ll * LST + q)
            insts.append(a)
    for i in range(EPT):
        a = []
        for ll, t in lanes(T, TPL, LPW, cols):
            q = f(t + i * TPL, c, sh)
            if q != f(t, c, sh) + f(i * TPL, c, sh):
                return False, 99, 99.0
            a.append(ll * LST + q)
        insts.append(a)
    worst, tot, n = 0, 0, 0
    for a in insts:
        for h in range(0, T, 32):
            banks = {}
            for x in set(a[h:h + 32]):
                banks[x % 32] = banks.get(x % 32, 0) + 1
            d = max(banks.values())
            worst, tot, n = max(worst, d), tot + d, n + 1
    return True, worst, tot / n


def choose(s, T, cols):
    """(c, s) per exchange and the line stride, or None when a line does not fit T threads."""
    M, EPT = m_of(s), ept_of(s)
    TPL = M // EPT
    if TPL > T or T % TPL:
        return None
    LPW = T // TPL
    nx = npass_of(s) - 1
    maps = [(1, 4)] * nx
    for _ in range(4):
        padm = max([M] + [f(M - 1, *m) + 1 for m in maps])
        LST = line_stride(padm, TPL, LPW, cols)
        new = []
        for P in range(nx):
            best = None
            for c, sh in CANDIDATES:
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
    return maps, LST, worst


def main():
    shapes = list(range(1, MAX_LOGM + 1)) + [F3_BASE + k for k in range(F3_MIN_K, F3_MAX_K + 1)]
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
                maps, LST, worst = r
                for P, (c, sh) in enumerate(maps):
                    lines.append(f"{{{s}, {T}, {cols}, {P}, {c}, {sh}}},  // worst {worst}")
    out = os.path.join(os.path.dirname(os.path.abspath(__file__)), "lds_maps.inc")
    with open(out, "w") as fh:
        fh.write("\n".join(lines) + "\n")
    print(f"wrote {out}: {len(lines) - 4} entries")


if __name__ == "__main__":
    main()
