"""Writes yz_pads.h: the LDS strides of the y-z kernels (fft_yz.h) for each
length and precision, chosen by counting bank conflicts.

A wave's 64 lanes are CPW columns of TM lanes, lane = c * TM + t.  LDS has 64
banks of 4 bytes; 16-byte accesses go 16 lanes at a time, 8-byte ones 32 and
4-byte ones all 64.  PS is the plane's column stride, RS the row stride of the
y exchange inside a column, CS, RX and RY the column and row strides of the
wave's z exchange (of single components).  Pads are limited to what leaves as
many waves on a CU as no padding would.

Run from the repository root: python amdkiit_amd/csrc/gen_yz_pads.py
"""
import os
import re

HERE = os.path.dirname(os.path.abspath(__file__))
LDS = 160 * 1024


def lengths():
    src = open(os.path.join(HERE, "amdk_api.hip")).read()
    body = src[src.index("#define AMDK_REG_SIZES(X)"):src.index("static bool reg_ok")]
    return [tuple(map(int, m)) for m in re.findall(r"X\((\d+), (\d+), (\d+)\)", body)]


def cycles(addr, lanes, words):
    """Passes of one access: lanes given as (active, element) pairs."""
    step, total = 64 // words, 0
    for h in range(0, 64, step):
        banks = {}
        for ok, e in addr[h:h + step]:
            if ok:
                for w in range(words):
                    banks.setdefault((e * words + w) % 64, set()).add(e)
        total += max([len(v) for v in banks.values()] or [0])
    return total


def choose(N, A, B, esize):
    TM = max(A, B)
    CPW = 64 // TM
    GZ = (N + CPW - 1) // CPW
    np_ = N // 2 + 1
    lanes = [(l // TM, l % TM) for l in range(64)]

    def cost(f, lim, words):
        return cycles([(c < CPW and t < lim, f(c, t)) for c, t in lanes], lanes, words)

    def lds(W, PS, CS):
        return np_ * 16 + (np_ * PS + 1) * esize + W * CPW * CS * (esize // 2)

    def blocks(W, PS, CS):
        return LDS // lds(W, PS, CS)
    W = 8 if 2 * lds(8, N + 1, N + 1) <= LDS else 16 if esize == 8 and lds(16, N + 1, N + 1) <= LDS else \
        12 if lds(12, N + 1, N + 1) <= LDS else 8
    W = min(W, GZ)
    want = max(1, min(blocks(W, N + 1, N + 1), 32 // W))
    wp, wx = esize // 4, esize // 8
    gy, runs = -(-np_ // CPW), sum(1 for k in range(B) if 4 * A * k <= N or 4 * (N - A * k - A + 1) <= N)
    ex = []
    for RX in range(B, B + 3):
        for RY in range(A, A + 3):
            for CS in range(max(A * RX, B * RY), max(A * RX, B * RY) + 33):
                c = B * cost(lambda c, t: c * CS + t * RX, A, wx) + A * cost(lambda c, t: c * CS + t, B, wx) + \
                    A * cost(lambda c, t: c * CS + t * RY, B, wx) + B * cost(lambda c, t: c * CS + t, A, wx)
                ex.append((2 * GZ * c, CS, RX, RY))
    ex.sort()
    best = None
    for RS in range(B, B + 2):
        for PS in range(max(N, A * RS), max(N, A * RS) + 25):
            y1 = cost(lambda c, t: c * PS + t * RS, A, wp)
            y2 = cost(lambda c, t: c * PS + t, B, wp)
            y3 = cost(lambda c, t: c * PS + t, A, wp)
            z = cost(lambda c, t: t * PS + c, A, wp)
            c = gy * (2 * B * y1 + 3 * A * y2 + B * y3) + 2 * runs * GZ * z
            for e in ex[:200]:
                if max(1, min(blocks(W, PS, e[1]), 32 // W)) >= want and lds(W, PS, e[1]) <= LDS:
                    if best is None or c + e[0] < best[0]:
                        best = (c + e[0], PS, RS) + e[1:]
                    break
    return best or (0, N + 1, B, N + 1, B, A)


def main():
    out = ["// LDS strides of the y-z kernels with the fewest bank conflicts (written by",
           "// gen_yz_pads.py, which says how they are chosen).", "#pragma once", "", "namespace amdk {", "",
           "// bytes: sizeof of a complex value (8 or 16)",
           "template <int N, int bytes> struct YzPads;"]
    for N, A, B in lengths():
        for esize in (8, 16):
            c, PS, RS, CS, RX, RY = choose(N, A, B, esize)
            out.append(f"template <> struct YzPads<{N}, {esize}> {{ static constexpr int PS = {PS}, RS = {RS}, CS = {CS}, "
                       f"RX = {RX}, RY = {RY}; }};")
    out += ["", "}  // namespace amdk"]
    with open(os.path.join(HERE, "yz_pads.h"), "w") as f:
        f.write("\n".join(out) + "\n")


if __name__ == "__main__":
    main()
