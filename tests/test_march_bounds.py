"""Host-side check of the addresses of the marching kernel (march_wave in
portlbm_amd/csrc/lbm_march.hip) and of the parts that lattices and batches are
cut into: for every wave of every lattice below, each element that it can
store belongs to a node of its own strip and rows (or to the places between
the row's last node and the next row, which no one else uses), no two waves
store the same element, every fluid node is stored, every read lies in the
allocation and every LDS access in the wave's slot.  The masks that drop stores
are taken as wide as they can be: each segment holds a fluid node.  The
arithmetic is the kernel's own, restated.
"""
import numpy as np
import pytest

ELEM = {"f64": 8, "f32": 4, "f16": 2}
K_OF = {"collision": 9, "stream": 1, "bundle": 3}
HALO, OWN = 4, 56
NOWHERE = 0xfffffff0


def _ru(n, a):
    return (n + a - 1) // a * a


def lattice_placement(Hx, Vx, elem):
    """P, X0, direction stride and bytes of a lattice's allocation."""
    X0 = 63
    P = _ru(X0 + Hx, 64)
    M = P * Vx
    Sd = _ru(M, ((2 << 20) if M * elem >= (32 << 20) else 4096) // elem) + 512 // elem
    return P, X0, Sd, 9 * Sd * elem + 64


def batch_placement(H, V, elem):
    """The same for a domain of a batch, which ends where the next one begins."""
    X0 = 15
    P = _ru(X0 + H, 16)
    return P, X0, P * V, 9 * P * V * elem


def wave(place, Hx, Vx, layout, elem, strip, y0, y1, T, skew=0):
    """(elements stored, byte ranges read, highest LDS byte) of one wave."""
    P, X0, Sd, _ = place
    N, K = 8 // elem, K_OF[layout]
    NA, VA = 9 // K, 64 * K // 2
    lane = np.arange(64)
    xw = 1 + strip * OWN * N - HALO * N + skew
    last = (Hx - 1 - xw) // N
    jb, je = max(y0 - T, 0), y1 - 1 + T
    wp = X0 + xw
    assert wp >= 0 and last >= HALO
    stride = Sd * K * elem
    stored, reads, lds = [], [], 0
    for j in range(jb, je + 2):  # fetch(jb) and fetch(j + 1) for j = jb .. je
        y = min(j, Vx - 1)
        reads.append(("code", 2 * (y * P + wp + np.minimum(lane, last) * N), 2 * N))
        row = (y * P + wp) * K * elem
        if layout == "stream":
            for d in range(9):
                reads.append(("lat", row + d * stride + np.minimum(lane, last) * 8, 8))
        else:
            top = ((min(last, 63) + 1) * 8 * K - 1) // 16
            for r in range(5):
                v, at = lane + 64 * r, np.full(64, row)
                if layout == "bundle":
                    if r == 1:
                        at, v = at + np.where(lane < 32, 0, stride), v - np.where(lane < 32, 0, VA)
                    elif r > 1:
                        at, v = at + (stride if r == 2 else 2 * stride), v - (VA if r == 2 else 2 * VA)
                reads.append(("lat", at + np.minimum(v, top) * 16, 16))
                lds = max(lds, (64 * r + 64) * 16)
    for y in range(y0, y1):
        row = (y * P + wp) * K * elem
        if layout == "stream":
            off = 8 * lane[(lane >= HALO) & (lane < 64 - HALO) & (lane <= last)]
            for d in range(9):
                stored.append((row + d * stride + off)[:, None] + np.arange(0, 8, elem))
        else:
            lanes = min(OWN, (Hx - 2 - xw) // N + 1 - HALO)
            nbytes = lanes * 8 * K
            for a in range(NA):
                base = row + HALO * 8 * K + a * stride
                lds = max(lds, 8 * (a * 64 * K + 63 * K + K))
                VO = OWN * K // 2
                for n in range((VO + 63) // 64):
                    v = 64 * n + lane
                    lds = max(lds, 16 * (a * VA + HALO * K // 2 + int(np.where(v < VO, v, 0).max()) + 1))
                    off = np.where(v * 16 < nbytes, v * 16, NOWHERE)
                    whole = off[(off != NOWHERE) & (off + 16 <= nbytes)]
                    half = off[(off != NOWHERE) & (off + 16 > nbytes)] if nbytes % 16 else off[:0]
                    assert all(o + 16 <= 64 * 8 * K for o in whole)  # the buffer's window
                    stored += [(base + whole)[:, None] + np.arange(0, 16, elem), (base + half)[:, None] + np.arange(0, 8, elem)]
    elements = np.concatenate([s.ravel() for s in stored]) // elem
    return elements, reads, lds


def check(place, Hx, Vx, layout, elem, parts, T, skew=0):
    P, X0, Sd, nbytes = place
    K, N = K_OF[layout], 8 // elem
    own = OWN * N
    owner = np.zeros(9 * Sd, dtype=np.int32)
    bad = 0
    for w, (strip, y0, y1) in enumerate(parts, 1):
        elements, reads, lds = wave(place, Hx, Vx, layout, elem, strip, y0, y1, T, skew)
        bad += int(np.any(elements < 0) or np.any(elements >= 9 * Sd) or np.unique(elements).size != elements.size)
        elements = elements[(elements >= 0) & (elements < 9 * Sd)]
        bad += int(np.any(owner[elements] != 0))
        owner[elements] = w
        a, r = elements // (K * Sd), elements % (K * Sd)
        n = r // K
        x, y = n % P - X0, n // P
        lo, hi = 1 + strip * own, min(1 + (strip + 1) * own, Hx)
        end = np.where(hi == Hx, Hx + N - 1, hi)  # places past the last column
        bad += int(np.any((y < y0) | (y >= y1) | (x < lo) | (x >= end)))
        for kind, at, size in reads:
            bad += int(np.any(at < 0))
            if kind == "code":
                bad += int(np.any(at + size > 2 * Sd))
            else:
                bad += int(np.any(at + size > nbytes))
        bad += int(lds > 320 * 16)
    y, x = np.mgrid[1:Vx - 1, 1:Hx - 1]
    n = (y * P + X0 + x).ravel()
    for d in range(9):
        bad += int(np.any(owner[(d // K) * K * Sd + K * n + d % K] == 0))
    return bad


def lattice_parts(Hx, Vx, elem, rows):
    own = OWN * 8 // elem
    strips, inner = (Hx - 2 + own - 1) // own, Vx - 2
    segs = (inner + rows - 1) // rows
    return [(s, 1 + g * rows, min(1 + (g + 1) * rows, Vx - 1)) for g in range(segs) for s in range(strips)]


@pytest.mark.parametrize("storage", ["f64", "f32", "f16"])
@pytest.mark.parametrize("layout", ["collision", "stream", "bundle"])
def test_lattices(layout, storage):
    elem = ELEM[storage]
    own = OWN * 8 // elem
    for width in (2, 3, own - 1, own, own + 1, own + 2, own + 5, 2 * own, 2 * own + own // 2 + 1):
        for inner, rows, T in ((9, 4, 4), (5, 8, 3), (7, 7, 2), (2, 4, 4)):
            Hx, Vx = width + 2, inner + 2
            assert check(lattice_placement(Hx, Vx, elem), Hx, Vx, layout, elem, lattice_parts(Hx, Vx, elem, rows), T) == 0


@pytest.mark.parametrize("storage", ["f64", "f32", "f16"])
def test_domains_of_a_batch(storage):
    """Rows split evenly into segments; the domain ends with its own places."""
    elem = ELEM[storage]
    own = OWN * 8 // elem
    for width in (2, 3, 15, 16, 28, own, own + 3):
        for inner, best in ((2, 8), (9, 8), (23, 8), (40, 13)):
            Hx, Vx = width + 2, inner + 2
            segs = (inner + best - 1) // best
            parts = [(s, 1 + inner * g // segs, 1 + inner * (g + 1) // segs) for g in range(segs)
                     for s in range((width + own - 1) // own)]
            assert check(batch_placement(Hx, Vx, elem), Hx, Vx, "stream", elem, parts, 4) == 0


def test_the_check_sees_misplaced_stores():
    for layout in K_OF:
        place = lattice_placement(130, 12, 8)
        parts = lattice_parts(130, 12, 8, 4)
        assert check(place, 130, 12, layout, 8, parts, 4, skew=1) > 0
        assert check(place, 130, 12, layout, 8, parts[:-1], 4) > 0
        assert check(place, 130, 12, layout, 8, parts + parts[:1], 4) > 0
