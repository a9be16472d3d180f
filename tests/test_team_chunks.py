"""The chunks in which the team kernel works a lattice (muca_amd/csrc/team_run.h),
restated with the rounds and order that the library's layout has for each L, and
enumerated over whole launches: they follow the reference's site order
(muca_delta_multigpu.cu:173), and none holds a site twice or two neighbouring
sites.  Odd L (passes over the even linear indices, chunks over row ends where a
chunk is no longer than the attempts between two neighbours) and even L whose
chunks run on into the next row."""
import pytest

import muca_amd as M
from test_team_layout import layout

FLOWING = [L for L in range(8, 84) if layout(L)["order"] == 2]


def _odd(L, NR, n):
    N, hw = L * L, (L - 1) // 2
    ox = oy = ot = op = rs = 0
    while rs < n:
        if hw >= 16 * NR:
            left = (N - 1 - oy * L - ox) // 2
        else:
            left = hw - ot if ot < hw else L - ot
        cnt = min(1 if op == 2 else left, 16 * NR, n - rs)
        sites = []
        for j in range(cnt):
            x, y = ox + 2 * j, oy
            if x >= L:
                x, y = x - L, y + 1
            assert 0 <= x < L and y < L
            sites.append(y * L + x)
        yield sites
        rs += cnt
        ox, ot = ox + 2 * cnt, ot + cnt
        while ox >= L:
            ox, oy = ox - L, oy + 1
        if ot == L:
            ot = 0
        if op == 2:
            ox = oy = ot = op = 0
        elif (ox, oy) == (L - 1, L - 1):
            ox, oy = (0, 0) if op == 0 else (L - 2, L - 1)
            ot, op = 0, op + 1


def _even(L, NR, n, over_rows):
    Rw = L // 2
    h = y = jb = rs = 0
    while rs < n:
        cnt = min(Rw if over_rows else Rw - jb, 16 * NR, n - rs)
        sites = []
        for j in range(cnt):
            x, yy, hh = 2 * (jb + j), y, h
            if x >= L:
                x, yy = x - L, (y + 1) % L
                hh = h ^ 1 if y + 1 == L else h
            sites.append(yy * L + x + hh)
        yield sites
        rs += cnt
        jb += cnt
        if jb >= Rw:
            jb, y = jb - Rw, y + 1
            if y == L:
                y, h = 0, h ^ 1


def _check(L, chunks, n):
    N = L * L
    half = N // 2
    i = 0
    for sites in chunks:
        s = set(sites)
        assert len(s) == len(sites)
        for e in sites:
            k = i % N
            assert e == (2 * k % N if k // half % 2 == 0 else (2 * k + 1) % N), (L, i)
            x, y = e % L, e // L
            around = {y * L + (x + 1) % L, y * L + (x - 1) % L, (y + 1) % L * L + x,
                      (y - 1) % L * L + x}
            assert not around & s, (L, e)
            i += 1
    assert i == n


@pytest.mark.parametrize("L", range(9, 84, 2))
def test_odd_chunks(L):
    seen = set()
    for prec, moments in ((M.REF32, False), (M.FP64, False), (M.FP64, True)):
        q = layout(L, prec=prec, moments=moments)
        if q["eligible"]:
            assert q["order"] == 1
            seen.add(q["rounds"])
    assert seen or L > 79
    N = L * L
    for NR in seen:
        for n in (2 * N + 7, N - 1, N // 2 + 3, 16 * NR + 1, 1):
            _check(L, _odd(L, NR, n), n)


@pytest.mark.parametrize("L", FLOWING + [80])
def test_even_chunks_over_row_ends(L):
    q = layout(L, prec=M.FP64, moments=L == 80)
    assert q["order"] == 2 and q["lat_lds"] and L % 32 // 2 <= 8
    N, NR = L * L, q["rounds"]
    assert 16 * NR <= L // 2
    for n in (2 * N + 7, N + L // 2 - 1, N // 2 + 3, 16 * NR + 1, 1):
        _check(L, _even(L, NR, n, True), n)


@pytest.mark.parametrize("L", [8, 10, 32, 56, 60, 80, 100, 128, 138, 256])
def test_even_chunks_within_rows(L):
    q = layout(L)
    assert q["eligible"] and q["order"] == 0
    N = L * L
    n = N + 3 * L + 5
    _check(L, _even(L, q["rounds"], n, False), n)


def test_sizes_that_the_flow_tests_run():
    """Two rounds and up to eight attempts over: L = 78 with and 80 without a
    histogram in LDS; L = 80 with one keeps its lattices in HBM, row by row."""
    assert {34, 48, 66, 72, 76, 78} <= set(FLOWING) and 80 not in FLOWING
    assert layout(78)["rounds"] == 2 and not layout(80)["lat_lds"]
    assert layout(80, prec=M.FP64, moments=True)["order"] == 2
