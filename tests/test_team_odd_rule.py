"""The chunks in which the team kernel works an odd lattice
(muca_amd/csrc/team_run.h, ODD), restated and enumerated over whole launches:
they follow the reference's site order (muca_delta_multigpu.cu:173) and none
holds two neighbouring sites."""
import pytest


def _chunks(L, NR, n):
    ox = oy = ot = op = rs = 0
    hw = (L - 1) // 2
    while rs < n:
        most = 1 if op == 2 else (hw - ot if ot < hw else L - ot)
        cnt = min(most, 16 * NR, n - rs)
        sites = []
        for j in range(cnt):
            x, y = ox + 2 * j, oy
            if x >= L:
                x, y = x - L, y + 1
            sites.append(y * L + x)
        yield sites
        rs += cnt
        ox += 2 * cnt
        ot += cnt
        while ox >= L:
            ox, oy = ox - L, oy + 1
        if ot == L:
            ot = 0
        if op == 2:
            ox = oy = ot = op = 0
        elif (ox, oy) == (L - 1, L - 1):
            ox, oy = (0, 0) if op == 0 else (L - 2, L - 1)
            ot, op = 0, op + 1


@pytest.mark.parametrize("L", [9, 11, 15, 31, 33, 45, 65, 71])
def test_chunks_follow_the_order_and_hold_no_neighbours(L):
    N = L * L
    half = N // 2
    order = [(2 * i) % N if (i // half) % 2 == 0 else (2 * i + 1) % N for i in range(N)]
    NR = min(4, ((L + 1) // 2 + 15) // 16)
    for n in (2 * N + 7, N - 1, half + 3, 1):
        got = []
        for sites in _chunks(L, NR, n):
            s = set(sites)
            for e in sites:
                x, y = e % L, e // L
                around = {y * L + (x + 1) % L, y * L + (x - 1) % L, (y + 1) % L * L + x,
                          (y - 1) % L * L + x}
                assert not around & s, (L, e)
            got += sites
        assert got == [order[i % N] for i in range(n)]
