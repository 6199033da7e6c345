"""The folded GEMM's launch plan on the host: every output tile computed once, inside the scratch rule,
and small tiles wherever they are the faster ones."""
import math
import random

import pytest

import _oracle as O
import _plan as P

FORMATS = [O.Q4_K, O.Q2_K, O.IQ3_S, O.Q4_0, O.Q8_0]


def tiles_of(p):
    """(tile_m, tile_n, K piece) of every workgroup, as mmqh_kernel maps its block index."""
    tr0, tc0, tiles = p.r0 // p.bm, p.c0 // p.bn, p.tiles_n * p.tiles_m
    count = p.main + (tiles - p.main) * p.pieces if p.pieces else p.main
    for z in range(p.splits):
        for b in range(count):
            if p.pieces and b >= p.main:
                q = b - p.main
                tt, width = q // p.pieces, p.tiles_n - tc0
                yield tr0 + tt // width, tc0 + tt % width, q % p.pieces
                continue
            t = (b % 8) * (p.main // 8) + b // 8 if p.main % 8 == 0 else b
            if p.rows and t >= tr0 * p.tiles_n:
                u = t - tr0 * p.tiles_n
                yield tr0 + u // tc0, u % tc0, z
            else:
                yield t // p.tiles_n, t % p.tiles_n, z


@pytest.mark.parametrize("qtype", FORMATS, ids=lambda t: O.NAMES[t])
def test_plan_covers_the_output(qtype):
    rng = random.Random(qtype)
    seen = set()

    def log_int(low, high):
        return int(math.exp(rng.uniform(math.log(low), math.log(high + 1))))

    for _ in range(400):
        m, n = log_int(17, 3000), log_int(1, 40000)
        k = 32 * log_int(1, 544) if O.BLOCK[qtype][0] == 32 else 256 * log_int(1, 68)
        p = P.folded(qtype, n, k, m)
        seen.add(p.id)
        assert p.tiles_n == -(-n // p.bn) and p.tiles_m == -(-m // p.bm)
        stages = -(-k // 256) * 4
        want = {(i, j): [] for i in range(p.tiles_m) for j in range(p.tiles_n)}
        for i, j, z in tiles_of(p):
            want[i, j].append(z)
        left = [t for t, z in want.items() if not z]
        if p.rest:  # the tiles from number `main` on, to a second launch in quarters
            assert p.splits == 1 and not p.pieces and p.bn == p.bm == 256
            assert sorted(left) == sorted((t // p.tiles_n, t % p.tiles_n) for t in range(p.main, p.main + p.rest))
        else:
            assert not left
        for (i, j), z in want.items():
            if z:
                tail = p.pieces and i * p.bm >= p.r0 and j * p.bn >= p.c0
                assert sorted(z) == list(range(p.pieces if tail else p.splits)), (n, k, m, p)
        if p.splits > 1:
            assert p.split_stages % 4 == 0 and (p.splits - 1) * p.split_stages < stages <= p.splits * p.split_stages
            assert p.splits * m * n * 4 <= p.sums
        if p.pieces:
            assert p.piece_stages % 4 == 0 and (p.pieces - 1) * p.piece_stages < stages <= p.pieces * p.piece_stages
            assert p.pieces * p.rows * p.cols * 4 <= p.sums
            assert (p.rows, p.cols) == (m - p.r0, n - p.c0) and p.r0 % p.bm == 0 and p.c0 % p.bn == 0
            assert p.r0 == 0 or p.c0 > 0 or p.r0 // p.bm * p.tiles_n == p.main
    assert len(seen) >= 8, seen


# n, K, rows whose products ran on tiles of 128 activation rows (128 x 128 with two K groups) in up to twice
# the time of the smaller tiles
SMALL = [(O.Q8_0, 512, 5120, 97), (O.Q8_0, 140, 1216, 312), (O.Q8_0, 4, 2624, 571), (O.Q8_0, 1536, 1056, 110),
         (O.Q4_0, 9892, 5792, 242), (O.Q2_K, 7548, 2560, 100), (O.Q2_K, 512, 5120, 1000)]


@pytest.mark.parametrize("qtype,n,k,m", SMALL)
def test_small_tiles_at_more_rows(qtype, n, k, m):
    assert P.folded(qtype, n, k, m).bm < 128
