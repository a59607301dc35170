"""bench.py's longest chain of column steps of the temporal-blocked solve against a schedule of its
tiles phase by phase, every tile starting as early as the words that its waves wait for allow and
one time unit per column step. Wave w runs block n in phase w + n and at its end holds block n + 1's
words: rows up to s1 + 63 of the row-tile before it (whose wave w stores them at the end of its
phase; all of a tile's waves lag alike), for wave 0 also rows up to s1 + TK - 1 of the sweep block
before it (stored by the last wave in its phase) and rows up to s1 + 63 + TK of the corner tile's last
wave, s1 being block n + 1's last step; rows past a tile's last clamp to it."""
import pytest
from test_bench_model import load_bench


def scheduled_finish(G, KB, rows, TK, BLK, W):
    nblk = rows // BLK
    start = {}

    def ends(tile, w, row):  # when the phase in which wave w of the tile ran this row ended
        return start[tile] + (w + min(row, rows - 1) // BLK + 1) * BLK

    finish = 0
    for g in range(G):
        for kb in range(KB):
            t = 0
            for n in range(-1, nblk - 1):  # the phase's number for wave 0; a later wave's is as much later on both sides
                s1 = (n + 1) * BLK + BLK - 1
                due = (n + 1) * BLK
                if g > 0:
                    t = max(t, ends((g - 1, kb), 0, s1 + 63) - due)
                if kb > 0:
                    t = max(t, ends((g, kb - 1), W - 1, s1 + TK - 1) - due)
                if g > 0 and kb > 0:
                    t = max(t, ends((g - 1, kb - 1), W - 1, s1 + 63 + TK) - due)
            start[(g, kb)] = t
            finish = max(finish, t + rows + (W - 1) * BLK)
    return finish


CASES = [(5, 10, 328, 4, 8), (5, 5, 328, 8, 8), (3, 3, 164, 8, 4), (10, 10, 584, 8, 8), (4, 6, 200, 16, 8),
         (6, 4, 320, 4, 4), (1, 1, 72, 2, 8), (67, 13, 4176, 16, 8), (7, 3, 400, 16, 4)]


@pytest.mark.parametrize("case", CASES, ids=["G%d_KB%d_rows%d_tk%d_blk%d" % c for c in CASES])
def test_longest_chain_matches_the_schedule(case):
    G, KB, rows, TK, BLK = case
    layout = dict(sweeps_per_tile=TK, cols_per_block=BLK, handoff_lag=1, row_tiles=G, sweep_blocks=KB,
                  steps_per_tile=rows)
    bench = load_bench()
    assert bench.longest_chain_steps(layout) == scheduled_finish(G, KB, rows, TK, BLK, bench.tile_waves(TK))
