"""The host rules of the matrix-core FFT passes (stwo-gpu_amd/csrc/fft_matrix.hpp), built by the host
compiler: how a pass is split into blocks, and which calls take the matrix cores."""
import heapq
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


@pytest.fixture(scope="module")
def ask(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("rules") / "matrix_rules_check")
    subprocess.run(["g++", "-std=c++17", "-O1", "-I" + os.path.join(ROOT, "stwo-gpu_amd", "csrc"),
                    os.path.join(HERE, "matrix_rules_check.cpp"), "-o", out], check=True, capture_output=True)

    def run(queries):
        text = "".join(" ".join(str(w) for w in q) + "\n" for q in queries)
        got = [int(v) for v in subprocess.run([out], input=text, capture_output=True, check=True, text=True).stdout.split()]
        assert len(got) == len(queries)
        return got

    return run


def _makespan(n_groups, tiles, fill, per_block):
    """Length of the launch in groups: each XCD takes its eighth of the blocks in order, fill / 8 at a
    time, a block costing its groups and a start of 0.3."""
    chunks = -(-n_groups // per_block)
    blocks = chunks * tiles
    q, rem = divmod(blocks, 8)
    worst, first = 0.0, 0
    for x in range(8):
        n = q + (1 if x < rem else 0)
        running = [0.0] * (fill // 8)
        for v in range(first, first + n):
            c = v // tiles
            size = min(per_block, n_groups - c * per_block)
            heapq.heapreplace(running, running[0] + size + 0.3)
        first += n
        worst = max(worst, max(running))
    return worst


# column groups, tiles and blocks at a time of the passes of an extension of n_cols columns of 2^n at 2^b
def _passes(n, n_cols, b):
    return [((n_cols + 1) // 2, 1 << (n - 12), 512), (n_cols, 1 << (n - 14), 256), ((n_cols + 1) // 2, 1 << (n + b - 12), 512)]


def test_blocks_are_even(ask):
    """No launch lasts much longer than its work spread over the chip: at most a fifth longer than the
    best of all splits up to 32 groups, over column counts that leave remainders."""
    queries = [q for n, cs in ((20, (24, 36, 48, 60, 67, 72, 96, 101, 200)), (18, (96, 192, 288)), (17, (384, 480, 577)))
               for c in cs for b in (1, 3) for q in _passes(n, c, b)]
    queries = sorted(set(queries))
    got = ask([("split", *q) for q in queries])
    for (g, t, fill), p in zip(queries, got):
        assert 1 <= p <= 32
        mine = _makespan(g, t, fill, p)
        best = min(_makespan(g, t, fill, k) for k in (1, 2, 3, 4, 5, 6, 8, 9, 12, 16, 18, 24, 32))
        assert mine <= 1.2 * best, (g, t, fill, p, mine, best)


def test_one_tile_beyond_the_caches(ask):
    """One tile: a single round while the columns fit the caches, at least four rounds beyond."""
    for g in (1, 100, 512, 2048, 2560, 6144):
        (p,) = ask([("split", g, 1, 512)])
        assert -(-g // p) <= 512
    for g in (8192, 16384, 1 << 18):
        (p,) = ask([("split", g, 1, 512)])
        assert -(-g // p) >= 4 * 512


# calls timed with both forms in one process (median of 25, four times in turn): the matrices' time
# over the butterflies', by log, values in millions (2^20) and kind
BUTTERFLIES_FASTER = [(10, 16, 0), (10, 16, 2), (10, 16, 3), (10, 16, 8), (10, 20, 8), (11, 16, 0), (11, 16, 3), (11, 20, 1),
                      (11, 20, 8), (11, 40, 3), (12, 16, 0), (12, 20, 2), (12, 24, 0), (12, 24, 8), (12, 28, 3), (12, 40, 3),
                      (12, 52, 3), (11, 20, 24)]
MATRICES_FASTER = [(10, 128, 0), (10, 64, 1), (10, 64, 2), (10, 64, 3), (10, 128, 8), (10, 32, 24), (10, 32, 16),
                   (11, 48, 0), (11, 36, 1), (11, 64, 2), (11, 80, 3), (11, 96, 8), (11, 32, 24), (12, 40, 0), (12, 40, 1),
                   (12, 64, 2), (12, 80, 3), (12, 36, 8), (12, 24, 24), (12, 32, 16)]


def test_small_columns_take_the_faster_form(ask):
    q = [("tile", log, (m << 20) >> log, kind) for log, m, kind in BUTTERFLIES_FASTER + MATRICES_FASTER]
    assert ask(q) == [0] * len(BUTTERFLIES_FASTER) + [1] * len(MATRICES_FASTER)


def test_small_columns_that_the_matrices_do_not_take(ask):
    """Other sizes of domain, blowups above 8, and a source larger than the domain."""
    assert ask([("tile", 9, 1 << 20, 0), ("tile", 13, 1 << 20, 0), ("tile", 12, 1 << 20, 4), ("tile", 12, 1 << 20, 7)]) == [0] * 4
