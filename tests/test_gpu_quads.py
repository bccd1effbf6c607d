"""Edges that share a vertex within one wavefront of the four-edge path.

Four light edges go to a wavefront in lock-step, in the order of their records
where every record is an edge of its own.  Each four here hold a delete at x
that lowers x's colour and inserts that join x to a vertex with a histogram, in
every order; fours share nothing, so words, rows (as sets: which free slot an
insert meets depends on the order) and histograms are the sequential oracle's.
"""
import numpy as np
import pytest

import streamgc_amd as S
import test_gpu_apply
from test_gpu_parity import _pair

pytestmark = pytest.mark.gpu

FOURS = 2304   # 9,216 edges: whole blocks of 256 records, and enough for the four-edge path
LEAVES = 9     # of each histogram vertex


def _graph():
    """Each four's vertices: x, its neighbours a and p, two stars b0 and b1 with their leaves, and two pairs of loose
    vertices; colours 3, 1, 1, 4 and 5, 1, and 1 and 2 (x can fall to 2 when it loses a)."""
    size = 3 + 2 * (1 + LEAVES) + 4
    at = np.arange(FOURS) * size
    edges, colour = [], np.ones(FOURS * size, np.uint32)
    for i in at.tolist():
        edges += [(i, i + 1), (i, i + 2)]
        for k in range(2):
            b = i + 3 + k * (1 + LEAVES)
            edges += [(b, b + 1 + j) for j in range(LEAVES)]
            colour[b] = 4 + k
        colour[[i, size + i - 3, size + i - 1]] = 3, 2, 2
    return S.csr_from_edges(FOURS * size, edges), colour, at, size


def _rows(csr):
    """The slots with each row's sorted."""
    rp, col = csr
    row = np.repeat(np.arange(len(rp) - 1), np.diff(rp.astype(np.int64)))
    return col[np.lexsort((col, row))]


@pytest.mark.parametrize("threshold", [1, LEAVES - 1])   # x has a histogram as well, or a bitmap
def test_deletes_and_inserts_at_one_vertex(threshold):
    g, colour, at, size = _graph()
    gpu, orc, og = _pair(g, epoch_size=1 << 20, batch_size=1 << 20, histogram_threshold=threshold,
                         exact_histogram=True)
    words = (colour | 1 << 16).astype(np.uint32)
    for eng in (gpu, orc):
        eng.set_words(words)
        eng.finish()
    recs = []
    for k, x in enumerate(at.tolist()):
        b0, b1, loose = x + 3, x + 4 + LEAVES, x + size - 4
        gone, in0, in1, pair = (x, x + 1, 1), (x, b0, 0), (b1, x, 0), (loose, loose + 1, 0)
        four = [[gone, in0, in1, pair], [in0, gone, pair, in1], [pair, in1, in0, gone], [in0, (x + 1, x, 1), pair,
                (loose + 2, loose + 3, 0)]][k % 4]
        recs += four
    batch = S.make_updates(*(list(c) for c in zip(*recs)))
    gpu.apply(batch)
    orc.submit(batch["u"], batch["v"], batch["type"])
    assert gpu.totals()["recolors"] >= FOURS
    assert np.array_equal(gpu.words(), orc.words())
    assert np.array_equal(_rows(gpu.csr()), _rows(orc.csr()))
    assert np.array_equal(gpu.hist(), orc.hist())
    assert np.all(orc.bitmaps() & ~gpu.bitmaps() == 0)   # (no neighbour's colour is missing)


@pytest.mark.parametrize("slack,cap", [(300, 0), (0, 1), (50, 2)])
@pytest.mark.parametrize("graphs", [1, 3])
def test_light_edges_by_four(graphs, slack, cap, monkeypatch):
    """The disjoint light edges of test_gpu_apply, more of them and over twice as many vertices as updates."""
    plain = test_gpu_apply._light_graph

    def sparse():
        g = plain()
        return S.CSRGraph(g.n + 12000, np.concatenate([g.row_ptr, np.full(12000, g.row_ptr[-1])]), g.col_idx)
    monkeypatch.setattr(test_gpu_apply, "PAIRS", 6500)
    monkeypatch.setattr(test_gpu_apply, "_light_graph", sparse)
    test_gpu_apply.test_light_edges_keep_the_oracles_slots(graphs, slack, cap)


@pytest.mark.parametrize("pairs", [4097, 8192, 8193, 8196, 9217])
def test_where_light_edges_go_by_four(pairs):
    """Launches at and past the least number of updates, and with one to two vertices and one more."""
    g = S.csr_from_edges(2 * pairs, [(2 * i, 2 * i + 1) for i in range(pairs)])
    gpu, orc, og = _pair(g, epoch_size=1 << 20, batch_size=1 << 20)
    u = 2 * np.arange(pairs, dtype=np.uint32)
    for extra, kind in ((0, 1), (1, 0), (0, 1)):
        recs = S.make_updates(np.concatenate([u, u[:extra]]), np.concatenate([u + 1, u[:extra] + 1]),
                              np.full(pairs + extra, kind, np.uint8))
        gpu.apply(recs)
        orc.submit(recs["u"], recs["v"], recs["type"])
        assert np.array_equal(gpu.csr()[1], orc.csr()[1]), (pairs, extra)
        assert np.array_equal(gpu.words() & 0xFFFF, orc.words() & 0xFFFF), (pairs, extra)


@pytest.mark.parametrize("vertices,more", [(64, 0), (22, 80000), (4, 0)])
def test_long_rows_among_light_edges(vertices, more):
    """Long rows' searches in launches of light edges: by four with long trips (64 vertices to an update), by four
    with short ones (a graph with few heavy edges), and one edge to a wavefront (most edges heavy)."""
    bed, pairs = 4000, 8200
    rng = np.random.default_rng(8)
    edges = [(bed + k, int(x)) for k, d in enumerate(test_gpu_apply.LONG) for x in rng.choice(bed, size=d, replace=False)]
    first = bed + len(test_gpu_apply.LONG)
    edges += [(first + 2 * i, first + 2 * i + 1) for i in range(pairs + more)]
    g = S.csr_from_edges(vertices * (pairs + 100), edges)
    gpu, orc, og = _pair(g, epoch_size=1 << 20, batch_size=1 << 20, slack_pct=3)
    u = first + 2 * np.arange(pairs, dtype=np.uint32)
    live = test_gpu_apply._live
    for k in range(6):   # one update of each long row a launch: deletes, a re-insert, inserts, a delete
        rows, used, recs = orc.csr(), set(), []
        for x in range(bed, first):
            row = [w for w in live(rows, x) if w not in used]
            out = [w for w in range(bed) if w not in used and w not in set(row)]
            w = row[(0, len(row) // 2, len(row) - 1)[(x + k) % 3]]
            recs.append([(x, w, 1), (w, x, 1), (x, out[x % 5], 0), (x, w, 0), (out[0], x, 0), (x, w, 1)][k])
            used |= {recs[-1][0], recs[-1][1]}
        a, b, t = (np.array(c) for c in zip(*recs))
        batch = S.make_updates(np.concatenate([a, u]), np.concatenate([b, u + 1]),
                               np.concatenate([t, np.full(pairs, 1 - k % 2)]).astype(np.uint8))
        gpu.apply(batch)
        orc.submit(batch["u"], batch["v"], batch["type"])
        got, want = gpu.csr()[1], orc.csr()[1]
        assert np.array_equal(got, want), (k, np.nonzero(got != want)[0][:8])
    assert gpu.overflow_count() == orc.overflow_count()


@pytest.mark.parametrize("order", [{"repair_every_epoch": True}, {}])
def test_shared_vertices_keep_every_invariant(order):
    """Churn and growth whose updates share vertices at random: the live edges are the oracle's, every bitmap
    row's bits hold its neighbours' colours, and a repaired epoch is proper."""
    g = S.gen_chung_lu(40000, 200000, 2.3, 300.0, seed=3, permute=True)
    gpu, orc, og = _pair(g, epoch_size=12000, batch_size=12000, exact_histogram=True, histogram_threshold=40, **order)
    init = S.generate_init_stream(g)
    gpu.process_stream(init)
    gpu.finish()
    orc.submit(init["u"], init["v"], init["type"])
    orc.finish()
    for stream in (S.generate_bench_stream_edges(g, 24000, 50, 6), S.dense_growth_stream(g, 24000, seed=7)):
        gpu.process_stream(stream)
        orc.submit(stream["u"], stream["v"], stream["type"])
        if not order:
            gpu.finish()
        assert gpu.overflow_count() == orc.overflow_count() == 0
        assert gpu.validate()[:2] == (0, 0)
        rp, col = gpu.csr()
        row = np.repeat(np.arange(g.n), np.diff(rp.astype(np.int64)))
        live = col != 0xFFFFFFFF
        assert np.array_equal(_rows((rp, col)), _rows(orc.csr()))
        colour = gpu.colors().astype(np.int64)[col[live]]
        held = gpu.bitmaps()[row[live]]
        few = (colour <= 64) & (g.degree[row[live]] <= 40)   # (histogram rows' bitmaps are never rebuilt)
        assert np.all(held[few] >> (colour[few] - 1).astype(np.uint64) & np.uint64(1))
