"""Deterministic replay in windows: bit-exact with the oracle where a window can go wrong.

The replay kernel judges several updates at once and runs the plain ones
before the first that is not together (16 to a window, 256 records staged at a
time).  The streams here end a window, or a staged chunk, at every remainder,
put two updates of one vertex into one window, recolour in the middle of one,
fill rows to their end, and mix in records that change nothing.
"""
import numpy as np
import pytest

import oracle_lib as O
import streamgc_amd as S
from test_gpu_parity import _pair, _same_state

pytestmark = pytest.mark.gpu


def _replay(g, parts, **cfg):
    gpu, orc, og = _pair(g, deterministic=True, epoch_size=1 << 20, batch_size=4096, repair_every_epoch=True, **cfg)
    init = S.generate_init_stream(g)
    gpu.process_stream(init)
    orc.submit(init["u"], init["v"], init["type"])
    assert gpu.finish() == orc.finish()
    for k, part in enumerate(parts):
        gpu.process_stream(part)
        orc.submit(part["u"], part["v"], part["type"])
        _same_state(gpu, orc, f"part {k} of {len(part)} updates")
    assert gpu.finish() == orc.finish()
    assert np.array_equal(gpu.snapshot(), orc.snapshot())


@pytest.mark.parametrize("exact", [False, True])
@pytest.mark.parametrize("name", ["delaunay1k", "rmat_s10"])
def test_window_and_chunk_remainders(name, exact, graph_path):
    g = S.load_graph_csr(graph_path(name))
    lengths = [1, 2, 15, 16, 17, 32, 33, 255, 256, 257, 529]
    stream = S.generate_bench_stream_edges(g, sum(lengths), 50, 3)
    cuts = np.cumsum([0] + lengths)
    _replay(g, [stream[a:b] for a, b in zip(cuts, cuts[1:])], exact_histogram=exact)


@pytest.mark.parametrize("threshold", [0, 8, 64])
def test_updates_of_one_vertex_in_one_window(threshold, graph_path):
    """Every update at the hub, and every second one; the hub and its leaves in both selection modes."""
    g = S.load_graph_csr(graph_path("rmat_s10"))
    hub = int(np.argmax(g.degree))
    row = g.col_idx[g.row_ptr[hub]:g.row_ptr[hub + 1]]
    rng = np.random.default_rng(1)
    pick = rng.choice(row, size=60, replace=False).astype(np.uint32)
    at = np.full(60, hub, np.uint32)
    gone, back = S.make_updates(at, pick, np.ones(60, np.uint8)), S.make_updates(pick, at, np.zeros(60, np.uint8))
    other = S.generate_bench_stream_edges(g, 120, 50, 4)
    mixed = np.empty(240, S.EDGE_UPDATE)
    mixed[0::2] = np.concatenate([gone, back])
    mixed[1::2] = other
    _replay(g, [gone, back, mixed], histogram_threshold=threshold, exact_histogram=True)


def test_rows_filled_to_their_end_and_records_without_effect(graph_path):
    """Growth into rows with no slack (overflow in the middle of windows), self-loops, ids out of range, other kinds."""
    g = S.load_graph_csr(graph_path("delaunay1k"))
    rng = np.random.default_rng(2)
    u, v = rng.integers(0, g.n + 3, 900).astype(np.uint32), rng.integers(0, g.n, 900).astype(np.uint32)
    t = rng.choice([0, 0, 0, 1, 2, 200], 900).astype(np.uint8)
    v[::37] = u[::37]
    _replay(g, [S.make_updates(u[:450], v[:450], t[:450]), S.make_updates(u[450:], v[450:], t[450:])],
            slack_pct=20, min_row_capacity=2, overflow_capacity=64)


@pytest.mark.parametrize("graphs", [3, 520])
def test_pool_segments_few_and_many(graphs, graph_path):
    """A block per graph, and (above 512 graphs) a wavefront per graph: each graph as the oracle has it."""
    g = S.load_graph_csr(graph_path("star6" if graphs > 100 else "rmat_s10"))
    cfg = S.StreamGCConfig(epoch_size=64, batch_size=64, overflow_capacity=16)
    pool = S.GraphPool(max_graphs=graphs, batch_capacity=1 << 16, deterministic=True, repair_every_epoch=True)
    gids = [pool.add(g, cfg) for _ in range(graphs)]
    init = S.generate_init_stream(g)
    streams = [np.concatenate([init, S.generate_bench_stream_edges(g, 29, 50, k % 8)]) for k in range(8)]
    pool.submit(np.concatenate([S.tag_graph(streams[gid % 8], gid) for gid in gids]))
    pool.finish()
    for k in range(min(8, graphs)):
        orc = O.Engine(O.Csr(g.n, g.row_ptr, g.col_idx, g.degree),
                       O.default_config(epoch_size=64, batch_size=64, overflow_capacity=16,
                                        flags=O.FLAG_REPAIR_EVERY_EPOCH))
        s = streams[k]
        orc.submit(s["u"], s["v"], s["type"])
        orc.finish()
        for gid in (k, graphs - 8 + k) if graphs > 8 else (k,):
            if gid % 8 == k:
                assert np.array_equal(pool.words(gid), orc.words()), gid
