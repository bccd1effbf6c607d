"""Maintenance sweeps with several rows to a wavefront.

A sweep over more rows than its grid has wavefronts takes four rows at a time,
16 lanes each, for rows of at most 64 slots, and the whole wavefront for longer
ones.  The graphs here have rows of every length around 16, 64 and 128 slots,
and a grid of one block makes every sweep take the shared form.
"""
import numpy as np
import pytest

import oracle_lib as O
import streamgc_amd as S
from test_gpu_parity import _pair, _same_state

pytestmark = pytest.mark.gpu

LENGTHS = [1, 2, 15, 16, 17, 31, 32, 33, 47, 48, 49, 62, 63, 64, 65, 66, 127, 128, 129, 130, 257]


def _graph(seed=5):
    """Vertices of the degrees above (three of each) over a bed of 900 others."""
    rng = np.random.default_rng(seed)
    edges, at = [], 900
    for d in LENGTHS * 3:
        edges += [(at, int(x)) for x in rng.choice(900, size=d, replace=False)]
        at += 1
    edges += [(int(a), int(b)) for a, b in rng.integers(0, 900, (700, 2)) if a != b]
    return S.csr_from_edges(at, edges)


@pytest.mark.parametrize("full", [False, True])
@pytest.mark.parametrize("slack", [30, 300])
@pytest.mark.parametrize("threshold", [64, 1000])
def test_shared_sweeps_bit_exact(threshold, slack, full):
    """Compaction, rebuild and the Tier-2 check, with rows that overflow (slack 30) and rows that do not."""
    g = _graph()
    gpu, orc, og = _pair(g, deterministic=True, epoch_size=300, batch_size=300, repair_every_epoch=True,
                         exact_histogram=True, histogram_threshold=threshold, slack_pct=slack, full_sweeps=full)
    gpu.set_tuning(sweep_blocks=1, apply_blocks=1)
    init = S.generate_init_stream(g)
    assert gpu.process_stream(init) == orc.submit(init["u"], init["v"], init["type"])
    _same_state(gpu, orc, "init")
    churn = S.generate_bench_stream_edges(g, 1800, 40, 9)
    assert gpu.process_stream(churn) == orc.submit(churn["u"], churn["v"], churn["type"])
    _same_state(gpu, orc, "churn")
    assert gpu.finish() == orc.finish()
    assert np.array_equal(gpu.snapshot(), orc.snapshot())


@pytest.mark.parametrize("ablations", [(), ("live_degree",), ("force_bitmap",)])
@pytest.mark.parametrize("graphs", [1, 3])
def test_shared_tier1_repairs_to_proper(graphs, ablations):
    """Parallel Tier-1: random colours uploaded over every row, graphs straddling a wavefront's four rows."""
    gs = [_graph(5 + k) for k in range(graphs)]
    rng = np.random.default_rng(3)
    words = [((1 << 16) | rng.integers(0, 4, g.n)).astype(np.uint32) for g in gs]
    if graphs == 1:
        eng = S.GPUPartition(gs[0], S.StreamGCConfig(repair_every_epoch=True, exact_histogram=True,
                                                     ablations=ablations))
        eng.set_tuning(sweep_blocks=1, serial_repair=0)
        eng.set_words(words[0])
        st = eng.finish()
        assert st["t2_remaining"] == 0
        assert eng.validate() == (0, 0, st["max_color"])
        # again from a settled state: selection from the exact neighbour colours
        eng.process_stream(S.generate_bench_stream_edges(gs[0], 900, 50, 2))
        assert eng.finish()["t2_remaining"] == 0
        assert eng.validate()[:2] == (0, 0)
    else:
        pool = S.GraphPool(max_graphs=4, repair_every_epoch=True, exact_histogram=True)
        pool.set_tuning(sweep_blocks=1, serial_repair=0)
        gids = [pool.add(g) for g in gs]
        for gid, w in zip(gids, words):
            pool.set_words(gid, w)
        assert all(s["t2_remaining"] == 0 for s in pool.finish())
        assert all(pool.validate(gid)[:2] == (0, 0) for gid in gids)


def test_shared_tier1_counts_what_single_rows_count():
    """A proper colouring has no conflict and a clash between two leaves one loser, however the rows are split."""
    g = _graph()
    orc = O.Engine(O.Csr(g.n, g.row_ptr, g.col_idx, g.degree), O.default_config())
    init = S.generate_init_stream(g)
    orc.submit(init["u"], init["v"], init["type"])
    orc.finish()
    words = orc.words()
    u, v = g.edges()
    long = [int(x) for x in range(900, g.n)]
    for blocks in (1, 2048):
        for w in long[::5]:
            k = int(np.nonzero(v == w)[0][0])
            clash = words.copy()
            clash[u[k]] = clash[v[k]]           # the leaf takes its neighbour's colour
            near = set(g.col_idx[g.row_ptr[u[k]]:g.row_ptr[u[k] + 1]].tolist())
            same = [x for x in near if (words[x] & 0xFFFF) == (words[v[k]] & 0xFFFF)]
            eng = S.GPUPartition(g, S.StreamGCConfig(repair_every_epoch=True, max_repair_iters=1))
            eng.set_tuning(sweep_blocks=blocks)
            eng.set_words(words)
            assert eng.finish()["t1_conflicts_last"] == 0
            eng.set_words(clash)
            assert 1 <= eng.finish()["t1_conflicts_last"] <= len(same) + 1
            assert eng.validate()[:2] == (0, 0)
