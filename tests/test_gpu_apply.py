"""The per-update kernel's two row scans: four light edges to a wavefront, and
long rows in trips of 1,024 slots.

Edges of one launch run in any order, so the launches here hold pairwise
disjoint edges: every row's outcome is then the oracle's, slot for slot.
"""
import numpy as np
import pytest

import streamgc_amd as S
from test_gpu_parity import _pair, _same_state

pytestmark = pytest.mark.gpu

LENGTHS = [1, 2, 3, 7, 8, 9, 15, 16, 17, 63, 64, 65, 126, 127, 128, 129, 130, 255, 256, 257, 511, 900]
LONG = [511, 512, 513, 514, 1023, 1024, 1025, 1026, 1535, 1537, 2047, 2049, 2050, 3001]
PAIRS = 5200   # more light edges than the launch spreads one to a wavefront


def _light_graph():
    """PAIRS edges (2i, 2i + 1), and vertices of the lengths above over the first 1,000 of their endpoints."""
    edges = [(2 * i, 2 * i + 1) for i in range(PAIRS)]
    rng, at = np.random.default_rng(3), 2 * PAIRS
    for d in LENGTHS:
        edges += [(at, int(x)) for x in rng.choice(1000, size=d, replace=False)]
        at += 1
    return S.csr_from_edges(at, edges)


def _live(rows, x):
    return [int(w) for w in rows[1][rows[0][x]:rows[0][x + 1]] if w != 0xFFFFFFFF]


@pytest.mark.parametrize("slack,cap", [(300, 0), (0, 1), (50, 2)])
@pytest.mark.parametrize("graphs", [1, 3])
def test_light_edges_keep_the_oracles_slots(graphs, slack, cap):
    g = _light_graph()
    cfg = dict(epoch_size=1 << 20, batch_size=1 << 20, slack_pct=slack, min_row_capacity=max(cap, 1),
               overflow_capacity=1 << 16)
    gpu, orc, og = _pair(g, **cfg)
    pool = None
    if graphs > 1:   # the same graph several times: a wavefront's edges straddle graphs
        pool = S.GraphPool(max_graphs=graphs, batch_capacity=1 << 18)
        gids = [pool.add(g, S.StreamGCConfig(**cfg)) for _ in range(graphs)]
    rng = np.random.default_rng(slack + cap)
    done = 0
    for launch in range(3):
        rows = orc.csr()
        used, groups = set(), []
        for x in range(2 * PAIRS, g.n):          # one edge of each longer row, at its start, middle or end
            row = [w for w in _live(rows, x) if w not in used]
            if row:
                w = row[(0, len(row) // 2, len(row) - 1)[(x + launch) % 3]]
                used |= {x, w}
                kind = x % 4
                groups.append([[(x, w, 1)], [(x, w, 1), (x, w, 0)], [(x, w, 1), (w, x, 0)],
                               [(x, w, 1), (x, w, 0), (x, w, 1)]][kind])
        for i in range(PAIRS):
            u, v = 2 * i, 2 * i + 1
            if u in used or v in used:
                continue
            live = v in _live(rows, u)
            kind = int(rng.integers(8))
            if kind == 7 and i + 1 < PAIRS and not {u + 2, v + 2} & used:   # an edge the rows have no room kept for
                groups.append([(u, v + 2, 0)])
                used |= {u, v + 2}
                continue
            if kind == 0:      # longer than a packed line
                groups.append([(u, v, 1), (u, v, 0), (u, v, 1), (u, v, 0), (u, v, 1)])
            elif kind == 1:    # again a live edge: found, or a second copy behind a hole
                groups.append([(u, v, 0), (v, u, 0)])
            elif kind == 2:    # a delete that finds nothing
                groups.append([(u, v, 1), (u, v, 1)])
            elif live:
                groups.append([(u, v, 1)] if kind < 5 else [(u, v, 1), (u, v, 0)])
            else:
                groups.append([(v, u, 0)] if kind < 5 else [(u, v, 0), (u, v, 1)])
            used |= {u, v}
        owner = np.concatenate([np.full(len(q), k) for k, q in enumerate(groups)])
        rng.shuffle(owner)
        at, recs = [0] * len(groups), []
        for k in owner.tolist():
            recs.append(groups[k][at[k]])
            at[k] += 1
        batch = S.make_updates(*(list(c) for c in zip(*recs)))
        orc.submit(batch["u"], batch["v"], batch["type"])
        done += len(batch)
        want = orc.csr()
        if pool is None:
            gpu.apply(batch)
            got = gpu.csr()
            assert np.array_equal(got[0], want[0])
            assert np.array_equal(got[1], want[1]), (launch, np.nonzero(got[1] != want[1])[0][:8])
            assert gpu.overflow_count() == orc.overflow_count()
            assert gpu.totals()["updates"] == done
        else:
            parts = [S.tag_graph(batch, gid) for gid in gids]
            pool.apply(np.stack(parts, axis=1).reshape(-1))   # the graphs' records in turn
            for gid in gids:
                got = pool.csr(gid)
                assert np.array_equal(got[1], want[1]), (launch, gid, np.nonzero(got[1] != want[1])[0][:8])
    if cap == 1:
        assert orc.overflow_count() > 0


@pytest.mark.parametrize("deterministic", [True, False])
def test_long_rows_keep_the_oracles_slots(deterministic):
    """Searches that end before, at and past the edges of a trip, from odd and even first slots."""
    bed = 4000
    rng = np.random.default_rng(8)
    edges = [(bed + k, int(x)) for k, d in enumerate(LONG) for x in rng.choice(bed, size=d, replace=False)]
    g = S.csr_from_edges(bed + len(LONG), edges)
    gpu, orc, og = _pair(g, deterministic=deterministic, epoch_size=1 << 20, batch_size=1 << 20, slack_pct=3)
    for k in range(6):
        # one update of each long row per launch: a delete, its re-insert, an insert past a packed row, ...
        rows, used, recs = orc.csr(), set(), []
        for x in range(bed, g.n):
            row = [w for w in _live(rows, x) if w not in used]
            out = [w for w in range(bed) if w not in used and w not in set(_live(rows, x))]
            w = row[(0, len(row) // 2, len(row) - 1)[(x + k) % 3]]
            recs.append([(x, w, 1), (w, x, 1), (x, out[x % 5], 0), (x, w, 0), (out[0], x, 0), (x, w, 1)][k])
            used |= {recs[-1][0], recs[-1][1]}
        batch = S.make_updates(*(list(c) for c in zip(*recs)))
        gpu.apply(batch)
        orc.submit(batch["u"], batch["v"], batch["type"])
        got, want = gpu.csr(), orc.csr()
        assert np.array_equal(got[0], want[0])
        assert np.array_equal(got[1], want[1]), (k, np.nonzero(got[1] != want[1])[0][:8])
    assert gpu.overflow_count() == orc.overflow_count()
    if deterministic:
        _same_state(gpu, orc, "long rows")
