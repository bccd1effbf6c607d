"""Epoch steps whose graphs do not all sweep next alike: their worklists are not built ahead.

An epoch's first worklist comes with that of the sweep after the drain where
every graph starts with the same one.  Here one graph was repaired before and
another was not, or one has no Tier-1 sweeps at all; every colouring published
must be proper, and stay so while the mix changes.
"""
import numpy as np
import pytest

import streamgc_amd as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("iters", [(20, 20), (20, 0), (0, 0)])
@pytest.mark.parametrize("captured", [False, True])
def test_settled_and_new_graphs_in_one_step(captured, iters):
    rng = np.random.default_rng(2)
    pool = S.GraphPool(max_graphs=4, repair_every_epoch=True, exact_histogram=True)
    graphs, gids = [], []
    for k in range(4):
        g = S.gen_rmat(9 + k % 2, 12.0, seed=k) if k % 2 else S.gen_delaunay(700 + 31 * k, seed=k)
        graphs.append(g)
        gids.append(pool.add(g, S.StreamGCConfig(epoch_size=200, batch_size=200, max_repair_iters=iters[k % 2])))
        # random colours: conflicts in every new graph; those before it are settled
        pool.set_words(gids[k], ((1 << 16) | rng.integers(1, 9, g.n)).astype(np.uint32))
        parts = [S.tag_graph(S.generate_bench_stream_edges(h, 200, 50, 10 * k + j), gids[j])
                 for j, h in enumerate(graphs)]
        if captured and k % 2:
            pool.batch_prepare(np.concatenate(parts))
            pool.batch_run()
            pool.batch_release()
        else:
            pool.submit(np.concatenate(parts))
        for gid in gids:
            assert pool.validate(gid)[:2] == (0, 0), (k, gid)
            assert np.array_equal(pool.snapshot(gid), pool.colors(gid)), (k, gid)
