"""Full sweeps on a grid with a wavefront for every row, and on one without."""
import numpy as np
import pytest

import streamgc_amd as S
from test_gpu_parity import _pair, _same_state
from test_gpu_sweeps import _graph

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("blocks", [None, 3])
@pytest.mark.parametrize("slack", [30, 300])
def test_full_sweeps_bit_exact(slack, blocks):
    g = _graph(11)
    gpu, orc, og = _pair(g, deterministic=True, epoch_size=300, batch_size=300, repair_every_epoch=True,
                         exact_histogram=True, slack_pct=slack, full_sweeps=True)
    if blocks:
        gpu.set_tuning(apply_blocks=blocks)
    init = S.generate_init_stream(g)
    assert gpu.process_stream(init) == orc.submit(init["u"], init["v"], init["type"])
    churn = S.generate_bench_stream_edges(g, 1500, 40, 9)
    assert gpu.process_stream(churn) == orc.submit(churn["u"], churn["v"], churn["type"])
    _same_state(gpu, orc, "churn")
    assert gpu.finish() == orc.finish()


@pytest.mark.parametrize("blocks", [None, 3])
@pytest.mark.parametrize("graphs", [1, 3])
def test_full_parallel_repair_to_proper(graphs, blocks):
    gs = [_graph(11 + k) for k in range(graphs)]
    rng = np.random.default_rng(4)
    pool = S.GraphPool(max_graphs=4, repair_every_epoch=True, exact_histogram=True, full_sweeps=True)
    pool.set_tuning(serial_repair=0, **({"apply_blocks": blocks} if blocks else {}))
    gids = [pool.add(g) for g in gs]
    for gid, g in zip(gids, gs):
        pool.set_words(gid, ((1 << 16) | rng.integers(0, 4, g.n)).astype(np.uint32))
    assert all(s["t2_remaining"] == 0 for s in pool.finish())
    assert all(pool.validate(gid)[:2] == (0, 0) for gid in gids)
    assert pool.totals()["rows_compact"] == sum(g.n for g in gs)   # every row once
