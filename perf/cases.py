"""Performance cases of the streaming-colouring engine, through its public Python entry points.

A case is one user-visible call sequence on graphs that are resident on the
GPU already: an update stream applied and published, the captured rounds of a
prepared stream, a mix of many graphs, the request loop, a restored colouring.

Every graph starts from a proper first-fit colouring (made here, uploaded as a
checkpoint would be), so that a pass is the work of a stream on a coloured
graph and not the colouring of an empty one.  A state alternates between a
stream and the same stream undone (reversed, inserts and deletes swapped), so
that each pass finds the graph the first one found and does the same work.
"""
import functools
import random

import numpy as np
import torch

import streamgc_amd as S

# com-LiveJournal's shape; the largest single graph of the benchmark's plain workloads.
LIVEJOURNAL = (3997962, 34681189, 15000.0)


def listed():
    return [
        # A tenant that sends a few updates at a time and reads the colours of the vertices it touched:
        # launches, copies and waits are all there is.
        dict(name="calls_tenant", kind="stream", graph="delaunay", n=5003, updates=61, epochs=1, source="host",
             read="query"),
        # A planar mesh of 2^17 points with full-size epochs from host buffers, as the command line sends them.
        dict(name="churn_mesh", kind="stream", graph="delaunay", n=131072, updates=32768, epochs=1, source="host",
             read="snapshot"),
        # A social graph at full size: one epoch of a stream that lies in HBM, then the touched vertices' colours.
        dict(name="churn_social", kind="stream", graph="chung_lu", n=LIVEJOURNAL[0], m=LIVEJOURNAL[1],
             max_degree=LIVEJOURNAL[2], updates=32768, epochs=1, source="device", read="query"),
        # A skewed graph with small, odd epochs: several epoch steps to a call.
        dict(name="churn_skewed", kind="stream", graph="rmat", scale=16, edge_factor=24.0, updates=4099, epochs=3,
             source="host", read="snapshot"),
        # The reference's epoch order: snapshots without repair, then the end-of-stream drain and repair.
        dict(name="reference_order", kind="stream", graph="chung_lu", n=262139, m=2097143, max_degree=3000.0,
             updates=8191, epochs=5, source="host", read="snapshot", order="reference"),
        # Dense growth inside the k-core: two inserts to a delete, so conflicts, recolours and repair sweeps.
        dict(name="growth_core", kind="stream", graph="rmat", scale=18, edge_factor=24.0, updates=32768, epochs=2,
             source="device", read="snapshot", stream="growth"),
        # The social graph's stream as prepared, captured rounds: the plain workloads' headline figure.
        dict(name="rounds_social", kind="rounds", graph="chung_lu", n=LIVEJOURNAL[0], m=LIVEJOURNAL[1],
             max_degree=LIVEJOURNAL[2], updates=16384, epochs=2, read="query"),
        # Many graphs of mixed sizes in one pool, their streams as captured rounds (the batched pattern).
        dict(name="rounds_pool", kind="pool_rounds", graphs=64, low=10, high=15, updates=4096, epochs=2),
        # A checkpointed colouring uploaded to the social graph: every sweep visits every row once.
        dict(name="restore_social", kind="restore", graph="chung_lu", n=LIVEJOURNAL[0], m=LIVEJOURNAL[1],
             max_degree=LIVEJOURNAL[2]),
        # Audit replay of one graph: deterministic mode, updates in stream order.
        dict(name="replay_one", kind="stream", graph="delaunay", n=16384, updates=509, epochs=1, source="host",
             read="snapshot", deterministic=True),
        # Audit replay of a pool: each graph's updates in stream order, the graphs in parallel.
        dict(name="replay_pool", kind="pool", graphs=48, low=10, high=14, updates=1021, epochs=2, deterministic=True),
        # The request loop: requests of many tenants, then a flush that publishes them all.
        dict(name="served", kind="served", graphs=32, low=10, high=14, updates=4096, epochs=2, requests=5),
    ]


def _log_int(rng, low, high):
    return int(round(low * (high / low) ** rng.random()))


def _draw_graph(rng, low, high):
    """A graph of the shapes above with low..high vertices."""
    shape = rng.choice(("delaunay", "chung_lu", "rmat"))
    if shape == "rmat":
        return dict(graph="rmat", scale=rng.randint(low.bit_length(), high.bit_length() - 1),
                    edge_factor=round(rng.uniform(8, 32), 1))
    n = _log_int(rng, low, high)
    if shape == "delaunay":
        return dict(graph="delaunay", n=min(n, 262144))
    return dict(graph="chung_lu", n=n, m=int(n * rng.uniform(6, 9)), max_degree=float(round(6 * n ** 0.5)))


def _draw_updates(rng, low, g):
    """Updates an epoch: up to a full one on a mesh, up to an update to 64 vertices on the graphs with hubs."""
    n = g.get("n") or 1 << g["scale"]
    return _log_int(rng, low, min(32768, max(n // (4 if g["graph"] == "delaunay" else 64), 2 * low)))


def draw(rng):
    kind = rng.choice(("stream", "stream", "stream", "rounds", "pool_rounds", "restore", "replay", "pool", "served"))
    if kind == "stream":
        g = _draw_graph(rng, 4096, 1500000)
        return dict(kind="stream", **g, updates=_draw_updates(rng, 16, g), epochs=rng.randint(1, 2),
                    source=rng.choice(("host", "device")), read=rng.choice(("query", "snapshot")))
    if kind == "rounds":
        g = _draw_graph(rng, 65536, 1500000)
        return dict(kind="rounds", **g, updates=_draw_updates(rng, 1024, g), epochs=rng.randint(1, 3), read="query")
    if kind == "restore":
        return dict(kind="restore", **_draw_graph(rng, 65536, 1500000))
    if kind == "replay":
        return dict(kind="stream", **_draw_graph(rng, 2048, 65536), updates=_log_int(rng, 32, 768), epochs=1,
                    source="host", read="snapshot", deterministic=True)
    low = rng.randint(10, 11)
    if kind == "pool":
        return dict(kind="pool", graphs=_log_int(rng, 6, 48), low=low, high=low + 3, updates=_log_int(rng, 64, 1024),
                    epochs=rng.randint(1, 2), deterministic=True)
    case = dict(kind=kind, graphs=_log_int(rng, 32, 64), low=low, high=low + 3, updates=_log_int(rng, 3072, 4096),
                epochs=rng.randint(1, 2))
    if kind == "served":
        case["requests"] = rng.randint(1, 6)
    return case


# ---------------------------------------------------------------- graphs, colourings, streams
@functools.lru_cache(maxsize=None)
def _one_graph(shape, n, m, max_degree, scale, edge_factor, seed):
    if shape == "delaunay":
        return S.gen_delaunay(n, seed=seed)
    if shape == "rmat":
        return S.gen_rmat(scale, edge_factor, seed=seed)
    return S.gen_chung_lu(n, m, 2.3, max_degree, seed=seed, permute=True)


def _graph(case):
    return _one_graph(case["graph"], case.get("n"), case.get("m"), case.get("max_degree"), case.get("scale"),
                      case.get("edge_factor"), 42)


def _graphs(case):
    """The graphs of a pool: Delaunay and R-MAT in turn, sizes spread over 2^low..2^high vertices."""
    rng = random.Random(42)
    out = []
    for i in range(case["graphs"]):
        if i % 2 == 0:
            n = _log_int(rng, 1 << case["low"], 1 << case["high"])
            out.append(_one_graph("delaunay", n, None, None, None, None, 42 + i))
        else:
            out.append(_one_graph("rmat", None, None, None, rng.randint(case["low"], case["high"]),
                                  float(rng.randint(8, 24)), 42 + i))
    return out


def _colour(graphs, seed):
    """The packed words (version 1) of a first-fit colouring of each graph, ties broken by the seed: each round, every
    uncoloured vertex takes the lowest colour no coloured neighbour holds, and of two neighbours with the same choice
    the one of the lower degree waits."""
    dev = torch.device("cuda")
    starts = np.cumsum([0] + [g.n for g in graphs])
    n = int(starts[-1])
    deg = torch.from_numpy(np.concatenate([np.diff(g.row_ptr.astype(np.int64)) for g in graphs])).to(dev)
    b = torch.cat([torch.from_numpy(g.col_idx.view(np.int32)).to(dev).long() + int(s) for g, s in zip(graphs, starts)])
    a = torch.repeat_interleave(torch.arange(n, device=dev), deg)
    order = torch.from_numpy(np.random.default_rng(seed).permutation(n)).to(dev)
    rank = deg * n + order
    colour = torch.where(deg == 0, 1, 0)
    width = 1 << 16
    while a.numel():
        held = colour[b]
        pairs = torch.unique(a[held > 0] * width + held[held > 0])   # (vertex, neighbour colour), sorted
        v = pairs // width
        place = torch.arange(pairs.numel(), device=dev) - torch.searchsorted(v, v) + 1
        gap = pairs % width != place                                 # the first place without its colour
        pick = torch.bincount(v, minlength=n) + 1
        pick = pick.scatter_reduce(0, v[gap], place[gap], "amin")
        wait = torch.zeros(n, dtype=torch.bool, device=dev)
        wait[a[(held == 0) & (pick[a] == pick[b]) & (rank[a] < rank[b])]] = True
        colour = torch.where((colour == 0) & ~wait, pick, colour)
        keep = colour[a] == 0
        a, b = a[keep], b[keep]
    words = (colour.cpu().numpy() | 1 << 16).astype(np.uint32)
    return [words[s:e] for s, e in zip(starts, starts[1:])]


@functools.lru_cache(maxsize=None)
def _edges(g):
    return g.edges()


@functools.lru_cache(maxsize=None)
def _core(g):
    return S.core_numbers(g)


def _churn(g, size, rng, insert_pct=50):
    """A churn stream: deletes of random edges, inserts of edges deleted before (the mix of the churn generator,
    without its pass over the whole graph)."""
    eu, ev = _edges(g)
    at, kind, gone, absent = [], [], [], set()
    while len(at) < size:
        if gone and rng.random() * 100 < insert_pct:
            k = rng.randrange(len(gone))
            e = gone[k]
            gone[k] = gone[-1]
            gone.pop()
            absent.discard(e)
            kind.append(S.UPDATE_ADD)
        else:
            e = rng.randrange(len(eu))
            if e in absent:
                continue
            absent.add(e)
            gone.append(e)
            kind.append(S.UPDATE_DEL)
        at.append(e)
    return S.make_updates(eu[at], ev[at], np.array(kind, np.uint8))


def _stream(case, g, size, rng):
    if case.get("stream") == "growth":
        return S.dense_growth_stream(g, size, seed=rng.randrange(1 << 30), core=_core(g))
    return _churn(g, size, rng)


def _undone(records):
    back = records[::-1].copy()
    back["type"] = 1 - back["type"]
    return back


def _touched(records):
    return np.concatenate([records["u"], records["v"]])


# ---------------------------------------------------------------- one case
def _config(case):
    return S.StreamGCConfig(epoch_size=case.get("updates", 32768), batch_size=case.get("updates", 32768),
                            exact_histogram=True, deterministic=case.get("deterministic", False),
                            repair_every_epoch=case.get("order") != "reference")


def _engine(case, seed):
    g = _graph(case)
    eng = S.GPUPartition(g, _config(case))
    eng.set_words(_colour([g], seed)[0])
    eng.finish()
    return g, eng


def _pool(case, seed, rng):
    """A pool of coloured graphs and each one's stream (odd lengths: up to `epochs` of its epochs)."""
    graphs = _graphs(case)
    size = case["updates"]
    pool = S.GraphPool(max_graphs=len(graphs), batch_capacity=1 << 18, deterministic=case.get("deterministic", False),
                       repair_every_epoch=True, exact_histogram=True)
    streams = []
    for g, words in zip(graphs, _colour(graphs, seed)):
        gid = pool.add(g, S.StreamGCConfig(epoch_size=size, batch_size=size))
        pool.set_words(gid, words)
        length = rng.randint(max(size * case["epochs"] // 2, 1), size * case["epochs"])
        streams.append(S.tag_graph(_churn(g, length, rng, rng.randint(40, 60)), gid))
    pool.finish()
    return pool, streams


def _snapshots(pool):
    return np.concatenate([pool.snapshot(gid) for gid in sorted(pool.graphs)])


def prepare(case, seed):
    rng = random.Random(seed)
    kind, state = case["kind"], dict(case=case, turn=0)
    if kind in ("stream", "rounds"):
        g, state["engine"] = _engine(case, seed)
        records = _stream(case, g, case["updates"] * case["epochs"], rng)
        state["ids"] = _touched(records)
        both = [records, _undone(records)]
        if kind == "rounds":   # the plan holds the stream and its undoing: every run starts from the same edges
            state["engine"].batch_prepare(np.concatenate(both))
        elif case["source"] == "device":
            state["streams"] = [S.DeviceStream(r) for r in both]
        else:
            state["streams"] = both
    elif kind == "restore":
        g, state["engine"] = _engine(case, seed + 1)
        state["words"] = _colour([g], seed)[0]   # the checkpoint: another colouring of the same edges
    else:
        state["pool"], streams = _pool(case, seed, rng)
        if kind == "pool_rounds":
            mixed = [np.concatenate([s, _undone(s)]) for s in streams]
            state["pool"].batch_prepare(np.concatenate(mixed))
        elif kind == "pool":
            state["streams"] = [np.concatenate(streams), np.concatenate([_undone(s) for s in streams])]
        else:
            state["server"] = S.GraphServer(state["pool"], max_batch=65536)
            for gid in sorted(state["pool"].graphs):
                state["server"].attach(gid, case["updates"])
            state["requests"] = []
            for way in (streams, [_undone(s) for s in streams]):
                parts = [(gid, part) for gid, s in enumerate(way) for part in np.array_split(s, case["requests"])]
                # arrival order: the tenants' requests interleaved, each tenant's own in order
                order = [gid for gid, _ in parts]
                rng.shuffle(order)
                queue = {gid: [p for h, p in parts if h == gid] for gid in set(order)}
                state["requests"].append([(gid, queue[gid].pop(0)) for gid in order])
    return state


def run(state):
    case = state["case"]
    kind, turn = case["kind"], state["turn"]
    if kind == "stream":
        state["turn"] = 1 - turn
        eng, records = state["engine"], state["streams"][turn]
        if case["source"] == "device":
            eng.submit_device(records.ptr, records.count)
        else:
            eng.process_stream(records)
        if case.get("order") == "reference":
            eng.finish()
        return eng.query(state["ids"]) if case["read"] == "query" else eng.snapshot()
    if kind == "rounds":
        state["engine"].batch_run()
        return state["engine"].query(state["ids"])
    if kind == "restore":
        state["engine"].set_words(state["words"])
        state["engine"].finish()
        return state["engine"].snapshot()
    if kind == "pool_rounds":
        state["pool"].batch_run()
        return _snapshots(state["pool"])
    state["turn"] = 1 - turn
    if kind == "pool":
        state["pool"].submit(state["streams"][turn])
        state["pool"].finish()
        return _snapshots(state["pool"])
    for gid, records in state["requests"][turn]:
        state["server"].submit(gid, records)
    state["server"].flush()
    return _snapshots(state["pool"])


def work(case):
    """Bytes a pass cannot do without: per update its record, its two slots read and written, its endpoints' words
    and bitmaps read; per epoch each vertex's word read and its colour published; the colours handed out."""
    kind = case["kind"]
    if kind in ("stream", "rounds", "restore"):
        n = case.get("n") or 1 << case["scale"]
        edges = case.get("m") or (3 * n if case["graph"] == "delaunay" else int(n * case["edge_factor"]))
        if kind == "restore":   # every row's slots and its neighbours' words; words in, bitmaps and colours out
            return {"bytes": 16.0 * edges + (4 + 4 + 8 + 2 + 2) * n, "flops": 0.0}
        updates, epochs = case["updates"] * case["epochs"], case["epochs"]
        if kind == "rounds":
            updates, epochs = 2 * updates, 2 * epochs
        out = 12 * updates if case.get("read") == "query" else 2 * n
    else:
        n = case["graphs"] * ((1 << case["low"]) + (1 << case["high"])) // 2
        updates = case["graphs"] * case["updates"] * case["epochs"] * 3 // 4
        epochs = case["epochs"]
        if kind == "pool_rounds":
            updates, epochs = 2 * updates, 2 * epochs
        out = 2 * n
    return {"bytes": float(updates * (16 + 2 * (4 + 4 + 4 + 8)) + epochs * 6 * n + out), "flops": 0.0}


def exact(case, seed):
    """Colours are whole numbers and a stream's are the outcome of its engine's order; only a restored colouring is
    known without running it."""
    if case["kind"] != "restore":
        return None
    return (_colour([_graph(case)], seed)[0] & 0xFFFF).astype(np.uint16)
