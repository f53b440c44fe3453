"""Native batched Leiden (ckv_batched_leiden, ckv_aggregate_coo,
ckv_densify_*) against the oracle's restatement of the reference
(oracle/leiden.py).  Dyadic edge weights make every float sum exact, so labels
must match bit for bit; with arbitrary float weights the sums are formed in
another order and the labels are still expected to match (a flip needs two
gains within an ulp)."""

from __future__ import annotations

import time

import numpy as np
import pytest
import torch

from community_kv_amd.graph.leiden import algorithm
from oracle import leiden as L
from tests import _leiden_graphs as lg

pytestmark = pytest.mark.gpu


def _dev(device, *arrays):
    return [torch.from_numpy(np.ascontiguousarray(a)).to(device) for a in arrays]


def _native_level(device, src, dst, w, G, S, **kw):
    s, d, x = _dev(device, src, dst, w)
    mod = algorithm._load_module()
    labels, q = mod.batched_leiden(s, d, x, G, S, 6, kw.get("resolution", 1.0), kw.get("theta", 0.01),
                                   kw.get("max_inner_iter", 16), kw.get("seed", 0), kw.get("use_boltzmann", False))
    torch.cuda.synchronize()
    return labels.cpu().numpy(), q.cpu().numpy()


LEVEL_CASES = [
    # seed, graphs, seq_len, communities, kwargs for planted(), kwargs for Leiden
    (1, 3, 500, 8, dict(), dict()),
    (2, 2, 800, 12, dict(self_loops=6, isolated=7, duplicates=20), dict(max_inner_iter=4)),
    (3, 4, 300, 5, dict(edges_per_vertex=10.0), dict(resolution=0.5, seed=7)),
    (4, 1, 2000, 30, dict(p_in=0.6), dict(resolution=2.0, max_inner_iter=1)),
    (5, 2, 600, 10, dict(dyadic=False), dict()),
    (6, 3, 400, 6, dict(dyadic=False, self_loops=3), dict(resolution=1.5, seed=3)),
]


@pytest.mark.parametrize("seed,G,S,k,gkw,lkw", LEVEL_CASES)
def test_batched_leiden_level_matches_oracle(device, seed, G, S, k, gkw, lkw):
    print(f"leiden level seed={seed} G={G} S={S} {gkw} {lkw}", flush=True)
    src, dst, w = lg.planted(seed, G, S, k, **gkw)
    got, q = _native_level(device, src, dst, w, G, S, **lkw)
    ref, q_ref = L.batched_leiden(src, dst, w, graphs=G, seq_len=S, **lkw)
    np.testing.assert_array_equal(got, ref)
    np.testing.assert_allclose(q, q_ref, rtol=1e-9, atol=1e-12)


@pytest.mark.parametrize("leaves", [3000, 1500, 1100, 300, 100])
def test_hub_vertex_over_table_capacity(device, leaves):
    """Degree 3000, 1500 and 1100 (workgroup kernel: the row is walked 1024
    entries at a time and the first 1024 communities along it are kept), 300
    (hub kernel, hashed table) and 100 (small-row kernel).  The workgroup
    table never overflows; if it did, the call would mark its modularity NaN
    (checked finite here) and run_leiden would raise."""
    src, dst, w, S = lg.hub(4, leaves, 40)
    print(f"leiden hub S={S} edges={src.size}", flush=True)
    got, q = _native_level(device, src, dst, w, 1, S)
    ref, _ = L.batched_leiden(src, dst, w, graphs=1, seq_len=S)
    np.testing.assert_array_equal(got, ref)
    assert np.isfinite(q).all()


def test_boltzmann_refinement_close_to_oracle(device):
    """Gumbel noise goes through logf: the device and numpy logarithms may
    differ in the last ulp, which can move a near-tied sample."""
    src, dst, w = lg.planted(8, 2, 700, 9)
    print("leiden boltzmann", flush=True)
    got, q = _native_level(device, src, dst, w, 2, 700, use_boltzmann=True, theta=0.05, seed=5)
    ref, q_ref = L.batched_leiden(src, dst, w, graphs=2, seq_len=700, use_boltzmann=True, theta=0.05, seed=5)
    assert (got == ref).mean() > 0.98
    np.testing.assert_allclose(q, q_ref, atol=5e-3)


def test_no_edges_marks_every_vertex_isolated(device):
    e = np.zeros(0, np.int32)
    got, q = _native_level(device, e, e, np.zeros(0, np.float32), 2, 5)
    assert (got == -1).all() and (q == 0).all()


def test_aggregate_coo_matches_oracle(device):
    src, dst, w = lg.planted(12, 3, 400, 7, self_loops=5)
    lab, _ = L.batched_leiden(src, dst, w, graphs=3, seq_len=400)
    lab = np.where(lab < 0, np.arange(1200), lab).astype(np.int32)
    dense, width = L.densify_per_graph(lab, 3, 400)
    print(f"aggregate width={width}", flush=True)
    s, d, x, dl = _dev(device, src, dst, w, dense)
    out = algorithm._load_module().aggregate_coo(s, d, x, dl, 3 * width)
    ref = L.aggregate_coo(src, dst, w, dense, 3 * width)
    for a, b in zip(out[:2], ref[:2]):
        np.testing.assert_array_equal(a.cpu().numpy(), b)
    np.testing.assert_array_equal(out[2].cpu().numpy(), ref[2])  # dyadic: exact sums


def test_densify_matches_oracle(device):
    rng = np.random.default_rng(3)
    G, S = 4, 777
    lab = (rng.integers(0, 50, (G, S)) * 7 % S + np.arange(G)[:, None] * S).astype(np.int32).ravel()
    lab[rng.random(lab.size) < 0.05] = -1
    print("densify", flush=True)
    dense, width = algorithm._densify_per_graph(torch.from_numpy(lab).to(device), G, S)
    own = np.where(lab < 0, np.arange(G * S), lab)
    ref, ref_w = L.densify_per_graph(own, G, S)
    assert width == ref_w
    np.testing.assert_array_equal(dense.cpu().numpy(), ref)


@pytest.mark.parametrize("dyadic", [True, False])
def test_run_leiden_multilevel_matches_oracle(device, dyadic):
    src, dst, w = lg.planted(31, 3, 1500, 40, edges_per_vertex=6.0, dyadic=dyadic, isolated=9)
    print(f"run_leiden multilevel dyadic={dyadic}", flush=True)
    s, d, x = _dev(device, src, dst, w)
    vertex, part, q = algorithm.run_leiden(s, d, x, G=3, seq_len=1500, max_inner_iter=8, seed=2)
    rv, rp, rq = L.run_leiden(src, dst, w, graphs=3, seq_len=1500, max_inner_iter=8, seed=2)
    np.testing.assert_array_equal(vertex.cpu().numpy(), rv)
    np.testing.assert_array_equal(part.cpu().numpy(), rp)
    assert q == pytest.approx(rq, abs=1e-9)


def test_ring_of_cliques_end_to_end(device):
    src, dst, w, S = lg.ring_of_cliques(2, 6, 5, seq_len=34)
    s, d, x = _dev(device, src, dst, w)
    vertex, part, q = algorithm.run_leiden(s, d, x, G=2, seq_len=S)
    by_clique = part.cpu().numpy().reshape(2, 6, 5)
    assert (by_clique == by_clique[..., :1]).all() and np.unique(by_clique[..., 0]).size == 12


@pytest.mark.parametrize("aggregation", ["query_group", "per_query_head", "layer_wise"])
def test_partition_graphs_matches_oracle_pipeline(device, aggregation):
    """Top-k prefill edges -> build_adjacency -> Leiden -> dense community ids
    (partition.py:289-353), against the oracle's composition; then
    build_partitioned_layer (538-618) on the same edges: community count over
    all positions (sink singletons included) and the token table."""
    from community_kv_amd.graph import partition as P
    from oracle import ckv_oracle as co

    rng = np.random.default_rng(17)
    Hq, Hkv, S, sinks, kappa = 8, 2, 1200, 4, 8
    rows = S - sinks - kappa + 1
    comm = rng.integers(0, 25, S)
    idx = np.empty((Hq, rows, kappa), np.int32)
    for r in range(rows):
        p = sinks + kappa - 1 + r
        pool = np.nonzero(comm[sinks:p + 1] == comm[p])[0] + sinks
        pool = pool if pool.size >= kappa else np.arange(sinks, p + 1)
        for h in range(Hq):
            idx[h, r] = rng.choice(pool, kappa, replace=False)
    sc = (rng.integers(1, 32, idx.shape) / 32.0).astype(np.float32)
    print(f"partition_graphs pipeline {aggregation}", flush=True)
    ti, ts = torch.from_numpy(idx).to(device), torch.from_numpy(sc).to(device)
    res = P.partition_graphs(ti, ts, aggregation=aggregation, num_kv_heads=Hkv, prefill_seq_len=S, num_sink=sinks,
                             lam=0.5, leiden_resolution=1.0, leiden_seed=0)
    gi, gs, pos = P._reshape_by_aggregation(torch.from_numpy(idx), torch.from_numpy(sc), aggregation=aggregation,
                                            num_kv_heads=Hkv, num_sink=sinks)
    graphs = gi.shape[0]
    src, dst, w = co.build_adjacency(gi.numpy(), gs.numpy(), pos.numpy(), seq_len=S, lam=0.5)
    ids, q = L.partition_labels(src, dst, w, graphs=graphs, seq_len=S, resolution=1.0, max_inner_iter=3, seed=0)
    np.testing.assert_array_equal(res.community_ids.cpu().numpy(), ids)
    assert res.community_counts.cpu().tolist() == (ids.max(axis=1) + 1).tolist()
    assert res.modularity == pytest.approx(q, abs=1e-9)
    keys = torch.randn(Hkv, S, 128, generator=torch.Generator().manual_seed(2)).to(torch.bfloat16).to(device)
    layer = P.build_partitioned_layer(layer_idx=0, topk_indices=ti, topk_scores=ts, keys=keys, num_sink=sinks,
                                      lam=0.5, leiden_resolution=1.0, leiden_seed=0, max_decode_tokens=4,
                                      aggregation=aggregation)
    assert layer.community_counts.cpu().tolist() == (ids.max(axis=1) + 1).tolist()
    np.testing.assert_array_equal(layer.token_communities[:, :S].cpu().numpy(), ids)
    assert (layer.token_communities[:, S:] == -1).all()


def test_build_adjacency_known_answers(device):
    """The reference tests' coalescing / discard cases (test_partition.py:212-250) through ckv_build_adjacency."""
    import json
    import os

    from community_kv_amd.graph.partition import build_adjacency

    golden = json.load(open(os.path.join(os.path.dirname(__file__), "golden", "reference_known_answers.json")))
    for name in ("adjacency_coalesces", "adjacency_discards_outside"):
        ka = golden[name]
        src, dst, w = build_adjacency(torch.tensor(ka["indices"], dtype=torch.int32, device=device),
                                      torch.tensor(ka["scores"], dtype=torch.float32, device=device),
                                      torch.tensor(ka["query_positions"], dtype=torch.int64, device=device),
                                      seq_len=ka["seq_len"], lam=ka["lam"])
        got = sorted(zip(src.tolist(), dst.tolist(), w.tolist()))
        assert got == sorted(tuple(p) for p in ka["pairs"]), name


@pytest.mark.parametrize("lam,dyadic", [(0.5, True), (1.0, False), (0.0, True), (0.3, False)])
def test_build_adjacency_matches_oracle(device, lam, dyadic):
    from community_kv_amd.graph.partition import build_adjacency
    from oracle import ckv_oracle as co

    rng = np.random.default_rng(int(lam * 10) + dyadic)
    G, R, kappa, S = 3, 2000, 8, 1500
    idx = rng.integers(0, S, (G, R, kappa)).astype(np.int32)
    idx[rng.random(idx.shape) < 0.05] = -1
    idx[rng.random(idx.shape) < 0.02] = S + 5
    sc = (rng.integers(1, 32, idx.shape) / 32.0 if dyadic else rng.random(idx.shape)).astype(np.float32)
    pos = rng.integers(0, S, (G, R)).astype(np.int64)
    print(f"build_adjacency lam={lam} dyadic={dyadic}", flush=True)
    s, d, w = build_adjacency(*_dev(device, idx, sc, pos), seq_len=S, lam=lam)
    rs, rd, rw = co.build_adjacency(idx, sc, pos, seq_len=S, lam=lam)
    np.testing.assert_array_equal(s.cpu().numpy(), rs)
    np.testing.assert_array_equal(d.cpu().numpy(), rd)
    if dyadic:
        np.testing.assert_array_equal(w.cpu().numpy(), rw)
    else:
        np.testing.assert_allclose(w.cpu().numpy(), rw, rtol=2e-6)


@pytest.mark.parametrize("R,S", [(9000, 3000), (4000, 40000), (300, 900)])
def test_build_adjacency_weights_that_cancel(device, R, S):
    """Edges whose weights add up to zero, or are all zero of either sign, are
    edges all the same (raw scores may be negative), however they are gathered."""
    from community_kv_amd.graph.partition import build_adjacency
    from oracle import ckv_oracle as co

    rng = np.random.default_rng(R)
    idx = rng.integers(0, S, (1, R, 8)).astype(np.int32)
    idx[..., 0] = 5
    sc = (rng.integers(-2, 3, idx.shape) / 8.0).astype(np.float32)
    sc[rng.random(sc.shape) < 0.1] = -0.0
    sc[:, :, 0] = np.where(rng.random((1, R)) < 0.5, 0.0, 0.25)
    pos = rng.integers(0, S, (1, R)).astype(np.int64)
    print(f"build_adjacency cancelling weights R={R} S={S}", flush=True)
    got = build_adjacency(*_dev(device, idx, sc, pos), seq_len=S, lam=0.5)
    ref = co.build_adjacency(idx, sc, pos, seq_len=S, lam=0.5)
    for a, b in zip(got, ref):
        np.testing.assert_array_equal(a.cpu().numpy(), b)


def test_build_adjacency_heavy_column_keeps_pace(device):
    """A column that every row names costs little beside the same rows without
    it (one workgroup reading all rows for it: 7 times with one graph)."""
    from community_kv_amd.graph.partition import build_adjacency

    g = torch.Generator(device=device).manual_seed(3)
    heads, R, S = 32, 30000, 30000
    pos = torch.arange(R, device=device).repeat(heads).unsqueeze(0)
    idx = (pos.unsqueeze(-1) - torch.randint(0, 300, (1, heads * R, 8), device=device, generator=g)).clamp_min(0).int()
    sc = torch.rand(1, heads * R, 8, device=device, generator=g)
    heavy = idx.clone()
    heavy[..., 0] = 3

    def best_ms(columns):
        best = float("inf")
        for _ in range(5):
            t0 = time.perf_counter()
            build_adjacency(columns, sc, pos, seq_len=S, lam=0.5)
            torch.cuda.synchronize()
            best = min(best, (time.perf_counter() - t0) * 1e3)
        return best

    plain, with_it = best_ms(idx), best_ms(heavy)
    print(f"build_adjacency {plain:.2f} ms, with a heavy column {with_it:.2f} ms", flush=True)
    assert with_it < 2.5 * plain


def test_build_adjacency_direct_edges_scratch_and_pace(device):
    """Without co-occurrence edges (lam = 1) a graph has one edge per column: it
    needs no more scratch per edge at 64 columns a row than at 8, and building
    it takes no longer than with them (where postings that bring all columns
    stood for the one edge, 3.9 and 1.8 times)."""
    from community_kv_amd import _native
    from community_kv_amd.graph.partition import build_adjacency

    lib, rows = _native.lib(), 1 << 20
    per_edge = [lib.ckv_adjacency_workspace_bytes(1, rows, k, 1.0) / (rows * k) for k in (8, 64)]
    assert max(per_edge) < 64
    g = torch.Generator(device=device).manual_seed(3)
    G, R, kappa, S = 8, 30000, 16, 30000
    pos = torch.arange(R, device=device).expand(G, R)
    idx = (pos.unsqueeze(-1) - torch.randint(0, 300, (G, R, kappa), device=device, generator=g)).clamp_min(0).int()
    sc = torch.rand(G, R, kappa, device=device, generator=g)

    def best_ms(lam):
        best = float("inf")
        for _ in range(6):
            t0 = time.perf_counter()
            build_adjacency(idx, sc, pos, seq_len=S, lam=lam)
            torch.cuda.synchronize()
            best = min(best, (time.perf_counter() - t0) * 1e3)
        return best

    direct, both = best_ms(1.0), best_ms(0.5)
    print(f"build_adjacency lam 1 {direct:.2f} ms, lam 0.5 {both:.2f} ms", flush=True)
    assert direct < 1.1 * both


def test_run_leiden_rejects_edges_across_graphs(device):
    s, d, w = _dev(device, np.array([0, 3], np.int32), np.array([1, 5], np.int32), np.ones(2, np.float32))
    with pytest.raises(ValueError, match="same graph"):
        algorithm.run_leiden(s, d, w, G=2, seq_len=4)


def test_overflow_raised_during_local_moving_reaches_the_caller(device):
    """A table overflow flagged by the local-moving sweeps must survive the
    refinement's control reset and make run_leiden raise (the hook raises the
    device flag after local moving, as a broken table bound would)."""
    from community_kv_amd import _native

    src, dst, w = lg.planted(3, 2, 300, 6)
    s, d, x = _dev(device, src, dst, w)
    print("overflow flag after local moving", flush=True)
    lib = _native.lib()
    lib.ckv_leiden_test_raise_overflow(1)
    try:
        with pytest.raises(RuntimeError, match="overflowed"):
            algorithm.run_leiden(s, d, x, G=2, seq_len=300)
    finally:
        lib.ckv_leiden_test_raise_overflow(0)
    torch.cuda.synchronize()
    _vertex, _part, q = algorithm.run_leiden(s, d, x, G=2, seq_len=300)
    assert np.isfinite(q)


ADJACENCY_TIERS = [
    # graphs, rows, kappa, seq_len, hub columns and the share of rows that name them
    (2, 1500, 8, 900, 0, 0.0),       # short and long runs, fewer vertices than the workgroup table
    (1, 400, 16, 3000, 2, 0.2),      # the width with its own code; runs of 80 rows: the id bitmap orders them
    (1, 300, 5, 2000, 1, 1.0),       # any other width
    (2, 6000, 8, 5000, 2, 1.0),      # more neighbours than the table: one pass of ranked sums
    (1, 4000, 8, 40000, 1, 1.0),     # two passes
    (1, 2500, 8, 290000, 1, 1.0),    # three bitmaps of ids
    (1, 9000, 8, 3000, 2, 1.0),      # runs in parts
    (2, 9000, 8, 500, 1, 1.0),       # of a graph whose vertices all fit the table
    (1, 30000, 8, 70000, 1, 0.6),    # runs just long enough for a sum per id,
    (1, 30000, 8, 70000, 1, 0.45),   # and too short for that
    (1, 20000, 3, 9000, 2, 1.0),     # parts of a width without its own code
    (1, 700, 8, 140000, 1, 0.15),    # more vertices than the bitmap holds: ordered by counting
    (1, 57, 8, 300, 1, 1.0),         # a run one posting past the short ones
    (1, 1, 1, 1, 0, 0.0),            # the smallest graph: one vertex, one self loop
    (2, 3000, 1, 900, 0, 0.0),       # one column a row: entries sorted by pair, as all graphs at lam = 1
    (2, 3000, 2, 900, 1, 0.5),       # two: gathered
]


@pytest.mark.parametrize("G,R,kappa,S,hubs,share", ADJACENCY_TIERS)
def test_build_adjacency_run_lengths(device, G, R, kappa, S, hubs, share):
    """Every way a vertex's edges are gathered (one wave, one workgroup, several
    workgroups, by rank) and ordered, with columns on both sides of the row's position,
    repeated within a row and outside the sequence; dyadic scores make the sums
    exact, so the edge list must equal the oracle's bit for bit."""
    from community_kv_amd.graph.partition import build_adjacency
    from oracle import ckv_oracle as co

    rng = np.random.default_rng(R + S)
    idx = rng.integers(0, S, (G, R, kappa)).astype(np.int32)
    if kappa > 1:
        for h in range(hubs):
            named = rng.random((G, R)) < share
            idx[..., h][named] = (7 + 11 * h) % S
        idx[:, ::5, -1] = idx[:, ::5, -2]
        idx[rng.random(idx.shape) < 0.03] = -1
        idx[rng.random(idx.shape) < 0.02] = S
    sc = (rng.integers(1, 9, idx.shape) / 16.0).astype(np.float32)
    pos = rng.integers(0, S, (G, R)).astype(np.int64)
    print(f"build_adjacency tiers G={G} R={R} kappa={kappa} S={S} hubs={hubs} share={share}", flush=True)
    for lam in (0.5, 1.0):
        got = build_adjacency(*_dev(device, idx, sc, pos), seq_len=S, lam=lam)
        ref = co.build_adjacency(idx, sc, pos, seq_len=S, lam=lam)
        for a, b in zip(got, ref):
            np.testing.assert_array_equal(a.cpu().numpy(), b)


CONTRACTIONS = [
    # seed, graphs, seq_len, hub leaves, isolated, shuffled: rows of one member, many members, a workgroup's and dense
    (41, 2, 700, 0, 5, False),
    (42, 1, 2400, 1500, 0, False),
    (43, 3, 500, 0, 0, True),
    (44, 1, 20000, 17000, 100, False),
    (45, 1, 20000, 17000, 0, True),
]


@pytest.mark.parametrize("seed,G,S,leaves,isolated,shuffled", CONTRACTIONS)
def test_run_leiden_contractions(device, seed, G, S, leaves, isolated, shuffled):
    """The whole native run on sorted edge lists and on shuffled ones (general
    sort), with hubs whose contracted rows take one wave, one workgroup and
    dense windows of ids: labels equal the oracle's level by level (dyadic
    weights: every sum exact), degrees equal the rows' sums."""
    src, dst, w = lg.planted(seed, G, S, 12, edges_per_vertex=5.0, self_loops=4, isolated=isolated)
    if leaves:  # one vertex joined to many, as a token every row attends to
        rng = np.random.default_rng(seed)
        far = rng.choice(np.arange(1, S - isolated), leaves, replace=False).astype(np.int32)
        src = np.concatenate([src, np.zeros(leaves, np.int32)])
        dst = np.concatenate([dst, far])
        w = np.concatenate([w, (rng.integers(1, 5, leaves) / 64.0).astype(np.float32)])
        total = int(G * S)
        key, inv = np.unique(np.minimum(src, dst).astype(np.int64) * total + np.maximum(src, dst), return_inverse=True)
        src, dst = (key // total).astype(np.int32), (key % total).astype(np.int32)
        w = np.bincount(inv, weights=w).astype(np.float32)
    else:
        order = np.lexsort((dst, src))
        src, dst, w = src[order], dst[order], w[order]
    if shuffled:
        order = np.random.default_rng(seed).permutation(src.size)
        src, dst, w = src[order], dst[order], w[order]
    print(f"leiden run G={G} S={S} edges={src.size} leaves={leaves} shuffled={shuffled}", flush=True)
    s, d, x = _dev(device, src, dst, w)
    vertex, part, q = algorithm.run_leiden(s, d, x, G=G, seq_len=S, max_inner_iter=5, seed=seed)
    rv, rp, rq = L.run_leiden(src, dst, w, graphs=G, seq_len=S, max_inner_iter=5, seed=seed)
    np.testing.assert_array_equal(vertex.cpu().numpy(), rv)
    np.testing.assert_array_equal(part.cpu().numpy(), rp)
    assert q == pytest.approx(rq, abs=1e-9)
    labels, degree, width, _ = algorithm.native_run(s, d, x, G=G, seq_len=S, max_level=6, resolution=1.0, theta=0.01,
                                                    max_inner_iter=5, seed=seed, use_boltzmann=False)
    k = np.bincount(src, weights=w, minlength=G * S) + np.bincount(dst, weights=w, minlength=G * S)
    np.testing.assert_array_equal(degree.cpu().numpy(), k)
    assert (labels.cpu().numpy() < 0).sum() == G * S - rv.size and int(labels.max()) < G * width


def test_dense_communities_match_oracle(device):
    """Native fill of isolated vertices and dense renumbering against the oracle's two steps."""
    from community_kv_amd import _native as nat

    rng = np.random.default_rng(9)
    for G, S, W in ((3, 257, 40), (1, 64, 1), (2, 5, 0)):
        lab = np.full((G, S), -1, np.int32)
        if W:
            lab = (rng.integers(0, W, (G, S)) + np.arange(G)[:, None] * W).astype(np.int32)
            lab[rng.random(lab.shape) < 0.2] = -1
        t = torch.from_numpy(lab).to(device)
        ids = torch.empty_like(t)
        counts = torch.empty(G, dtype=torch.int32, device=device)
        ws = torch.empty(nat.lib().ckv_dense_communities_workspace_bytes(G, S, W), dtype=torch.uint8, device=device)
        print(f"dense communities G={G} S={S} W={W}", flush=True)
        nat.check(nat.lib().ckv_dense_communities(t.data_ptr(), G, S, W, ids.data_ptr(), counts.data_ptr(),
                                                  ws.data_ptr(), nat.stream_handle(t.device)))
        ref = L.dense_remap(L.fill_isolated(lab))
        np.testing.assert_array_equal(ids.cpu().numpy(), ref)
        assert counts.cpu().tolist() == (ref.max(axis=1) + 1).tolist()


SWEEP_ROWS = [
    # seed, row lengths, vertices, self loops, sweeps: each side of the row classes' edges; more sweeps than one ring of
    # marks; the longest row of a graph that needs no workgroup of 1,024 threads, and of one that does
    (51, (1, 2, 31, 32, 33, 63, 64, 65), 400, 3, 5),
    (52, (127, 128, 129, 130), 700, 0, 4),
    (53, (255, 256, 257, 511, 512, 513), 1500, 0, 4),
    (54, (1022, 1021), 1023, 1, 3),
    (55, (1023, 1022), 1024, 1, 3),
    (56, (1023, 1024, 1025), 2200, 1, 3),
    (57, (40, 90), 300, 0, 130),
]


@pytest.mark.parametrize("ordered", [True, False])
@pytest.mark.parametrize("seed,rows,S,loops,sweeps", SWEEP_ROWS)
def test_sweep_row_classes(device, seed, rows, S, loops, sweeps, ordered):
    """Rows at the edges of the sweeps' classes (half a wave, a workgroup of
    256, one of 1,024), on an ascending list (each row names a neighbour once:
    the first sweeps build no table) and on a shuffled one: labels equal the
    oracle's (dyadic weights: every sum exact)."""
    rng = np.random.default_rng(seed)
    src, dst, w = lg.planted(seed, 2, S, 10, edges_per_vertex=4.0, self_loops=loops)
    key = {}
    for a, b, x in zip(src.tolist(), dst.tolist(), w.tolist()):
        key[min(a, b), max(a, b)] = x
    for i, n in enumerate(rows):  # vertex i of the second graph gets a row of exactly n other vertices
        v = S + i
        have = {b if a == v else a for a, b in key if (a == v) != (b == v)}
        far = [u for u in rng.permutation(np.arange(S + len(rows), 2 * S)).tolist() if u not in have]
        for u in far[:max(0, n - len(have))]:
            key[v, u] = int(rng.integers(1, 9)) / 64.0
    if loops:
        key[S, S] = 0.25
    order = sorted(key)
    if not ordered:
        order = [order[i] for i in rng.permutation(len(order))]
    src, dst = (np.array([p[i] for p in order], np.int32) for i in (0, 1))
    w = np.array([key[p] for p in order], np.float32)
    print(f"leiden rows {rows} S={S} edges={src.size} ordered={ordered} sweeps={sweeps}", flush=True)
    s, d, x = _dev(device, src, dst, w)
    kw = dict(seq_len=S, max_level=1, max_inner_iter=sweeps, seed=seed)
    vertex, part, _ = algorithm.run_leiden(s, d, x, G=2, **kw)
    rv, rp, _ = L.run_leiden(src, dst, w, graphs=2, **kw)
    np.testing.assert_array_equal(vertex.cpu().numpy(), rv)
    np.testing.assert_array_equal(part.cpu().numpy(), rp)
    # with noise in the scores, the same sweeps through the general path (logf is the device's on both sides)
    vertex, part, _ = algorithm.run_leiden(s, d, x, G=2, use_boltzmann=True, **kw)
    general, _ = _native_level(device, src, dst, w, 2, S, use_boltzmann=True, max_inner_iter=sweeps, seed=seed)
    general = general[vertex.cpu().numpy()]
    pairs = np.unique(np.stack([general, part.cpu().numpy()]), axis=1).shape[1]
    assert pairs == np.unique(general).size == np.unique(part.cpu().numpy()).size


def test_run_leiden_ranks_on_both_paths(device):
    """Labels are ranked by a bitmap in LDS up to 262,144 vertices a graph and by
    a scan above: one vertex without edges more gives the same communities."""
    rng = np.random.default_rng(9)
    S = 1 << 18
    v = rng.choice(S, 3000, replace=False).astype(np.int64)
    a, b = v[rng.integers(0, v.size, 12000)], v[rng.integers(0, v.size, 12000)]
    key = np.unique(np.minimum(a, b)[a != b] * (S + 1) + np.maximum(a, b)[a != b])
    w = (rng.integers(1, 64, key.size) / 64.0).astype(np.float32)
    s, d, x = _dev(device, (key // (S + 1)).astype(np.int32), (key % (S + 1)).astype(np.int32), w)
    print(f"leiden ranks edges={key.size}", flush=True)
    got = [algorithm.run_leiden(s, d, x, G=1, seq_len=n, max_level=3, max_inner_iter=3, seed=2) for n in (S, S + 1)]
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])
    assert got[0][2] == pytest.approx(got[1][2], abs=1e-12)


@pytest.mark.parametrize("at", ["front", "middle", "back", "spread"])
def test_run_leiden_sparse_edge_lists(device, at):
    """Vertices without edges before, between and behind those with edges, in
    gaps on both sides of the length that one thread fills, in one graph of
    three: labels equal the oracle's (dyadic weights: every sum exact)."""
    rng = np.random.default_rng(len(at))
    G, S, n = 3, 5000, 240
    if at == "spread":
        live = np.cumsum(np.concatenate([[0], np.tile([1, 2, 15, 16, 17, 18, 33, 64], 30)]))[:n]
    else:
        live = np.arange(n) + {"front": 0, "middle": 2300, "back": S - n}[at]
    graph = {"front": 0, "middle": 1, "back": 2, "spread": 1}[at]
    a, b = live[rng.integers(0, n, 900)], live[rng.integers(0, n, 900)]
    key = np.unique((np.minimum(a, b) * S + np.maximum(a, b)))
    src, dst = (key // S + graph * S).astype(np.int32), (key % S + graph * S).astype(np.int32)
    w = (rng.integers(1, 64, key.size) / 64.0).astype(np.float32)
    s, d, x = _dev(device, src, dst, w)
    print(f"leiden sparse {at} edges={key.size}", flush=True)
    vertex, part, q = algorithm.run_leiden(s, d, x, G=G, seq_len=S, max_inner_iter=4, seed=1)
    rv, rp, rq = L.run_leiden(src, dst, w, graphs=G, seq_len=S, max_inner_iter=4, seed=1)
    np.testing.assert_array_equal(vertex.cpu().numpy(), rv)
    np.testing.assert_array_equal(part.cpu().numpy(), rp)
    assert q == pytest.approx(rq, abs=1e-9)


def test_run_leiden_graphs_without_edges_cost_little(device):
    """Edges in the last of 32 graphs of 32,768 vertices: the run takes at most
    a few times as long as on that graph alone (what a vertex without edges
    costs; one thread that fills the others' row starts made it 60 times)."""
    rng = np.random.default_rng(2)
    G, S = 32, 32768
    a = rng.integers(0, S - 200, 100000)
    key = np.unique(a * S + a + rng.integers(1, 200, a.size))
    w = torch.from_numpy((rng.integers(1, 64, key.size) / 64.0).astype(np.float32)).to(device)

    def best_us(graphs):
        off = (graphs - 1) * S
        s, d = _dev(device, (key // S + off).astype(np.int32), (key % S + off).astype(np.int32))
        best = float("inf")
        for _ in range(6):
            t0 = time.perf_counter()
            algorithm.run_leiden(s, d, w, G=graphs, seq_len=S, max_inner_iter=4)
            torch.cuda.synchronize()
            best = min(best, (time.perf_counter() - t0) * 1e6)
        return best

    alone, among = best_us(1), best_us(G)
    print(f"leiden one graph {alone:.0f} us, among {G} {among:.0f} us", flush=True)
    assert among < 8.0 * alone


def test_run_leiden_sweeps_after_the_end_cost_little(device):
    """Sweeps queued behind a phase's end leave the vertices alone: 64 sweeps of
    a graph that settles in a few (30,000 leaves around one vertex, one
    community in the end) take little longer than 8 (every vertex adding its
    degree to that community's total once more a sweep: 5 times)."""
    S = 30001
    rng = np.random.default_rng(4)
    s, d, w = _dev(device, np.zeros(S - 1, np.int32), np.arange(1, S, dtype=np.int32),
                   (rng.integers(1, 64, S - 1) / 64.0).astype(np.float32))

    def best_us(sweeps):
        best = float("inf")
        for _ in range(5):
            t0 = time.perf_counter()
            algorithm.run_leiden(s, d, w, G=1, seq_len=S, max_inner_iter=sweeps)
            torch.cuda.synchronize()
            best = min(best, (time.perf_counter() - t0) * 1e6)
        return best

    few, many = best_us(8), best_us(64)
    print(f"leiden 8 sweeps {few:.0f} us, 64 sweeps {many:.0f} us", flush=True)
    assert many < 2.5 * few


@pytest.mark.parametrize("S", [64, 127, 5000])
def test_run_leiden_members_of_one_community(device, S):
    """Members of a community counted and placed a wave at a time: whole waves of
    one community, a few of it among others, fewer than are worth it, and a last
    wave that is not full.  Labels equal the oracle's (dyadic weights)."""
    rng = np.random.default_rng(S)
    hubs = np.array([0, S // 2, S // 2 + 1])
    home = np.where(np.arange(S) < S // 2, hubs[0], hubs[1 + (np.arange(S) % 16 == 0)])
    pairs = {(min(a, b), max(a, b)) for a, b in zip(home.tolist(), range(S)) if a != b}
    order = sorted(pairs)
    src, dst = (np.array([p[i] for p in order], np.int32) for i in (0, 1))
    w = (rng.integers(1, 64, src.size) / 64.0).astype(np.float32)
    print(f"leiden members S={S}", flush=True)
    s, d, x = _dev(device, src, dst, w)
    vertex, part, q = algorithm.run_leiden(s, d, x, G=1, seq_len=S, max_inner_iter=6, seed=3)
    rv, rp, rq = L.run_leiden(src, dst, w, graphs=1, seq_len=S, max_inner_iter=6, seed=3)
    np.testing.assert_array_equal(vertex.cpu().numpy(), rv)
    np.testing.assert_array_equal(part.cpu().numpy(), rp)
    assert q == pytest.approx(rq, abs=1e-9)


@pytest.mark.parametrize("ordered", [True, False])
@pytest.mark.parametrize("S", [32760, 32761, 40000])
def test_sweeps_on_both_sides_of_the_grid_split(device, S, ordered):
    """Up to 4,095 chunks of eight vertices the long rows have workgroups of
    their own, from 4,096 on every workgroup takes hubs, mids and chunks in turn
    from one table: rows of each class among short ones, several chunks a
    workgroup, on ascending and on shuffled lists; one level's labels equal the
    oracle's (dyadic weights: every sum exact)."""
    rng = np.random.default_rng(S)
    a = rng.integers(0, S, 3 * S)
    b = np.clip(a + rng.integers(1, 40, a.size), 0, S - 1)
    long_rows = [(129, 40), (200, 40), (256, 20), (257, 20), (600, 30), (1023, 10), (1025, 4), (3000, 2)]
    heads = rng.choice(S, sum(n for _, n in long_rows), replace=False)
    at = 0
    for length, many in long_rows:
        for v in heads[at:at + many]:
            a = np.concatenate([a, np.full(length, v)])
            b = np.concatenate([b, rng.choice(S, length, replace=False)])
        at += many
    key = np.unique((np.minimum(a, b) * S + np.maximum(a, b))[a != b])
    if not ordered:
        key = rng.permutation(key)
    src, dst = (key // S).astype(np.int32), (key % S).astype(np.int32)
    w = (rng.integers(1, 64, key.size) / 64.0).astype(np.float32)
    print(f"leiden grid split S={S} edges={key.size} ordered={ordered}", flush=True)
    s, d, x = _dev(device, src, dst, w)
    kw = dict(seq_len=S, max_level=1, max_inner_iter=3, seed=5)
    vertex, part, _ = algorithm.run_leiden(s, d, x, G=1, **kw)
    rv, rp, _ = L.run_leiden(src, dst, w, graphs=1, **kw)
    np.testing.assert_array_equal(vertex.cpu().numpy(), rv)
    np.testing.assert_array_equal(part.cpu().numpy(), rp)


def test_native_run_applies_environment_overrides(device, monkeypatch):
    """The reference's environment variables reach the native run (sweeps and
    temperature of the noise, and the noise itself)."""
    src, dst, w = lg.planted(7, 2, 600, 9)
    s, d, x = _dev(device, src, dst, w)
    kw = dict(G=2, seq_len=600, seed=3)
    explicit = algorithm.run_leiden(s, d, x, max_inner_iter=2, theta=0.5, use_boltzmann=True, **kw)
    plain = algorithm.run_leiden(s, d, x, **kw)
    monkeypatch.setenv("COMMUNITY_KV_LEIDEN_MAX_INNER_ITER", "2")
    monkeypatch.setenv("COMMUNITY_KV_LEIDEN_THETA", "0.5")
    monkeypatch.setenv("COMMUNITY_KV_LEIDEN_BOLTZMANN", "1")
    got = algorithm.run_leiden(s, d, x, **kw)
    assert torch.equal(got[1], explicit[1]) and got[2] == explicit[2]
    assert plain[1].shape != got[1].shape or not torch.equal(plain[1], got[1])


@pytest.mark.parametrize("dyadic", [True, False])
def test_partition_modularity_of_an_edge_list(device, dyadic):
    """ckv_partition_modularity (any labels, any edge order) against the same
    formula in float64 on the host: sums of some 10^4 f64 terms."""
    src, dst, w = lg.planted(11, 2, 900, 14, self_loops=5, isolated=20, dyadic=dyadic)
    rng = np.random.default_rng(1)
    order = rng.permutation(src.size)
    src, dst, w = src[order], dst[order], w[order]
    lab = rng.integers(0, 30, 1800).astype(np.int32)
    print(f"partition modularity edges={src.size}", flush=True)
    s, d, x, l = _dev(device, src, dst, w, lab)
    got = algorithm._compute_disjoint_modularity(s, d, x, l, 1.25)
    ref = algorithm._compute_disjoint_modularity(*(torch.from_numpy(a) for a in (src, dst, w, lab)), 1.25)
    assert got == pytest.approx(ref, abs=1e-12)
