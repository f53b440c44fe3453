"""GPU state assembly from labels (``ckv_label_counts`` + ``ckv_build_layer_state``)
against the oracle's restatement of the reference's compute_centroids /
build_member_csr / init_modularity_state (graph/partition.py:382-535): CSR,
sizes, token table and centroids bit for bit (the kernel adds keys in
ascending position order, as the oracle does); modularity weights within
float-summation tolerance (both the reference and this build add them with
float atomics)."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from community_kv_amd.graph.kernels.state_build import build_layer_state, label_counts
from oracle import ckv_oracle as co

pytestmark = pytest.mark.gpu


def _labels(rng, graphs, seq_len, maxc, num_sink, zipf=False):
    if zipf:
        w = 1.0 / np.arange(1, maxc + 1) ** 1.1
        ids = rng.choice(maxc, size=(graphs, seq_len), p=w / w.sum())
    else:
        ids = rng.integers(0, maxc, size=(graphs, seq_len))
    ids[:, :num_sink] = rng.integers(0, 3, size=(graphs, num_sink))  # sink labels are ignored
    return ids.astype(np.int32)


def _edges(rng, graphs, seq_len, num_sink, n):
    g = rng.integers(0, graphs, n)
    a = rng.integers(num_sink, seq_len, n)
    b = rng.integers(num_sink, seq_len, n)
    order = np.lexsort((b, a, g))
    src = (g * seq_len + a)[order].astype(np.int32)
    dst = (g * seq_len + b)[order].astype(np.int32)
    w = rng.random(n).astype(np.float32)
    return src, dst, w


CASES = [
    # graphs, seq_len, num_sink, maxc, to_graph, to_kv, key dtype, fp8, zipf, edges
    (2, 5000, 10, 300, [0, 1], [0, 1], torch.bfloat16, True, False, 20000),
    (1, 3000, 4, 40, [0, 0, 0, 0], [0, 1, 2, 3], torch.float32, False, False, 5000),
    (3, 64, 0, 1, [0, 1, 2], [2, 1, 0], torch.bfloat16, True, False, 0),
    (4, 9000, 10, 2000, [0, 1, 2, 3], [0, 1, 2, 3], torch.bfloat16, True, True, 0),
    # more communities than the kernels' LDS counters (16,384): the rest counted in global memory
    (2, 60000, 10, 30000, [0, 1], [0, 1], torch.bfloat16, True, False, 100000),
    # config 2 shape: 8 graphs x 32k positions, 512 Zipf communities, prefill-sized edge list
    (8, 32768, 10, 512, list(range(8)), list(range(8)), torch.bfloat16, True, True, 400000),
]


@pytest.mark.parametrize("graphs,seq_len,num_sink,maxc,to_graph,to_kv,kdt,fp8,zipf,n_edges", CASES)
def test_state_build_matches_oracle(device, graphs, seq_len, num_sink, maxc, to_graph, to_kv, kdt, fp8, zipf,
                                    n_edges):
    print(f"state build graphs={graphs} S={seq_len} sinks={num_sink} maxc={maxc} heads={len(to_graph)} "
          f"{kdt} fp8={fp8} edges={n_edges}", flush=True)
    rng = np.random.default_rng(seq_len + maxc)
    ids = _labels(rng, graphs, seq_len, maxc, num_sink, zipf)
    if graphs > 1:
        ids[-1, num_sink:] %= max(1, maxc // 2)  # graphs with different community counts
    kv_heads = max(to_kv) + 1
    cache = torch.randn(kv_heads, seq_len + 77, 128, generator=torch.Generator().manual_seed(3)) * 2.0
    cache = cache.to(kdt)
    keys = cache.to(device)[:, :seq_len]  # token stride 128, cache longer than the prompt
    edges = _edges(rng, graphs, seq_len, num_sink, n_edges) if n_edges else None
    tg = torch.tensor(to_graph, dtype=torch.int32, device=device)
    tk = torch.tensor(to_kv, dtype=torch.int32, device=device)
    max_decode = 16
    st = build_layer_state(torch.from_numpy(ids).to(device), keys, retrieval_to_graph=tg, retrieval_to_kv=tk,
                           num_sink=num_sink, max_decode_tokens=max_decode, fp8=fp8,
                           edges=None if edges is None else tuple(torch.from_numpy(e).to(device) for e in edges))
    torch.cuda.synchronize()
    counts = (ids[:, num_sink:].max(axis=1) + 1).astype(np.int32)
    assert st.community_counts.cpu().numpy().tolist() == counts.tolist()
    off, pos = co.build_member_csr(ids, counts, num_sink=num_sink)
    np.testing.assert_array_equal(st.member_offsets.cpu().numpy(), off)
    np.testing.assert_array_equal(st.member_positions.cpu().numpy(), pos)
    keys_np = cache[:, :seq_len].float().numpy()
    cent, sizes = co.compute_centroids(ids, counts, keys_np, to_graph=np.asarray(to_graph, np.int32),
                                       to_kv=np.asarray(to_kv, np.int32), num_sink=num_sink,
                                       max_decode_tokens=max_decode, fp8=fp8)
    np.testing.assert_array_equal(st.community_sizes.cpu().numpy(), sizes)
    got = st.centroids.cpu()
    if fp8:
        np.testing.assert_array_equal(got.view(torch.uint8).numpy(), cent)
    else:
        np.testing.assert_array_equal(got.numpy().view(np.uint32), cent.view(np.uint32))
    tok = st.token_communities.cpu().numpy()
    np.testing.assert_array_equal(tok[:, :seq_len], ids)
    assert (tok[:, seq_len:] == -1).all()
    if edges is not None:
        cw, tw = co.init_modularity_state(ids, *edges, community_capacity=st.community_weight.shape[1],
                                          seq_len=seq_len)
        np.testing.assert_allclose(st.community_weight.cpu().numpy(), cw, rtol=2e-5, atol=1e-4)
        np.testing.assert_allclose(st.total_weight.cpu().numpy(), tw, rtol=2e-5)
    else:
        assert not st.community_weight.any() and not st.total_weight.any()


def test_label_counts_flags_negative_labels(device):
    ids = torch.tensor([[5, 1, 2, -3, 0], [7, 7, 0, 1, 4]], dtype=torch.int32, device=device)
    assert label_counts(ids, num_sink=1).cpu().tolist() == [-1, 8]
    assert label_counts(ids, num_sink=4).cpu().tolist() == [1, 5]
    keys = torch.zeros(2, 5, 128, dtype=torch.bfloat16, device=device)
    tg = torch.arange(2, dtype=torch.int32, device=device)
    with pytest.raises(ValueError, match="nonnegative"):
        build_layer_state(ids, keys, retrieval_to_graph=tg, retrieval_to_kv=tg, num_sink=1, max_decode_tokens=4)


@pytest.mark.parametrize("lam,kappa", [(0.5, 8), (1.0, 8), (0.3, 16)])
def test_state_build_topk_edges_match_coalesced_graph(device, lam, kappa):
    """Modularity weights from the prefill top-k edges directly must equal
    those of the reference's graph (build_adjacency + init_modularity_state)."""
    from community_kv_amd.graph.kernels.state_build import TopkEdges

    print(f"state build top-k edges lam={lam} kappa={kappa}", flush=True)
    rng = np.random.default_rng(int(lam * 10) + kappa)
    graphs, group, seq_len, num_sink, maxc = 2, 4, 3000, 10, 120
    ids = _labels(rng, graphs, seq_len, maxc, num_sink)
    row0 = num_sink + kappa - 1
    rows = seq_len - row0
    heads = graphs * group
    idx = rng.integers(num_sink, seq_len, size=(heads, rows, kappa)).astype(np.int32)
    idx[rng.random(idx.shape) < 0.05] = -1                 # dropped columns
    idx[rng.random(idx.shape) < 0.02] = seq_len + 3        # outside the sequence
    sc = rng.random((heads, rows, kappa)).astype(np.float32)
    keys = torch.randn(graphs, seq_len, 128, generator=torch.Generator().manual_seed(5)).to(torch.bfloat16)
    tg = torch.arange(graphs, dtype=torch.int32, device=device)
    st = build_layer_state(torch.from_numpy(ids).to(device), keys.to(device), retrieval_to_graph=tg,
                           retrieval_to_kv=tg, num_sink=num_sink, max_decode_tokens=8,
                           topk_edges=TopkEdges(indices=torch.from_numpy(idx).to(device),
                                                scores=torch.from_numpy(sc).to(device), row0=row0, group=group,
                                                lam=lam))
    torch.cuda.synchronize()
    pos = np.tile(np.arange(row0, row0 + rows), group)[None].repeat(graphs, 0)
    src, dst, w = co.build_adjacency(idx.reshape(graphs, group * rows, kappa), sc.reshape(graphs, group * rows, kappa),
                                     pos, seq_len=seq_len, lam=lam)
    cw, tw = co.init_modularity_state(ids, src, dst, w, community_capacity=st.community_weight.shape[1],
                                      seq_len=seq_len)
    np.testing.assert_allclose(st.community_weight.cpu().numpy(), cw, rtol=1e-4, atol=1e-3)
    # the totals add ~10^5-10^6 edge weights: the device's (per-row closed
    # form, per-workgroup partial sums) sits within 1e-5 of the float64 sum;
    # the oracle's one long float32 chain drifts further (checked loosely)
    tw64 = np.array([2.0 * w[src // seq_len == g].astype(np.float64).sum() for g in range(graphs)])
    np.testing.assert_allclose(st.total_weight.cpu().numpy(), tw64, rtol=1e-5)
    np.testing.assert_allclose(tw, tw64, rtol=1e-3)


@pytest.mark.parametrize("kdt,fp8", [(torch.bfloat16, True), (torch.bfloat16, False), (torch.float32, True)])
def test_state_build_block_edges(device, kdt, fp8):
    """Communities whose sizes sit at the edges of the block sums (4, 16 and
    64 rows loaded; one block finished at once, several added later), newest
    members in partial 64-position groups, and label counts around a power of
    two: CSR, sizes and centroids bit for bit."""
    sizes = [1, 4, 5, 16, 17, 63, 64, 65, 128, 129, 200, 3]
    for extra in (4, 5, 6):  # 16, 17 and 18 labels: 4, 5 and 5 label bits
        rng = np.random.default_rng(extra)
        lab = np.repeat(np.arange(len(sizes) + extra), sizes + [2] * extra).astype(np.int32)
        rng.shuffle(lab)
        ids = np.concatenate([np.zeros(3, np.int32), lab])[None]
        seq_len = ids.shape[1]
        keys = (torch.randn(1, seq_len, 128, generator=torch.Generator().manual_seed(extra)) * 3.0).to(kdt)
        print(f"state build block edges {kdt} fp8={fp8} S={seq_len} labels={len(sizes) + extra}", flush=True)
        one = torch.zeros(1, dtype=torch.int32, device=device)
        st = build_layer_state(torch.from_numpy(ids).to(device), keys.to(device), retrieval_to_graph=one,
                               retrieval_to_kv=one, num_sink=3, max_decode_tokens=2, fp8=fp8)
        counts = np.array([len(sizes) + extra], np.int32)
        off, pos = co.build_member_csr(ids, counts, num_sink=3)
        np.testing.assert_array_equal(st.member_offsets.cpu().numpy(), off)
        np.testing.assert_array_equal(st.member_positions.cpu().numpy(), pos)
        cent, csizes = co.compute_centroids(ids, counts, keys.float().numpy(), to_graph=np.zeros(1, np.int32),
                                            to_kv=np.zeros(1, np.int32), num_sink=3, max_decode_tokens=2, fp8=fp8)
        np.testing.assert_array_equal(st.community_sizes.cpu().numpy(), csizes)
        got = st.centroids.cpu()
        if fp8:
            np.testing.assert_array_equal(got.view(torch.uint8).numpy(), cent)
        else:
            np.testing.assert_array_equal(got.numpy().view(np.uint32), cent.view(np.uint32))


@pytest.mark.parametrize("kappa,offset", [(8, 0), (8, 1), (16, 0), (16, 3), (5, 0)])
def test_state_build_topk_load_widths(device, kappa, offset):
    """Top-k edges read with 16-byte loads (8 or 16 edges a row, aligned) and
    one by one (any other width, or a view that starts off a 16-byte address)
    give the weights of the float64 closed form: at most about 3,400 x 9 float
    terms per community, so 1e-4 relative."""
    from community_kv_amd.graph.kernels.state_build import TopkEdges

    rng = np.random.default_rng(kappa + offset)
    graphs, group, seq_len, num_sink, maxc, lam = 2, 2, 1700, 4, 37, 0.5
    ids = _labels(rng, graphs, seq_len, maxc, num_sink)
    row0 = num_sink + kappa - 1
    rows, heads = seq_len - row0, graphs * group
    idx = rng.integers(0, seq_len, size=(heads, rows, kappa)).astype(np.int32)
    idx[rng.random(idx.shape) < 0.1] = -1
    sc = rng.random((heads, rows, kappa)).astype(np.float32)

    def shifted(a):
        flat = torch.zeros(a.size + offset, dtype=torch.from_numpy(a).dtype, device=device)
        flat[offset:] = torch.from_numpy(a).to(device).flatten()
        return flat[offset:].view(a.shape)

    print(f"state build top-k widths kappa={kappa} offset={offset}", flush=True)
    tg = torch.arange(graphs, dtype=torch.int32, device=device)
    keys = torch.zeros(graphs, seq_len, 128, dtype=torch.bfloat16, device=device)
    st = build_layer_state(torch.from_numpy(ids).to(device), keys, retrieval_to_graph=tg, retrieval_to_kv=tg,
                           num_sink=num_sink, max_decode_tokens=8,
                           topk_edges=TopkEdges(indices=shifted(idx), scores=shifted(sc), row0=row0, group=group,
                                                lam=lam))
    weight = np.zeros((graphs, st.community_weight.shape[1]))
    total = np.zeros(graphs)
    for h in range(heads):
        g = h // group
        p = np.where(idx[h] >= 0, sc[h], 0.0).astype(np.float64)
        s, s2 = p.sum(1), (p * p).sum(1)
        w = lam / 2 * p + (1 - lam) * p * (s[:, None] + p)
        np.add.at(weight[g], ids[g][np.maximum(idx[h], 0)], w)
        np.add.at(weight[g], ids[g][row0:], lam / 2 * s)
        total[g] += (lam * s + (1 - lam) * (s * s + s2)).sum()
    np.testing.assert_allclose(st.community_weight.cpu().numpy(), weight, rtol=1e-4, atol=1e-4)
    np.testing.assert_allclose(st.total_weight.cpu().numpy(), total, rtol=1e-5)


@pytest.mark.parametrize("graphs,seq_len,n", [(1, 300, 200), (3, 1000, 5000), (2, 4000, 40000), (5, 700, 9000)])
def test_state_build_weights_from_degrees(device, graphs, seq_len, n):
    """Weights from the vertices' degrees and totals from the edges equal those
    of the edge list alone (dyadic weights, sums below 2^11: exact), with graphs
    that end inside a block of 8,192 edges, span several, or share one."""
    rng = np.random.default_rng(n)
    ids = rng.integers(0, 50, (graphs, seq_len)).astype(np.int32)
    src, dst, _ = _edges(rng, graphs, seq_len, 0, n)
    w = (rng.integers(1, 64, n) / 4096.0).astype(np.float32)
    degree = (np.bincount(src, weights=w, minlength=graphs * seq_len)
              + np.bincount(dst, weights=w, minlength=graphs * seq_len))
    keys = torch.zeros(graphs, seq_len, 128, dtype=torch.bfloat16, device=device)
    tg = torch.arange(graphs, dtype=torch.int32, device=device)
    edges = tuple(torch.from_numpy(e).to(device) for e in (src, dst, w))
    print(f"state build degrees graphs={graphs} S={seq_len} edges={n}", flush=True)
    kw = dict(retrieval_to_graph=tg, retrieval_to_kv=tg, num_sink=0, max_decode_tokens=4, edges=edges)
    a = build_layer_state(torch.from_numpy(ids).to(device), keys, **kw)
    b = build_layer_state(torch.from_numpy(ids).to(device), keys, vertex_degree=torch.from_numpy(degree).to(device), **kw)
    assert torch.equal(a.community_weight, b.community_weight) and torch.equal(a.total_weight, b.total_weight)
    np.testing.assert_array_equal(b.total_weight.cpu().numpy(),
                                  np.bincount(src // seq_len, weights=2.0 * w, minlength=graphs).astype(np.float32))
    with pytest.raises(ValueError, match="edge list"):
        build_layer_state(torch.from_numpy(ids).to(device), keys, retrieval_to_graph=tg, retrieval_to_kv=tg, num_sink=0,
                          max_decode_tokens=4, vertex_degree=torch.from_numpy(degree).to(device))


@pytest.mark.parametrize("order", ["shuffled", "descending", "rotated", "outside"])
@pytest.mark.parametrize("graphs,seq_len,n", [(3, 1000, 5000), (2, 4000, 40000), (1, 300, 8193)])
def test_state_build_degree_weights_any_edge_order(device, graphs, seq_len, n, order):
    """Totals beside given degrees do not depend on the order of the edge list
    (shuffled, graphs descending, graphs in blocks of their own but rotated),
    and edges whose source lies outside the graphs are left out of them (dyadic
    weights, sums below 2^12: exact)."""
    rng = np.random.default_rng(n + graphs)
    ids = rng.integers(0, 50, (graphs, seq_len)).astype(np.int32)
    src, dst, _ = _edges(rng, graphs, seq_len, 0, n)
    w = (rng.integers(1, 64, n) / 4096.0).astype(np.float32)
    V = graphs * seq_len
    if order == "outside":
        src[:: 7] = rng.choice([-1, -seq_len, -2**31, V, V + seq_len, 2**31 - 1], src[::7].size)
        src[0] = V
    else:
        at = {"shuffled": rng.permutation(n), "descending": np.arange(n)[::-1],
              "rotated": np.roll(np.arange(n), n // 2)}[order]
        src, dst, w = src[at].copy(), dst[at].copy(), w[at].copy()
    ok = (src >= 0) & (src < V)
    degree = (np.bincount(src[ok], weights=w[ok], minlength=V) + np.bincount(dst[ok], weights=w[ok], minlength=V))
    tg = torch.arange(graphs, dtype=torch.int32, device=device)
    print(f"state build degrees {order} graphs={graphs} S={seq_len} edges={n}", flush=True)
    st = build_layer_state(torch.from_numpy(ids).to(device),
                           torch.zeros(graphs, seq_len, 128, dtype=torch.bfloat16, device=device),
                           retrieval_to_graph=tg, retrieval_to_kv=tg, num_sink=0, max_decode_tokens=4,
                           edges=tuple(torch.from_numpy(e).to(device) for e in (src, dst, w)),
                           vertex_degree=torch.from_numpy(degree).to(device))
    np.testing.assert_array_equal(st.total_weight.cpu().numpy(),
                                  np.bincount(src[ok] // seq_len, weights=2.0 * w[ok], minlength=graphs))
    by_label = np.stack([np.bincount(ids[g], weights=degree.reshape(graphs, seq_len)[g],
                                     minlength=st.community_weight.shape[1]) for g in range(graphs)])
    np.testing.assert_array_equal(st.community_weight.cpu().numpy(), by_label)


@pytest.mark.parametrize("count,extra", [(8186, 6), (8186, 7), (8192, 3), (8193, 3), (16384, 3), (16385, 3), (19000, 3)])
def test_state_build_topk_many_communities(device, count, extra):
    """Community counts on both sides of the line between sums in doubles and in
    floats (8,192 communities, 64 KB of LDS either way) and of the one above
    which the rest is added in global memory (16,384), against the float64
    closed form: some 10 float terms a community, so 1e-5 relative."""
    from community_kv_amd.graph.kernels.state_build import TopkEdges

    rng = np.random.default_rng(count + extra)
    seq_len, num_sink, kappa, lam = 9000 if count < 9000 else 20000, 2, 8, 0.5
    row0 = num_sink + kappa - 1
    rows = seq_len - row0
    ids = rng.integers(0, count, (1, seq_len)).astype(np.int32)
    ids[0, -1] = count - 1
    idx = rng.integers(-1, seq_len + 1, size=(1, rows, kappa)).astype(np.int32)
    sc = rng.random((1, rows, kappa)).astype(np.float32)
    one = torch.zeros(1, dtype=torch.int32, device=device)
    st = build_layer_state(torch.from_numpy(ids).to(device),
                           torch.zeros(1, seq_len, 128, dtype=torch.bfloat16, device=device), retrieval_to_graph=one,
                           retrieval_to_kv=one, num_sink=num_sink, max_decode_tokens=extra,
                           topk_edges=TopkEdges(indices=torch.from_numpy(idx).to(device),
                                                scores=torch.from_numpy(sc).to(device), row0=row0, group=1, lam=lam))
    weight = np.zeros(st.community_weight.shape[1])
    print(f"state build many communities capacity={weight.size}", flush=True)
    ok = (idx[0] >= 0) & (idx[0] < seq_len)
    p = np.where(ok, sc[0], 0.0).astype(np.float64)
    s, s2 = p.sum(1), (p * p).sum(1)
    np.add.at(weight, ids[0][np.where(ok, idx[0], 0)], lam / 2 * p + (1 - lam) * p * (s[:, None] + p))
    np.add.at(weight, ids[0][row0:], lam / 2 * s)
    np.testing.assert_allclose(st.community_weight.cpu().numpy()[0], weight, rtol=1e-5, atol=1e-5)
    np.testing.assert_allclose(st.total_weight.cpu().numpy()[0], (lam * s + (1 - lam) * (s * s + s2)).sum(), rtol=1e-5)
