"""Batched multi-source engines on the GPU: every column of a batched run equals the single-source run of
its source, bit for bit, at every column width, and the single-source runs equal the oracle.

Min-plus columns (SSSP distances, BFS depths) are compared with the oracle's Dijkstra / BFS queue and
with g1_sssp's BLAS engine (apps/sssp_blas.cu:17-84); personalized PageRank columns with g1_ppr
(apps/pagerank_blas.cu:16-125 with a restart vector) bit for bit, and with the FP64 oracle within L1 1e-5.
"""
import os
import subprocess
import sys

import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

WIDTHS = [8, 16, 32, 64]


@pytest.fixture(scope="module")
def graphs(gpu):
    import graphone_amd as g1
    out = []
    h = g1.HostGraph.rmat(13, 16, seed=21).assign_weights(1, 255, seed=22)
    out.append(("rmat13", h, g1.Graph(h)))
    h = g1.HostGraph.grid(48, 48, 0.6, seed=5).assign_weights(1, 64, seed=6, symmetric=True)
    out.append(("grid48", h, g1.Graph(h, symmetric=True)))
    return out


def _sources(h, count, seed):
    rng = np.random.default_rng(seed)
    deg = h.out_degrees()
    src = list(rng.integers(0, h.n, size=count - 3))
    src.append(int(np.argmax(deg)))                       # hub
    src.append(int(np.flatnonzero(deg == 0)[0]) if np.any(deg == 0) else 0)  # leaf / isolated
    src.append(src[0])                                      # duplicate source
    return [int(s) for s in src]


@pytest.mark.parametrize("k", WIDTHS)
def test_sssp_batch_columns_bitexact(graphs, k):
    for name, h, g in graphs:
        srcs = _sources(h, 19, seed=k)
        got = g.sssp_batch(srcs, k=k)
        assert got.values.shape == (len(srcs), h.n)
        assert got.stats["k"] == k and got.stats["tiles"] == -(-len(srcs) // k)
        for c, s in enumerate(srcs):
            want = oracle.dijkstra(h.row_offsets, h.col_indices, h.weights, s)
            assert np.array_equal(got.values[c], want), (name, k, c, s)


@pytest.mark.parametrize("k", [8, 64])
def test_bfs_batch_columns_bitexact(graphs, k):
    for name, h, g in graphs:
        srcs = _sources(h, 11, seed=100 + k)
        got = g.sssp_batch(srcs, k=k, weighted=False)
        for c, s in enumerate(srcs):
            want = oracle.bfs_queue(h.row_offsets, h.col_indices, s)
            assert np.array_equal(got.values[c], want), (name, k, c, s)


@pytest.mark.parametrize("tile", [512, 1024, 2048, 4096])
def test_minplus_merge_tiles_bitexact(graphs, tile):
    """The k = 64 min-plus kernel on each merge partition the autotuner may pick (rows + nonzeros per
    tile): SSSP and BFS columns equal the oracle's, and so does the 32-bit rerun of a batch whose
    distances outgrow 16 bits (a 400-vertex path: 3 tiles of 512, 1 of 4096)."""
    import graphone_amd as g1
    try:
        for name, h, g in graphs:
            g.set_merge_tile(tile)
            srcs = _sources(h, 64, seed=tile)
            got = g.sssp_batch(srcs, k=64)
            assert got.stats["merge_tile"] == tile
            bfs = g.sssp_batch(srcs, k=64, weighted=False)
            for c, s in enumerate(srcs):
                want = oracle.dijkstra(h.row_offsets, h.col_indices, h.weights, s)
                assert np.array_equal(got.values[c], want), (name, tile, c, s)
                want = oracle.bfs_queue(h.row_offsets, h.col_indices, s)
                assert np.array_equal(bfs.values[c], want), (name, tile, c, s)
    finally:
        for _, _, g in graphs:
            g.set_merge_tile(2048)
    n = 400
    src = np.arange(n - 1, dtype=np.uint32)
    h = g1.HostGraph.from_edges(n, src, src + 1, np.full(n - 1, 250, dtype=np.uint32), directed=False)
    g = g1.Graph(h)
    g.set_merge_tile(tile)
    srcs = [int(s) for s in np.linspace(0, n - 1, 64).astype(np.uint32)]
    got = g.sssp_batch(srcs, k=64)
    assert int(got.values.max()) > 0xFFFF
    for c, s in enumerate(srcs):
        assert np.array_equal(got.values[c], oracle.dijkstra(h.row_offsets, h.col_indices, h.weights, s)), (tile, c)
    with pytest.raises(g1.G1Error):
        g.set_merge_tile(3000)


def test_sssp_batch_equals_single_source_engine(graphs):
    name, h, g = graphs[0]
    srcs = _sources(h, 7, seed=3)
    got = g.sssp_batch(srcs, k=16)
    for c, s in enumerate(srcs):
        assert np.array_equal(got.values[c], g.sssp(s, "merge").values)


@pytest.mark.parametrize("k", WIDTHS)
def test_ppr_batch_columns_bit_identical(graphs, k):
    """A batched PPR column is the single-seed g1_ppr result bit for bit (same row-sum fold order, same
    per-column L1 tree and stop rule), including seeds that stop at different iterations."""
    for name, h, g in graphs:
        seeds = _sources(h, 13, seed=200 + k)
        got = g.ppr_batch(seeds, restart=0.15, max_iter=60, tol=1e-7, k=k)
        iters = set()
        for c, s in enumerate(seeds):
            single = g.ppr(s, restart=0.15, max_iter=60, tol=1e-7)
            iters.add(single.stats["iterations"])
            assert np.array_equal(got.values[c].view(np.uint32), single.values.view(np.uint32)), (name, k, c, s)
        if name == "rmat13":
            assert len(iters) > 1, "seeds should stop at different iterations"


def test_ppr_batch_matches_oracle(graphs):
    for name, h, g in graphs:
        t = h.transpose()
        seeds = _sources(h, 5, seed=9)
        got = g.ppr_batch(seeds, restart=0.15, max_iter=100, tol=1e-9, k=8)
        for c, s in enumerate(seeds):
            want, _ = oracle.pagerank_f64(h.row_offsets, h.weights, t.row_offsets, t.col_indices, t.weights,
                                          0.85, max_iter=100, tol=1e-9, seed=s, restart=0.15)
            l1 = float(np.abs(got.values[c].astype(np.float64) - want).sum())
            assert l1 <= 1e-5, (name, c, s, l1)


def test_autotune_and_default_width(graphs):
    name, h, g = graphs[0]
    srcs = _sources(h, 9, seed=1)
    k = g.autotune("minplus", srcs, weighted=True)
    assert k in WIDTHS
    got = g.sssp_batch(srcs)  # k = 0: the tuned width
    assert got.stats["k"] == k
    assert got.stats["merge_tile"] in (512, 1024, 2048, 4096)
    for c, s in enumerate(srcs):
        assert np.array_equal(got.values[c], oracle.dijkstra(h.row_offsets, h.col_indices, h.weights, s))
    kp = g.autotune("ppr", srcs)
    assert kp in WIDTHS
    assert g.ppr_batch(srcs[:3]).stats["k"] == kp


def test_batch_edge_cases(graphs):
    import graphone_amd as g1
    name, h, g = graphs[0]
    # one source, and an empty batch
    one = g.sssp_batch([5], k=64)
    assert np.array_equal(one.values[0], oracle.dijkstra(h.row_offsets, h.col_indices, h.weights, 5))
    empty = g.sssp_batch([], k=8)
    assert empty.values.shape == (0, h.n) and empty.stats["tiles"] == 0
    with pytest.raises(g1.G1Error):
        g.sssp_batch([h.n], k=8)
    with pytest.raises(g1.G1Error):
        g.sssp_batch([0, 1], k=12)
    with pytest.raises(g1.G1Error):
        g.ppr_batch([0], restart=0.0, k=8)


def test_road_batch_matches_oracle(graphs):
    """One workgroup per query on a low-degree graph (the grid): mixed BFS / SSSP queries, bit-exact
    against the oracle, including more queries than one launch takes."""
    import graphone_amd as g1
    name, h, g = graphs[1]
    assert name == "grid48"
    rng = np.random.default_rng(5)
    srcs = [int(s) for s in rng.integers(0, h.n, size=70)]
    kinds = ["sssp" if i % 3 else "bfs" for i in range(len(srcs))]
    got = g.road_batch(srcs, kinds)
    for c, (s, k) in enumerate(zip(srcs, kinds)):
        if k == "sssp":
            want = oracle.dijkstra(h.row_offsets, h.col_indices, h.weights, s)
        else:
            want = oracle.bfs_queue(h.row_offsets, h.col_indices, s)
        assert np.array_equal(got.values[c], want), (c, s, k)
    with pytest.raises(g1.G1Error):
        graphs[0][2].road_batch([0])  # RMAT: hubs far above the road engine's degree bound


def test_sssp_batch_distances_past_16_bits(gpu):
    """k = 64 keeps distances in 16 bits while they fit; on a long heavy path (distances up to
    ~100,000 > 0xFFFF) the batch must notice and redo the run with 32-bit storage, still bit-exact.
    A second, light path checks the 16-bit run itself (all distances < 0xFFFF)."""
    import graphone_amd as g1
    n = 400
    src = np.arange(n - 1, dtype=np.uint32)
    dst = src + 1
    for wv in (250, 3):
        h = g1.HostGraph.from_edges(n, src, dst, np.full(n - 1, wv, dtype=np.uint32), directed=False)
        g = g1.Graph(h)
        srcs = [int(s) for s in np.linspace(0, n - 1, 64).astype(np.uint32)]
        got = g.sssp_batch(srcs, k=64)
        for c, s in enumerate(srcs):
            want = oracle.dijkstra(h.row_offsets, h.col_indices, h.weights, s)
            assert np.array_equal(got.values[c], want), (wv, c, s)
        if wv == 250:
            assert int(got.values.max()) > 0xFFFF


@pytest.mark.parametrize("shape", ["alone", "chain", "hub", "sparse", "dense"])
def test_batch64_row_shapes(gpu, shape):
    """The k = 64 min-plus kernel takes 64 merge steps (nonzeros and row ends) at a time, a quarter of a merge tile
    a wave: a vertex alone, one in-edge a row (every other step an end), a row across several tiles, blocks
    that are nothing but row ends, and rows of about a block; on every merge tile, weighted (16-bit storage, and
    with long edges the 32-bit rerun) and as BFS, against Dijkstra and the queue BFS."""
    import graphone_amd as g1
    rng = np.random.default_rng(len(shape))
    if shape == "alone":
        n, src, dst = 1, [], []
    elif shape == "chain":
        n = 300
        src, dst = np.arange(n - 1), np.arange(1, n)
    elif shape == "hub":
        n = 6001  # everything leads to vertex 6000, which leads back to a third of it
        src = np.concatenate([np.arange(6000), np.full(2000, 6000)])
        dst = np.concatenate([np.full(6000, 6000), rng.choice(6000, 2000, replace=False)])
    elif shape == "sparse":
        n = 20000
        src, dst = rng.integers(0, 40, 900) * 500, rng.integers(0, n, 900)
    else:
        n = 257
        src, dst = np.repeat(np.arange(n), 63), rng.integers(0, n, 63 * n)
    srcs = rng.integers(0, n, size=64 if n > 1 else 3)
    for hi in (200, 70000):
        w = rng.integers(1, hi + 1, size=len(src)).astype(np.uint32)
        h = g1.HostGraph.from_edges(n, src, dst, w)
        g = g1.Graph(h)
        few = sorted(set(int(s) for s in srcs))[:4]
        want = {s: (oracle.dijkstra(h.row_offsets, h.col_indices, h.weights, s),
                    oracle.bfs_queue(h.row_offsets, h.col_indices, s)) for s in few}
        for tile in (512, 1024, 2048, 4096):
            g.set_merge_tile(tile)
            for weighted in (True, False):
                got = g.sssp_batch(srcs, k=64, weighted=weighted).values
                for c, s in enumerate(srcs):
                    if int(s) in want:
                        assert np.array_equal(got[c], want[int(s)][0 if weighted else 1]), (tile, weighted, c)


@pytest.mark.parametrize("n", [(1 << 18) - 1, 1 << 18])
def test_ppr_batch64_scale_array(gpu, n):
    """The 64-column PPR product gathers its sources' scales below 2^18 vertices and streams them in the in-edges'
    order from there: either way a column has the single-seed run's bits, with another restart (other scales) on the
    same graph as well. Two thirds of the edges leave 500 hubs; most vertices have neither in- nor out-edges."""
    import graphone_amd as g1
    rng = np.random.default_rng(n)
    m = 400_003
    src = np.where(rng.random(m) < 0.66, rng.integers(0, 500, m), rng.integers(0, n, m))
    dst = rng.integers(0, n // 3, m)
    h = g1.HostGraph.from_edges(n, src, dst, rng.integers(1, 50, m).astype(np.uint32), directed=True)
    g = g1.Graph(h)
    seeds = [0, 1, n - 1] + [int(v) for v in src[:64]]  # more than one tile of 64
    for restart in (0.15, 0.4):
        got = g.ppr_batch(seeds, restart=restart, max_iter=9, tol=0.0, k=64)
        for c in (0, 2, 40, 66):
            single = g.ppr(seeds[c], restart=restart, max_iter=9, tol=0.0)
            assert np.array_equal(got.values[c].view(np.uint32), single.values.view(np.uint32)), (restart, c)


def test_batch64_idle_iterations(gpu):
    """A k = 64 min-plus batch of more merge tiles than the chip holds at once (its kernel then looks a whole quarter
    over where the first block has no active source): 40 iterations with one changed vertex a source, at ids on both
    ends of the activity bitmaps' words and bytes, then a dense spread from the path's end through 4.3 million
    edges, into a hub of 30,000 in-edges as well; weighted and as BFS, on two merge tiles, against the oracle."""
    import graphone_amd as g1
    rng = np.random.default_rng(3)
    n, m = 500_003, 4_300_000
    path = np.array([0, 63, 64, 511, 512, 2047, 2048, n - 1, n - 3] + list(range(5000, 5031)))
    body = np.setdiff1d(np.arange(n), path)
    src = np.concatenate([rng.choice(body, m), rng.choice(body, 30000), path[:-1], np.full(5, path[-1])])
    dst = np.concatenate([rng.choice(body, m), np.full(30000, body[7]), path[1:], rng.choice(body, 5)])
    h = g1.HostGraph.from_edges(n, src, dst, rng.integers(1, 200, src.size).astype(np.uint32))
    g = g1.Graph(h)
    srcs = [int(path[0]), int(path[3]), int(path[8]), int(body[11])] * 16
    for tile in (2048, 4096):
        g.set_merge_tile(tile)
        for weighted in (True, False):
            got = g.sssp_batch(srcs, k=64, weighted=weighted).values
            for c in range(4):
                want = (oracle.dijkstra(h.row_offsets, h.col_indices, h.weights, srcs[c]) if weighted else
                        oracle.bfs_queue(h.row_offsets, h.col_indices, srcs[c]))
                assert np.array_equal(got[c], want) and np.array_equal(got[60 + c], want), (tile, weighted, c)


def test_switched_off_wave_kernels_give_the_same_bits(gpu, tmp_path):
    """G1_PPR_WAVE=0 (the 64-column PPR product by rounds, with x and y arrays and a rank kernel) and G1_MINPLUS_WAVE=0
    with G1_MINPLUS_U16=0 (the min-plus batch on the chunked kernel): the bits of the default kernels, more seeds than
    a tile holds and fewer, columns that converge before others."""
    import graphone_amd as g1
    code = """
import sys
import numpy as np
import graphone_amd as g1
h = g1.HostGraph.rmat(13, 12, seed=9).assign_weights(1, 300, seed=10)
g = g1.Graph(h)
rng = np.random.default_rng(4)
out = {}
for count in (5, 70):
    ids = rng.integers(0, h.n, count)
    out[f"ppr{count}"] = g.ppr_batch(ids, max_iter=31, tol=1e-4, k=64).values.view(np.uint32)
    out[f"sssp{count}"] = g.sssp_batch(ids, k=64).values
np.savez(sys.argv[1], **out)
"""
    got = []
    for name, env in (("on", {}), ("off", {"G1_PPR_WAVE": "0", "G1_MINPLUS_WAVE": "0", "G1_MINPLUS_U16": "0"})):
        path = str(tmp_path / f"{name}.npz")
        root = os.path.dirname(os.path.dirname(os.path.abspath(g1.__file__)))
        subprocess.run([sys.executable, "-c", code, path], check=True, timeout=100,
                       env={**os.environ, **env, "PYTHONPATH": root})
        got.append(np.load(path))
    for key in got[0].files:
        assert np.array_equal(got[0][key], got[1][key]), key


@pytest.mark.parametrize("n", [(1 << 17) - 1, 1 << 17])
def test_ppr_batch64_fusion_line(gpu, n):
    """Below 2^17 vertices an iteration of the 64-column PPR is a product and a rank kernel, from there one kernel that
    writes the ranks: a column has the single-seed run's bits and iteration either way, with fewer seeds than columns
    and columns that converge at different iterations."""
    import graphone_amd as g1
    rng = np.random.default_rng(n)
    m = 300_001
    src, dst = rng.integers(0, n, m) // 3, rng.integers(0, n, m)
    h = g1.HostGraph.from_edges(n, src, dst, rng.integers(1, 50, m).astype(np.uint32), directed=True)
    g = g1.Graph(h)
    seeds = [0, n - 1, int(src[5]), int(src[6]), int(dst[9])]
    for tol, iters in ((0.0, 7), (1e-3, 40)):
        got = g.ppr_batch(seeds, max_iter=iters, tol=tol, k=64)
        for c, s in enumerate(seeds):
            single = g.ppr(s, max_iter=iters, tol=tol)
            assert np.array_equal(got.values[c].view(np.uint32), single.values.view(np.uint32)), (tol, c)
