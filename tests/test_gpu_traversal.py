"""GPU parity for BFS, SSSP and multi-source BFS: bit-exact against the CPU oracle."""
import json
import pathlib

import numpy as np
import pytest

import medusa_amd as md
from medusa_amd import workloads as wl
from conftest import csr_from_edges, random_graph

pytestmark = pytest.mark.gpu
GOLDEN = json.loads((pathlib.Path(__file__).parent / "golden" / "golden.json").read_text())
U32MAX = 0xFFFFFFFF


@pytest.fixture(autouse=True)
def _announce(request):
    print(f"\n[case] {request.node.nodeid}", flush=True)


def _dirs():
    return [md.DIR_PUSH, md.DIR_PULL, md.DIR_AUTO]


# ---- BFS -------------------------------------------------------------------------

@pytest.mark.parametrize("name", sorted(GOLDEN))
def test_bfs_golden(name):
    g = GOLDEN[name]
    rp, col, _ = csr_from_edges(g["n"], g["edges"], g["weights"])
    with md.Graph(rp, col) as G:
        for s, want in g["bfs"].items():
            for d in _dirs():
                lv, st = G.bfs(int(s), direction=d)
                assert lv.tolist() == want, (s, d)
                assert st.reached == sum(1 for x in want if x >= 0)


@pytest.mark.parametrize("seed", range(4))
def test_bfs_random_vs_oracle(oracle, seed):
    n = 3000 + 500 * seed
    rp, col, _ = random_graph(n, 8 * n, seed)
    with md.Graph(rp, col) as G:
        for src in (0, n - 1, seed * 97 % n):
            want = oracle.bfs_queue(rp, col, src)
            for d in _dirs():
                lv, _ = G.bfs(src, direction=d)
                assert np.array_equal(lv, want), (src, d)


def test_bfs_hubs_use_large_path(oracle):
    # a few hubs with thousands of out-edges, and a small threshold so the
    # workgroup-split kernel handles them
    rng = np.random.default_rng(3)
    n = 20000
    src = np.concatenate([rng.integers(0, n, 60000), np.repeat([5, 77, 901], 9000)])
    dst = rng.integers(0, n, len(src))
    rp, col, _ = csr_from_edges(n, np.stack([src, dst], 1))
    with md.Graph(rp, col) as G:
        for large in (0, 64, 1):
            for s in (5, 3):
                lv, _ = G.bfs(s, direction=md.DIR_PUSH, large_degree=large)
                assert np.array_equal(lv, oracle.bfs_queue(rp, col, s)), (large, s)


@pytest.mark.parametrize("n", [1023, 1024, 2049, 40_001])
def test_bfs_rounds_per_workgroup(oracle, n):
    """Two workgroups walk the vertex rounds of the pull and the compaction (20 rounds each at the
    largest size, past the 16 whose visited words load at once), with in-degrees on both sides of
    the lane limit of 32 and winners of exact claims in both workgroups' segments."""
    rng = np.random.default_rng(n)
    src = [rng.integers(0, n, 3 * n)]
    dst = [rng.integers(0, n, 3 * n)]
    for d in (31, 32, 33, 200):
        v = rng.integers(0, n, 8)
        src.append(rng.integers(0, n, 8 * d))
        dst.append(np.repeat(v, d))
    rp, col, _ = csr_from_edges(n, np.stack([np.concatenate(src), np.concatenate(dst)], 1))
    s = wl.max_outdeg_vertex(rp)
    want = oracle.bfs_queue(rp, col, s)
    with md.Graph(rp, col) as G:
        for d in _dirs():
            for grid in (2, 0):
                assert np.array_equal(G.bfs(s, direction=d, grid=grid, large_degree=4)[0], want), (d, grid)


@pytest.mark.parametrize("n", [4096, 4097, 20000])
@pytest.mark.parametrize("width,fan", [(1023, 1), (1024, 1), (1025, 1), (4095, 1), (341, 3), (342, 3), (1365, 3),
                                       (1366, 3), (7, 585), (7, 586), (64, 600)])
def test_bfs_frontiers_of_one_workgroup(oracle, n, width, fan):
    """Second frontiers of `width` vertices with `fan` out-edges each, on both sides of the 1024 and
    4096 out-edges that one workgroup takes, then a chain (thin supersteps to the end); hubs in the
    frontiers handed over; host outputs, device-driven and host-driven runs, runs of different
    lengths on one handle, and more sources than the starting kernel takes."""
    rng = np.random.default_rng(width * fan + n)
    width = min(width, n - 2)
    first = np.arange(1, width + 1)
    chain = np.arange(n - 41, n - 1)
    edges = np.concatenate([
        np.stack([np.zeros(width, np.int64), first], 1),
        np.stack([np.repeat(first, fan), rng.integers(0, n - 40, width * fan)], 1),
        np.stack([chain, chain + 1], 1),
    ])
    rp, col, _ = csr_from_edges(n, edges)
    sources = rng.integers(0, n, 4000).astype(np.uint32)
    with md.Graph(rp, col) as G:
        for s in (0, n - 41, 1, 0):
            want = oracle.bfs_queue(rp, col, s)
            for d in _dirs():
                for large in (0, 100):
                    lv, st = G.bfs(s, direction=d, large_degree=large)
                    assert np.array_equal(lv, want), (s, d, large)
            host = G.bfs(s, timing=True)[1]
            dev = G.bfs(s)[1]
            assert (host.supersteps, host.push_steps, host.pull_steps) == (dev.supersteps, dev.push_steps, dev.pull_steps)
            assert (host.reached, host.edges_traversed) == (dev.reached, dev.edges_traversed)
        # as many sources as the starting kernel takes, and more (duplicates): one edge short of a
        # search from a vertex that points at all of them
        rp2 = np.append(rp, rp[-1] + len(np.unique(sources))).astype(np.uint32)
        col2 = np.append(col, np.unique(sources)).astype(np.uint32)
        want = np.maximum(oracle.bfs_queue(rp2, col2, n) - 1, -1)[:n]
        for k in (4096, 5000):
            assert np.array_equal(G.bfs_multi(np.resize(sources, k))[0], want), k


@pytest.mark.parametrize("n", [32 * 1024 + 1, 140_000, 262_144])
@pytest.mark.parametrize("fan", [700, 60_000])
def test_bfs_held_joins(oracle, n, fan):
    """Waves with several rounds of vertices (one segment for all of a workgroup's at 32 and 64
    workgroups, one each at 33): a source whose targets all join at once, so a wave's list of joins
    fills up and is appended in the middle, then a random graph that leaves some vertices to pulls of
    sparsely unvisited words; hubs among the joins."""
    rng = np.random.default_rng(n + fan)
    first = rng.permutation(np.arange(1, n))[:min(fan, n - 1)]
    dense = np.arange(1, min(fan, n - 1) + 1)
    src = np.concatenate([np.zeros(len(first), np.int64), np.full(len(dense), first[0]), rng.integers(0, n, 2 * n)])
    dst = np.concatenate([first, dense, rng.integers(0, n, 2 * n)])
    rp, col, _ = csr_from_edges(n, np.stack([src, dst], 1))
    want = oracle.bfs_queue(rp, col, 0)
    with md.Graph(rp, col) as G:
        for d in _dirs():
            for grid in (2, 32, 33, 64, 0):
                got, st = G.bfs(0, direction=d, grid=grid, large_degree=6)
                assert np.array_equal(got, want), (d, grid)
                assert st.reached == (want >= 0).sum(), (d, grid)


@pytest.mark.parametrize("parents", [1, 3, 64])
@pytest.mark.parametrize("total", [4097, 8192])
def test_bfs_few_vertices_with_many_out_edges(oracle, parents, total):
    """A frontier of at most 64 vertices with more out-edges than two or seven workgroups take at once
    (1024 each), up to a queue segment's 8192: every out-edge counts on every grid, in both drivers."""
    n = 262_144  # segments of 8192
    rng = np.random.default_rng(parents + total)
    ids = rng.permutation(np.arange(1, n))
    par, kids = ids[:parents], ids[parents:parents + total]
    src = [np.zeros(parents, np.int64), par[np.arange(total) * parents // total], rng.integers(1, n, 2 * n)]
    dst = [par, kids, rng.integers(1, n, 2 * n)]
    keep = ~np.isin(src[2], par)  # the parents' only out-edges are those to their children
    src[2], dst[2] = src[2][keep], dst[2][keep]
    rp, col, _ = csr_from_edges(n, np.stack([np.concatenate(src), np.concatenate(dst)], 1))
    want = oracle.bfs_queue(rp, col, 0)
    with md.Graph(rp, col) as G:
        for grid in (2, 7, 0):
            for d in (md.DIR_AUTO, md.DIR_PUSH):
                for timing in (0, 1):
                    lv, st = G.bfs(0, direction=d, grid=grid, timing=timing)
                    assert np.array_equal(lv, want), (grid, d, timing)
                    assert st.reached == (want >= 0).sum(), (grid, d, timing)


def test_bfs_edge_cases(oracle):
    with md.Graph(np.array([0, 0], np.uint32), np.array([], np.uint32)) as G:
        lv, st = G.bfs(0)
        assert lv.tolist() == [0] and st.supersteps == 1
    # isolated source in a larger graph, self-loops and duplicates
    rp, col, _ = csr_from_edges(6, [(1, 1), (1, 2), (1, 2), (2, 3), (3, 1)])
    with md.Graph(rp, col) as G:
        assert G.bfs(0)[0].tolist() == [0, -1, -1, -1, -1, -1]
        assert G.bfs(1)[0].tolist() == [-1, 0, 1, 2, -1, -1]
        with pytest.raises(md.MedusaError):
            G.bfs(6)


def test_bfs_er_config(oracle):
    rp, col = wl.er_graph()
    want = oracle.bfs_queue(rp, col, 0)
    sweep, steps = oracle.bfs_sweep(rp, col, 0)
    assert np.array_equal(want, sweep)
    with md.Graph(rp, col) as G:
        for d in _dirs():
            lv, st = G.bfs(0, direction=d)
            assert np.array_equal(lv, want), d
            assert st.supersteps == steps  # one superstep per level plus the empty one
        out = np.zeros_like(want)
        deg = np.diff(rp.astype(np.int64))
        assert G.bfs(0, out=out)[1].edges_traversed == deg[want >= 0].sum()


@pytest.mark.slow
def test_bfs_rmat20(oracle):
    rp, col = wl.rmat_graph()
    with md.Graph(rp, col) as G:
        for s in (0, wl.max_outdeg_vertex(rp), 123457):
            want = oracle.bfs_queue(rp, col, s)
            for d in _dirs():
                lv, _ = G.bfs(s, direction=d)
                assert np.array_equal(lv, want), (s, d)


def test_bfs_device_output_and_repeatability(oracle):
    torch = pytest.importorskip("torch")
    rp, col, _ = random_graph(5000, 40000, 9)
    with md.Graph(rp, col) as G:
        out = torch.empty(5000, dtype=torch.int32, device="cuda")
        G.bfs(17, out=out)
        a = out.cpu().numpy()
        b, _ = G.bfs(17)
        assert np.array_equal(a, b)
        assert np.array_equal(a, oracle.bfs_queue(rp, col, 17))


# ---- SSSP ------------------------------------------------------------------------

@pytest.mark.parametrize("name", sorted(GOLDEN))
def test_sssp_golden(name):
    g = GOLDEN[name]
    rp, col, w = csr_from_edges(g["n"], g["edges"], g["weights"])
    with md.Graph(rp, col, w) as G:
        for s, want in g["sssp"].items():
            want = [U32MAX if x is None else x for x in want]
            for delta in (0, 1, 3, U32MAX):
                d, _ = G.sssp(int(s), delta=delta)
                assert d.tolist() == want, (s, delta)


@pytest.mark.parametrize("seed", range(3))
def test_sssp_random_vs_dijkstra(oracle, seed):
    n = 4000
    rp, col, _ = random_graph(n, 6 * n, seed)
    w = np.random.default_rng(seed).integers(1, 1001, len(col)).astype(np.uint32)
    with md.Graph(rp, col, w) as G:
        for src in (0, 1234):
            want = oracle.sssp_dijkstra(rp, col, w, src)
            for delta in (0, 1, 50, 1000, U32MAX):
                d, _ = G.sssp(src, delta=delta)
                assert np.array_equal(d, want), (src, delta)


def test_sssp_large_weights_and_unweighted_error(oracle):
    rp, col, w = csr_from_edges(4, [(0, 1), (1, 2), (0, 2), (2, 3)], [0x7FFFFFFF, 0x7FFFFFFF, 0xFFFFFF00, 0xF0])
    with md.Graph(rp, col, w) as G:
        d, _ = G.sssp(0)
        assert d.tolist() == oracle.sssp_dijkstra(rp, col, w, 0).tolist()
    with md.Graph(rp, col) as G:
        with pytest.raises(md.MedusaError) as e:
            G.sssp(0)
        assert e.value.code == -4


def test_sssp_lattice_small(oracle):
    rp, col, w = wl.lattice_graph(64, 64, seed=3)
    src = wl.lattice_source(64, 64)
    want = oracle.sssp_dijkstra(rp, col, w, src)
    assert np.array_equal(want, oracle.sssp_bsp(rp, col, w, src)[0])
    with md.Graph(rp, col, w) as G:
        for delta in (0, 1, 500, 5000, U32MAX):
            d, _ = G.sssp(src, delta=delta)
            assert np.array_equal(d, want), delta


@pytest.mark.slow
def test_sssp_lattice_config(oracle, delta_policy):
    """The 1400x1400 lattice at full size: the default width, a fixed width and the learned width
    (the policy trained on smaller lattices; device- and host-driven) all give Dijkstra's
    distances."""
    rp, col, w = wl.lattice_graph()
    src = wl.lattice_source()
    want = oracle.sssp_dijkstra(rp, col, w, src)
    deg = np.diff(rp.astype(np.int64))
    with md.Graph(rp, col, w) as G:
        for delta in (0, 2000):
            d, st = G.sssp(src, delta=delta)
            assert np.array_equal(d, want), delta
            assert st.edges_traversed == deg[want != U32MAX].sum()
        for timing in (0, 1):
            d, st = G.sssp(src, policy=delta_policy, timing=timing)
            assert np.array_equal(d, want), ("learned width", timing)
            assert st.edges_traversed == deg[want != U32MAX].sum()


# ---- multi-source BFS ----------------------------------------------------------------

def test_mbfs_small(oracle):
    rp, col, _ = random_graph(3000, 15000, 5)
    with md.Graph(rp, col) as G:
        for srcs in ([0], [0, 0, 5], list(range(0, 3000, 47))[:64], [2999] * 3):
            want = oracle.mbfs(rp, col, np.array(srcs, np.uint32))
            for d in _dirs():
                out, st = G.mbfs(srcs, direction=d)
                assert np.array_equal(out, want), (len(srcs), d)


@pytest.mark.parametrize("n", [1, 3, 1023, 4095, 4097, 12290])
@pytest.mark.parametrize("k", [1, 8, 9, 16, 17, 32, 33, 64])
def test_mbfs_level_planes(oracle, n, k):
    """Every width of the level planes, vertex counts around the update's tile of 4096 and the 4
    vertices of a finishing lane, levels on both sides of 16 (the fifth plane) and 255 (saturated),
    repeated sources, host and device outputs, both drivers, and a BFS in between whose buffers
    replace the ones the supersteps were captured with."""
    torch = pytest.importorskip("torch")
    rng = np.random.default_rng(n * 64 + k)
    chain = np.arange(min(n - 1, 300))  # levels past 255, the rest at random behind its ends
    src = np.concatenate([chain, rng.integers(n // 2, n, 2 * n)])
    dst = np.concatenate([chain + 1, rng.integers(n // 2, n, 2 * n)])
    rp, col, _ = csr_from_edges(n, np.stack([src, dst], 1))
    srcs = rng.integers(0, n, k).astype(np.uint32)
    srcs[0], srcs[k // 2] = 0, min(n - 1, 284)
    want = oracle.mbfs(rp, col, srcs)
    dev = torch.full((k, n), 7, dtype=torch.uint8, device="cuda")
    with md.Graph(rp, col) as G:
        for opts in ({}, {"timing": 1}, {"direction": md.DIR_PULL, "large_degree": 2}, {}):
            out, st = G.mbfs(srcs, **opts)
            assert np.array_equal(out, want), opts
            G.mbfs(srcs, out=dev, **opts)
            assert np.array_equal(dev.cpu().numpy(), want), opts
            G.bfs(0)
        saturated = any(oracle.bfs_queue(rp, col, int(v)).max() >= 255 for v in np.unique(srcs))
        assert G.mbfs(srcs)[1].reserved[0] == int(saturated)


@pytest.mark.parametrize("n", [70, 4096, 9000])
def test_mbfs_hubs_and_slices(oracle, n):
    """In-degrees on both sides of the 64 of a lane and of the 256 of a hub's round, in windows of
    mixed degrees and vertices without in-edges, pulled by two workgroups (many rounds of slices and
    hubs each) and by the default; pull to push and back by the heuristic."""
    rng = np.random.default_rng(n)
    src = [rng.integers(0, n, 2 * n)]
    dst = [rng.integers(0, n // 2, 2 * n)]
    for d in (63, 64, 65, 255, 256, 257, 1000):
        v = rng.integers(0, n, 12)
        src.append(rng.integers(0, n, 12 * d))
        dst.append(np.repeat(v, d))
    rp, col, _ = csr_from_edges(n, np.stack([np.concatenate(src), np.concatenate(dst)], 1))
    with md.Graph(rp, col) as G:
        for k in (1, 5, 64):
            srcs = rng.integers(0, n, k).astype(np.uint32)
            want = oracle.mbfs(rp, col, srcs)
            for d in _dirs():
                for grid in (2, 0):
                    out, st = G.mbfs(srcs, direction=d, grid=grid, large_degree=8)
                    assert np.array_equal(out, want), (k, d, grid)
                    host = G.mbfs(srcs, direction=d, grid=grid, large_degree=8, timing=1)[1]
                    assert (st.supersteps, st.push_steps, st.pull_steps, st.edges_traversed) == (
                        host.supersteps, host.push_steps, host.pull_steps, host.edges_traversed)


def test_mbfs_widths_in_turn_on_one_handle(oracle):
    """Calls of every plane width in turn on one handle, each width's captured supersteps used again after
    the others, with a width's buffers growing in between."""
    rp, col = wl.rmat_graph(scale=13, edge_factor=8, seed=3)
    rng = np.random.default_rng(5)
    with md.Graph(rp, col) as G:
        for k in (3, 12, 3, 30, 12, 64, 3, 30, 8, 16, 64, 12):
            srcs = rng.integers(0, len(rp) - 1, k).astype(np.uint32)
            assert np.array_equal(G.mbfs(srcs)[0], oracle.mbfs(rp, col, srcs)), k


@pytest.mark.parametrize("where", ["device", "host"])
def test_mbfs_device_time_covers_the_levels(where):
    """device_ms covers the making of the level bytes: without edges, 64 sources differ from 33 by 31 rows
    of levels alone (the masks and planes are as wide), and the GPU cannot write those faster than its
    memory-side cache takes them (17.2 TB/s)."""
    torch = pytest.importorskip("torch")
    n = 1 << 24
    ms = {}
    with md.Graph(np.zeros(n + 1, np.uint32), np.zeros(0, np.uint32)) as G:
        for k in (33, 64):
            out = torch.empty((k, n), dtype=torch.uint8, device="cuda") if where == "device" else np.empty((k, n), np.uint8)
            srcs = np.arange(k, dtype=np.uint32)
            ms[k] = min(G.mbfs(srcs, out=out)[1].device_ms for _ in range(5))
    print(f"[mbfs levels {where}] 33 sources {ms[33]:.4f} ms, 64 sources {ms[64]:.4f} ms", flush=True)
    assert ms[64] - ms[33] >= 31 * n / 17.2e12 * 1e3


def test_mbfs_rows_in_pieces():
    """A host output of more bytes than the row buffer holds: no vertex but the sources is reached."""
    n, k = 5_000_001, 64
    with md.Graph(np.zeros(n + 1, np.uint32), np.zeros(0, np.uint32)) as G:
        srcs = (np.arange(k) * 70_001).astype(np.uint32)
        out, _ = G.mbfs(srcs)
    assert np.array_equal(out[np.arange(k), srcs], np.zeros(k))
    out[np.arange(k), srcs] = 255
    assert (out == 255).all()


def test_mbfs_matches_plain_bfs(oracle):
    rp, col = wl.er_graph(8192, 65536, seed=1)
    srcs = wl.mbfs_sources(rp, 64, seed=4)
    with md.Graph(rp, col) as G:
        out, st = G.mbfs(srcs)
        for i, s in enumerate(srcs):
            lv, _ = G.bfs(int(s))
            assert np.array_equal(out[i], np.where(lv < 0, 255, lv).astype(np.uint8))


@pytest.mark.slow
def test_mbfs_rmat20_config(oracle, mbfs_policy):
    """RMAT-20 with 64 sources at full size: the heuristic engine, the learned direction (policy
    trained on smaller RMAT graphs) and the autotuned launch shape (with and without the policy)
    all give the oracle's per-source levels."""
    rp, col = wl.rmat_graph()
    srcs = wl.mbfs_sources(rp, 64, seed=4)
    want = oracle.mbfs(rp, col, srcs)
    deg = np.diff(rp.astype(np.int64))
    reached = sum(deg[want[i] != 255].sum() for i in range(len(srcs)))
    with md.Graph(rp, col) as G:
        out, st = G.mbfs(srcs)
        assert np.array_equal(out, want)
        assert st.edges_traversed == reached
        out, st = G.mbfs(srcs, policy=mbfs_policy)
        assert np.array_equal(out, want), "learned direction"
        t = G.autotune(md.TUNE_MBFS, srcs, reps=1)
        assert t.large_degree > 0 and t.grid > 0
        for pol in (None, mbfs_policy):
            out, st = G.mbfs(srcs, policy=pol)
            assert np.array_equal(out, want), ("autotuned", pol is not None)
            assert st.edges_traversed == reached


@pytest.mark.parametrize("layers", [0, 5, 7, 8, 9, 17, 40])
def test_bfs_first_run_of_a_handle(oracle, layers):
    """The first run of a handle launches its kernels one by one and may need replays after them: wide
    layers of vertices, too many edges for one workgroup, whose count is around the eight slots of a
    first sequence; later runs on the handle are shorter, equal and longer."""
    wide = 6000
    n = 1 + layers * wide
    at = np.arange(wide)
    edges = [np.stack([np.zeros(wide, np.int64), 1 + at], 1)] if layers else [np.zeros((0, 2), np.int64)]
    for k in range(1, layers):
        for step in (0, 1, 77, 2500):
            edges.append(np.stack([1 + (k - 1) * wide + at, 1 + k * wide + (at + step) % wide], 1))
    rp, col, _ = csr_from_edges(n, np.concatenate(edges))
    for first, d in ((0, md.DIR_AUTO), (0, md.DIR_PUSH), (1 + (layers // 2) * wide if layers > 1 else 0, md.DIR_AUTO)):
        with md.Graph(rp, col) as G:
            for s in (first, 0, n - 1, 0, first):
                got, st = G.bfs(s, direction=d)
                want = oracle.bfs_queue(rp, col, s)
                assert np.array_equal(got, want), (first, s)
                assert st.reached == int((want >= 0).sum()), (first, s)


@pytest.mark.parametrize("n", [1, 1023, 1025, 9000])
def test_sssp_runs_of_different_lengths(oracle, n):
    """Runs on one handle whose slot counts differ by more than a replay (a path of `n` vertices
    from its start, its middle and its end), so the first replay is too short, too long and
    right; between them a multi-source BFS, whose level planes replace the stamps; host and device
    outputs, reached counts on both sides of a closing workgroup's 1024 vertices."""
    torch = pytest.importorskip("torch")
    rp, col, _ = csr_from_edges(n, np.stack([np.arange(n - 1), np.arange(1, n)], 1))
    w = np.random.default_rng(n).integers(1, 1001, len(col)).astype(np.uint32)
    dev = torch.empty(n, dtype=torch.int32, device="cuda")
    with md.Graph(rp, col, w) as G:
        for s in (0, n - 1, n // 2, 0, 0, n - 1):
            want = oracle.sssp_dijkstra(rp, col, w, s)
            for opts in ({}, {"local_rounds": 0xFFFFFFFF, "delta": 100000}, {"far_limit": 1}, {"timing": 1}):
                if n > 1025 and "delta" not in opts and "timing" in opts:
                    continue  # thousands of host-driven supersteps
                got, st = G.sssp(s, **opts)
                assert np.array_equal(got, want), (s, opts)
                assert (st.reached, st.edges_traversed) == (n - s, n - 1 - s), (s, opts)
                st = G.sssp(s, out=dev, **opts)[1]
                assert np.array_equal(dev.cpu().numpy().view(np.uint32), want), (s, opts)
                assert (st.reached, st.edges_traversed) == (n - s, n - 1 - s), (s, opts)
            G.mbfs(np.arange(min(n, 64), dtype=np.uint32))


@pytest.mark.parametrize("far_limit", [1, 7, 64])
def test_sssp_far_queue_limit_rebuilds(oracle, far_limit):
    """A far queue capped far below its need is rebuilt from the distances at every split;
    distances stay exact on both drivers, for every bucket width, and with local rounds (whose
    split slot relaxes the vertices it moves, also after a rescan) on a random graph and a
    lattice."""
    rp, col, _ = random_graph(6000, 36000, 31)
    w = np.random.default_rng(31).integers(1, 1001, len(col)).astype(np.uint32)
    lrp, lcol, lw = wl.lattice_graph(60, 70, seed=13)
    for rp, col, w, src in ((rp, col, w, 7), (lrp, lcol, lw, wl.lattice_source(60, 70))):
        want = oracle.sssp_dijkstra(rp, col, w, src)
        with md.Graph(rp, col, w) as G:
            for lr in (0, 32, U32MAX):
                for delta in (0, 50, 400):
                    for timing in (0, 1):
                        d, _ = G.sssp(src, delta=delta, far_limit=far_limit, timing=timing, local_rounds=lr)
                        assert np.array_equal(d, want), (lr, delta, timing)


def test_sssp_zero_weights_duplicates_and_self_loops(oracle):
    """The reference draws weights from rand32() % 1000, so 0 occurs; duplicates and self
    loops are kept."""
    rng = np.random.default_rng(8)
    n, m = 4000, 30000
    src = rng.integers(0, n, m)
    dst = rng.integers(0, n, m)
    src[:500] = dst[:500]                         # self loops
    src[500:1500] = src[1500:2500]                # duplicate arcs
    dst[500:1500] = dst[1500:2500]
    w = rng.integers(0, 1000, m).astype(np.uint32)
    w[::7] = 0
    rp, col, wc = csr_from_edges(n, np.stack([src, dst], 1), w)
    want = oracle.sssp_dijkstra(rp, col, wc, 11)
    with md.Graph(rp, col, wc) as G:
        for delta in (0, 1, 37, 0xFFFFFFFF):
            for timing in (0, 1):
                d, _ = G.sssp(11, delta=delta, timing=timing)
                assert np.array_equal(d, want), (delta, timing)


@pytest.mark.parametrize("case", ["lattice", "random", "zero_weights", "hubs"])
def test_sssp_local_rounds(oracle, case):
    """Workgroups relaxing the vertices they lowered themselves for up to 1, 3 or 64 further
    rounds, or none, in both loop drivers: distances stay Dijkstra's.  The cases cover a
    thin frontier (lattice), a dense random graph, zero weights with duplicate arcs and self
    loops (offers that tie), and hubs wider than one near-queue slice (never kept locally)."""
    rng = np.random.default_rng(21)
    if case == "lattice":
        rp, col, w = wl.lattice_graph(120, 150, seed=9)
        src = wl.lattice_source(120, 150)
    elif case == "random":
        rp, col, _ = random_graph(6000, 60000, 21)
        w = rng.integers(1, 1001, len(col)).astype(np.uint32)
        src = 3
    elif case == "zero_weights":
        n, m = 3000, 9000
        e = rng.integers(0, n, (m, 2))
        e[:300, 0] = e[:300, 1]
        e[300:900] = e[900:1500]
        w = rng.integers(0, 20, m).astype(np.uint32)
        w[::3] = 0
        rp, col, w = csr_from_edges(n, e, w)
        src = 5
    else:
        n = 20000
        hub = np.stack([np.zeros(3000, np.int64), rng.integers(1, n, 3000)], 1)
        rest = np.stack([rng.integers(0, n, 40000), rng.integers(0, n, 40000)], 1)
        rp, col, _ = csr_from_edges(n, np.concatenate([hub, rest]))
        w = rng.integers(1, 1001, len(col)).astype(np.uint32)
        src = 0
    want = oracle.sssp_dijkstra(rp, col, w, src)
    with md.Graph(rp, col, w) as G:
        for lr in (1, 3, 64, U32MAX, 0):
            for delta in ((0, 300, U32MAX) if case == "lattice" else (0, 1, 300, U32MAX)):
                for timing in (0, 1):
                    d, _ = G.sssp(src, delta=delta, timing=timing, local_rounds=lr)
                    assert np.array_equal(d, want), (lr, delta, timing)
        with pytest.raises(md.MedusaError):
            G.sssp(src, local_rounds=65)


@pytest.mark.parametrize("deg", [1, 7, 8, 63, 128, 129])
def test_sssp_wave_rounds(oracle, deg):
    """Local rounds at the edges of the wave rounds: out-degrees up to a record's 7 edges, beyond it,
    the largest (128) and one past it (block-wide rounds instead), zero and large weights, a source
    whose neighbours all have that degree (rings that overflow into the near queue), few and many
    rounds, and a far queue that overflows; both drivers, distances equal Dijkstra's."""
    rng = np.random.default_rng(deg)
    n = 6000
    src = [np.zeros(deg, np.int64), np.repeat(np.arange(1, 600), deg), rng.integers(600, n, 3 * n)]
    dst = [np.arange(1, deg + 1), rng.integers(0, n, 599 * deg), rng.integers(0, n, 3 * n)]
    rp, col, _ = csr_from_edges(n, np.stack([np.concatenate(src), np.concatenate(dst)], 1))
    w = rng.integers(0, 1001, len(col)).astype(np.uint32)
    w[rng.integers(0, len(w), 20)] = 0xF0000000  # sums past 32 bits
    want = oracle.sssp_dijkstra(rp, col, w, 0)
    with md.Graph(rp, col, w) as G:
        for rounds in (1, 2, 64):
            for timing, delta, far in ((0, 0, 0), (1, 300, 0), (0, 50, 40), (0, 0xFFFFFFFF, 0)):
                d, st = G.sssp(0, local_rounds=rounds, timing=timing, delta=delta, far_limit=far)
                assert np.array_equal(d, want), (rounds, timing, delta, far)


def test_sssp_wide_frontiers_with_local_rounds(oracle):
    """A uniform graph without hubs whose frontiers and far queues pass the 131,072 entries up to which
    the wave rounds run, with supersteps on both sides of that, rebuilt far queues among them: distances
    equal Dijkstra's in both drivers."""
    n = 1 << 20
    rp, col = wl.er_graph(n, 4 * n, seed=11)
    w = np.random.default_rng(11).integers(0, 1001, len(col)).astype(np.uint32)
    src = wl.max_outdeg_vertex(rp)
    want = oracle.sssp_dijkstra(rp, col, w, src)
    with md.Graph(rp, col, w) as G:
        for opts in ({}, {"delta": 0xFFFFFFFF}, {"delta": 500}, {"far_limit": 1000}, {"local_rounds": 2},
                     {"timing": 1}, {"timing": 1, "delta": 500}):
            d, st = G.sssp(src, **opts)
            assert np.array_equal(d, want), opts
            assert st.reached == (want != 0xFFFFFFFF).sum(), opts
        G.sssp(src, delta=500, trace=1)
        assert G.trace()[:, 1].max() > 131_072  # far entries at a split


def test_sssp_local_rounds_on_wide_frontiers_cost_little():
    """On a uniform graph of 2^22 vertices and mean out-degree 4 most edges are relaxed in frontiers of a
    million vertices, where local rounds only repeat work: the default run may not take more than 1.25
    times one without rounds (1.05 measured; 2.05 with rounds in every superstep).  The same width and
    the same distances."""
    n = 1 << 22
    rp, col = wl.er_graph(n, 4 * n, seed=1)
    w = np.random.default_rng(6).integers(1, 1001, len(col)).astype(np.uint32)
    src = wl.max_outdeg_vertex(rp)
    with md.Graph(rp, col, w) as G:
        ms, dist = {}, {}
        for rounds in (0, 0xFFFFFFFF):
            dist[rounds], _ = G.sssp(src, local_rounds=rounds, delta=4000)
            ms[rounds] = min(G.sssp(src, local_rounds=rounds, delta=4000)[1].device_ms for _ in range(5))
    print(f"[sssp er 2^22] default rounds {ms[0]:.3f} ms, none {ms[0xFFFFFFFF]:.3f} ms", flush=True)
    assert np.array_equal(dist[0], dist[0xFFFFFFFF])
    assert ms[0] <= 1.25 * ms[0xFFFFFFFF]


def test_sssp_sparse_power_law_local_rounds(oracle):
    """A sparse skewed graph (Chung-Lu, mean out-degree about 2, so local rounds are on by
    default) whose hubs span many near-queue slices and are never kept locally, and whose
    frontier grows past the queue length up to which the rounds run: distances stay Dijkstra's
    with the default rounds, with none, and with the widest bucket."""
    rp, col = wl.chung_lu_graph(n=200_000, m=420_000, seed=17, max_degree=20_000)
    w = wl.weighted(rp, col, seed=17)
    src = wl.max_outdeg_vertex(rp)
    want = oracle.sssp_dijkstra(rp, col, w, src)
    with md.Graph(rp, col, w) as G:
        for kw in ({}, {"local_rounds": U32MAX}, {"delta": U32MAX}, {"local_rounds": 64, "delta": 300},
                   {"timing": 1}):
            d, st = G.sssp(src, **kw)
            assert np.array_equal(d, want), kw
            assert st.reached == int((want != U32MAX).sum())


def test_sssp_wide_bucket_split_moves_most_vertices(oracle):
    """A sparse graph of more than 2^20 vertices with local rounds on and a bucket so wide that
    the first split moves almost every vertex below the threshold: the split appends the
    vertices it moves and its local rounds append the ones they lower again, so one slot may
    append a vertex twice.  Distances stay Dijkstra's for several wide widths."""
    rp, col = wl.chung_lu_graph(n=1_200_000, m=2_500_000, seed=29, max_degree=5_000)
    w = wl.weighted(rp, col, seed=29)
    src = wl.max_outdeg_vertex(rp)
    want = oracle.sssp_dijkstra(rp, col, w, src)
    with md.Graph(rp, col, w) as G:
        for delta in (20_000, 200_000, 1 << 30):
            d, st = G.sssp(src, delta=delta, local_rounds=64)
            assert np.array_equal(d, want), delta
            assert st.reached == int((want != U32MAX).sum())


def test_sssp_hub_source_slices(oracle):
    """A source whose out-degree spans many near-queue slices, plus hubs inside the graph."""
    rng = np.random.default_rng(12)
    n = 50000
    hub = np.stack([np.zeros(20000, np.int64), rng.integers(1, n, 20000)], 1)
    hubs2 = np.stack([np.repeat(rng.integers(0, n, 8), 3000), rng.integers(0, n, 24000)], 1)
    rest = rng.integers(0, n, (150000, 2))
    rp, col, _ = csr_from_edges(n, np.concatenate([hub, hubs2, rest]))
    w = rng.integers(1, 1001, len(col)).astype(np.uint32)
    want = oracle.sssp_dijkstra(rp, col, w, 0)
    with md.Graph(rp, col, w) as G:
        for delta in (0, 100, 0xFFFFFFFF):
            for timing in (0, 1):
                d, _ = G.sssp(0, delta=delta, timing=timing)
                assert np.array_equal(d, want), (delta, timing)


@pytest.mark.parametrize("case", ["n1_empty", "n1_selfloop", "n2_empty", "n3_chain"])
def test_tiny_graphs_every_engine(oracle, case):
    """The smallest inputs through every engine and driver: one vertex with and without a
    self loop, two isolated vertices, a 3-chain."""
    edges, n = {"n1_empty": ([], 1), "n1_selfloop": ([(0, 0)], 1), "n2_empty": ([], 2),
                "n3_chain": ([(0, 1), (1, 2)], 3)}[case]
    rp, col, w = csr_from_edges(n, np.array(edges, np.int64).reshape(-1, 2), [7] * len(edges))
    w = np.asarray(w if w is not None else [], np.uint32)
    with md.Graph(rp, col, w) as G:
        for src in range(n):
            want = oracle.bfs_queue(rp, col, src)
            for d in _dirs():
                for timing in (0, 1):
                    assert np.array_equal(G.bfs(src, direction=d, timing=timing)[0], want)
            dwant = oracle.sssp_dijkstra(rp, col, w, src)
            for timing in (0, 1):
                assert np.array_equal(G.sssp(src, timing=timing)[0], dwant)
            srcs = np.array([src, src], np.uint32)
            mwant = oracle.mbfs(rp, col, srcs)
            for timing in (0, 1):
                assert np.array_equal(G.mbfs(srcs, timing=timing)[0], mwant)
        r, _ = G.pagerank(0.85, 4)
        assert np.array_equal(r.view(np.uint32), oracle.pagerank_f32(rp, col, 0.85, 4).view(np.uint32))


def test_one_handle_from_several_threads(oracle):
    """Calls on one handle from several host threads are serialised by the handle's lock:
    every thread gets its own source's exact levels, distances and ranks."""
    import threading
    n = 20000
    rp, col, _ = random_graph(n, 8 * n, 21)
    w = np.random.default_rng(21).integers(1, 1001, len(col)).astype(np.uint32)
    sources = [0, 17, 999, 4321, 12345, 19999]
    want_lv = {s: oracle.bfs_queue(rp, col, s) for s in sources}
    want_d = {s: oracle.sssp_dijkstra(rp, col, w, s) for s in sources}
    errors = []
    with md.Graph(rp, col, w) as G:
        want_pr = G.pagerank(steps=10)[0]

        def work(s):
            try:
                for _ in range(3):
                    lv, _ = G.bfs(s)
                    d, _ = G.sssp(s)
                    pr, _ = G.pagerank(steps=10)
                    mb, _ = G.mbfs([s, (s + 1) % n])
                    if not (np.array_equal(lv, want_lv[s]) and np.array_equal(d, want_d[s])
                            and np.array_equal(pr, want_pr) and np.array_equal(mb[0], np.where(
                                want_lv[s] < 0, 0xFF, want_lv[s]).astype(np.uint8))):
                        errors.append(s)
            except Exception as e:  # reported below
                errors.append((s, repr(e)))

        threads = [threading.Thread(target=work, args=(s,)) for s in sources]
        for t in threads:
            t.start()
        for t in threads:
            t.join(timeout=120)
        assert not any(t.is_alive() for t in threads)
    assert errors == []


@pytest.mark.slow
def test_rmat22_four_times_the_configs(oracle):
    """RMAT scale 22 (4,194,304 vertices, 67,108,864 arcs), four times the RMAT-20 configs:
    BFS, SSSP and 8-source MBFS stay bit-exact against the oracle."""
    rp, col = wl.rmat_graph(scale=22, edge_factor=16, seed=22)
    w = wl.weighted(rp, col, seed=23)
    src = wl.max_outdeg_vertex(rp)
    want = oracle.bfs_queue(rp, col, src)
    with md.Graph(rp, col, w) as G:
        for d in _dirs():
            lv, _ = G.bfs(src, direction=d)
            assert np.array_equal(lv, want), d
        dist, _ = G.sssp(src)
        assert np.array_equal(dist, oracle.sssp_dijkstra(rp, col, w, src))
        srcs = wl.mbfs_sources(rp, 8, seed=24)
        out, _ = G.mbfs(srcs)
        assert np.array_equal(out, oracle.mbfs(rp, col, srcs))
