"""Solves inside one workgroup with the vertex state in LDS: sizes at the edges of what fits, of the
hub handling and of the hand-over to the grid-wide kernels, against Dinic, certified."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def arcs_graph(mf, n, parts, s, t, seed, top=1000):
    u = np.concatenate([np.broadcast_to(a, np.broadcast(a, b).shape).ravel() for a, b in parts])
    v = np.concatenate([np.broadcast_to(b, np.broadcast(a, b).shape).ravel() for a, b in parts])
    cap = np.random.default_rng(seed).integers(1, top + 1, size=u.size)
    return mf.Graph.from_arcs(n, u, v, cap, s, t)


def chains(mf, width, length, seed):
    """width chains of length vertices into t; s feeds every vertex, so the first worklist holds
    all of them while no BFS frontier is wider than width."""
    n = width * length + 2
    x = 2 + np.arange(width * length).reshape(length, width)
    parts = [(np.array([0]), x.ravel()), (x[:-1], x[1:]), (x[-1], np.array([1]))]
    parts.append((x[1:], np.roll(x[:-1], 1, axis=1)))  # and back, to the chain beside it
    return arcs_graph(mf, n, parts, 0, 1, seed)


def dense_layers(mf, k, layers, seed):
    """Complete bipartite arcs between layers of k vertices: every inner vertex has 2k slots."""
    x = 2 + np.arange(k * layers).reshape(layers, k)
    parts = [(np.array([0]), x[0]), (x[-1], np.array([1]))]
    parts += [(x[i][:, None], x[i + 1][None, :]) for i in range(layers - 1)]
    return arcs_graph(mf, k * layers + 2, parts, 0, 1, seed)


def check(mf, orc, ctx, g):
    value = orc.dinic_maxflow(g)
    for g2 in (g, mf.Graph.from_arcs(g.n, g.dst, g.tails(), g.cap, g.t, g.s)):
        # one instance to a CU; in more than there are CUs, with small ones beside
        assert ctx.batch_solve([g2])[0].tolist() == [value]
    tiny = chains(mf, 3, 4, seed=1)
    values = ctx.batch_solve([tiny] * 300 + [g])[0]
    assert values[300] == value and set(values[:300]) == {orc.dinic_maxflow(tiny)}
    tails = g.tails()
    for layout in (mf.LAYOUT_BCSR, mf.LAYOUT_BCSR2, mf.LAYOUT_RCSR):
        dg = ctx.upload(g, layout)
        try:
            for algo in (mf.ALGO_VC, mf.ALGO_TC):  # the second restores the residuals first
                r = dg.solve(algo)
                assert r.value == value and r.pushes > 0
                assert orc.certify(g, dg.read_flow(return_excess=False), value,
                                   preflow=True)[0] == "ok"
                assert orc.certify(g, dg.read_flow(), value) == ("ok", value)
                side = dg.read_cut()
                assert g.cap[(side[tails] == 0) & (side[g.dst] == 1)].sum(dtype=np.int64) == value
        finally:
            dg.close()


@pytest.mark.parametrize("width,length", [
    (63, 17), (64, 16), (1, 300),  # bitmap words, single-vertex frontiers
    (1500, 15),    # excesses in LDS, worklists longer than their lists
    (1300, 19),    # about as many vertices as fit with their excesses
    (1301, 20),    # more: excesses in global memory
    (1500, 41),    # nearly as many as fit at all
    (1600, 42),    # too many: on the grid, its global relabels in one workgroup
    (9000, 8),     # their frontiers handed to grid-wide levels and back
    (20000, 4),    # frontiers longer than the LDS lists
    (2048, 13), (2049, 13),  # the widest frontiers that stay with excesses in global memory, and wider
    (2800, 8), (2801, 8), (4000, 2),  # and in LDS; two wide frontiers stay
])
def test_chains(mf, orc, ctx, width, length):
    check(mf, orc, ctx, chains(mf, width, length, seed=width + length))


@pytest.mark.parametrize("k,layers", [
    (47, 6), (48, 6), (49, 6),  # 94, 96 and 98 slots: the last are hubs
    (130, 4),                   # hubs of one and a half rounds of a wave
    (290, 3),                   # more hubs at a time than wait in LDS
])
def test_hubs(mf, orc, ctx, k, layers):
    check(mf, orc, ctx, dense_layers(mf, k, layers, seed=k))


@pytest.mark.parametrize("frontier", [1, 2, 300])
@pytest.mark.parametrize("direction", [0, 1, 2])
def test_relabel_takeover(mf, orc, ctx, frontier, direction):
    # the one-workgroup search takes over behind grid-wide levels, top-down and bottom-up, at the
    # smallest frontier, at most of them and where only some fit
    for g in (chains(mf, 200, 420, seed=5), mf.gen_bipartite(40000, 41000, 6.0, 7),
              mf.gen_rmat(14, 16, seed=3)):
        value = orc.dinic_maxflow(g)
        dg = ctx.upload(g, mf.LAYOUT_BCSR)
        try:
            r = dg.solve(mf.ALGO_VC, bfs_block_frontier=frontier, bfs_direction=direction)
            assert r.value == value and 0 <= r.bfs_grid_levels <= r.bfs_levels
            assert orc.certify(g, dg.read_flow(return_excess=False), value,
                               preflow=True)[0] == "ok"
        finally:
            dg.close()


def test_threads_of_different_sizes(mf, orc):
    # graphs that ask for little and for nearly all LDS, solved side by side, a context each
    from concurrent.futures import ThreadPoolExecutor

    graphs = [chains(mf, 3, 4, 1), chains(mf, 1300, 19, 2), chains(mf, 1500, 41, 3),
              chains(mf, 2000, 60, 4)]
    want = [orc.dinic_maxflow(g) for g in graphs]

    def solve(g):
        ctx = mf.Context(0)
        try:
            return [ctx.solve(g).value for _ in range(10)]
        finally:
            ctx.close()

    with ThreadPoolExecutor(len(graphs)) as pool:
        assert list(pool.map(solve, graphs)) == [[v] * 10 for v in want]


@pytest.mark.parametrize("coop", [0, 1])
@pytest.mark.parametrize("width,length", [
    (2801, 8),    # abandoned at the third wide frontier
    (2049, 13),   # at the first one, level 1
    (9000, 6),    # a frontier longer than the LDS list
    (0, 0),       # a matching: the sink's neighbours
])
def test_grid_goes_on_from_an_abandoned_search(mf, orc, ctx, width, length, coop):
    g = chains(mf, width, length, seed=9) if width else mf.gen_bipartite(17000, 16500, 8.0, seed=9)
    value = orc.dinic_maxflow(g)
    for layout in (mf.LAYOUT_BCSR, mf.LAYOUT_BCSR2, mf.LAYOUT_RCSR):
        dg = ctx.upload(g, layout)
        try:
            for algo in (mf.ALGO_VC, mf.ALGO_TC):
                r = dg.solve(algo, bfs_cooperative=coop)
                assert r.value == value and r.bfs_levels > 0
                assert coop or r.bfs_grid_levels > 0  # (else its frontier's own level at least)
                assert orc.certify(g, dg.read_flow(return_excess=False), value,
                                   preflow=True)[0] == "ok"
        finally:
            dg.close()
    assert ctx.solve_noalloc(g, mf.ALGO_VC, bfs_cooperative=coop).value == value


@pytest.mark.parametrize("left,right,both_lines", [
    # the sink takes less: frontiers up to 9,400 stay, those of left vertices (but for a few without arcs)
    (9400, 9200, True), (9430, 9200, False),
    (9600, 9550, True),                           # hardly less
    (11400, 11800, True), (11400, 11801, False),  # more: up to 11,800
])
def test_wide_frontiers_by_layout(mf, orc, ctx, left, right, both_lines):
    # matchings in one workgroup: any width on BCSR, what RCSR and BCSR2 read a slot's two lines for
    g = mf.gen_bipartite(left, right, 8.0, seed=left)
    value = orc.dinic_maxflow(g)
    for layout in (mf.LAYOUT_BCSR, mf.LAYOUT_BCSR2, mf.LAYOUT_RCSR):
        dg = ctx.upload(g, layout)
        try:
            r = dg.solve(mf.ALGO_VC)
            assert r.value == value
            assert (r.bfs_grid_levels == 0) == (layout == mf.LAYOUT_BCSR or both_lines)
            assert orc.certify(g, dg.read_flow(return_excess=False), value,
                               preflow=True)[0] == "ok"
        finally:
            dg.close()


def test_graphs_destroyed_by_another_thread(mf, orc):
    # a garbage collector's thread closes graphs of a context that is solving, launches being captured
    import threading

    ctx = mf.Context(0)
    g = mf.gen_rmat(13, 8, seed=2)
    value = orc.dinic_maxflow(g)
    old = [ctx.upload(mf.gen_washington_rlg(8, 8, 100, i), mf.LAYOUT_BCSR) for i in range(400)]
    done = threading.Event()

    def collect():
        while old and not done.is_set():
            old.pop().close()
            done.wait(0.0002)

    thread = threading.Thread(target=collect)
    thread.start()
    try:
        for cycles in range(6, 66, 6):
            dg = ctx.upload(g, mf.LAYOUT_BCSR)
            assert dg.solve(mf.ALGO_VC, cycle_graphs=1, cycles_per_relabel=cycles).value == value
            dg.close()
    finally:
        done.set()
        thread.join()
        for dg in old:
            dg.close()
        ctx.close()
