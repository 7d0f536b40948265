"""Paths that small graphs and batches no longer take by themselves: the grid-wide cycles with their tile
widths and forwarding, the general batch kernel, and the one-workgroup solvers' hubs where the excesses are
in global memory.  Against Dinic, certified."""
import numpy as np
import pytest

from conftest import generated_graph
from test_one_workgroup_gpu import chains
from test_solver_gpu import LANE_PRESETS

pytestmark = pytest.mark.gpu


def solve_on_grid(mf, orc, ctx, g, algo, value, **options):
    """A solve whose cycles are timed is one on the grid."""
    dg = ctx.upload(g, mf.LAYOUT_BCSR)
    try:
        r = dg.solve(algo, profile_kernels=4, **options)
        assert r.value == value and r.profiled_launches > 0
        assert orc.certify(g, dg.read_flow(return_excess=False), value, preflow=True)[0] == "ok"
        assert orc.certify(g, dg.read_flow(), value) == ("ok", value)
    finally:
        dg.close()


@pytest.mark.parametrize("lanes", LANE_PRESETS)
@pytest.mark.parametrize("name", ["genrmf16_s1", "bip_3000_2000_s9"])
def test_class_lanes_on_the_grid(mf, orc, ctx, golden, name, lanes):
    g, value = generated_graph(mf, golden, name)
    solve_on_grid(mf, orc, ctx, g, mf.ALGO_VC, value, class_lanes=lanes)


@pytest.mark.parametrize("hops", [-1, 1, 64])
@pytest.mark.parametrize("name", ["rlg32_s7", "genrmf16_s1", "bip_3000_2000_s9"])
def test_push_forwarding_on_the_grid(mf, orc, ctx, golden, name, hops):
    g, value = generated_graph(mf, golden, name)
    for algo in (mf.ALGO_TC, mf.ALGO_VC):
        solve_on_grid(mf, orc, ctx, g, algo, value, forward_hops=hops)


@pytest.mark.parametrize("algo", [0, 1])
@pytest.mark.parametrize("hops", [-1, 2, 32])
def test_batch_of_more_vertices_than_the_lds_kernels_take(mf, orc, ctx, golden, algo, hops):
    # 2^19 + 2 vertices go to the general batch kernel, 2^19 - 2 and the small ones stay
    rng = np.random.default_rng(4)
    graphs = []
    for width in (131072, 131071):
        x = 2 + np.arange(4 * width).reshape(4, width)
        u = np.concatenate([np.zeros(width, np.int64), x[0], x[1], x[2], x[3]])
        v = np.concatenate([x[0], x[1], x[2], x[3], np.ones(width, np.int64)])
        graphs.append(mf.Graph.from_arcs(2 + 4 * width, u, v, rng.integers(1, 100, u.size), 0, 1))
    assert graphs[0].n == 2**19 + 2 and graphs[1].n == 2**19 - 2
    small = [generated_graph(mf, golden, n) for n in ("rlg16_s3", "genrmf8_s7", "rmat10_s5")]
    values = [orc.dinic_maxflow(g) for g in graphs] + [v for _, v in small]
    graphs += [g for g, _ in small]
    assert ctx.batch_solve(graphs, batch_algo=algo, forward_hops=hops)[0].tolist() == values


def hubs_over_chains(mf, width, length, slots, seed):
    """Chains (see there) with a hub every second level: arcs from random vertices of that level and the
    next, and to half as many of later levels; hubs have `slots` residual slots."""
    base = chains(mf, width, length, seed)
    rng = np.random.default_rng(seed)
    x = 2 + np.arange(width * length).reshape(length, width)
    u, v = [base.tails()], [base.dst]
    n = base.n
    into = slots * 2 // 3
    for level in range(0, length - 8, 2):
        near = x[level:level + 2].ravel()
        far = x[level + 3:level + 8].ravel()
        u += [rng.choice(near, into, replace=False), np.full(slots - into, n)]
        v += [np.full(into, n), rng.choice(far, slots - into, replace=False)]
        n += 1
    u, v = np.concatenate(u), np.concatenate(v)
    cap = np.concatenate([base.cap, rng.integers(1, 1000, u.size - base.m)])
    return mf.Graph.from_arcs(n, u, v, cap, 0, 1)


@pytest.mark.parametrize("slots", [96, 97, 250])
@pytest.mark.parametrize("width,length", [(300, 100), (650, 108)])
def test_hubs_with_excesses_in_global_memory(mf, orc, ctx, width, length, slots):
    # 30,000 vertices: heights in LDS; 70,000: batched, both in global memory
    g = hubs_over_chains(mf, width, length, slots, seed=slots)
    value = orc.dinic_maxflow(g)
    tiny = chains(mf, 3, 4, seed=1)
    assert ctx.batch_solve([g])[0].tolist() == [value]
    values = ctx.batch_solve([tiny] * 300 + [g])[0]
    assert values[300] == value and set(values[:300]) == {orc.dinic_maxflow(tiny)}
    for layout in (mf.LAYOUT_BCSR, mf.LAYOUT_BCSR2, mf.LAYOUT_RCSR):
        dg = ctx.upload(g, layout)
        try:
            for _ in range(2):
                r = dg.solve(mf.ALGO_VC)
                assert r.value == value
                assert (r.bfs_grid_levels == 0) or width > 300
                assert orc.certify(g, dg.read_flow(return_excess=False), value,
                                   preflow=True)[0] == "ok"
        finally:
            dg.close()


def test_autotune_leaves_out_what_has_no_effect(mf, orc, ctx):
    inert = ("tile_lanes", "class_lanes", "forward_hops", "batch_algo", "bfs_block_frontier",
             "bfs_cooperative")
    start = mf.options(class_lanes=[4, 8, 16, 64, 256], forward_hops=8,
                       bfs_block_frontier=1024).to_dict()
    g = chains(mf, 40, 60, seed=2)
    best, _, trials = ctx.batch_autotune([g] * 8 + [chains(mf, 20, 30, seed=3)] * 8, sample=8, **start)
    assert {k: best[k] for k in inert} == {k: start[k] for k in inert} and trials >= 18
    dg = ctx.upload(g, mf.LAYOUT_BCSR)
    try:
        best, _, trials = dg.autotune(mf.ALGO_VC, **start)
        assert best["cycle_graphs"] or {k: best[k] for k in inert} == {k: start[k] for k in inert}
        assert dg.solve(mf.ALGO_VC, **best).value == orc.dinic_maxflow(g)
    finally:
        dg.close()
