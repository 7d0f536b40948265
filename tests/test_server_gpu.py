"""Served requests at the edges of what the serving kernel takes, and beside what runs alone."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOP = 2**31 - 1


def serve(srv, ids, seconds=60):
    """Values by request id."""
    left, t0 = set(ids), time.time()
    while left and time.time() - t0 < seconds:
        srv.progress(wait=True)
        left.difference_update(srv.completed())
    assert not left
    return [srv.result(i)[0] for i in ids]


@pytest.mark.parametrize("into_t,value", [(5, 10), (TOP // 2, TOP - 1), (TOP, None)])
def test_more_than_an_int32_out_of_the_source(mf, ctx, into_t, value):
    # two paths s -> a -> t, s -> b -> t: excesses are 32-bit, so the request is solved from t if
    # the capacity into t fits, and refused if neither does
    g = mf.Graph.from_arcs(4, np.array([0, 0, 1, 2]), np.array([1, 2, 3, 3]),
                           np.array([TOP, TOP, into_t, into_t]), 0, 3)
    srv = mf.Server(ctx, hbm_budget_bytes=16 << 20, max_inflight_launches=1)
    try:
        if value is None:
            with pytest.raises(mf.MFError) as ei:
                srv.submit(g)
            assert ei.value.name == "MF_ERR_OVERFLOW"
        else:
            assert serve(srv, [srv.submit(g)]) == [value]
    finally:
        srv.close()


def beside_backlog(mf, orc, ctx, big, budget=4 << 30, alone_at_a_time=4):
    """For as many requests as may run alone at a time: how many of 600 small ones of 13 to 22 ms each,
    published before it, were unfinished when it had its result."""
    small = mf.gen_genrmf(16, 60, 1, 10000, 3)
    srv = mf.Server(ctx, hbm_budget_bytes=budget, max_inflight_launches=alone_at_a_time)
    try:
        first = [srv.submit(small) for _ in range(600)]
        t0 = time.time()
        while srv.stats()["admitted"] < len(first) and time.time() - t0 < 60:
            srv.progress()
        alone = [srv.submit(big) for _ in range(alone_at_a_time)]
        values = serve(srv, first + alone)
        assert set(values[:600]) == {orc.dinic_maxflow(small)}
        assert set(values[600:]) == {orc.dinic_maxflow(big)}
        assert [srv.times(i)["batched"] for i in alone] == [0] * len(alone)
        ends = np.array([srv.times(i)["finish_ms"] for i in first])
        return [int((ends > srv.times(i)["finish_ms"]).sum()) for i in alone]
    finally:
        srv.close()


@pytest.mark.parametrize("gen,args", [("gen_genrmf", (20, 45, 1, 10000, 5)),    # in one workgroup
                                      ("gen_bipartite", (20000, 15000, 8.0, 77))])  # on the grid
def test_large_request_beside_a_backlog(mf, orc, ctx, gen, args):
    # more small requests than there are CUs are queued: a large one does not wait for them to
    # leave the serving kernel
    assert max(beside_backlog(mf, orc, ctx, getattr(mf, gen)(*args))) >= 256


@pytest.mark.parametrize("scale,factor", [(13, 16), (14, 4), (14, 15)])
def test_power_law_requests(mf, orc, ctx, scale, factor):
    # frontiers wider than 2,800 vertices and hubs: solved with the vertex state in LDS all the same.
    # One lane for a hub's whole scan took 30 to 100 ms; 20 is well above the 5 to 18 of a wave
    graphs = [mf.gen_rmat(scale, factor, seed=40 + i) for i in range(4)]
    srv = mf.Server(ctx, hbm_budget_bytes=1 << 30, max_inflight_launches=1)
    try:
        ids = [srv.submit(g) for g in graphs]
        assert serve(srv, ids) == [orc.dinic_maxflow(g) for g in graphs]
        assert all(srv.times(i)["batched"] == 1 for i in ids)
        assert min(srv.times(i)["device_ms"] for i in ids) < 20
    finally:
        srv.close()


def test_large_request_frees_nothing_beside_a_backlog(mf, orc, ctx):
    # hipFree waits for the serving kernel: the arrays of a request of 70 MB are kept for the next one
    assert max(beside_backlog(mf, orc, ctx, mf.gen_rmat(16, 16, seed=4))) >= 256


def test_one_large_request_at_a_time_beside_a_backlog(mf, orc, ctx):
    # wherever its workgroups' turn is: whichever shader engine that is has a CU free
    others = [mf.Context(0) for _ in range(2)]
    big = mf.gen_genrmf(20, 45, 1, 10000, 5)
    behind = [beside_backlog(mf, orc, ctx, big, alone_at_a_time=1)[0] for _ in range(4)]
    for c in others:
        c.close()
    assert sorted(behind)[1] >= 256, behind  # (one server's streams may share a hardware queue)


@pytest.mark.parametrize("others", [0, 1, 2])
@pytest.mark.parametrize("alone_at_a_time", [1, 4])
def test_no_stream_waits_for_the_serving_kernel(mf, orc, ctx, others, alone_at_a_time):
    # whatever streams there were before the server's: none of a large request's work shares a hardware
    # queue with the serving kernel
    others = [mf.Context(0) for _ in range(others)]
    big = mf.gen_bipartite(20000, 15000, 8.0, 77)
    behind = beside_backlog(mf, orc, ctx, big, alone_at_a_time=alone_at_a_time)
    for c in others:
        c.close()
    assert min(behind) >= 256, behind


def test_small_requests_behind_large_ones(mf, orc, ctx):
    # eight large requests, one of them perhaps in the serving kernel's hardware queue, then small ones:
    # the serving kernel is launched when that one has finished
    large = [mf.gen_genrmf(18, 56, 1, 10000, i) for i in range(8)]
    small = [mf.gen_washington_rlg(20 + i, 30, 10000, i) for i in range(24)]
    values = [orc.dinic_maxflow(g) for g in large + small]
    srv = mf.Server(ctx, hbm_budget_bytes=4 << 30, max_inflight_launches=4)
    try:
        for _ in range(3):
            ids = [srv.submit(g) for g in large]
            srv.progress()
            ids += [srv.submit(g) for g in small]
            assert serve(srv, ids) == values
    finally:
        srv.close()
