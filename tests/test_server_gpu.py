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
