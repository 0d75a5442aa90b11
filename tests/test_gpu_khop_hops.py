"""Batches whose hops differ by orders of magnitude, so that each pass takes a table, words and scans of
its own size: growing and shrinking hops, hops that draw nothing, requests with fewer hops than others and
with none, one table for all passes and one for each.  Against the oracle."""
import numpy as np
import pytest

from conftest import load_case

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def env(oracle_mod):
    import grass_amd
    import torch
    assert torch.cuda.is_available()
    c = load_case("rmat12")
    gb, ob = c["gt_graph"].tobytes(), c["gt_offset"].tobytes()
    return grass_amd.Graph.from_bytes(gb, ob, "gt"), oracle_mod.Graph(gb, ob, "gt")


@pytest.mark.parametrize("requests,seeds,fanouts", [
    (33, 700, [[10, 10, 5]]),            # 23 k, 0.2 M, 2 M entries: all tables at once
    (60, 3000, [[60, 1, 1, 2]]),         # the second pass the largest; one table shared by the passes
    (40, 600, [[0, 9], [0, 0, 3]]),      # nothing drawn
    (30, 900, [[3, 0, 4], [2]]),         # a pass in the middle without entries for anyone
    (50, 500, [[1], [1, 1, 1, 20], [], [12, 3]]),
    (3000, 6, [[30], [], [1, 2]]),       # more requests than a scan takes along
])
def test_hops(env, requests, seeds, fanouts):
    g, og = env
    print(f"[khop hops] requests={requests} seeds={seeds} fanouts={fanouts}", flush=True)
    rng = np.random.default_rng(requests)
    sl = [rng.integers(0, g.n, size=max(seeds - i % 5, 0)).astype(np.uint32) for i in range(requests)]
    fl = [fanouts[i % len(fanouts)] for i in range(requests)]
    H = max(map(len, fl))
    res, exp = g.khop_batch(sl, fl, seed=8), og.khop(sl, fl, seed=8)
    src, dst, off = (np.asarray(res[k]) for k in ("src", "dst", "offsets"))
    assert res["total"] == len(exp["dst"])
    for r in range(requests):
        e = np.concatenate([np.arange(off[h, r], off[h, r + 1]) for h in range(H)]).astype(np.int64)
        a, b = int(exp["edge_off"][r]), int(exp["edge_off"][r + 1])
        np.testing.assert_array_equal(src[e].view(np.uint32), exp["src"][a:b], err_msg=f"request {r}")
        np.testing.assert_array_equal(dst[e].view(np.uint32), exp["dst"][a:b], err_msg=f"request {r}")
