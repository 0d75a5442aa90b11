"""k-hop passes and blocks around the limits of the one-workgroup kernels: 4096 seeds, requests or
destinations of a pass, 8192 positions and 1024 requests of blocks, and blocks whose table takes more than
64 KB of LDS (over 5461 positions).  Edges must equal the oracle's, blocks the numbering by first appearance."""
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


def _check(env, sl, fl):
    g, og = env
    res = g.khop_minibatch(sl, fl, seed=17)
    src, dst, nodes, lsrc, ldst = (res[k].cpu().numpy().view(np.uint32) for k in ("src", "dst", "nodes", "lsrc", "ldst"))
    off, node_off = res["offsets"].cpu().numpy(), res["node_off"].cpu().numpy()
    exp = og.khop(sl, fl, seed=17)
    assert res["total"] == len(exp["dst"])
    for r, seeds in enumerate(sl):
        e = np.concatenate([np.arange(off[h, r], off[h, r + 1]) for h in range(len(off))]).astype(np.int64)
        a, b = int(exp["edge_off"][r]), int(exp["edge_off"][r + 1])
        np.testing.assert_array_equal(src[e], exp["src"][a:b])
        np.testing.assert_array_equal(dst[e], exp["dst"][a:b])
        seq = np.concatenate([seeds, dst[e]])
        uniq, first = np.unique(seq, return_index=True)
        ids = np.empty(len(uniq), np.int64)
        ids[np.argsort(first)] = np.arange(len(uniq))
        np.testing.assert_array_equal(nodes[node_off[r]:node_off[r + 1]], seq[np.sort(first)])
        np.testing.assert_array_equal(ldst[e], ids[np.searchsorted(uniq, dst[e])])
        np.testing.assert_array_equal(lsrc[e], ids[np.searchsorted(uniq, src[e])])
    return sum(map(len, sl)) + res["total"]


@pytest.mark.parametrize("seeds", [4095, 4096, 4097])
@pytest.mark.parametrize("requests", [1, 5])
def test_seeds(env, seeds, requests):
    print(f"[one workgroup] {requests} x {seeds} seeds", flush=True)
    rng = np.random.default_rng(seeds)
    cut = np.sort(rng.integers(0, seeds + 1, size=requests - 1))
    sl = np.split(rng.integers(0, env[0].n, size=seeds).astype(np.uint32), cut)
    _check(env, sl, [[3, 2]] * requests)


@pytest.mark.parametrize("seeds,fanout", [(273, 15), (256, 16), (241, 17)])  # 4095, 4096, 4097 destinations at most
def test_destinations(env, seeds, fanout):
    print(f"[one workgroup] {seeds} seeds x {fanout}", flush=True)
    g, og = env
    hubs = np.argsort([-og.degree(v) for v in range(g.n)], kind="stable")[:seeds]  # (all have 100 neighbours)
    _check(env, [hubs.astype(np.uint32)], [[fanout, 2]])


@pytest.mark.parametrize("positions", [5460, 5461, 5462, 8191, 8192, 8193])
def test_positions(env, positions):
    print(f"[one workgroup] {positions} positions", flush=True)
    n = env[0].n
    distinct = min(n, positions // 2)
    v = np.random.default_rng(positions).permutation(n)[:distinct]
    seeds = np.concatenate([v, np.resize(v, positions - 2 * distinct)]).astype(np.uint32)
    assert _check(env, [seeds], [[1]]) == positions  # (every vertex has a neighbour)


@pytest.mark.parametrize("requests", [1023, 1024, 1025, 4096, 4097])
def test_requests(env, requests):
    print(f"[one workgroup] {requests} requests", flush=True)
    rng = np.random.default_rng(requests)
    sl = [rng.integers(0, env[0].n, size=0 if requests > 4000 and i % 3 else 1).astype(np.uint32) for i in range(requests)]
    _check(env, sl, [[2, 2]] * requests)
