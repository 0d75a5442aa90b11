"""k-hop batches whose offsets come out of the scans themselves: as many requests as one round of a tile's
threads reads, one less and one more, as many as the scan takes and more; requests that end at, before
and after a tile (4096 frontier items, 262144 positions); empty requests at the front, inside and at
the end; hops that draw nothing.  Against the oracle, blocks against the numbering by first appearance."""
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


def _check(env, sl, fanouts):
    g, og = env
    R, H = len(sl), len(fanouts)
    res = g.khop_minibatch(sl, [fanouts] * R, seed=5)
    exp = og.khop(sl, [fanouts] * R, seed=5)
    src, dst = (res[k].cpu().numpy().view(np.uint32) for k in ("src", "dst"))
    off, node_off = res["offsets"].cpu().numpy(), res["node_off"].cpu().numpy()
    nodes = res["nodes"].cpu().numpy().view(np.uint32)
    assert res["total"] == len(exp["dst"]) == off[H - 1, R]
    for r in range(R):
        e = np.concatenate([np.arange(off[h, r], off[h, r + 1]) for h in range(H)]).astype(np.int64)
        a, b = int(exp["edge_off"][r]), int(exp["edge_off"][r + 1])
        np.testing.assert_array_equal(src[e], exp["src"][a:b], err_msg=f"request {r}")
        np.testing.assert_array_equal(dst[e], exp["dst"][a:b], err_msg=f"request {r}")
        seq = np.concatenate([sl[r], dst[e]])
        _, first = np.unique(seq, return_index=True)
        np.testing.assert_array_equal(nodes[node_off[r]:node_off[r + 1]], seq[np.sort(first)], err_msg=f"request {r}")


@pytest.mark.parametrize("requests", [10, 255, 256, 257, 1023, 1024, 1025])
def test_requests(env, requests):
    """Distinct seeds, so that request sizes are item counts; over a million destinations a hop."""
    n = env[0].n
    rng = np.random.default_rng(requests)
    print(f"[scan marks] requests={requests}", flush=True)
    sizes = [0, 2048, 2048, 1, 0, 2047, 2049, 0]
    more = requests - len(sizes) - 1
    sizes += [max(1, min(n, 110_000 // more))] * more + [0]
    _check(env, [rng.permutation(n)[:k].astype(np.uint32) for k in sizes], [10, 2])


def test_positions(env):
    """Seeds past a million positions: the ends of requests are the ends of tiles of words."""
    rng = np.random.default_rng(9)
    print("[scan marks] positions", flush=True)
    sizes = [0, 262144, 262143, 1, 262208, 64, 0, 262080, 5, 0]
    _check(env, [rng.integers(0, env[0].n, size=k).astype(np.uint32) for k in sizes], [2, 1])


def test_no_draws(oracle_mod):
    """Seeds without neighbours: the second hop has no items, though its bound takes several tiles."""
    import grass_amd
    from grass_amd import ingest
    n = 20_000
    col = np.append(np.arange(1, 100), n - 1).astype(np.uint32)
    gb, ob = ingest.csr_from_sorted_edges(np.zeros(100, np.uint32), col).compress("le", threads=2)
    env = grass_amd.Graph.from_bytes(gb, ob, "le"), oracle_mod.Graph(gb, ob, "le")
    assert env[0].n == n
    print("[scan marks] no draws", flush=True)
    rng = np.random.default_rng(4)
    _check(env, [(1 + rng.permutation(n - 1)[:6000]).astype(np.uint32) for _ in range(3)], [60, 2])
