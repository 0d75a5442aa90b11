"""k-hop batches and their blocks at the sizes where the pipeline changes: frontiers and sequences that
one workgroup scans and ones that take a scan of several, dedup tables all at once and one shared by
the passes, few requests and more than one workgroup prepares, and requests that end inside a
64-position word.  Edges must equal the oracle's, blocks the numbering by first appearance."""
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
    (1, 30, [15, 10]),           # one workgroup scans everything
    (3, 63, [5]),                # one hop: no destinations are deduplicated
    (7, 400, [25, 10]),          # a frontier bound past one workgroup's scan
    (42, 3369, [10, 10, 2]),     # all tables together too large, the shared one not
    (40, 3369, [20, 20]),        # over a million positions: the word scan takes several launches
    (9000, 3, [4, 4]),           # more requests than one workgroup prepares
])
def test_passes(env, requests, seeds, fanouts):
    g, og = env
    print(f"[khop passes] requests={requests} seeds={seeds} fanouts={fanouts}", flush=True)
    rng = np.random.default_rng(requests)
    sl = [rng.integers(0, g.n, size=seeds - (i % 3 if seeds > 3 else 0)).astype(np.uint32) for i in range(requests)]
    fl = [fanouts] * requests
    res = g.khop_minibatch(sl, fl, seed=11)
    src, dst = (res[k].cpu().numpy().view(np.uint32) for k in ("src", "dst"))
    off = res["offsets"].cpu().numpy()
    exp = og.khop(sl, fl, seed=11)
    assert res["total"] == len(exp["dst"])
    nodes, node_off = res["nodes"].cpu().numpy().view(np.uint32), res["node_off"].cpu().numpy()
    lsrc, ldst = res["lsrc"].cpu().numpy(), res["ldst"].cpu().numpy()
    for r in range(requests):
        e = np.concatenate([np.arange(off[h, r], off[h, r + 1]) for h in range(len(fanouts))])
        a, b = int(exp["edge_off"][r]), int(exp["edge_off"][r + 1])
        np.testing.assert_array_equal(src[e], exp["src"][a:b])
        np.testing.assert_array_equal(dst[e], exp["dst"][a:b])
        seq = np.concatenate([sl[r], dst[e]])
        uniq, first = np.unique(seq, return_index=True)
        ids = np.empty(len(uniq), np.int64)  # local id of each distinct vertex: rank of its first position
        ids[np.argsort(first)] = np.arange(len(uniq))
        mine = nodes[node_off[r]:node_off[r + 1]]
        np.testing.assert_array_equal(mine, seq[np.sort(first)])
        np.testing.assert_array_equal(ldst[e], ids[np.searchsorted(uniq, dst[e])])
        np.testing.assert_array_equal(lsrc[e], ids[np.searchsorted(uniq, src[e])])
