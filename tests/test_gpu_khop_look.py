"""Frontiers of as many entries as make the deduplication read its slots before it claims them (2^19), and
of one fewer: distinct entries, and repeats of few, against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

N = 600_000


@pytest.fixture(scope="module")
def env(oracle_mod):
    import grass_amd
    import torch
    from grass_amd import ingest
    assert torch.cuda.is_available()
    src = np.arange(N, dtype=np.uint32)  # a cycle
    gb, ob = ingest.graph_sort(src, ((src + 1) % N).astype(np.uint32), threads=4).compress("le", threads=4)
    return grass_amd.Graph.from_bytes(gb, ob, "le"), oracle_mod.Graph(gb, ob, "le")


@pytest.mark.parametrize("entries", [(1 << 19) - 1, 1 << 19])
@pytest.mark.parametrize("kind", ["distinct", "repeats"])
def test_entries(env, kind, entries):
    g, og = env
    print(f"[khop look] {kind} {entries}", flush=True)
    rng = np.random.default_rng(entries)
    if kind == "distinct":
        v = rng.permutation(N)[:entries].astype(np.uint32)
    else:
        v = rng.integers(0, 900, size=entries).astype(np.uint32)
    sl = [v[:1000], v[1000:300_000], v[300_000:]]
    res, exp = g.khop_batch(sl, [[2, 1]] * 3, seed=6), og.khop(sl, [[2, 1]] * 3, seed=6)
    src, dst, off = (np.asarray(res[k]) for k in ("src", "dst", "offsets"))
    assert res["total"] == len(exp["dst"])
    for r in range(3):
        e = np.concatenate([np.arange(off[h, r], off[h, r + 1]) for h in range(2)]).astype(np.int64)
        a, b = int(exp["edge_off"][r]), int(exp["edge_off"][r + 1])
        np.testing.assert_array_equal(src[e].view(np.uint32), exp["src"][a:b])
        np.testing.assert_array_equal(dst[e].view(np.uint32), exp["dst"][a:b])
