"""Blocks of batches large enough to go by partition: requests that end at, before and after a tile of 8192
positions, requests of one position and of none, most positions repeats of few vertices or none
repeated, and vertices chosen so that one bucket holds more distinct ones than its table, which must
fall back.  Numbering by first appearance, against numpy; the table in memory gives the same."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

N = 2_400_000


@pytest.fixture(scope="module")
def graph():
    """A cycle: every vertex has the two neighbours next to it."""
    import torch

    import grass_amd
    from grass_amd import ingest
    assert torch.cuda.is_available()
    src = np.arange(N, dtype=np.uint32)
    csr = ingest.graph_sort(src, ((src + 1) % N).astype(np.uint32), threads=8)
    assert csr.n == N
    return grass_amd.Graph.from_bytes(*csr.compress("le", threads=8), "le")


def _hash(v):
    """The partition's hash of a vertex; the bucket is the high word of its product with the count."""
    h = v.astype(np.uint64) * 0x9E3779B1 & 0xFFFFFFFF
    h ^= h >> 15
    h = h * 0x85EBCA77 & 0xFFFFFFFF
    return h ^ (h >> 13)


def _check(g, seeds, fanouts):
    fl = [fanouts] * len(seeds)
    res = g.khop_minibatch(seeds, fl, seed=3)
    src, dst, nodes = (res[k].cpu().numpy().view(np.uint32) for k in ("src", "dst", "nodes"))
    off, node_off = res["offsets"].cpu().numpy(), res["node_off"].cpu().numpy()
    lsrc, ldst = res["lsrc"].cpu().numpy(), res["ldst"].cpu().numpy()
    assert sum(map(len, seeds)) + res["total"] >= 1 << 20
    for r, s in enumerate(seeds):
        e = np.concatenate([np.arange(off[h, r], off[h, r + 1]) for h in range(len(fanouts))]).astype(np.int64)
        seq = np.concatenate([s, dst[e]])
        uniq, first = np.unique(seq, return_index=True)
        ids = np.empty(len(uniq), np.int64)
        ids[np.argsort(first)] = np.arange(len(uniq))
        np.testing.assert_array_equal(nodes[node_off[r]:node_off[r + 1]], seq[np.sort(first)], err_msg=f"request {r}")
        np.testing.assert_array_equal(ldst[e], ids[np.searchsorted(uniq, dst[e])], err_msg=f"request {r}")
        np.testing.assert_array_equal(lsrc[e], ids[np.searchsorted(uniq, src[e])], err_msg=f"request {r}")
    return nodes, node_off, lsrc, ldst


@pytest.mark.parametrize("kind", ["distinct", "repeats"])
def test_tiles(graph, kind, monkeypatch):
    rng = np.random.default_rng(1)
    sizes = [4096, 4095, 4097, 1, 0, 2, 8192, 8191, 60000, 300000, 120001, 2560, 2561]
    if kind == "repeats":  # (the next hop's frontier has each vertex once)
        sizes += [540_672, 16384]
    print(f"[block parts] {kind}", flush=True)
    ids = N if kind == "distinct" else 700
    seeds = [rng.integers(0, ids, size=k).astype(np.uint32) for k in sizes]
    a = _check(graph, seeds, [1, 2])
    monkeypatch.setenv("GRASS_EXPORT_SLOT", "16")
    for x, y in zip(a, _check(graph, seeds, [1, 2])):
        np.testing.assert_array_equal(x, y)


def _bucket_case(graph, buckets, few, rng):
    """One request of exactly `buckets` x 2560 positions: every vertex of `few`, repeats of them, and one
    destination for each of `few`."""
    print(f"[block parts] {len(few)} vertices", flush=True)
    seeds = few[rng.integers(0, len(few), size=buckets * 2560 - len(few))]
    seeds[:len(few)] = few
    _check(graph, [seeds], [1])


def test_buckets_nearly_full(graph):
    """60 of 625 buckets hold about 3500 distinct vertices each, of the 4096 their tables take."""
    rng = np.random.default_rng(2)
    v = np.arange(N, dtype=np.uint32)
    _bucket_case(graph, 625, v[(_hash(v) * 625 >> 32 < 60) & (rng.random(N) < 0.8)], rng)


def test_a_bucket_past_its_table(graph):
    """More than 5000 distinct vertices in one bucket."""
    v = np.arange(N, dtype=np.uint32)
    few = v[_hash(v) * 422 >> 32 == 7]
    assert len(few) > 5000
    _bucket_case(graph, 422, few, np.random.default_rng(3))
