"""graph_sort on the GPU where a wave, a tile of keys or a part of the edge list ends (1024, 16384 and 65536
edges), with repeats across them, and with long stretches of ids that have no larger, no smaller or
no neighbour at all: the same CSR as the host's."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _edges(kind, m, rng):
    if kind == "few ids":  # every key many times over
        return rng.integers(0, 5, m), rng.integers(0, 5, m)
    if kind == "star":  # late ids have no larger neighbour, or (directed) no entries
        return np.zeros(m, np.int64), np.arange(m) + 1
    if kind == "star in":
        return np.arange(m) + 1, np.zeros(m, np.int64)
    if kind == "path":
        return np.arange(m), np.arange(m) + 1
    if kind == "self loops":  # mostly dropped
        u = rng.integers(0, 1000, m)
        return u, np.where(rng.random(m) < 0.9, u, rng.integers(0, 1000, m))
    return rng.integers(0, max(2, m // 3), m), rng.integers(0, max(2, m // 3), m)


@pytest.mark.parametrize("directed", [False, True])
@pytest.mark.parametrize("kind", ["random", "few ids", "star", "star in", "path", "self loops"])
@pytest.mark.parametrize("m", [1, 1023, 1024, 16383, 16384, 65535, 65537, 262145])
def test_graph_sort_edges(m, kind, directed):
    import torch

    from grass_amd import ingest
    rng = np.random.default_rng(m)
    u, v = (np.ascontiguousarray(x, dtype=np.uint32) for x in _edges(kind, m, rng))
    rp, col = ingest.graph_sort(u, v, directed=directed, threads=2).arrays()
    s, d = (torch.from_numpy(x.view(np.int32)).cuda() for x in (u, v))
    drp, dcol = ingest.graph_sort_device(s, d, directed=directed)
    np.testing.assert_array_equal(drp.cpu().numpy().astype(np.uint64), rp)
    np.testing.assert_array_equal(dcol.cpu().numpy().view(np.uint32), col)
