"""Prefix sums at the lengths where the number of tiles (4096 values) or the choice between one launch
(at most four tiles) and two changes: the row pointers of a full decode, for n around each edge, with and
without the tiles' prefixes kept."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 255, 4095, 4096, 4097, 8192, 8193, 16383, 16384, 16385, 20481])
@pytest.mark.parametrize("fmt", ["le", "gt"])
def test_row_pointers(fmt, n):
    import grass_amd as ga
    from grass_amd import ingest
    print(f"[scan tiles] fmt={fmt} n={n}", flush=True)
    rng = np.random.default_rng(n)
    # (v, v + 1 .. v + deg) mod n, without repeats and self loops; the last id appears in row 0
    deg = rng.integers(0, min(n, 7), n)
    deg[0] = max(deg[0], 1)
    rows = [np.sort((v + 1 + np.arange(d)) % n) for v, d in enumerate(deg)]
    rows[0][-1] = n - 1
    col = np.concatenate(rows).astype(np.uint32)
    src = np.repeat(np.arange(n, dtype=np.uint32), deg)
    csr = ingest.csr_from_sorted_edges(src, col)
    assert csr.n == n
    g = ga.Graph.from_bytes(*csr.compress(fmt, threads=2), fmt)
    for _ in range(2):  # the first decode makes the tiles' prefixes, the second scans from them
        rp, cl = g.decode_csr()
        np.testing.assert_array_equal(rp, np.concatenate([[0], np.cumsum(deg)]).astype(np.uint64))
        np.testing.assert_array_equal(cl, col)
    g.close()
