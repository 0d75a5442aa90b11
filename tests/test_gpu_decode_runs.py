"""The run-based full decode at the shapes where a run, a pass of 64 runs or a wave's range of runs
ends: every degree up to 70, degrees around multiples of 64 and 256, one list of many passes,
stretches of more than 64 vertices without entries, and neighbours spread so widely that four
fields take a fifth 32-bit word.  The decode must equal the oracle's, which is the CSR that was
compressed (but for a GT self loop at a block head, which the format cannot hold)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ga():
    import grass_amd
    import torch
    assert torch.cuda.is_available()
    grass_amd.lib()
    return grass_amd


def _csr(n, spread):
    """n vertices, most of them without entries; rows sorted, unique, over all of [0, n) (`spread`) or
    close to their vertex."""
    rng = np.random.default_rng(7 + spread)
    degs = list(range(71)) + [127, 128, 129, 255, 256, 257, 1023, 1025, 9000]
    at = np.concatenate([np.arange(200), np.arange(400, 400 + len(degs)), [n - 70, n - 3]])
    deg = np.zeros(n, np.int64)
    deg[at[:200]] = rng.integers(0, 9, 200)
    deg[at[200:200 + len(degs)]] = degs
    deg[n - 70], deg[n - 3], deg[n - 1] = 300, 2, 1
    rowptr = np.zeros(n + 1, np.uint64)
    rowptr[1:] = np.cumsum(deg)
    cols = []
    for v in np.flatnonzero(deg):
        d = int(deg[v])
        if v == n - 1:  # the last id appears, so that the edge list has n vertices
            row = np.array([v])
        elif spread:
            row = np.sort(rng.choice(n, size=d, replace=False))
        else:
            lo = max(0, min(v - d, n - 2 * d - 8))
            row = np.sort(rng.choice(np.arange(lo, lo + 2 * d + 8), size=d, replace=False))
        cols.append(row.astype(np.uint32))
    return rowptr, np.concatenate(cols)


@pytest.mark.parametrize("spread", [0, 1])
@pytest.mark.parametrize("fmt", ["le", "gt"])
def test_decode_run_edges(ga, oracle_mod, fmt, spread):
    from grass_amd import ingest
    n = 6_000_000 if spread else 20_000
    print(f"[decode runs] fmt={fmt} n={n}", flush=True)
    rowptr, col = _csr(n, spread)
    src = np.repeat(np.arange(n, dtype=np.uint32), np.diff(rowptr.astype(np.int64)))
    csr = ingest.csr_from_sorted_edges(src, col)
    assert csr.n == n
    gb, ob = csr.compress(fmt, threads=4)
    erp, ecol = oracle_mod.Graph(gb, ob, fmt).decode_csr()
    np.testing.assert_array_equal(erp, rowptr)
    g = ga.Graph.from_bytes(gb, ob, fmt)
    for per_wave in (512, 1024, 8192):
        g.set_tuning(decode_edges_per_wave=per_wave)
        rp, cl = g.decode_csr()
        np.testing.assert_array_equal(rp, erp)
        np.testing.assert_array_equal(cl, ecol, err_msg=f"{per_wave} slots per wave")
    g.close()
