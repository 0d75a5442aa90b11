"""The encoder by slots at the sizes where a pass of 64 slots, a chunk of passes or a word ends: rows of
every length around multiples of 64, long stretches of empty rows and of rows of one entry, ids at both
ends of the range, lists of consecutive ids (one-bit gaps).  The images must equal the host compressor's,
and a graph encoded straight into its resident form must equal, in figures and content, the one loaded
from those images; rows that need the general encoder (a GT self loop, an id past the graph, an unsorted
row) give what they give through the images."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def env():
    import torch

    import grass_amd
    from grass_amd import ingest
    assert torch.cuda.is_available()
    grass_amd.lib()
    return torch, grass_amd, ingest


def _rows(n, deg, kind, seed):
    """A strictly ascending row without v itself for each of the degrees; row n - 2 holds the last id."""
    rng = np.random.default_rng(seed)
    cols = []
    for v, d in enumerate(deg):
        d = int(d)
        if kind == "dense":  # consecutive ids after v (mod n)
            row = np.sort((v + 1 + np.arange(d)) % n)
        else:
            row = rng.integers(0, n - 1, size=d) if d == 1 else rng.choice(n - 1, size=d, replace=False)
            row = np.sort(row + (row >= v))
        cols.append(row)
    deg[n - 2] = 1
    cols[n - 2] = np.array([n - 1])
    rowptr = np.zeros(n + 1, np.uint64)
    rowptr[1:] = np.cumsum(deg)
    return rowptr, np.concatenate(cols).astype(np.uint32)


def _cases():
    rng = np.random.default_rng(5)
    n = 3000
    ladder = np.zeros(n, np.int64)
    ladder[:len(range(0, 200))] = np.arange(200)
    ladder[300:308] = [255, 256, 257, 1023, 1024, 1025, 2047, 2990]
    yield "ladder", n, ladder
    yield "empty", 20000, np.zeros(20000, np.int64)
    ones = np.ones(20000, np.int64)
    ones[5000:9000] = 0
    yield "ones", 20000, ones
    mixed = rng.choice([0, 1, 2, 3, 62, 63, 64, 65, 700], size=6000, p=[.2, .2, .2, .2, .05, .05, .04, .05, .01])
    yield "mixed", 6000, mixed.astype(np.int64)
    yield "tiny", 3, np.array([2, 0, 0])
    hub = np.full(70000, 1, np.int64)
    hub[12345] = 66000
    yield "hub", 70000, hub


CASES = {name: (n, deg) for name, n, deg in _cases()}


def _device(torch, rowptr, col):
    return (torch.from_numpy(rowptr.astype(np.int64)).cuda(),
            torch.from_numpy(np.ascontiguousarray(col, dtype=np.uint32).view(np.int32)).cuda())


def _same(torch, a, b):
    assert str(a.info()) == str(b.info())
    for x, y in zip(a.decode_csr(), b.decode_csr()):
        np.testing.assert_array_equal(x, y)
    starts = torch.arange(min(a.n, 4096), dtype=torch.int32, device="cuda")
    pa, pb = (g.random_walk(walkers=len(starts), length=8, seed=3, starts=starts) for g in (a, b))
    assert torch.equal(torch.as_tensor(pa), torch.as_tensor(pb))


@pytest.mark.parametrize("kind", ["random", "dense"])
@pytest.mark.parametrize("case", list(CASES))
@pytest.mark.parametrize("fmt", ["le", "gt"])
def test_slots(env, fmt, case, kind):
    torch, ga, ingest = env
    n, deg = CASES[case]
    print(f"[encode slots] fmt={fmt} case={case} kind={kind}", flush=True)
    rowptr, col = _rows(n, deg.copy(), kind, 11)
    src = np.repeat(np.arange(n, dtype=np.uint32), np.diff(rowptr.astype(np.int64)))
    csr = ingest.csr_from_sorted_edges(src, col)
    assert csr.n == n
    eg, eo = csr.compress(fmt, threads=2)
    rp, cl = _device(torch, rowptr, col)
    gb, ob = ingest.compress_device(rp, cl, fmt)
    assert gb == eg and ob == eo
    direct, loaded = ga.Graph.from_csr_device(rp, cl, fmt), ga.Graph.from_bytes(eg, eo, fmt)
    _same(torch, direct, loaded)
    direct.close()
    loaded.close()


@pytest.mark.parametrize("p", ["2", "8", "64"])
def test_checkpoint_intervals(env, monkeypatch, p):
    torch, ga, ingest = env
    monkeypatch.setenv("GRASS_GT_CHECKPOINT", p)
    n, deg = CASES["ladder"]
    rowptr, col = _rows(n, deg.copy(), "random", 12)
    rp, cl = _device(torch, rowptr, col)
    gb, ob = ingest.compress_device(rp, cl, "gt")
    direct, loaded = ga.Graph.from_csr_device(rp, cl, "gt"), ga.Graph.from_bytes(gb, ob, "gt")
    _same(torch, direct, loaded)
    direct.close()
    loaded.close()


@pytest.mark.parametrize("what", ["self loop", "past the graph", "unsorted", "repeated"])
@pytest.mark.parametrize("fmt", ["le", "gt"])
def test_rows_for_the_general_encoder(env, fmt, what):
    torch, ga, ingest = env
    n, deg = CASES["ladder"]
    print(f"[encode slots] fmt={fmt} {what}", flush=True)
    rowptr, col = _rows(n, deg.copy(), "random", 13)
    at = int(rowptr[40])
    if what == "self loop":
        row = col[at:at + 40]
        row[0] = 40
        row.sort()
    elif what == "past the graph":
        col[at + 39] = n + 7
    elif what == "unsorted":
        col[at + 9], col[at + 30] = col[at + 30], col[at + 9]
    else:
        col[at + 9] = col[at + 8]
    rp, cl = _device(torch, rowptr, col)
    gb, ob = ingest.compress_device(rp, cl, fmt)
    if what == "self loop":
        src = np.repeat(np.arange(n, dtype=np.uint32), np.diff(rowptr.astype(np.int64)))
        assert (gb, ob) == ingest.csr_from_sorted_edges(src, col).compress(fmt, threads=2)
    direct, loaded = ga.Graph.from_csr_device(rp, cl, fmt), ga.Graph.from_bytes(gb, ob, fmt)
    assert str(direct.info()) == str(loaded.info())
    for x, y in zip(direct.decode_csr(), loaded.decode_csr()):
        np.testing.assert_array_equal(x, y)
    direct.close()
    loaded.close()
