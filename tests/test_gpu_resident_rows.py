"""Graphs built from rows on the GPU, straight into their resident form or through the images, against the
rows themselves and the oracle's walks: what the two ways share cannot hide in their comparison."""
import numpy as np
import pytest

from test_gpu_encode_slots import CASES, _device, _rows, env  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmt,interval", [("le", ""), ("gt", "2"), ("gt", "4"), ("gt", "8"), ("gt", "64")])
def test_resident(env, oracle_mod, monkeypatch, fmt, interval):  # noqa: F811
    if interval:
        monkeypatch.setenv("GRASS_GT_CHECKPOINT", interval)
    for case in CASES:
        for kind in ("random", "dense"):
            print(f"[resident rows] {fmt} {interval} {case} {kind}", flush=True)
            _check(env, oracle_mod, fmt, interval, case, kind)


def _check(env, oracle_mod, fmt, interval, case, kind):  # noqa: F811
    torch, ga, ingest = env
    n, deg = CASES[case]
    rowptr, col = _rows(n, deg.copy(), kind, 14)
    rp, cl = _device(torch, rowptr, col)
    gb, ob = ingest.compress_device(rp, cl, fmt)
    starts = np.arange(min(n, 4096), dtype=np.uint32)
    walks, _ = oracle_mod.Graph(gb, ob, fmt).random_walk(len(starts), 8, seed=3, starts=starts)
    starts_dev = torch.from_numpy(starts.view(np.int32)).cuda()
    for g in (ga.Graph.from_csr_device(rp, cl, fmt), ga.Graph.from_bytes(gb, ob, fmt)):
        assert g.info()["gt_checkpoint"] == (int(interval) if interval else 0)
        a, b = g.decode_csr()
        np.testing.assert_array_equal(a, rowptr)
        np.testing.assert_array_equal(b, col)
        mine = g.random_walk(len(starts), 8, seed=3, starts=starts_dev)
        np.testing.assert_array_equal(ga.to_numpy_u32(mine), walks)
        g.close()
