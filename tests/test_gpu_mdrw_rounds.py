"""The MDRW walk in rounds of guessed steps at the edges of its frontier sums (whole and partial rows
of 16 entries, blocks and groups; the largest frontier it takes and the first it does not), of its
draws (64 at a time) and of its limit on the degree sum, past which an instance is walked again one
step at a time.  Every edge must equal the oracle's."""
import numpy as np
import pytest

from conftest import load_case

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 15, 16, 17, 31, 255, 256, 257, 1000, 4095, 4096]


@pytest.fixture(scope="module")
def ga():
    import grass_amd
    import torch
    assert torch.cuda.is_available()
    grass_amd.lib()
    return grass_amd


def _check(g, og, sizes, target, seed):
    res, exp = g.mdrw(sizes, target=target, seed=seed), og.mdrw(sizes, target=target, seed=seed)
    for k in ("step_off", "step_src", "step_dst", "vert_off", "verts", "ind_off", "ind_src", "ind_dst"):
        np.testing.assert_array_equal(res[k], exp[k], err_msg=k)


@pytest.mark.parametrize("fmt", ["le", "gt"])
@pytest.mark.parametrize("case,target,sizes", [
    ("rmat12", 4300, SIZES),                 # 204 to 4299 steps per instance
    ("rmat12", 4160, [4097, 64, 4096]),      # a frontier past the rounds' limit takes the plain kernel
    ("rmat12", 1064, [1000, 1001, 999, 1063, 1064]),  # 64, 63, 65, 1 and 0 steps
    ("degrees", 600, [1, 3, 16, 40, 300]),   # few vertices, many without neighbours
])
def test_rounds_equal_oracle(ga, oracle_mod, fmt, case, target, sizes):
    print(f"[mdrw rounds] case={case} fmt={fmt} target={target}", flush=True)
    c = load_case(case)
    gb, ob = c[f"{fmt}_graph"].tobytes(), c[f"{fmt}_offset"].tobytes()
    _check(ga.Graph.from_bytes(gb, ob, fmt), oracle_mod.Graph(gb, ob, fmt), sizes, target, seed=17)


@pytest.mark.parametrize("wmax", [1, 2000, 30000])
def test_walked_again_past_the_sum_limit(ga, oracle_mod, monkeypatch, wmax):
    """Limits that every instance passes at once, that some pass on the way, and that few pass."""
    print(f"[mdrw rounds] wmax={wmax}", flush=True)
    monkeypatch.setenv("GRASS_MDRW_WMAX", str(wmax))
    c = load_case("rmat12")
    gb, ob = c["gt_graph"].tobytes(), c["gt_offset"].tobytes()
    _check(ga.Graph.from_bytes(gb, ob, "gt"), oracle_mod.Graph(gb, ob, "gt"), [4, 20, 60, 200, 700], 1500, seed=5)
