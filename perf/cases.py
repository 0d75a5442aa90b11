"""Workloads for timing the framework through its public entry points.

Every case builds its compressed graph on the GPU from its seed (R-MAT edges, graph_sort, device
encoder), as a program that owns a device edge list would, keeps the resident graph, and times one
operation on it:

  walk        one Graph.random_walk request
  walk_batch  many walk requests of different sizes in one grass_random_walk_batch call
  minibatch   a k-hop batch and its mini-batch blocks in local ids (grass_khop_batch, then
              grass_khop_blocks_build), into buffers the trainer keeps
  replay      one replay of a captured plan of walk and k-hop requests
  mdrw        Graph.mdrw_tensors: frontier samples and their induced edge lists, collected into the
              program's own padded batch buffers
  decode      the full decode of the resident graph to a CSR in device memory
  ingest      an edge list on the GPU -> CSR -> encoded, resident graph -> a first walk on it
  load        .graph/.offset images in host memory -> resident graph -> a first walk on it

A case fixes the sizes of its requests; the seed gives the graph, the seeds and starts, and the
draws.  How much comes back then still differs from seed to seed (drawn edges, distinct vertices),
so outputs are the program's whole buffers, sized for the case and zero past what was written.
They are vertex ids and offsets (whole numbers), so there is nothing to compare with a wider float
type: exact() gives None.
"""
import math
import random

import torch

import grass_amd
from grass_amd import ingest

C = grass_amd.C
DEVICE = "cuda:0"

# R-MAT quadrant probabilities: the skewed graphs of the benchmark, a milder skew, and no skew (a
# uniform random graph: no hubs, every list short).
SKEW = {"rmat": (0.57, 0.19, 0.19), "mild": (0.45, 0.22, 0.22), "uniform": (0.25, 0.25, 0.25)}


def listed():
    return [
        # a single user's few short walks on a small graph: launch and call latency
        dict(name="walk_one_le_s14", op="walk", fmt="le", scale=14, ef=16, skew="rmat", walkers=64, length=10,
             starts=True),
        # one DeepWalk pass: 2^20 walks of length 80
        dict(name="walk_epoch_le_s22", op="walk", fmt="le", scale=22, ef=16, skew="rmat", walkers=1 << 20,
             length=80, starts=False),
        # the benchmark's batch of walk requests at its scale
        dict(name="walk_batch_gt_s24", op="walk_batch", fmt="gt", scale=24, ef=16, skew="rmat", requests=256,
             walkers=4096),
        # an online GNN inference request: a handful of seeds
        dict(name="minibatch_one_gt_s18", op="minibatch", fmt="gt", scale=18, ef=16, skew="rmat", requests=1,
             seeds=48, fanouts="15,10"),
        # GNN training: 16 workers' mini-batches in one call
        dict(name="minibatch_train_gt_s24", op="minibatch", fmt="gt", scale=24, ef=16, skew="rmat", requests=16,
             seeds=8192, fanouts="25,10"),
        # 3-hop training on a graph without hubs
        dict(name="minibatch_3hop_le_s20", op="minibatch", fmt="le", scale=20, ef=8, skew="uniform", requests=33,
             seeds=700, fanouts="10,10,5"),
        # a steady serving step of small requests of both kinds, captured once and replayed
        dict(name="replay_small_gt_s22", op="replay", fmt="gt", scale=22, ef=16, skew="rmat", requests=16,
             walkers=4096, seeds=400, fanouts="25,10"),
        # graph statistics from frontier samples: a batch of the benchmark's instance shape
        dict(name="mdrw_gt_s22", op="mdrw", fmt="gt", scale=22, ef=16, skew="rmat", instances=64, target=16384,
             local=False),
        # a few small samples with local ids
        dict(name="mdrw_few_le_s18", op="mdrw", fmt="le", scale=18, ef=16, skew="mild", instances=5, target=3000,
             local=True),
        # full decode, LE at the size of the correctness tests and GT at the benchmark's
        dict(name="decode_le_s22", op="decode", fmt="le", scale=22, ef=16, skew="rmat"),
        dict(name="decode_gt_s24", op="decode", fmt="gt", scale=24, ef=16, skew="rmat"),
        # a new snapshot of a graph built on the GPU: sort, encode, load, first walks
        dict(name="ingest_gt_s22", op="ingest", fmt="gt", scale=22, ef=16, skew="rmat", directed=False,
             walkers=65536, length=20),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["walk", "walk_batch", "minibatch", "replay", "mdrw", "decode", "ingest", "load"])
    low, top = {"walk": (14, 23), "walk_batch": (16, 24), "minibatch": (16, 24), "replay": (20, 23), "mdrw": (16, 22),
                "decode": (14, 24), "ingest": (14, 22), "load": (14, 22)}[op]
    scale = rng.randint(low, top)
    ef = rng.choice([e for e in (3, 5, 8, 12, 16, 24) if e << scale <= 16 << top])
    case = dict(op=op, fmt=rng.choice(["le", "gt"]), scale=scale, ef=ef,
                skew=rng.choice(["rmat", "rmat", "mild", "uniform"]))
    if op == "walk":
        case.update(walkers=_log(rng, 40, 1 << 20), length=_log(rng, 5, 80), starts=rng.random() < 0.5)
    elif op == "walk_batch":
        case.update(requests=_log(rng, 2, 256), walkers=_log(rng, 30, 4096))
    elif op == "minibatch":
        seeds = _log(rng, 16, 8192)
        fans = rng.choice(["25,10", "15,10", "10,5", "20", "10,10,5"])
        most = 32768 if fans == "10,10,5" else 131072
        case.update(requests=_log(rng, 1, min(128, max(1, most // seeds))), seeds=seeds, fanouts=fans)
    elif op == "replay":
        case.update(ef=rng.choice([8, 12, 16]), skew=rng.choice(["rmat", "mild"]), requests=_log(rng, 2, 24),
                    walkers=_log(rng, 64, 4096), seeds=_log(rng, 16, 2000),
                    fanouts=rng.choice(["25,10", "15,10", "10,10,5"]))
    elif op == "mdrw":
        case.update(instances=_log(rng, 2, 64), target=_log(rng, 700, 16384), local=rng.random() < 0.3)
    elif op == "ingest":
        case.update(directed=rng.random() < 0.3, walkers=_log(rng, 1000, 65536), length=20)
    elif op == "load":
        case.update(walkers=_log(rng, 1000, 65536), length=20)
    return case


def _edges(case, seed):
    a, b, c = SKEW[case["skew"]]
    return ingest.rmat_edges_device(case["scale"], case["ef"], a, b, c, seed=seed & 0x7FFFFFFF)


def _graph(case, seed):
    src, dst = _edges(case, seed)
    rowptr, col = ingest.graph_sort_device(src, dst)
    del src, dst
    return grass_amd.Graph.from_csr_device(rowptr, col, case["fmt"])


def _ids(n, count, seed):
    gen = torch.Generator(device=DEVICE)
    gen.manual_seed(seed & 0x7FFFFFFF)
    return torch.randint(0, n, (count,), dtype=torch.int32, device=DEVICE, generator=gen)


def _zeros(count, dtype=torch.int32):
    return torch.zeros(count, dtype=dtype, device=DEVICE)


def _ptr(t):
    return C.c_void_p(t.data_ptr())


def _stream():
    return C.c_void_p(torch.cuda.current_stream().cuda_stream)


def _call(name, *args):
    grass_amd._check(getattr(ingest.lib(), name)(*args), name)


def _sizes(case, what):
    """The requests' sizes: the same for every seed."""
    return random.Random("%s %s %s" % (what, case["requests"], case.get("walkers")))


def _walk_requests(case):
    r = _sizes(case, "walks")
    return [dict(walkers=r.randint(1, case["walkers"]), length=r.randint(10, 100), instance=i)
            for i in range(case["requests"])]


def _seed_lists(case, g, seed):
    """One device tensor of seeds per request: `seeds` each in a training batch, about as many on
    average in a served one."""
    counts = [case["seeds"]] * case["requests"]
    if case["op"] == "replay":
        r = _sizes(case, "seeds")
        counts = [max(1, int(c * r.uniform(0.25, 1.75))) for c in counts]
    return list(torch.split(_ids(g.n, sum(counts), seed + 1), counts))


def _fanouts(case):
    return [int(x) for x in case["fanouts"].split(",")]


def _csr_buffers(case):
    """Row pointers and columns of any graph of the case's size."""
    return _zeros((1 << case["scale"]) + 1, torch.int64), _zeros(2 * case["ef"] << case["scale"])


def _induced_room(case):
    return int(1.5 * _induced(case)) + (2 << 20)


def prepare(case, seed):
    op = case["op"]
    st = dict(case=case, seed=seed & 0x7FFFFFFF)
    if op == "ingest":
        st["src"], st["dst"] = _edges(case, seed)
        st["rowptr"], st["col"] = _csr_buffers(case)
        return st
    if op == "load":
        rowptr, col = ingest.graph_sort_device(*_edges(case, seed))
        st["images"] = ingest.compress_device(rowptr, col, case["fmt"])
        return st
    g = st["g"] = _graph(case, seed)
    if op == "walk":
        st["starts"] = _ids(g.n, case["walkers"], seed + 1) if case["starts"] else None
    elif op == "walk_batch":
        reqs = _walk_requests(case)
        sizes = [r["walkers"] * (r["length"] + 1) for r in reqs]
        st["slab"] = _zeros(sum(sizes))
        st["reqs"], st["keep"] = g.rw_request_array(reqs, list(torch.split(st["slab"], sizes)))
    elif op == "minibatch":
        R, fans = case["requests"], _fanouts(case)
        st["reqs"], st["seeds"] = g.khop_request_array(_seed_lists(case, g, seed), [fans] * R)
        front, cap = R * case["seeds"], 0
        nodes = front
        for f in fans:
            front *= f
            cap += front
        out = st["out"] = dict(src=_zeros(cap), dst=_zeros(cap), offsets=_zeros(len(fans) * (R + 1), torch.int64),
                               lsrc=_zeros(cap), ldst=_zeros(cap), nodes=_zeros(nodes + cap),
                               node_off=_zeros(R + 1, torch.int64))
        st["edges"] = grass_amd.KhopOutput(out["src"].data_ptr(), out["dst"].data_ptr(), cap,
                                           out["offsets"].data_ptr(), 0, 0)
        st["blocks"] = grass_amd.KhopBlocks(out["nodes"].data_ptr(), nodes + cap, out["node_off"].data_ptr(),
                                            out["lsrc"].data_ptr(), out["ldst"].data_ptr(), 0)
    elif op == "replay":
        seeds = _seed_lists(case, g, seed)
        p = st["plan"] = g.plan(_walk_requests(case), seeds, [_fanouts(case)] * len(seeds), st["seed"])
        for t in (p.khop_src, p.khop_dst):  # sized by a bound: nothing undefined past the batch's edges
            t.zero_()
    elif op == "mdrw":
        r, top = random.Random(case["target"]), max(2, case["target"] // 4)
        st["frontiers"] = [r.randint(max(1, top // 8), top) for _ in range(case["instances"])]
        steps = sum(case["target"] - m for m in st["frontiers"])
        room = dict(step=steps, verts=case["instances"] * case["target"], ind=_induced_room(case))
        st["out"] = {k: _zeros(room[k.split("_")[0]]) for k in
                     ["step_src", "step_dst", "verts", "ind_src", "ind_dst"] +
                     (["ind_lsrc", "ind_ldst", "step_lsrc", "step_ldst"] if case["local"] else [])}
    elif op == "decode":
        st["rowptr"], st["col"] = _csr_buffers(case)
    return st


def run(st):
    case, seed, op = st["case"], st["seed"], st["case"]["op"]
    if op == "ingest":
        n, m = C.c_uint64(), C.c_uint64()
        _call("grass_graph_sort_device", _ptr(st["src"]), _ptr(st["dst"]), st["src"].numel(), int(case["directed"]), 0,
              _stream(), _ptr(st["rowptr"]), st["rowptr"].numel(), _ptr(st["col"]), st["col"].numel(), C.byref(n),
              C.byref(m))
        with grass_amd.Graph.from_csr_device(st["rowptr"][: n.value + 1], st["col"][: m.value], case["fmt"]) as g:
            walks = g.random_walk(case["walkers"], case["length"], seed)
            return [st["rowptr"], st["col"], walks, g.n, g.m, g.max_degree, g.total_bits]
    if op == "load":
        with grass_amd.Graph.from_bytes(*st["images"], case["fmt"]) as g:
            walks = g.random_walk(case["walkers"], case["length"], seed)
            return [walks, g.n, g.m, g.max_degree, g.total_bits]
    g = st["g"]
    if op == "walk":
        return g.random_walk(case["walkers"], case["length"], seed, starts=st["starts"])
    if op == "walk_batch":
        _call("grass_random_walk_batch", g.handle, st["reqs"], case["requests"], seed, _stream())
        return st["slab"]
    if op == "minibatch":
        _call("grass_khop_batch", g.handle, st["reqs"], case["requests"], seed, C.byref(st["edges"]), _stream())
        _call("grass_khop_blocks_build", g.handle, st["reqs"], case["requests"], C.byref(st["edges"]),
              C.byref(st["blocks"]), _stream())
        return st["out"]
    if op == "replay":
        p = st["plan"]
        p.launch()
        return [p.walks, p.khop_src, p.khop_dst, p.khop_offsets]
    if op == "mdrw":
        res = g.mdrw_tensors(st["frontiers"], case["target"], seed, local=case["local"])
        for k, buf in st["out"].items():
            buf[: res[k].numel()].copy_(res[k])
        return dict(st["out"], step_off=res["step_off"], vert_off=res["vert_off"], ind_off=res["ind_off"])
    _call("grass_decode_csr", g.handle, _ptr(st["rowptr"]), _ptr(st["col"]), _stream())
    return [st["rowptr"], st["col"]]


def exact(case, seed):
    return None


def _graph_size(case):
    """About (vertices, adjacency entries, compressed bytes per entry) of the undirected graph: an
    R-MAT graph repeats some edges and leaves some ids unused."""
    s, ef = case["scale"], case["ef"]
    ids = float(1 << s)
    if case["skew"] == "uniform":
        n, keep = ids * (1 - math.exp(-2 * ef)), 1.0
    elif case["skew"] == "mild":
        n, keep = ids * 0.93, 1 - 0.06 * 2 ** (-0.2 * (s - 12))
    else:
        n, keep = ids * (0.82 - 0.0243 * (s - 12)), 1 - 0.26 * 2 ** (-0.26 * (s - 12))
    m = 2.0 * ef * ids * keep
    per_entry = 1.2 + 0.0495 * s + (0.25 if case["skew"] != "rmat" else 0.0)
    return n, m, per_entry


def _induced(case):
    """About the induced edges of an MDRW batch (a little over, from runs of each kind of graph): an
    entry of a sampled vertex's list is in the sample more often the larger the sample, the denser
    the graph and the more skewed its degrees."""
    n, _, _ = _graph_size(case)
    size = min(case["target"], n)
    dense = (case["target"] / 16384) ** 0.55 * (case["ef"] / 16) ** 0.8
    per = {"rmat": 290 * dense, "mild": 45 * dense * 2 ** ((16 - case["scale"]) / 3), "uniform": 0.0}[case["skew"]]
    return case["instances"] * size * (2 + per + 2 * case["ef"] * size / n)


def work(case):
    """Bytes one pass cannot do without: inputs read once, outputs written once (a sampled neighbour
    costs its vertex's record start, its header, and its own bits)."""
    op = case["op"]
    n, m, bpe = _graph_size(case)
    per_draw = 8 + 4 + bpe  # record start, header, payload bits
    csr = 8 * (n + 1) + 4 * m
    if op == "walk":
        steps = case["walkers"] * case["length"]
        b = steps * (per_draw + 4) + 8 * case["walkers"]
    elif op == "walk_batch":
        steps = case["requests"] * case["walkers"] / 2 * 55
        b = steps * (per_draw + 4)
    elif op in ("minibatch", "replay"):
        front, edges, verts = case["requests"] * case["seeds"], 0.0, 0.0
        verts += front
        for h, f in enumerate(_fanouts(case)):
            drawn = front * f * (0.95 if h or case["skew"] == "uniform" else 0.4)
            edges += drawn
            front = 0.8 * drawn
            verts += front
        b = edges * (bpe + 8) + verts * 16
        if op == "minibatch":
            b += edges * 8 + verts * 4
        else:
            b += case["requests"] * case["walkers"] / 2 * 55 * (per_draw + 4)
    elif op == "mdrw":
        verts = case["instances"] * min(case["target"], n)
        b = verts * (per_draw + 12) + _induced(case) * (16 if case["local"] else 8)
    elif op == "decode":
        b = m * bpe + 3 * n + csr
    elif op == "ingest":
        b = 8.0 * case["ef"] * (1 << case["scale"]) + csr + m * bpe
    else:
        b = 2 * (m * bpe + 3 * n)
    return {"bytes": b, "flops": 0}
