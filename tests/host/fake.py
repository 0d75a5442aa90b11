"""libgrass_amd.so on fake_hip.cpp: for tests of host code (which kernels a call launches, what it does
when memory is short) that run in a process of their own, without torch.

A test module marks its bodies with @on_fake; pytest then runs each in a new process, `python module.py
body`, which ends in main()."""
import ctypes as C
import functools
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
REPO = os.path.dirname(os.path.dirname(HERE))
CHILD = "GRASS_FAKE_HIP"


def on_fake(body):
    @functools.wraps(body)
    def test(tmp_path):
        so = str(tmp_path / "fake_hip.so")
        subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-shared", "-fPIC", "-I/opt/rocm/include", "-o", so,
                        os.path.join(HERE, "fake_hip.cpp")], check=True, timeout=120)
        r = subprocess.run([sys.executable, sys.modules[body.__module__].__file__, body.__name__], timeout=120,
                           capture_output=True, text=True, env=dict(os.environ, **{CHILD: so}))
        assert r.returncode == 0, r.stdout[-3000:] + r.stderr[-3000:]
    test.body = body
    del test.__wrapped__  # (pytest takes the arguments from it)
    return test


def main(module):
    """Runs the body named on the command line."""
    sys.path.insert(0, REPO)
    sys.modules["torch"] = None  # its HIP runtime stays out
    fake = C.CDLL(os.environ[CHILD], mode=C.RTLD_GLOBAL)
    fake.fake_limit.argtypes = [C.c_size_t]
    fake.fake_limit_of.argtypes = [C.c_int, C.c_size_t]
    fake.fake_used.restype = fake.fake_room.restype = fake.fake_copies_in_capture.restype = C.c_size_t
    fake.fake_room.argtypes = [C.c_size_t]
    fake.fake_launches.restype = C.c_char_p
    import grass_amd
    module[sys.argv[1]].body(fake, grass_amd)


def used(fake):
    return fake.fake_used(0)


def unlimited(fake):
    fake.fake_limit(C.c_size_t(-1).value)


def launches(fake):
    """[(kernel's mangled name, workgroups, the first argument's first three words)] since the last call."""
    rows = [l.split() for l in fake.fake_launches().decode().splitlines()]
    return [(r[0], int(r[1]), [int(x) for x in r[2:]]) for r in rows]


def graph(ga, n, fmt=0):
    """A graph of n vertices without edges (no kernel ran)."""
    g, rp = C.c_void_p(), C.create_string_buffer(64)
    rc = ga.lib().grass_compress_device_open(rp, None, n, fmt, 0, None, C.byref(g))
    assert rc == ga.OK, rc
    return g


def requests(ga, counts, fanouts):
    """k-hop requests of so many seeds at an address that is not read."""
    reqs = (ga.KhopRequest * len(counts))()
    for q, k in zip(reqs, counts):
        q.seeds_dev, q.num_seeds, q.hops = 64, k, len(fanouts)
        for h, f in enumerate(fanouts):
            q.fanout[h] = f
    return reqs


def blocks(ga, g, counts, edges, hops=1, fanouts=(10,)):
    """grass_khop_blocks_build of such requests and `edges` batch edges."""
    b = ga.KhopOutput(src_dev=64, dst_dev=64, capacity=edges, offsets_dev=64, total=edges, max_hops=hops)
    out = ga.KhopBlocks(nodes_dev=64, node_capacity=1, node_off_dev=64, lsrc_dev=64, ldst_dev=64)
    reqs = requests(ga, counts, fanouts)
    return ga.lib().grass_khop_blocks_build(g, reqs, len(reqs), C.byref(b), C.byref(out), None)


def khop(ga, g, counts, fanouts):
    o = ga.KhopOutput(src_dev=64, dst_dev=64, capacity=1 << 20, offsets_dev=64)
    reqs = requests(ga, counts, fanouts)
    return ga.lib().grass_khop_batch(g, reqs, len(reqs), 1, C.byref(o), None)
