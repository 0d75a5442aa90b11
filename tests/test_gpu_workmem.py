"""Working memory kept between calls: several threads ingest, load and sample graphs of different sizes
at once, on streams of their own, over and over, so that blocks pass from one thread's call to
another's; every result must equal the one computed alone."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_blocks_shared_by_threads():
    import torch

    import grass_amd
    from grass_amd import ingest
    assert torch.cuda.is_available()
    grass_amd.lib()

    def work(scale, fmt, stream):
        with torch.cuda.stream(stream):
            src, dst = ingest.rmat_edges_device(scale, 8, seed=scale, stream=stream)
            stream.synchronize()
            rp, col = ingest.graph_sort_device(src, dst, stream=stream)
            g = grass_amd.Graph.from_csr_device(rp, col, fmt, stream=stream)
            gb, ob = ingest.compress_device(rp, col, fmt, stream=stream)
            h = grass_amd.Graph.from_bytes(gb, ob, fmt)
            out = [*g.decode_csr(stream=stream), *h.decode_csr(stream=stream)]
            m = g.mdrw([9, 40], target=300, seed=scale, stream=stream)
            out += [m[k] for k in ("step_dst", "verts", "ind_src", "ind_dst")]
            out += [rp.cpu().numpy(), col.cpu().numpy()]
            g.close()
            h.close()
        return out

    jobs = [(10, "le"), (12, "gt"), (14, "le"), (13, "gt")]
    expect = [work(s, f, torch.cuda.Stream()) for s, f in jobs]
    for e in expect:  # the decodes are the sorted CSR
        np.testing.assert_array_equal(e[0], e[-2].view(np.uint64))
        np.testing.assert_array_equal(e[1], e[-1].view(np.uint32))
        np.testing.assert_array_equal(e[1], e[3])
    failed = []

    def loop(i):
        try:
            stream = torch.cuda.Stream()
            for _ in range(4):
                for a, b in zip(work(*jobs[i], stream), expect[i]):
                    np.testing.assert_array_equal(a, b)
        except Exception as x:  # reported by the main thread
            failed.append((i, repr(x)))

    print("[work memory] 4 threads x 4 rounds", flush=True)
    threads = [threading.Thread(target=loop, args=(i,)) for i in range(len(jobs))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed, failed
