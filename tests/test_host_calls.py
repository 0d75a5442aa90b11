"""What calls do to streams and memory on the host's side (on a HIP runtime of host memory, tests/host)."""
import ctypes as C
import os
import sys

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "host"))
import fake as fk  # noqa: E402


@fk.on_fake
def test_sync_of_a_capturing_stream(fake, ga):
    """Refused, and nothing is left in the caller's graph."""
    g = fk.graph(ga, 1 << 12)
    s = C.c_void_p(4096)
    assert ga.lib().grass_sync(g, s) == ga.OK
    fake.fake_capturing(1)
    assert ga.lib().grass_sync(g, s) == ga.EDEVICE
    assert fake.fake_copies_in_capture() == 0
    fake.fake_capturing(0)
    assert ga.lib().grass_sync(g, s) == ga.OK


def _idle(fake, ga):
    """A graph whose building left memory idle, and no other: (graph, bytes idle)."""
    before = fk.used(fake)
    g = fk.graph(ga, 1 << 20)
    idle = fk.used(fake) - before - 20 * (1 << 20)  # (headers and degrees)
    assert idle > 16 << 20
    fake.fake_limit(0)
    return g, idle


@fk.on_fake
def test_device_alloc_on_idle_memory(fake, ga):
    g, idle = _idle(fake, ga)
    p = C.c_void_p()
    assert ga.lib().grass_device_alloc(g, idle // 2, C.byref(p)) == ga.OK


@fk.on_fake
def test_graph_on_idle_memory(fake, ga):
    g, idle = _idle(fake, ga)
    fk.graph(ga, 1 << 10)  # (its working memory does not fit any idle block)


@fk.on_fake
def test_session_on_idle_memory(fake, ga):
    from grass_amd import serve
    g, idle = _idle(fake, ga)
    cfg = serve.Config(idle // 2, 4, 1, 1, 1024)
    s = C.c_void_p()
    assert serve.lib().grass_session_create(g, C.byref(cfg), C.byref(s)) == ga.OK
    assert serve.lib().grass_session_destroy(s) == ga.OK


@fk.on_fake
def test_pinned_memory_that_fails(fake, ga):
    """A failure is in the status alone."""
    g = fk.graph(ga, 1 << 10)
    fake.fake_limit_of(1, 0)
    assert fk.khop(ga, g, [100] * 1000, (2, 2)) == ga.ENOMEM
    assert fake.hipGetLastError() == 0


def _left(fake, ga):
    """A graph on 4096 vertices, with the working memory of a larger one, closed, idle: (graph, bytes idle)."""
    g = fk.graph(ga, 1 << 12)
    ga.lib().grass_trim(0)
    before = fk.used(fake)
    big = fk.graph(ga, 1 << 20)
    assert ga.lib().grass_close(big) == ga.OK
    idle = fk.used(fake) - before
    assert idle > 16 << 20  # (kept for the next graph)
    return g, idle


@fk.on_fake
def test_trim(fake, ga):
    g, idle = _left(fake, ga)
    before = fk.used(fake)
    assert ga.lib().grass_trim(0) == ga.OK
    assert fk.used(fake) == before - idle and fake.fake_used(1) == 0
    assert ga.lib().grass_trim(-1) == ga.EINVAL and ga.lib().grass_trim(1) == ga.EINVAL


@fk.on_fake
def test_idle_memory_goes(fake, ga):
    """Blocks idle for 10 s go with the calls of a program that only samples."""
    def walks(g):
        r = ga.RwRequest(64, 4, 0, None, 64)
        return ga.lib().grass_random_walk_batch(g, C.byref(r), 1, 1, None)
    for call in (lambda g: ga.lib().grass_sync(g, C.c_void_p(4096)), lambda g: fk.khop(ga, g, [100], (2, 2)), walks):
        g, idle = _left(fake, ga)
        assert call(g) == ga.OK
        before = fk.used(fake)
        assert call(g) == ga.OK and fk.used(fake) == before
        fake.fake_later(11)
        assert call(g) == ga.OK
        assert fk.used(fake) == before - idle


if __name__ == "__main__":
    fk.main(globals())
