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


if __name__ == "__main__":
    fk.main(globals())
