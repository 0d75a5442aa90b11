"""Calls that go on when memory is short (on a HIP runtime of host memory, tests/host): what they fall
back to must work, and what they leave must fit the next call."""
import os
import sys

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "host"))
import fake as fk  # noqa: E402

P = (1 << 20) + 77  # positions that go by partition (31 bytes each of working memory, the table 20)


def _blocks(fake, ga, vertices, free):
    """The kernels of blocks of P positions, with so much device memory free beside the graph's."""
    g = fk.graph(ga, vertices)
    fk.launches(fake)
    fake.fake_limit(free)
    rc = fk.blocks(ga, g, [P - 50], 50)
    assert rc == ga.OK, ga.strerror(rc)
    return " ".join(k for k, _, _ in fk.launches(fake))


@fk.on_fake
def test_blocks_without_partition_memory(fake, ga):
    names = _blocks(fake, ga, 1 << 12, 25 * P)
    assert "rel_insert_kernel" in names and "rel_part" not in names


@fk.on_fake
def test_blocks_on_memory_others_left(fake, ga):
    """The partition's memory is there once the blocks that building the graph left idle are freed."""
    names = _blocks(fake, ga, 1 << 20, 25 * P)
    assert "rel_part_dedup_kernel" in names and "rel_insert" not in names


if __name__ == "__main__":
    fk.main(globals())
