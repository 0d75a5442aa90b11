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


def _table_fits(fake, ga, g):
    """A batch on the 16-byte table clears no more than the table's memory."""
    os.environ["GRASS_KHOP_SLOT"] = "16"
    fk.launches(fake)
    rc = fk.khop(ga, g, [5000], (10, 10))
    assert rc == ga.OK, ga.strerror(rc)
    clears = [a for k, _, a in fk.launches(fake) if "ht_clear_kernel" in k]
    assert clears  # (new memory holds anything)
    for slot, mask, _ in clears:
        assert fake.fake_room(slot) >= (mask + 1) * 16
    del os.environ["GRASS_KHOP_SLOT"]


@fk.on_fake
def test_khop_table_after_failed_blocks(fake, ga):
    """The 16-byte table's size is not remembered past its memory: blocks that failed gave that back, and
    smaller ones took less in its place."""
    g = fk.graph(ga, 1 << 12)
    os.environ["GRASS_KHOP_SLOT"] = "16"
    assert fk.khop(ga, g, [500_000], (10, 10)) == ga.OK
    del os.environ["GRASS_KHOP_SLOT"]
    fake.fake_limit(P)
    assert fk.blocks(ga, g, [4 * P], 50) == ga.ENOMEM
    fk.unlimited(fake)
    assert fk.blocks(ga, g, [20_000], 50) == ga.OK
    _table_fits(fake, ga, g)


@fk.on_fake
def test_khop_table_after_a_failed_one(fake, ga):
    """Nor past a larger table that could not be had (but the batch's other memory, 215 MB, could)."""
    g = fk.graph(ga, 1 << 12)
    os.environ["GRASS_KHOP_SLOT"] = "16"
    assert fk.khop(ga, g, [500_000], (10, 10)) == ga.OK
    fake.fake_limit(250 << 20)
    assert fk.khop(ga, g, [4 * P], (10, 10)) == ga.ENOMEM
    fk.unlimited(fake)
    _table_fits(fake, ga, g)


if __name__ == "__main__":
    fk.main(globals())
