"""Which blocks go by partition (on a HIP runtime of host memory, tests/host): requests whose distinct
vertices its buckets hold."""
import os
import sys

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "host"))
import fake as fk  # noqa: E402

DISTINCT = 8192 * 3072


def _parts(fake, ga, g, counts, edges, fanouts):
    fk.launches(fake)
    rc = fk.blocks(ga, g, counts, edges, len(fanouts), fanouts)
    assert rc == ga.OK, ga.strerror(rc)
    names = " ".join(k for k, _, _ in fk.launches(fake))
    assert ("rel_part_dedup_kernel" in names) != ("rel_insert_kernel" in names)
    return "rel_part_dedup_kernel" in names


@fk.on_fake
def test_a_request_of_many_distinct_vertices(fake, ga):
    g = fk.graph(ga, DISTINCT + 1)
    # (the graph has no edges, so only seeds can be distinct vertices)
    assert _parts(fake, ga, g, [DISTINCT - 10], 10, (1,))
    assert _parts(fake, ga, g, [DISTINCT], 10, (1,))
    assert not _parts(fake, ga, g, [DISTINCT + 1], 0, (1,))
    assert not _parts(fake, ga, g, [DISTINCT * 3], 10, (1,))
    assert not _parts(fake, ga, g, [1 << 20, DISTINCT * 2], 10, (1,))
    assert _parts(fake, ga, g, [DISTINCT // 2] * 4, 10, (1,))


@fk.on_fake
def test_few_vertices(fake, ga):
    """Any number of positions where the graph has no more vertices than that."""
    g = fk.graph(ga, DISTINCT)
    assert _parts(fake, ga, g, [DISTINCT * 3], 10, (1,))


@fk.on_fake
def test_positions_near_the_end_of_32_bits(fake, ga):
    """A bucket's positions are counted by 4096 in 32 bits."""
    g = fk.graph(ga, 1 << 12)
    last = 2 ** 32 - 4096 - 1
    assert _parts(fake, ga, g, [2 ** 31, last - 2 ** 31 - 5], 5, (1,))
    assert not _parts(fake, ga, g, [2 ** 31, last - 2 ** 31 - 4], 5, (1,))


if __name__ == "__main__":
    fk.main(globals())
