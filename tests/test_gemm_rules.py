"""Which form a GEMM launch takes, by its sizes: both sides of every line."""

import pytest
from gemm_rules import call, m_grouped_tile_rows, schedule


@pytest.mark.parametrize("groups,largest,rest,per_group,form", [
    # a tile of a whole share or more
    (64, 200, 4, 24, "parts"), (64, 50, 1, 24, "in order"),
    (16, 900, 1, 60, "parts"),
    # groups of few tiles, of which an eighth is two or three or none: never eighths, whatever the skew
    (128, 120, 10, 24, "parts"), (128, 36, 10, 24, "in order"), (120, 48, 25, 5, "parts"), (256, 60, 40, 1, "parts"), (64, 100, 60, 8, "parts"),
    (128, 70, 4, 24, "parts"),
    (128, 75, 5, 32, "eighths"), (128, 40, 9, 32, "in order"), (64, 40, 5, 36, "in order"),
    # from 40 tiles on: a group of a 25th of the work
    (64, 60, 13, 88, "eighths"), (64, 30, 13, 88, "in order"), (64, 20, 3, 40, "eighths"), (128, 60, 10, 48, "in order"), (128, 80, 8, 48, "eighths"),
    (32, 18, 5, 276, "eighths"), (128, 15, 10, 144, "eighths"), (128, 15, 10, 120, "in order"), (32, 4, 3, 40, "in order"), (8, 14, 4, 276, "eighths"),
    (6, 12, 2, 276, "in order"),
])
def test_schedule_of_skewed_groups(groups, largest, rest, per_group, form):
    blocks = [rest] * groups
    blocks[groups // 3] = largest
    got, share, most = schedule(blocks, per_group)
    assert got == form, (got, share, most)


def test_parts_of_a_share_that_are_dealt_out_one_by_one():
    assert [call("big_tile_parts", form, blocks * 256, 256) for form in (1, 2) for blocks in (56, 139, 140, 400)] == [8, 8, 16, 16, 8, 8, 8, 8]


def test_few_used_rows_are_counted_without_their_padding():
    assert [call("few_used_rows", rows, 128) for rows in (0, 128 * 16, 128 * 120, 128 * 120 + 1, 128 * 160)] == [1, 1, 1, 0, 0]



@pytest.mark.parametrize("groups,n,k", [(128, 1536, 2048), (128, 2048, 768), (64, 2816, 2048)])
def test_a_capacity_and_exact_sizes_take_the_same_tiles(groups, n, k):
    """The rows that count decide, not the padded rows that hold them: whole blocks of the routing's own sizes, or as many as
    any routing could need."""
    for rows in (16, 64, 96, 120, 121, 128, 136, 150):
        exact = groups * (128 if rows <= 110 else 128 * 3 // 2)  # a half of the groups past one block, of those with 128 rows in the mean
        capacity = (rows * groups + 127 * groups + 127) // 128 * 128
        answers = {m_grouped_tile_rows(padded, n, k, groups, rows * groups) for padded in (exact, capacity)}
        assert answers == {128 if rows <= 120 else 0}, rows


def test_weights_that_are_read_again_stay_in_the_memory_side_cache():
    """128 MiB and more of whole lines, for groups of up to one and a half tiles of 128 rows, counted with half a tile of padding
    where a capacity holds them; groups of 64 rows always."""

    def streams(rows, groups=16, n=4096, k=2048, used=None, ldb=None, few=0):
        return call("streams_weights", rows * groups, n, k, groups, used is not None, (used or 0) * groups, ldb or k, few)

    assert [streams(rows) for rows in (128, 192, 193, 256, 384, 640)] == [1, 1, 0, 0, 0, 0]
    assert [streams(rows + 127, used=rows) for rows in (16, 120, 128, 129, 300)] == [1, 1, 1, 0, 0]
    assert streams(192, used=192) and not streams(256, used=192)  # whole blocks of rows that all count
    assert streams(640, few=1) and not streams(128, n=4080) and not streams(128, groups=15) and not streams(128, ldb=2080)
