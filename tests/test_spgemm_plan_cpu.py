"""Arithmetic of the CSR x CSR launches (sapphire_amd/csrc/sph_spgemm_plan.h, reached through the
host harness; no device is needed)."""
import pytest

from tests import host_layer as hl


@pytest.mark.parametrize("rows_per_turn", range(1, 9))
def test_turns_cover_every_row_and_no_row_makes_no_turn(rows_per_turn):
    for M in [0, 1, 2, 7, 8, 9, 63, 64, 65, 8191, 65536, 2**32 - 9, 2**32 - 2, 2**32 - 1]:
        turns = hl.spgemm_turns(M, rows_per_turn)
        assert turns * rows_per_turn >= M
        assert max(turns - 1, 0) * rows_per_turn < M or (M == 0 and turns == 0), M


def test_staging_asks_for_less_when_the_device_is_full():
    M, capacity = 1000, 50000  # 50 entries per row
    plenty, lean = 3 * 50 + 64, 2 * 50 + 64
    assert hl.staging_slot(M, 10, capacity, 8 * plenty * M) == (plenty, [plenty])
    assert hl.staging_slot(M, 10, capacity, 8 * plenty * M - 1) == (lean, [plenty, lean])
    assert hl.staging_slot(M, 10, capacity, 8 * lean * M - 1) == (0, [plenty, lean])
    for empty in ((0, 10, 5), (10, 0, 5), (10, 10, 0)):
        assert hl.staging_slot(*empty, 2**40) == (0, [])


def test_a_kept_block_is_larger_only_where_there_is_room():
    for bytes, room, want in [(1000, 1250, (1250, [1250])), (1000, 1249, (1000, [1250, 1000])),
                              (1000, 1000, (1000, [1250, 1000])), (1000, 999, (0, [1250, 1000])),
                              (1800, 2000, (2000, [2000])), (1800, 1999, (1800, [2000, 1800])),
                              (2000, 1999, (0, [2000])), (2000, 2000, (2000, [2000])), (1, 1, (1, [1]))]:
        assert hl.take_with_room(bytes, 2000, room) == want, (bytes, room)


def test_staging_stays_below_the_limit_of_its_indexes():
    room = 2**60
    # one row: 3 * capacity + 64 against 2^31
    most = (2**31 - 1 - 64) // 3
    assert hl.staging_slot(1, 10, most, room)[0] == 3 * most + 64
    assert hl.staging_slot(1, 10, most + 1, room)[0] == 2 * (most + 1) + 64
    most = (2**31 - 1 - 64) // 2
    assert hl.staging_slot(1, 10, most, room)[0] == 2 * most + 64
    assert hl.staging_slot(1, 10, most + 1, room) == (0, [])
    assert hl.staging_slot(1, 10, 2**32 - 1, room) == (0, [])
    # the slots of all rows together
    rows = (2**31 - 1) // 64
    assert hl.staging_slot(rows, 10, rows - 1, room)[0] == 64
    assert hl.staging_slot(rows + 1, 10, rows, room) == (0, [])
    assert hl.staging_slot(2**32 - 2, 10, 2**32 - 1, room) == (0, [])
