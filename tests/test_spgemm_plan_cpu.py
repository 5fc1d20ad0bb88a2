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
