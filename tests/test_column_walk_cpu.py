"""How a group of lanes walks the columns of a row in the dense -> CSR count and fill passes
(sapphire_amd/csrc/sph_column_walk.h, reached through the host harness), and the widest row that
the entry points take; no device is needed."""
import ctypes

import pytest

from sapphire_amd import capi
from tests import host_layer as hl

WIDEST = 2**32 - 256


@pytest.mark.parametrize("lanes", [4, 8, 16, 32, 64])
def test_every_column_once_in_order(lanes):
    step = lanes * 4
    ends = [0, 1, 3, 4, 5, step - 1, step, step + 1, 4 * step - 1, 4 * step, 4 * step + 1,
            5 * step - 1, 5 * step, 5 * step + 1, 8191, 8192, 8193]
    if lanes == 64:  # a last batch or step that touches the end of 32 bits
        ends += [WIDEST - d for d in (0, 1, 255, 256, 257, 767, 768, 769, 1024)]
    for N in ends:
        seen, wrong, steps = hl.column_walk(N, lanes, 4)
        assert (seen, wrong) == (N, None), N
        assert steps == (N + step - 1) // step, N


def test_wider_rows_are_refused():
    """Before anything is enqueued: the addresses are never followed."""
    some = ctypes.create_string_buffer(64)
    p, N = ctypes.addressof(some), WIDEST + 1
    for entry, args in (("sph_csr_row_offsets_f32", (p, p, 1, N, N, None)),
                        ("sph_csr_row_offsets_noalloc_f32", (p, p, 1, N, N)),
                        ("sph_csr_from_dense_f32", (p, p, p, 1, p, 1, N, N, None)),
                        ("sph_csr_fill_f32", (p, p, p, p, 1, N, N))):
        with pytest.raises(capi.SphError, match="columns"):
            capi.call(entry, *args)
