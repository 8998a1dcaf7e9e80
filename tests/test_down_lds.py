"""The routed down's LDS copies against the arrays they go to, on the CPU.

From stage Q's rows on, a pick batch's scales are copied into LDS in whole 16-byte pieces, from the
16-byte boundary below the batch's first byte: V4.1's 20 scale bytes a pick start a batch up to 12
bytes into a piece, and the copy ends up to 12 bytes past its last byte.
"""

import pytest

UNITS = range(9)  # the compiled shapes


@pytest.mark.parametrize("unit", UNITS)
def test_pick_batch_copies_stay_in_their_arrays(unit):
    from sgl_amd_mono.moe import _lib

    slack = _lib.testing_lib().mkmoe_host_pick_copy_slack
    over = {rows: slack(unit, rows) for rows in range(1, 49) if slack(unit, rows) < 0}
    assert not over, over
