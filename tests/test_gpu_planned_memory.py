"""What a program plans a case's memory by (ih_grid_bytes) covers what the case comes
to hold, the buffer that its first transfer of an unpinned host array allocates among
it: a grid of less than the buffer's 4 MiB, one at it and larger ones."""
import numpy as np
import pytest

import impact_hip as ih

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [(8, 8, 8), (57, 121, 57), (118, 71, 91), (505, 9, 129), (129, 65, 65)],
                         ids=lambda n: "x".join(map(str, n)))
def test_a_transfer_is_planned_for(N):
    c = ih.Case(N, (1,) * 6)
    planned = c.lib.ih_grid_bytes(ih.grid_desc(N, (1,) * 6))
    before = c.bytes()
    a = np.zeros(c.shape)
    c.upload(ih.PRE, a)
    grown = c.bytes() - before
    rows = min((N[1] + 7) * (N[2] + 7), (4 << 20) // (8 * (N[0] + 7)))
    assert grown == 8 * (N[0] + 7) * rows
    c.download(ih.PRE)
    assert c.bytes() == before + grown <= planned
    # the coefficient tables and partial sums, which the case does not count: at least
    # 81 values a position, and four buffers of one value a tile of 16 x 16 x 32 points
    parts = 4 * 8 * int(np.prod([-(-n // t) for n, t in zip(N, (16, 16, 32))]))
    assert c.bytes() + 81 * 8 * sum(N) + parts <= planned
    c.close()
