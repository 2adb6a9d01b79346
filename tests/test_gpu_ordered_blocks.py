"""The ordered plasma depositions against the oracle, bit for bit, on grids large enough for the larger
deposition blocks (the smallest ones serve the grids of the other tests): near a lattice, crossing,
with more particles in a window than are sequenced at a time, wrapped and shuffled, and sizes that
leave remainders of a block.
"""
import pytest

pytest.importorskip("torch")

import test_gpu_ordered as ordered  # noqa: E402

pytestmark = pytest.mark.gpu

# nx, ny, ppc, amp (cells), wrapped, shuffled, tile
CASES = [(363, 377, 1, 0.1, 0, False, 32), (361, 379, 2, 3.0, 300, False, 24), (131, 1029, 3, 2.0, 0, False, 32),
         (505, 523, 1, 1.0, 0, False, 32), (523, 509, 3, 2.0, 100, False, 9), (1031, 301, 1, 1.0, 0, True, 64)]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(str(v) for v in c))
@pytest.mark.parametrize("order,dtype", [(2, 2), (3, 2), (0, 1)])
def test_ordered_blocks(case, order, dtype):
    ordered.test_ordered_depositions(case, order, dtype)
