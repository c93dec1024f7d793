"""The FFN's dispatch rules on the host (credit_amd/csrc/ffn_plan.hpp).  No GPU."""
import shutil

import pytest

from ffn_plan import gemm_plan

pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")

# Multiples of 128 up to the sizes of a large model, denser at the small end.
ROWS = [128 * i for i in (1, 2, 3, 4, 6, 8, 9, 12, 15, 16, 17, 24, 25, 32, 64)]
WIDTHS = [128 * i for i in (1, 2, 3, 5, 6, 8, 10, 14, 16, 17, 18, 25, 32, 34, 44, 54, 64, 75, 86,
                            88, 96, 111, 112, 128, 129, 130, 148, 192, 224, 257, 258, 300)]


def order(plan):
    """What a product's bits depend on (the 256-tile kernel has no skew)."""
    return plan.slices, 0 if plan.big else plan.skew


def test_order_of_additions_does_not_depend_on_the_layout():
    """The same for a [N, K] and a [K, N] B, whichever kernels run; the slices
    also with M and N exchanged (the weight gradients, which take no skew)."""
    for m in ROWS:
        for n in WIDTHS:
            for k in WIDTHS:
                a, b = gemm_plan(m, n, k, False), gemm_plan(m, n, k, True)
                assert order(a) == order(b), (m, n, k, a, b)
                assert a.slices == gemm_plan(n, m, k, False).slices, (m, n, k)
