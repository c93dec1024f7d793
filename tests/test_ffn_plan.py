"""The FFN's dispatch rules on the host (credit_amd/csrc/ffn_plan.hpp).  No GPU."""
import shutil

import pytest

from ffn_plan import gemm_plan, kernel, products

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


@pytest.mark.parametrize("m,n,k", [(1920, 3200, 9600), (2176, 9600, 2432), (1408, 3584, 9600)])
def test_an_unsplit_product_is_priced_on_the_kernel_that_runs_it(m, n, k):
    """Products that the ring kernel would run faster in two K slices and the
    held kernel faster whole."""
    assert kernel(gemm_plan(m, n, k, False)) == "held"
    assert gemm_plan(m, n, k, True).slices == 1


@pytest.mark.parametrize("m,n,k,two", [(4736, 3328, 5376, True), (2176, 6912, 2304, True),
                                       (4096, 2944, 1024, False), (2816, 9600, 1792, False), (1024, 13440, 768, False),
                                       (4224, 8576, 2176, False)])
def test_held_workgroups_to_a_cu(m, n, k, two):
    """Two to a CU where the third would leave a round nearly empty."""
    plan = gemm_plan(m, n, k, False)
    assert plan.held
    lds = 36864 + plan.extra_lds
    assert lds <= 65536 and ((160 << 10) // lds == 2) == two


@pytest.mark.parametrize("rows,d,f", [(2176, 2304, 6912), (4224, 2176, 8576)])
def test_backward_workspace_holds_no_copy_of_the_input(lib, rows, d, f):
    """Where no product is split the backward's workspace is its own regions
    (rstd; u, du, h^T, du^T; dout^T, a^T; da): the rounded copy of x that these
    shapes read passes through da, so that no workspace is too small for it."""
    assert all(p.slices == 1 for p in products(rows, d, f, False).values())
    own = [4 * rows] + 4 * [2 * rows * f] + 2 * [2 * rows * d] + [4 * rows * d]
    fixed = 256 + (1 << 20) + (4 << 20)
    assert lib.credit_ffn_bwd_workspace_bytes(rows, d, f) <= fixed + sum(own) + 256 * len(own)
