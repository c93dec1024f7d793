"""The FFN's GEMM kernels on shapes that are known to reach them: the dispatch
is asked first (tests/ffn_plan.py), so that a changed rule fails here and does
not move the coverage.

Each shape runs the training forward and both backwards in both weight layouts.
The contract is bit equality between the layouts and between the saved and the
recomputing backward; against the float64 oracle every output holds the
tolerances of test_gpu_ffn.py and test_gpu_ffn_backward.py (bf16 outputs, rtol
1e-2 and atol 1e-2, for the weight gradients of their largest element)."""
import numpy as np
import pytest
import torch

from credit_amd import hip_lib
from credit_amd.workloads import make_ffn_backward_inputs
from ffn_plan import kernel, products
from oracle import reference as ref

pytestmark = pytest.mark.gpu

EPS = hip_lib.FFN_EPS


def run(x, w1, w2, dout, kn):
    """out, u, h, dx, dw1, dw2 of the training pair, gradients as [d, f] and
    [f, d]; the plain forward and the recomputing backward give the same bits."""
    rows, f = x.shape[0], w1.shape[1 if kn else 0]
    out, plain = (torch.full_like(x, float("nan")) for _ in range(2))
    rstd = torch.full((rows,), float("nan"), device=x.device)
    u, h = (torch.full((rows, f), float("nan"), device=x.device, dtype=torch.bfloat16)
            for _ in range(2))
    saved, again = ([torch.full_like(t, float("nan")) for t in (x, w1, w2)] for _ in range(2))
    cfg = hip_lib.make_cfg()
    hip_lib.ffn(x, w1, w2, plain, EPS, cfg, layout="in_out" if kn else "linear")
    hip_lib.ffn_train_forward(x, w1, w2, out, rstd, u, h, EPS, cfg, kn)
    hip_lib.ffn_backward_saved(x, w1, w2, dout, rstd, u, h, *saved, cfg, kn)
    hip_lib.ffn_backward(x, w1, w2, dout, *again, EPS, cfg, kn)
    torch.cuda.synchronize()
    assert torch.equal(plain, out)
    for a, b in zip(saved, again):
        assert torch.equal(a, b)
    dx, dw1, dw2 = saved
    return [out, u, h, dx] + ([dw1, dw2] if kn else [dw1.t(), dw2.t()])


def check(gpu, rows, d, f, sample=None):
    """`sample`: against the oracle only these rows of out and dx (each depends on
    its own row of x and dout alone)."""
    inputs = make_ffn_backward_inputs(rows, d, torch.Generator().manual_seed(rows + d + f),
                                      ffn_dim=f)
    x, k1, k2, dout = (t.to(gpu) for t in inputs)
    linear = run(x, k1.t().contiguous(), k2.t().contiguous(), dout, False)
    for name, a, b in zip(("out", "u", "h", "dx", "dw1", "dw2"), linear,
                          run(x, k1, k2, dout, True)):
        assert torch.equal(a, b), (name, int((a != b).sum()))
    nx, n1, n2, ng = (t.float().numpy() for t in inputs)
    out, _, _, *got = linear if sample is None else [t[sample] for t in linear[:4]] + linear[4:]
    if sample is not None:
        nx, ng = nx[sample], ng[sample]
    round_a = not (rows % 256 == 0 and f % 256 == 0 and rows * f // 65536 % 8 == 0)
    np.testing.assert_allclose(out.float().cpu().numpy(),
                               ref.ffn_rmsnorm_gelu(nx, n1, n2, EPS, round_a=round_a),
                               rtol=1e-2, atol=1e-2)
    expect = ref.ffn_rmsnorm_gelu_backward(nx, n1, n2, ng, EPS)
    for name, g, e in list(zip(("dx", "dw1", "dw2"), got, expect))[:None if sample is None else 1]:
        scale = 1.0 if name == "dx" else np.abs(e).max()
        excess = np.abs(g.double().cpu().numpy() - e) - 1e-2 * (np.abs(e) + scale)
        assert excess.max() <= 0, (name, excess.max())


# Kernels of a shape's products, by layout where they differ (nn.Linear, [in,
# out]).  256-row ring tiles with every epilogue, on one M-tile skewed; the
# 256-tile kernel with every epilogue, on 136 to 200 tiles, at its shortest K of
# two steps and at six; the held kernel likewise.
SHAPES = [
    ((768, 512, 5504), {"gemm1": "ring 256", "du": "ring 256"}),
    ((1280, 3328, 512), {"gemm2": "ring 256", "da": "ring 256"}),
    ((256, 512, 20480), {"gemm1": "ring 256", "du": "ring 256", "dw1": ("held", "256-tile"),
                         "dw2": ("held", "256-tile")}),
    ((2048, 384, 6400), {"gemm1": "256-tile", "du": "256-tile"}),
    ((5120, 2560, 384), {"gemm2": "256-tile", "da": "256-tile"}),
    ((2048, 128, 4352), {"gemm1": ("held", "256-tile"), "du": ("256-tile", "held")}),
    ((4352, 2048, 128), {"gemm2": ("held", "256-tile"), "da": ("256-tile", "held")}),
    ((384, 2048, 6400), {"dw1": "256-tile", "dw2": "256-tile"}),
    ((640, 640, 6912), {"gemm1": ("held", "ring 128"), "dw1": ("ring 256", "ring 128"),
                         "dw2": ("held", "ring 256")}),
]


def assert_kernels(shape, expected):
    for kn in (False, True):
        plans = products(*shape, kn)
        for product, name in expected.items():
            want = name if isinstance(name, str) else name[kn]
            assert kernel(plans[product]) == want, (shape, kn, product)


@pytest.mark.parametrize("shape,kernels", SHAPES, ids=["x".join(map(str, s)) for s, _ in SHAPES])
def test_kernels(gpu, shape, kernels):
    print(f"ffn kernels {shape} {kernels}", flush=True)
    assert_kernels(shape, kernels)
    check(gpu, *shape)


def test_tall_tiles_split(gpu):
    """256-row tiles with K in two slices (GEMM2 and da): no smaller shape has
    them."""
    shape = (768, 5504, 9600)
    assert_kernels(shape, {"gemm2": "ring 256 split 2", "da": "ring 256 split 2"})
    check(gpu, *shape, sample=np.array([0, 1, 127, 128, 255, 256, 400, 511, 512, 700, 766, 767]))


def test_held_two_to_a_cu(gpu):
    """810 tiles of 32 steps: launched with LDS that keeps the third workgroup off."""
    shape = (1152, 2048, 11520)
    assert_kernels(shape, {"gemm1": ("held", "ring 128"), "du": ("ring 128", "held")})
    assert products(*shape, False)["gemm1"].extra_lds > 0
    check(gpu, *shape, sample=np.array([0, 1, 127, 128, 255, 500, 1023, 1024, 1151]))


def test_one_tall_tile_of_rows_is_skewed():
    for kn in (False, True):
        plan = products(256, 512, 20480, kn)["gemm1"]
        assert (kernel(plan), plan.skew) == ("ring 256", 1)


# 256 rows and more 128-tiles than CUs: the two layouts run different kernels.
@pytest.mark.parametrize("rows,d,f", [(256, 384, 16512), (256, 768, 32896)])
def test_one_tall_tile_of_rows_unskewed(gpu, rows, d, f):
    for kn, name in ((False, "held"), (True, "ring 256")):
        plan = products(rows, d, f, kn)["gemm1"]
        assert (kernel(plan), plan.skew) == (name, 0)
    check(gpu, rows, d, f)
