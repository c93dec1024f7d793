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


def check(gpu, rows, d, f):
    inputs = make_ffn_backward_inputs(rows, d, torch.Generator().manual_seed(rows + d + f),
                                      ffn_dim=f)
    x, k1, k2, dout = (t.to(gpu) for t in inputs)
    linear = run(x, k1.t().contiguous(), k2.t().contiguous(), dout, False)
    for name, a, b in zip(("out", "u", "h", "dx", "dw1", "dw2"), linear,
                          run(x, k1, k2, dout, True)):
        assert torch.equal(a, b), (name, int((a != b).sum()))
    nx, n1, n2, ng = (t.float().numpy() for t in inputs)
    got = [t.float().cpu().numpy() for t in linear]
    round_a = not (rows % 256 == 0 and f % 256 == 0 and d % 128 == 0 and
                   rows * f // 65536 % 8 == 0)
    np.testing.assert_allclose(got[0], ref.ffn_rmsnorm_gelu(nx, n1, n2, EPS, round_a=round_a),
                               rtol=1e-2, atol=1e-2)
    expect = ref.ffn_rmsnorm_gelu_backward(nx, n1, n2, ng, EPS)
    for name, g, e, scale in zip(("dx", "dw1", "dw2"), got[3:], expect,
                                 (1.0, np.abs(expect[1]).max(), np.abs(expect[2]).max())):
        excess = np.abs(g.astype(np.float64) - e) - 1e-2 * (np.abs(e) + scale)
        assert excess.max() <= 0, (name, excess.max())


# 256 rows and more 128-tiles than CUs: the two layouts run different kernels.
@pytest.mark.parametrize("rows,d,f", [(256, 384, 16512), (256, 768, 32896)])
def test_one_tall_tile_of_rows_unskewed(gpu, rows, d, f):
    for kn, name in ((False, "held"), (True, "ring 256")):
        plan = products(rows, d, f, kn)["gemm1"]
        assert (kernel(plan), plan.skew) == (name, 0)
    check(gpu, rows, d, f)
