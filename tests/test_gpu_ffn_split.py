"""The FFN's BM x 128 tile GEMM: K split over workgroups, and the same product
without room for its partial sums.

Every product is one sum per element: bf16 products exact in fp32, added in
fp32 in a fixed order.  Against the float64 oracle the outputs carry the bf16
roundings the oracle restates (a, h) and their own: within the rtol 1e-2 / atol
1e-2 of every bf16 output.  A caller workspace too small for the partial sums
changes the launch, not the order of the additions, so those outputs agree bit
for bit."""
import numpy as np
import pytest
import torch

from credit_amd import hip_lib
from credit_amd.workloads import make_ffn_inputs
from oracle import reference as ref

pytestmark = pytest.mark.gpu

EPS = hip_lib.FFN_EPS
WS_FIXED = 256 + (1 << 20) + (4 << 20)  # header, counters, slots

# (rows, d, f), 128-row tiles: one M-tile with GEMM2's K split 15, 16 and an
# uneven 7 ways (74 K-steps), two with 6, and without a split 200 to 128 tiles
# and odd multiples of 128 in every dimension.
SHAPES = [(128, 128, 8192), (128, 256, 16384), (128, 384, 4736), (256, 2048, 6400),
          (1024, 2048, 3200), (384, 640, 1152)]


def make(rows, d, f, layout, gpu):
    x, w1, w2 = (t.to(gpu) for t in make_ffn_inputs(
        rows, d, torch.Generator().manual_seed(rows + d + f), ffn_dim=f))
    if layout == "linear":
        w1, w2 = w1.t().contiguous(), w2.t().contiguous()
    return x, w1, w2


def run(x, w1, w2, layout, workspace=None):
    out = torch.full_like(x, float("nan"))
    hip_lib.ffn(x, w1, w2, out, EPS, hip_lib.make_cfg(workspace=workspace), layout=layout)
    torch.cuda.synchronize()
    return out


@pytest.mark.parametrize("layout", ["linear", "in_out"])
@pytest.mark.parametrize("rows,d,f", SHAPES)
def test_split_products(gpu, rows, d, f, layout):
    print(f"ffn split rows={rows} d={d} f={f} {layout}", flush=True)
    x, w1, w2 = make(rows, d, f, layout, gpu)
    out = run(x, w1, w2, layout)
    k1, k2 = (w1, w2) if layout == "in_out" else (w1.t(), w2.t())
    expect = ref.ffn_rmsnorm_gelu(x.float().cpu().numpy(), k1.float().cpu().numpy(),
                                  k2.float().cpu().numpy(), EPS)
    np.testing.assert_allclose(out.float().cpu().numpy(), expect, rtol=1e-2, atol=1e-2)
    # The least workspace the call takes: rstd and h, no room for anything else.
    least = torch.zeros(WS_FIXED + 4 * rows + 2 * rows * f, dtype=torch.uint8, device=gpu)
    assert torch.equal(run(x, w1, w2, layout, least), out)
    full = torch.zeros(hip_lib.workspace_bytes("ffn", rows, f), dtype=torch.uint8, device=gpu)
    assert torch.equal(run(x, w1, w2, layout, full), out)


@pytest.mark.parametrize("layout", ["linear", "in_out"])
@pytest.mark.parametrize("rows,d,f", [(128, 256, 8192), (384, 640, 1152), (2048, 256, 256)])
def test_output_in_place_of_x(gpu, rows, d, f, layout):
    """The output holds the normalised copy of x until the last product writes
    it, but not where it is x: the same bits, with room for a copy or none."""
    print(f"ffn in place rows={rows} d={d} f={f} {layout}", flush=True)
    x, w1, w2 = make(rows, d, f, layout, gpu)
    out = run(x, w1, w2, layout)
    least = torch.zeros(WS_FIXED + 4 * rows + 2 * rows * f, dtype=torch.uint8, device=gpu)
    for workspace in (None, least):
        y = x.clone()
        hip_lib.ffn(y, w1, w2, y, EPS, hip_lib.make_cfg(workspace=workspace), layout=layout)
        torch.cuda.synchronize()
        assert torch.equal(y, out)


@pytest.mark.parametrize("rows,d,f", [(128, 256, 8192), (1024, 2048, 3200)])
def test_train_forward_captured_first(gpu, rows, d, f):
    """The training forward as a stream's first call, under capture (it can
    allocate nothing there): replays give the eager call's bits."""
    x, w1, w2 = make(rows, d, f, "linear", gpu)

    def outputs():
        return (torch.zeros_like(x), torch.zeros(rows, device=gpu),
                torch.zeros(rows, f, device=gpu, dtype=torch.bfloat16),
                torch.zeros(rows, f, device=gpu, dtype=torch.bfloat16))

    captured, eager = outputs(), outputs()
    graph = torch.cuda.CUDAGraph()
    stream = torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=stream):
        hip_lib.ffn_train_forward(x, w1, w2, *captured, EPS, hip_lib.make_cfg())
    for i in range(3):
        x.mul_(-1.0)
        hip_lib.ffn_train_forward(x, w1, w2, *eager, EPS, hip_lib.make_cfg())
        graph.replay()
        torch.cuda.synchronize()
        for a, b in zip(captured, eager):
            assert torch.equal(a, b), i


# More 128-tiles than CUs in GEMM1 (258 tiles of two K-steps; 270 of five), in
# GEMM2 (272 of 18) and in the weight gradients.
@pytest.mark.parametrize("rows,d,f", [(384, 128, 11008), (640, 640, 6912), (2176, 2048, 1152)])
def test_more_tiles_than_cus(gpu, rows, d, f):
    """Several workgroups to a CU in the nn.Linear layout, the ring kernel in the
    [in, out] one: the same additions in the same order."""
    print(f"ffn held rows={rows} d={d} f={f}", flush=True)
    x, w1, w2 = make(rows, d, f, "linear", gpu)
    k1, k2 = w1.t().contiguous(), w2.t().contiguous()
    out = run(x, w1, w2, "linear")
    assert torch.equal(run(x, k1, k2, "in_out"), out)
    expect = ref.ffn_rmsnorm_gelu(x.float().cpu().numpy(), k1.float().cpu().numpy(),
                                  k2.float().cpu().numpy(), EPS)
    np.testing.assert_allclose(out.float().cpu().numpy(), expect, rtol=1e-2, atol=1e-2)
    dout = torch.randn(rows, d, generator=torch.Generator().manual_seed(f)).to(gpu, torch.bfloat16)
    grads = []
    for a, b, kn in ((w1, w2, False), (k1, k2, True)):
        y, rstd = torch.empty_like(x), torch.empty(rows, device=gpu)
        u = torch.empty(rows, f, device=gpu, dtype=torch.bfloat16)
        h, g = torch.empty_like(u), (torch.empty_like(x), torch.empty_like(a), torch.empty_like(b))
        hip_lib.ffn_train_forward(x, a, b, y, rstd, u, h, EPS, hip_lib.make_cfg(), kn)
        hip_lib.ffn_backward_saved(x, a, b, dout, rstd, u, h, *g, hip_lib.make_cfg(), kn)
        torch.cuda.synchronize()
        assert torch.equal(y, out)
        grads.append((g[0], g[1].t() if kn else g[1], g[2].t() if kn else g[2]))
    for a, b in zip(*grads):
        assert torch.equal(a, b)
