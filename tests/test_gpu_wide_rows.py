"""Few wide rows in two launches of chunks: both sides of the width and row
rules, the widest row, chunks of a few columns less than the others, a last
column by itself, whole vectors, outputs in place of an input, special values,
and a captured call (which takes another kernel).

fp32 within rtol 1e-5 / atol 1e-6 of the float64 oracle (maxima, int8 codes and
scales bit for bit), bf16 within rtol 1e-2 / atol 1e-2."""
import numpy as np
import pytest
import torch

from credit_amd import hip_lib
from credit_amd.workloads import WORKLOADS
from oracle import reference as ref
from test_gpu_ragged_rows import BF16, FP32, check_guards, output, place, sample

pytestmark = pytest.mark.gpu

# rows, cols, elements past a 16-byte address
SHAPES = [(1, 16385, 0), (3, 20001, 1), (128, 16391, 0), (129, 33001, 0), (1, 262143, 0),
          (2, 262144, 3), (2, 262145, 0), (5, 98309, 2), (300, 66001, 0), (32, 24580, 0),
          (16, 131072, 0), (17, 262144, 0), (1, 262144, 0), (33, 32768, 0),
          (7, 65540, 0)]


@pytest.mark.parametrize("rows,cols,shift", SHAPES)
def test_wide_softmax(gpu, rows, cols, shift):
    print(f"wide softmax {rows} x {cols} + {shift}", flush=True)
    x, dy = WORKLOADS["softmax_fwd"].make_inputs(rows, cols, seed=rows + cols)
    xs, ds = place(x, shift, gpu), place(dy, shift, gpu)
    p, gp = output((rows, cols), torch.float32, shift, gpu)
    m, lse = torch.empty(rows, device=gpu), torch.empty(rows, device=gpu)
    hip_lib.softmax_fwd(xs, p, m, lse, hip_lib.make_cfg())
    gx, gg = output((rows, cols), torch.float32, shift, gpu)
    hip_lib.softmax_bwd(p, ds, gx, hip_lib.make_cfg())
    lx, gl = output((rows, cols), torch.float32, shift, gpu)
    hip_lib.softmax_logits_backward(xs, ds, lx, hip_lib.make_cfg())
    torch.cuda.synchronize()
    check_guards(gp, gg, gl)
    i = sample(rows)
    ep, em, el = ref.softmax_fwd(x[i].numpy())
    np.testing.assert_allclose(p[i].cpu().numpy(), ep, **FP32)
    assert np.array_equal(m[i].cpu().numpy(), em.astype(np.float32))
    np.testing.assert_allclose(lse[i].cpu().numpy(), el, **FP32)
    np.testing.assert_allclose(gx[i].cpu().numpy(),
                               ref.softmax_bwd(p[i].cpu().numpy(), dy[i].numpy()), **FP32)
    np.testing.assert_allclose(lx[i].cpu().numpy(),
                               ref.softmax_logits_backward(x[i].numpy(), dy[i].numpy()), **FP32)
    for t in (p, gx, lx):
        assert not bool(torch.isnan(t).any())
    # In place of the logits.
    hip_lib.softmax_logits_backward(xs, ds, xs, hip_lib.make_cfg())
    assert torch.equal(xs, lx)


@pytest.mark.parametrize("rows,cols,shift", SHAPES)
def test_wide_quant(gpu, rows, cols, shift):
    print(f"wide quant {rows} x {cols} + {shift}", flush=True)
    (x,) = WORKLOADS["rowwise_quant"].make_inputs(rows, cols, seed=rows + cols)
    x[rows // 2] = 0.0
    q, gq = output((rows, cols), torch.int8, shift, gpu)
    scale = torch.empty(rows, device=gpu)
    hip_lib.rowwise_quant(place(x, shift, gpu), q, scale, hip_lib.make_cfg())
    torch.cuda.synchronize()
    check_guards(gq)
    i = sample(rows)
    eq, es = ref.rowwise_quant(x[i].numpy())
    assert np.array_equal(q[i].cpu().numpy(), eq)
    assert np.array_equal(scale[i].cpu().numpy(), es.astype(np.float32))


@pytest.mark.parametrize("rows,cols,shift", SHAPES)
def test_wide_layernorm_backward(gpu, rows, cols, shift):
    print(f"wide layernorm backward {rows} x {cols} + {shift}", flush=True)
    x, dy, gamma = WORKLOADS["layernorm_backward"].make_inputs(rows, cols, seed=rows + cols)
    x = x + 3.0
    xs, ds, gs = (place(t, shift, gpu) for t in (x, dy, gamma))
    dx, gd = output((rows, cols), torch.float32, shift, gpu)
    hip_lib.layernorm_backward(xs, ds, gs, dx, hip_lib.LAYERNORM_EPS, hip_lib.make_cfg())
    torch.cuda.synchronize()
    check_guards(gd)
    i = sample(rows)
    np.testing.assert_allclose(dx[i].cpu().numpy(),
                               ref.layernorm_backward(x[i].numpy(), dy[i].numpy(), gamma.numpy()),
                               **FP32)
    # In place of x: no chunk reads an element that another has written.
    hip_lib.layernorm_backward(xs, ds, gs, xs, hip_lib.LAYERNORM_EPS, hip_lib.make_cfg())
    assert torch.equal(xs, dx)


@pytest.mark.parametrize("cols", [40003, 65536])
def test_wide_softmax_edge_rows(gpu, cols):
    """Rows of -inf, with +inf, with NaN, of the lowest float, and one whose
    first chunks are -inf: p, max and lse as torch gives them."""
    x = torch.randn(5, cols, generator=torch.Generator().manual_seed(1))
    x[0] = -float("inf")
    x[1, 77] = float("inf")
    x[2, cols - 1] = float("nan")
    x[3] = torch.finfo(torch.float32).min
    x[4, :30000] = -float("inf")
    xs = x.to(gpu)
    p, m, lse = hip_lib.allocate_outputs("softmax_fwd", (xs,))
    hip_lib.softmax_fwd(xs, p, m, lse, hip_lib.make_cfg())
    assert torch.equal(m.cpu().isnan(), x.amax(1).isnan())
    assert torch.equal(m.cpu().nan_to_num(7.0), x.amax(1).nan_to_num(7.0))
    assert bool(p[:3].isnan().all())
    np.testing.assert_allclose(p[3:].cpu().numpy(), torch.softmax(x[3:].double(), 1), **FP32)
    assert lse[0].item() == -float("inf") and bool(lse[1:3].isnan().all())
    dy, g, dx = torch.rand_like(xs), torch.ones(cols, device=gpu), torch.empty_like(xs)
    hip_lib.layernorm_backward(xs, dy, g, dx, hip_lib.LAYERNORM_EPS, hip_lib.make_cfg())
    assert bool(dx[:3].isnan().all()) and bool(dx[4].isnan().all())


def test_wide_softmax_captured(gpu):
    """Replays beside eager calls on the stream of the capture."""
    xs = [torch.randn(3, 40003, generator=torch.Generator().manual_seed(i)).to(gpu)
          for i in range(2)]
    eager = [hip_lib.allocate_outputs("softmax_fwd", (x,)) for x in xs]
    captured = hip_lib.allocate_outputs("softmax_fwd", (xs[0],))
    stream = torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        hip_lib.softmax_fwd(xs[0], *eager[0], hip_lib.make_cfg())
    with torch.cuda.graph(graph, stream=stream):
        hip_lib.softmax_fwd(xs[0], *captured, hip_lib.make_cfg())
    for _ in range(3):
        for t in captured:
            t.zero_()
        graph.replay()
        with torch.cuda.stream(stream):
            hip_lib.softmax_fwd(xs[1], *eager[1], hip_lib.make_cfg())
        torch.cuda.synchronize()
        for a, b in zip(captured, eager[0]):
            np.testing.assert_allclose(a.cpu().numpy(), b.cpu().numpy(), **FP32)
    e = ref.softmax_fwd(xs[1].cpu().numpy())
    np.testing.assert_allclose(eager[1][0].cpu().numpy(), e[0], **FP32)


@pytest.mark.parametrize("name,rows,cols", [
    ("softmax_fwd", 16, 131072), ("softmax_bwd", 16, 131072),
    ("softmax_logits_backward", 8, 262144), ("layernorm_backward", 8, 131072),
    ("layernorm_fwd", 16, 131072), ("layernorm_backward_bf16", 16, 131072),
    ("rowwise_quant", 16, 131072)])
def test_wide_aligned_captured_after_a_warm_up(gpu, name, rows, cols):
    """One eager call on a new stream readies it for the captured one, which
    runs SPLIT: its workspace is there."""
    print(f"captured {name} {rows} x {cols}", flush=True)
    ins = tuple(t.to(gpu) for t in WORKLOADS[name].make_inputs(rows, cols, seed=5))
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    eager, captured = (hip_lib.allocate_outputs(name, ins) for _ in range(2))
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        hip_lib.bind(name, ins, eager)()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=stream):
        hip_lib.bind(name, ins, captured)()
    for _ in range(3):
        for t in captured:
            t.zero_()
        graph.replay()
        with torch.cuda.stream(stream):
            hip_lib.bind(name, ins, eager)()
        torch.cuda.synchronize()
        for a, b in zip(captured, eager):
            tol = BF16 if a.dtype == torch.bfloat16 else FP32
            np.testing.assert_allclose(a.float().cpu().numpy(), b.float().cpu().numpy(), **tol)


# bf16: odd widths (chunks of odd rows start inside a dword), even ones, whole
# vectors, a last chunk of few elements.
HALF_SHAPES = [(1, 16385, 0), (4, 20001, 2), (129, 33001, 0), (3, 262143, 0), (2, 262142, 2),
               (5, 98311, 0), (7, 32770, 0), (32, 24584, 0), (16, 131072, 0), (300, 66003, 0),
               (6, 40003, 1)]


@pytest.mark.parametrize("rows,cols,shift", HALF_SHAPES)
def test_wide_layernorm_bf16(gpu, rows, cols, shift):
    print(f"wide bf16 layernorm {rows} x {cols} + {shift}", flush=True)
    x, gamma, beta = WORKLOADS["layernorm_fwd"].make_inputs(rows, cols, seed=rows + cols)
    x[: rows // 2] += 3.0
    xs, gs, bs = (place(t, shift, gpu) for t in (x, gamma, beta))
    y, gy = output((rows, cols), torch.bfloat16, shift, gpu)
    mean, rstd = torch.empty(rows, device=gpu), torch.empty(rows, device=gpu)
    hip_lib.layernorm_fwd(xs, gs, bs, y, mean, rstd, hip_lib.LAYERNORM_EPS, hip_lib.make_cfg())
    dy = WORKLOADS["layernorm_backward_bf16"].make_inputs(rows, cols, seed=rows + cols)[1]
    ds = place(dy, shift, gpu)
    dx, gd = output((rows, cols), torch.bfloat16, shift, gpu)
    hip_lib.layernorm_backward(xs, ds, gs, dx, hip_lib.LAYERNORM_EPS, hip_lib.make_cfg())
    torch.cuda.synchronize()
    check_guards(gy, gd)
    i = sample(rows)
    ey, em, er = ref.layernorm_fwd(x[i].float().numpy(), gamma.float().numpy(),
                                   beta.float().numpy())
    np.testing.assert_allclose(y[i].float().cpu().numpy(), ey, **BF16)
    np.testing.assert_allclose(mean[i].cpu().numpy(), em, **FP32)
    np.testing.assert_allclose(rstd[i].cpu().numpy(), er, **FP32)
    expect = ref.layernorm_backward(x[i].float().numpy(), dy[i].float().numpy(),
                                    gamma.float().numpy())
    np.testing.assert_allclose(dx[i].float().cpu().numpy(), expect, **BF16)
    assert not bool(torch.isnan(y).any()) and not bool(torch.isnan(dx).any())


@pytest.mark.parametrize("cols", [40003, 65536])
def test_wide_layernorm_edge_rows(gpu, cols):
    """Rows that start with, hold or are infinities, and with a NaN: outputs,
    mean and rstd as the READ variant gives them."""
    x = torch.randn(5, cols, generator=torch.Generator().manual_seed(2))
    x[0, 0] = float("inf")
    x[1, cols - 1] = -float("inf")
    x[2] = float("inf")
    x[3, 0] = float("nan")
    gamma, beta = torch.ones(cols, device=gpu).bfloat16(), torch.zeros(cols, device=gpu).bfloat16()
    ins = (x.bfloat16().to(gpu), gamma, beta)
    got, want = (hip_lib.allocate_outputs("layernorm_fwd", ins) for _ in range(2))
    hip_lib.layernorm_fwd(*ins, *got, hip_lib.LAYERNORM_EPS, hip_lib.make_cfg())
    hip_lib.layernorm_fwd(*ins, *want, hip_lib.LAYERNORM_EPS, hip_lib.make_cfg(variant="read"))
    for g, w, tol in zip(got, want, (BF16, FP32, FP32)):
        np.testing.assert_allclose(g.float().cpu().numpy(), w.float().cpu().numpy(), **tol)
