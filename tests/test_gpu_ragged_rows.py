"""Rows that fit no 16-byte layout, on the kernels that hold one in a
workgroup's registers and on the streaming ones past their width: odd widths,
the edges of each register table, buffers at 4-byte addresses, more rows than
the persistent grid holds.

fp32 within rtol 1e-5 / atol 1e-6 of the float64 oracle (maxima, int8 codes and
scales bit for bit), bf16 within rtol 1e-2 / atol 1e-2."""
import numpy as np
import pytest
import torch

from credit_amd import hip_lib
from credit_amd.workloads import WORKLOADS
from oracle import reference as ref

pytestmark = pytest.mark.gpu

FP32 = dict(rtol=1e-5, atol=1e-6)
BF16 = dict(rtol=1e-2, atol=1e-2)
GUARD = 8


def place(t, shift, gpu):
    """A copy of t on the GPU, `shift` elements behind a 16-byte address."""
    flat = torch.empty(t.numel() + 16, dtype=t.dtype, device=gpu)
    out = flat[shift:shift + t.numel()].view(t.shape)
    out.copy_(t)
    return out


def output(shape, dtype, shift, gpu):
    """NaN (or 85) everywhere, with guard elements on both sides of the view."""
    n = int(np.prod(shape))
    fill = 85 if dtype == torch.int8 else float("nan")
    flat = torch.full((n + 2 * GUARD + 8,), fill, dtype=dtype, device=gpu)
    view = flat[GUARD + shift:GUARD + shift + n].view(shape)
    return view, (flat, GUARD + shift, n)


def check_guards(*guards):
    for flat, start, n in guards:
        for edge in (flat[:start], flat[start + n:]):
            assert bool(torch.isnan(edge).all() if edge.is_floating_point() else (edge == 85).all())


# Widths: below one vector, the edges of the register tables (1024, 4096, 8192,
# 16384, 32768, 53248, 65536 elements), past the last; rows past the grid.
SHAPES = [(3, 1, 0), (5, 3, 1), (7, 1023, 0), (9, 1025, 0), (4, 4096, 1), (5000, 1003, 0),
          (700, 8191, 0), (600, 16385, 0), (300, 32767, 0), (270, 50001, 0), (3, 53247, 0),
          (5, 53249, 0), (2, 65535, 3), (2, 65537, 0), (1200, 66001, 0)]


def sample(rows):
    return np.unique(np.linspace(0, rows - 1, 40).astype(int))


@pytest.mark.parametrize("rows,cols,shift", SHAPES)
def test_ragged_softmax(gpu, rows, cols, shift):
    print(f"ragged softmax {rows} x {cols} + {shift}", flush=True)
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


def test_ragged_softmax_edge_rows(gpu):
    """Rows of -inf, with +inf, with NaN and of the lowest float beside a plain
    one: p, max and lse as torch gives them."""
    x = torch.randn(5, 1003, generator=torch.Generator().manual_seed(1))
    x[0] = -float("inf")
    x[1, 77] = float("inf")
    x[2, 1002] = float("nan")
    x[3] = torch.finfo(torch.float32).min
    xs = x.to(gpu)
    p, m, lse = hip_lib.allocate_outputs("softmax_fwd", (xs,))
    hip_lib.softmax_fwd(xs, p, m, lse, hip_lib.make_cfg())
    assert torch.equal(m.cpu().isnan(), x.amax(1).isnan())
    assert torch.equal(m.cpu().nan_to_num(7.0), x.amax(1).nan_to_num(7.0))
    assert bool(p[:3].isnan().all())
    np.testing.assert_allclose(p[3:].cpu().numpy(), torch.softmax(x[3:].double(), 1), **FP32)
    assert lse[0].item() == -float("inf") and bool(lse[1:3].isnan().all())


@pytest.mark.parametrize("rows,cols,shift", SHAPES)
def test_ragged_quant(gpu, rows, cols, shift):
    print(f"ragged quant {rows} x {cols} + {shift}", flush=True)
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


# Even and odd widths (odd: every other row starts inside a dword), buffers at
# 4-byte (shift 2) and 2-byte (shift 1, streamed) addresses, both edges of the
# register tables and the first width past them.
NORM_SHAPES = [(3, 30, 2), (4, 31, 0), (5, 1002, 0), (6, 1023, 0), (4000, 1030, 0), (4001, 1001, 2),
               (700, 5003, 0), (9, 2047, 0), (9, 2049, 0), (600, 8194, 0), (601, 8191, 0),
               (300, 16390, 2), (300, 16383, 0), (270, 32766, 0), (270, 32767, 0), (3, 32770, 0),
               (3, 32769, 1), (2, 65534, 0), (3, 65535, 0), (2, 65538, 0), (3, 65537, 0)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows,cols,shift", NORM_SHAPES)
def test_ragged_layernorm_backward(gpu, rows, cols, shift, dtype):
    print(f"ragged layernorm backward {rows} x {cols} + {shift} {dtype}", flush=True)
    name = "layernorm_backward" + ("_bf16" if dtype == torch.bfloat16 else "")
    x, dy, gamma = WORKLOADS[name].make_inputs(rows, cols, seed=rows + cols)
    x = (x + 3.0).to(dtype)  # an offset the shifted sums take out
    dx, gd = output((rows, cols), dtype, shift, gpu)
    hip_lib.layernorm_backward(place(x, shift, gpu), place(dy, shift, gpu),
                               place(gamma, shift, gpu), dx, hip_lib.LAYERNORM_EPS,
                               hip_lib.make_cfg())
    torch.cuda.synchronize()
    check_guards(gd)
    i = sample(rows)
    expect = ref.layernorm_backward(x[i].float().numpy(), dy[i].float().numpy(),
                                    gamma.float().numpy())
    np.testing.assert_allclose(dx[i].float().cpu().numpy(), expect,
                               **(FP32 if dtype == torch.float32 else BF16))
    assert not bool(torch.isnan(dx).any())


@pytest.mark.parametrize("rows,cols,shift", NORM_SHAPES)
def test_ragged_layernorm_forward(gpu, rows, cols, shift):
    print(f"ragged layernorm forward {rows} x {cols} + {shift}", flush=True)
    x, gamma, beta = WORKLOADS["layernorm_fwd"].make_inputs(rows, cols, seed=rows + cols)
    x[: rows // 2] += 3.0  # an offset the variance takes out
    y, gy = output((rows, cols), torch.bfloat16, shift, gpu)
    mean, rstd = torch.empty(rows, device=gpu), torch.empty(rows, device=gpu)
    hip_lib.layernorm_fwd(place(x, shift, gpu), place(gamma, shift, gpu), place(beta, shift, gpu),
                          y, mean, rstd, hip_lib.LAYERNORM_EPS, hip_lib.make_cfg())
    torch.cuda.synchronize()
    check_guards(gy)
    i = sample(rows)
    ey, em, er = ref.layernorm_fwd(x[i].float().numpy(), gamma.float().numpy(),
                                   beta.float().numpy())
    np.testing.assert_allclose(y[i].float().cpu().numpy(), ey, **BF16)
    np.testing.assert_allclose(mean[i].cpu().numpy(), em, **FP32)
    np.testing.assert_allclose(rstd[i].cpu().numpy(), er, **FP32)
    assert not bool(torch.isnan(y).any())
