"""Ragged rows of a few to a few hundred columns, from one row to more than the
persistent grids hold: where AUTO changes between kernels that hold a row in a
wave's registers and READ, and where those change between vectors and single
elements.  Checked as the wider ones are (test_gpu_ragged_rows.py)."""
import pytest
import torch

import test_gpu_ragged_rows as ragged

pytestmark = pytest.mark.gpu

# rows, cols, elements past a 16-byte address.  From 3 columns on: a row of one
# column has variance 0, so its LayerNorm backward multiplies the rounding of
# one product (2^-24) by 1 / sqrt(eps) = 316, 2e-5 where the answer is 0.
SHAPES = [(1, 3, 0), (100, 3, 3), (300, 7, 1), (2047, 9, 2), (2049, 6, 0), (3000, 15, 0),
          (4097, 17, 2), (500, 62, 0), (600, 63, 0), (9000, 62, 2), (513, 255, 0), (512, 201, 0),
          (2500, 254, 0), (3000, 257, 0), (4096, 511, 0), (4097, 509, 0), (700, 513, 3),
          (9001, 258, 0), (20000, 5, 0)]


@pytest.mark.parametrize("rows,cols,shift", SHAPES)
def test_narrow_softmax(gpu, rows, cols, shift):
    ragged.test_ragged_softmax(gpu, rows, cols, shift)


@pytest.mark.parametrize("rows,cols,shift", SHAPES)
def test_narrow_quant(gpu, rows, cols, shift):
    ragged.test_ragged_quant(gpu, rows, cols, shift)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows,cols,shift", SHAPES)
def test_narrow_layernorm_backward(gpu, rows, cols, shift, dtype):
    ragged.test_ragged_layernorm_backward(gpu, rows, cols, shift, dtype)


@pytest.mark.parametrize("rows,cols,shift", SHAPES)
def test_narrow_layernorm_forward(gpu, rows, cols, shift):
    ragged.test_ragged_layernorm_forward(gpu, rows, cols, shift)


# LayerNorm backward: the last and the first width of the tables' entries of five
# and six vectors a lane (fp32 5120, 10240 and 12288 columns, bf16 twice that).
@pytest.mark.parametrize("cols,shift,dtype", [
    (5119, 0, torch.float32), (5121, 0, torch.float32), (10239, 1, torch.float32),
    (10241, 0, torch.float32), (12287, 0, torch.float32), (12289, 0, torch.float32),
    (10239, 0, torch.bfloat16), (10242, 0, torch.bfloat16), (20479, 2, torch.bfloat16),
    (20478, 0, torch.bfloat16), (20481, 0, torch.bfloat16), (24574, 0, torch.bfloat16),
    (24577, 0, torch.bfloat16)])
def test_layernorm_backward_table_edges(gpu, cols, shift, dtype):
    ragged.test_ragged_layernorm_backward(gpu, 270, cols, shift, dtype)


# Softmax: the same of the entry of three vectors a lane.
@pytest.mark.parametrize("rows,cols", [(900, 2049), (1000, 2051), (2100, 3071), (700, 3073)])
def test_softmax_table_edges(gpu, rows, cols):
    ragged.test_ragged_softmax(gpu, rows, cols, 0)
