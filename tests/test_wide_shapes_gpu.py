"""Products of up to 16 rows with more columns than two tiles a compute unit: the launch shapes at their edges, bfloat16 and float32
outputs, with and without the norm's factor."""
import pytest
import torch

from test_rows_plan_gpu import near

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.fixture(scope="module")
def ops():
    from tiny_llm_infer_amd.kernels.ops import HipOps
    return HipOps(DEV)


# columns: the last of two tiles a compute unit and the first after it, the same of three and of four; an odd number of tiles, a partial one
@pytest.mark.parametrize("cols", [8192, 8193, 8240, 12288, 12289, 16368, 16384])
@pytest.mark.parametrize("rows, k", [(1, 136), (16, 1024), (5, 4096)])
def test_launch_shapes(ops, cols, rows, k):
    from tiny_llm_infer_amd.kernels.ops import NormedRows
    from tiny_llm_infer_amd.parts.base import BuildEnv
    from tiny_llm_infer_amd.parts.linear import as_matrix
    env = BuildEnv(dtype=torch.bfloat16, device=torch.device(DEV), ops=ops, max_model_len=64)
    g = torch.Generator(device=DEV).manual_seed(cols + rows)
    x = torch.randn((rows, k), generator=g, device=DEV).to(torch.bfloat16)
    w = torch.randn((cols, k), generator=g, device=DEV).mul_(0.05).to(torch.bfloat16)
    matrix = as_matrix(w, env)
    y = ops.linear(x, matrix)
    assert near(y, x, w)
    wide = ops.linear(x, matrix, out_dtype=torch.float32)
    assert near(wide, x, w) and torch.equal(wide.to(torch.bfloat16), y)
    # the factor of a row of squares that sum to 4 k is a half, but for eps: the same products, halved
    normed = NormedRows(x, torch.full((1, rows), 4.0 * k, device=DEV), 0.0)
    assert torch.equal(ops.linear(normed, matrix), (0.5 * wide).to(torch.bfloat16))
    assert torch.equal(ops.linear(normed, matrix, out_dtype=torch.float32), 0.5 * wide)


# columns at both sides of 9 and of 12 tiles for four compute units; k under which the shapes have different numbers of waves
@pytest.mark.parametrize("cols, as_before", [(8208, True), (9200, True), (9201, False), (12288, False), (12289, True), (16368, True)])
@pytest.mark.parametrize("rows", [1, 16])
def test_row_major_matrices(ops, cols, as_before, rows):
    """Right, and in the shape of two tiles and eight waves where the others are slower."""
    g = torch.Generator(device=DEV).manual_seed(cols + rows)
    x = torch.randn((rows, 2048), generator=g, device=DEV).to(torch.bfloat16)
    w = torch.randn((cols, 2048), generator=g, device=DEV).mul_(0.05).to(torch.bfloat16)
    y = ops.linear(x, w, out_dtype=torch.float32)
    assert near(y, x, w)
    ops.skinny_cfg = 28
    try:
        pairs = ops.linear(x, w, out_dtype=torch.float32)
    finally:
        ops.skinny_cfg = 0
    assert torch.equal(y, pairs) == as_before
