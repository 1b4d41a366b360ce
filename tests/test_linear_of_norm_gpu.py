"""A product that norms its rows on their way in beside the norm and the product in launches of their own, and float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
BF = torch.bfloat16


@pytest.fixture(scope="module")
def ops():
    from tiny_llm_infer_amd.kernels.ops import HipOps
    return HipOps(DEV)


# rows, columns of the product, k, column of the first element, columns of the rows: half tiles, one and two tiles a workgroup by
# four and by eight waves; fewer steps of k than waves, as many, several each
SIZES = [(1, 96, 128, 0, 128), (16, 3072, 1024, 0, 1040), (7, 250, 640, 8, 720), (8, 4112, 256, 16, 272), (3, 9000, 1152, 64, 1216), (5, 13000, 384, 0, 400)]


@pytest.mark.parametrize("size", SIZES)
def test_product_of_normed_rows(ops, size):
    from tiny_llm_infer_amd.parts.base import BuildEnv
    from tiny_llm_infer_amd.parts.linear import as_matrix
    M, N, K, at, width = size
    env = BuildEnv(dtype=BF, device=torch.device(DEV), ops=ops, max_model_len=64)
    g = torch.Generator(device=DEV).manual_seed(N)
    proj = torch.randn((M, width), generator=g, device=DEV).mul_(3).to(BF)
    weight = 1 + 0.3 * torch.randn((K,), generator=g, device=DEV)
    w = torch.randn((N, K), generator=g, device=DEV).mul_(K ** -0.5).to(BF)
    matrix = as_matrix(w, env)
    got = ops.linear_of_norm(proj, at, K, weight, 1e-5, matrix)
    apart = ops.linear(ops.norm_rows(proj, at, K, weight, 1e-5), matrix)
    x = proj[:, at:at + K].double()
    rows = weight.double() * x / torch.sqrt((x * x).mean(dim=1, keepdim=True) + 1e-5)
    want, terms = rows @ w.double().T, rows.abs() @ w.double().abs().T
    # an element of a row is rounded to bfloat16 once (2^-9 to 2^-8 of it), independently: 2^-8 of the terms' sizes at most; the result once more; the
    # float32 sums and the factor are far below
    slack = 2.0 ** -8 * (terms + want.abs()) + 1e-6 * terms
    assert bool(((got.double() - want).abs() <= slack).all()) and bool(((apart.double() - want).abs() <= slack).all())
    # and no further off than the two launches are, but for which elements happen to be rounded up
    off = [float((y.double() - want).norm() / want.norm()) for y in (got, apart)]
    assert off[0] <= 1.1 * off[1]


def test_rows_that_it_does_not_take_go_through_the_norm(ops):
    from tiny_llm_infer_amd.parts.base import BuildEnv
    from tiny_llm_infer_amd.parts.linear import as_matrix
    env = BuildEnv(dtype=BF, device=torch.device(DEV), ops=ops, max_model_len=64)
    for rows, k, at, width in ((17, 128, 0, 128), (4, 136, 0, 136), (4, 128, 4, 136), (4, 128, 0, 132)):
        proj, w = torch.randn((rows, width), device=DEV).to(BF), as_matrix(torch.randn((64, k), device=DEV).to(BF), env)
        weight = torch.ones(k, device=DEV)
        assert torch.equal(ops.linear_of_norm(proj, at, k, weight, 1e-5, w), ops.linear(ops.norm_rows(proj, at, k, weight, 1e-5), w))


# rows, columns, k at both sides of the rule: 16 and 17 rows, k 1,024, 2,048 and a step more, two tiles a compute unit and a tile more
@pytest.mark.parametrize("size, together", [((16, 64, 2048), True), ((17, 64, 128), False), ((8, 256, 2176), False), ((3, 8192, 1152), True), ((3, 8208, 1152), False),
                                            ((3, 8208, 1024), True), ((2, 12288, 2048), False)])
def test_where_the_norm_is_taken_in(ops, size, together):
    """Longer rows, and many columns of rows that are not short, go through the norm: the same bits as both launches."""
    from tiny_llm_infer_amd.parts.base import BuildEnv
    from tiny_llm_infer_amd.parts.linear import as_matrix
    M, N, K = size
    env = BuildEnv(dtype=BF, device=torch.device(DEV), ops=ops, max_model_len=64)
    g = torch.Generator(device=DEV).manual_seed(K)
    proj, weight = torch.randn((M, K), generator=g, device=DEV).to(BF), 1 + 0.3 * torch.randn((K,), generator=g, device=DEV)
    matrix = as_matrix(torch.randn((N, K), generator=g, device=DEV).mul_(K ** -0.5).to(BF), env)
    got, apart = ops.linear_of_norm(proj, 0, K, weight, 1e-5, matrix), ops.linear(ops.norm_rows(proj, 0, K, weight, 1e-5), matrix)
    assert torch.equal(got, apart) != together
    assert float((got.double() - apart.double()).norm() / apart.double().norm()) < 2.0 ** -7        # (a rounding to bfloat16 of each side's rows)
