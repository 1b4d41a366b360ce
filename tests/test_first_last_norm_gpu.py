"""The first norm of a model in the embedding's launch and the last one in the head's product: beside the separate kernels."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
BF = torch.bfloat16


@pytest.fixture(scope="module")
def ops():
    from tiny_llm_infer_amd.kernels.ops import HipOps
    return HipOps(DEV)


@pytest.mark.parametrize("dtype", [torch.float32, BF])
@pytest.mark.parametrize("rows, n", [(1, 4), (3, 252), (8, 4096), (5, 4100), (2, 8192), (300, 1024), (2, 16384)])
def test_embedding_and_norm_in_one_pass(ops, rows, n, dtype):
    """The same bits as the two passes; ids outside the table read its first row, as there."""
    g = torch.Generator(device=DEV).manual_seed(rows + n)
    table = torch.randn(50, n, generator=g, device=DEV).to(dtype)
    ids = torch.randint(0, 50, (rows + 2,), generator=g, device=DEV).to(torch.int32)
    ids[rows - 1] = 50
    weight = torch.randn(n, generator=g, device=DEV)
    resid, out = ops.embed_rmsnorm(table, ids, rows, weight, 1e-6)
    want = ops.embed(table, ids, rows)
    assert torch.equal(resid, want) and torch.equal(out, ops.add_rmsnorm(want, None, weight, 1e-6, dtype))


def test_what_the_embedding_leaves_to_the_norm(ops):
    ids = torch.zeros(2, dtype=torch.int32, device=DEV)
    for n in (6, 16388):
        assert ops.embed_rmsnorm(torch.zeros(4, n, device=DEV), ids, 2, torch.ones(n, device=DEV), 1e-6) is None


@pytest.mark.parametrize("rows", [1, 4, 8, 9, 16])
@pytest.mark.parametrize("N, K", [(1000, 4096), (70, 512), (4096, 2048), (9000, 136), (16384, 256), (16400, 4096)])
def test_float32_products_of_rows_that_owe_their_norm(ops, rows, N, K):
    """The norm's factor applied to float32 outputs: half tiles, one and two tiles a workgroup, x through LDS and not; bfloat16 rows
    of w h with the factor behind the product, against float64: rounding of those rows only (2^-9 of an element each, at random)."""
    from tiny_llm_infer_amd.kernels.ops import PendingProduct
    from tiny_llm_infer_amd.parts.base import BuildEnv
    from tiny_llm_infer_amd.parts.linear import as_matrix
    g = torch.Generator(device=DEV).manual_seed(rows + N)
    env = BuildEnv(dtype=BF, device=torch.device(DEV), ops=ops, max_model_len=64)
    rnd = lambda *shape: torch.randn(*shape, generator=g, device=DEV)
    before, head = as_matrix((rnd(K, 64) / 8).to(BF), env), (rnd(N, K) * K ** -0.5).to(BF)
    x, resid, weight = rnd(rows, 64).to(BF), rnd(rows, K), rnd(K) * 0.1 + 1
    h = resid.double() + x.double() @ before.w.double().T if before.w is not None else None
    if h is None:
        h = resid.double() + x.double() @ ops.untile_matrix(before.tiled, (K, 64)).double().T
    normed = ops.add_rmsnorm(resid, PendingProduct(x, before), weight, 1e-6, BF, lazy=True)
    y = ops.linear(normed, as_matrix(head.clone(), env), out_dtype=torch.float32)
    want = (h * torch.rsqrt((h * h).mean(1, keepdim=True) + 1e-6) * weight.double()) @ head.double().T
    assert y.dtype == torch.float32 and y.shape == want.shape
    assert float((y.double() - want).norm() / want.norm()) < 2 ** -9
