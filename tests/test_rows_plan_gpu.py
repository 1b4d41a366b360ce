"""Products of many rows: workgroups dealt out over the dies at the edges of the dealing (column groups that make no whole round of
eight, short last chunks of 2,048 rows), every launch shape, with and without ranges of k."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.fixture(scope="module")
def ops():
    from tiny_llm_infer_amd.kernels.ops import HipOps
    return HipOps(DEV)


def product(ops, x, tiled, N, splits, cfg, deferred=False):
    M, K = x.shape
    ops.rows_splits, ops.rows_cfg = splits, cfg
    try:
        y = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=DEV)
        return ops._linear_rows(x, tiled, y, M, N, K, 0, deferred)
    finally:
        ops.rows_splits = ops.rows_cfg = 0


def near(y, x, w):
    """bfloat16 results of float32 sums: half a unit in the last place of the result (8 bits of it: 2^-8 of its size at most), and K 2^-24 of the sum of the terms' sizes
    (at most K roundings of the sums, whatever their order)."""
    want = x.double() @ w.double().T
    slack = 2.0 ** -8 * want.abs() + x.shape[1] * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)
    return bool(((y.double() - want).abs() <= slack).all())


# rows, outputs: one column group; groups of every launch shape that leave some over after a round of dies; a chunk and a row, two and a half
@pytest.mark.parametrize("mn", [(129, 16), (300, 1040), (513, 4112), (2049, 784), (5000, 272)])
@pytest.mark.parametrize("cfg", [0, 1, 2, 3, 4, 5, 6])
def test_every_output_is_written_once(ops, mn, cfg):
    M, N = mn
    K = 512
    g = torch.Generator(device=DEV).manual_seed(M + N)
    x = torch.randn((M, K), generator=g, device=DEV).to(torch.bfloat16)
    w = torch.randn((N, K), generator=g, device=DEV).mul_(0.05).to(torch.bfloat16)
    tiled = ops.tile_matrix(w)
    for splits in (1, 2):
        y = product(ops, x, tiled, N, splits, cfg)
        assert near(y, x, w), splits
        if splits > 1:
            left = product(ops, x, tiled, N, splits, cfg, deferred=True)
            assert tuple(left.parts.shape) == (splits, M, N) and torch.equal(ops.resolve(left), y)


# k of one slice, of fewer than two ranges' worth, of an odd number of slices; few and many columns; rows at the edges of a block of 128
@pytest.mark.parametrize("mnk", [(257, 16, 128), (385, 1040, 904), (640, 2048, 2048), (641, 2048, 4096), (1000, 3072, 1024), (1537, 512, 1152), (2048, 256, 8192)])
def test_plan(ops, mnk):
    """The plan's ranges and launch shape: right, and the ranges within what their sums are laid out for."""
    M, N, K = mnk
    g = torch.Generator(device=DEV).manual_seed(K)
    x = torch.randn((M, K), generator=g, device=DEV).to(torch.bfloat16)
    w = torch.randn((N, K), generator=g, device=DEV).mul_(0.05).to(torch.bfloat16)
    splits = ops.lib.tli_gemm_rows_splits(M, N, K)
    assert 1 <= splits <= 16 and (splits == 1 or splits * 4 <= (K + 127) // 128)
    assert near(product(ops, x, ops.tile_matrix(w), N, 0, 0), x, w)
