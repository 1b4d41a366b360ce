"""The float32 products on the matrix cores beside float64, at the edges of their tiles (16 to 64 rows of either
operand, steps of 16 k, eight ranges of k), and a row's independence of the rows beside it."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.fixture(scope="module")
def ops():
    from tiny_llm_infer_amd.kernels.ops import HipOps
    return HipOps(DEV)


def rnd(shape, seed, std=1.0):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return torch.randn(shape, generator=g, device=DEV) * std


# (rows, outputs, k): one row; partial tiles of both; k of less than a step, of a partial last step, of fewer steps than
# ranges, of many batches; each launch shape: up to 16, 32 and more rows; parts of a tile (four or eight columns), one tile, two
SIZES = [(1, 96, 64), (5, 301, 4), (9, 1500, 68), (16, 2100, 100), (7, 16400, 260), (17, 77, 1028), (20, 1999, 132), (24, 4100, 260),
         (32, 16448, 64), (33, 130, 4096), (64, 1040, 36), (100, 4100, 132), (65, 16385, 132), (200, 8200, 1100), (130, 2050, 516)]


def bound(x, w):
    """Eight ranges of K / 8 sums each, then their sum: at most K / 8 + 11 roundings of 2^-24 (and one for the result) of
    the sum of the terms' sizes."""
    terms = x.double().abs() @ w.double().abs().T
    return (x.shape[1] / 8 + 12) * 2.0 ** -24 * terms


@pytest.mark.parametrize("mnk", SIZES)
def test_product(ops, mnk):
    M, N, K = mnk
    x, w = rnd((M, K), 1), rnd((N, K), 2, 0.05)
    y = ops.linear(x, w)
    assert bool(((y.double() - x.double() @ w.double().T).abs() <= bound(x, w)).all())
    for lo, hi in ((0, 1), (M // 2, M), (M - 1, M), (0, min(M, 16)), (0, min(M, 32))):
        assert torch.equal(ops.linear(x[lo:hi].clone(), w), y[lo:hi]), "a row's sums depend on the rows beside it"


@pytest.mark.parametrize("mnk", [(1, 32, 64), (5, 48, 100), (16, 24, 36), (17, 40, 100), (32, 1000, 516), (33, 1000, 1028), (100, 50, 260),
                                 (200, 4100, 516)])
@pytest.mark.parametrize("activation", ["silu", "gelu_tanh"])
def test_gated_product(ops, mnk, activation):
    from tiny_llm_infer_amd.parts.base import BuildEnv
    from tiny_llm_infer_amd.parts.linear import GatedMatrix
    M, N, K = mnk
    env = BuildEnv(dtype=torch.float32, device=torch.device(DEV), ops=ops, max_model_len=64)
    x, gate, up = rnd((M, K), 3), rnd((N, K), 4, 2 / math.sqrt(K)), rnd((N, K), 5, 2 / math.sqrt(K))
    y = ops.linear_swiglu(x, GatedMatrix(gate, up, env), activation=activation, scale=0.7)
    g, u = x.double() @ gate.double().T, x.double() @ up.double().T
    act = torch.nn.functional.silu(g) if activation == "silu" else torch.nn.functional.gelu(g, approximate="tanh")
    # a gate's error counts at most 1.13 times (the steepest slope of either activation), the exponential and the division
    # are good to a few roundings
    allowed = 0.7 * (1.13 * bound(x, gate) * u.abs() + act.abs() * bound(x, up)) + 16 * 2.0 ** -24 * (0.7 * act * u).abs() + 1e-7
    assert bool(((y.double() - 0.7 * act * u).abs() <= allowed).all())
    for lo, hi in ((0, 1), (0, min(M, 16)), (M // 2, M), (0, min(M, 32))):
        assert torch.equal(ops.linear_swiglu(x[lo:hi].clone(), GatedMatrix(gate, up, env), activation=activation, scale=0.7), y[lo:hi])


def test_operands_that_are_not_in_whole_pieces_go_to_the_plain_kernel(ops):
    x, w = rnd((5, 70), 6), rnd((40, 70), 7)
    assert torch.equal(ops.linear(x, w), ops.linear_plain(x, w))
    flat = rnd((5 * 64 + 1,), 8)
    x, w = flat[1:].view(5, 64), rnd((40, 64), 9)
    assert torch.equal(ops.linear(x, w), ops.linear_plain(x, w))
