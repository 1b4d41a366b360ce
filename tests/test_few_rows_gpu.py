"""Decode products whose columns are taken in half tiles of eight (up to 2,048 outputs and 16 rows), beside float64 at
the edges of their tiles; and decode attention where a row's keys are cut into many short splits."""
import math

import pytest
import torch

from test_long_context_gpu import close, fill, make_step, ref_attention_dev, rnd_dev

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
BF = torch.bfloat16


@pytest.fixture(scope="module")
def ops():
    from tiny_llm_infer_amd.kernels.ops import HipOps
    return HipOps(DEV)


def allowed(x, w, extra=0.0):
    """K float32 additions of exact products, and the rounding of the result to bfloat16."""
    terms = x.double().abs() @ w.double().abs().T + extra
    return (x.shape[1] * 2.0 ** -24) * terms


# (rows, outputs, k): either end of the range into the residual and one past it on both sides, and few outputs; outputs that end inside a half tile, between the
# halves of one and not in whole float4s; k of one step and of a ragged last one; 1, 4, 5, 8, 9 and 16 rows (the rows' loads)
HALF_SIZES = [(1, 1024, 128), (4, 1500, 264), (5, 2048, 1032), (8, 1030, 72), (9, 1031, 640), (16, 1992, 2056), (3, 1016, 256),
              (2, 2064, 256), (17, 1024, 256), (2, 8, 128), (16, 17, 264), (6, 250, 2048), (11, 72, 4096)]


@pytest.mark.parametrize("mnk", HALF_SIZES)
def test_half_tiles(ops, mnk):
    from tiny_llm_infer_amd.parts.base import BuildEnv
    from tiny_llm_infer_amd.parts.linear import Matrix
    M, N, K = mnk
    env = BuildEnv(dtype=BF, device=torch.device(DEV), ops=ops, max_model_len=64)
    x, w = rnd_dev((M, K), 1), rnd_dev((N, K), 2, 0.05)
    m = Matrix(w, env)
    want, tol = x.double() @ w.double().T, allowed(x, w)
    y32 = ops.linear(x, m, out_dtype=torch.float32)
    assert bool(((y32.double() - want).abs() <= tol).all())
    y = ops.linear(x, m)
    assert bool(((y.double() - want).abs() <= tol + 2.0 ** -8 * want.abs()).all())
    unit = ops.linear_act(x, m, "relu2")
    relu = want.clamp(min=0)
    assert bool(((unit.double() - relu * relu).abs() <= 2 * relu * tol + tol * tol + 2.0 ** -7 * relu * relu).all())
    if M > 16:
        return
    # into the residual: the sum, the next norm's rows and their sums of squares
    resid, nw = rnd_dev((M, N), 3).float(), 1 + rnd_dev((N,), 4, 0.2).float()
    r = resid.clone()
    normed = ops.add_rmsnorm(r, ops.linear(x, m, deferred=True), nw, 1e-5, BF, lazy=True)
    h = resid.double() + want
    slack = allowed(x, w, resid.double().abs()) + 2.0 ** -23 * h.abs()
    assert bool(((r.double() - h).abs() <= slack).all())
    assert torch.allclose(normed.ssq.sum(0).double(), (h * h).sum(-1), rtol=1e-4)
    # and from normed rows, back to a product of half tiles
    back = rnd_dev((1536, N), 5, 0.05)
    if N % 8 == 0:
        z = ops.linear(normed, Matrix(back, env))
        n = nw.double() * h / torch.sqrt((h * h).mean(-1, keepdim=True) + 1e-5)
        # the normed rows are rounded to bfloat16 once, the result once
        limit = 2.0 ** -8 * (n.abs() @ back.double().abs().T) + 2.0 ** -8 * (n @ back.double().T).abs() + 1e-3
        assert bool(((z.double() - n @ back.double().T).abs() <= limit).all())


# heads, kv heads, head_dim, page, lengths, splits: eight splits of 128 keys at the first length that is split; sixteen and
# more of 256; counts that are no multiple of eight; two workgroups a compute unit; rows far too short for most splits
SPLITS = [(32, 8, 128, 16, [513], 8), (32, 8, 128, 16, [1024, 1, 129, 640], 8), (16, 2, 64, 8, [4096], 16),
          (8, 4, 256, 16, [4097], 32), (32, 8, 128, 16, [2100, 2049, 700], 11), (32, 8, 128, 16, [1500] * 9, 4),
          (32, 8, 128, 32, [3000, 5, 2900, 2500, 3100, 4000, 2049, 128, 3000, 3500, 127, 3300], 6)]


@pytest.mark.parametrize("case", SPLITS, ids=lambda c: f"{len(c[4])}x{c[4][0]}-{c[1]}x{c[2]}")
def test_short_splits(ops, case):
    heads, kv_heads, hd, page, lens, splits = case
    num_pages = sum((n + page - 1) // page for n in lens) + 5
    step, tables, pos, seq = make_step(lens, [1] * len(lens), page, num_pages, 5, kv_heads, hd, BF, None)
    if ops.DECODE_WORKGROUPS == 256:
        assert ops._decode_splits(len(lens), step.reach, step.cache.group, heads, kv_heads, hd, None)[0] == splits
    ks, vs = fill(step, tables, lens, kv_heads, hd, 100)
    q = rnd_dev((len(pos), heads * hd), 50)
    scale = 1 / math.sqrt(hd)
    out = ops.paged_attention(q, step, step.cache, heads, kv_heads, hd, scale, None)
    close(out, ref_attention_dev(q, ks, vs, pos, seq, heads, kv_heads, scale, None), "short splits")


@pytest.mark.parametrize("n", [4112, 4128, 16400])
def test_an_odd_number_of_tiles_two_a_workgroup(ops, n):
    """Workgroups of two tiles of 16 columns, the last of them with one: right sums, and no sums of squares beyond a row's own
    (the NaNs behind them stay)."""
    M, K, parts = 5, 136, (n + 15) // 16
    x, w = rnd_dev((M, K), 1), rnd_dev((n, K), 2, 0.05)
    tiled = ops.tile_matrix(w)
    resid, nw = rnd_dev((M, n), 3).float(), 1 + rnd_dev((n,), 4, 0.2).float()
    r, ssq, xw = resid.clone(), torch.full((parts + 2, M), math.nan, device=DEV), torch.empty((M, n), dtype=BF, device=DEV)
    ops._call(ops.lib.tli_gemm_skinny_fused_bf16, x.data_ptr(), tiled.data_ptr(), None, M, n, K, 0, None, 0, 0.0, r.data_ptr(), nw.data_ptr(),
              xw.data_ptr(), ssq.data_ptr(), 0, 0, 1.0, 0, ops._stream())
    h = resid.double() + x.double() @ w.double().T
    assert bool(((r.double() - h).abs() <= allowed(x, w, resid.double().abs()) + 2.0 ** -23 * h.abs()).all())
    assert torch.allclose(ssq[:parts].sum(0).double(), (h * h).sum(-1), rtol=1e-4)
    assert bool(ssq[parts:].isnan().all())


@pytest.mark.parametrize("cfg", [0, 8, 14, 18, 24, 28])
@pytest.mark.parametrize("n", [1024, 1500, 2048, 2064, 4112])
def test_partial_sums_of_every_launch_shape(ops, n, cfg):
    """Into the residual through each launch shape: as many sums of squares a row as tli_gemm_skinny_parts says, all of them
    written (there are NaNs before), and no more."""
    M, K = 5, 256
    x, w = rnd_dev((M, K), 1), rnd_dev((n, K), 2, 0.05)
    tiled = ops.tile_matrix(w)
    resid, nw = rnd_dev((M, n), 3).float(), 1 + rnd_dev((n,), 4, 0.2).float()
    parts = ops.lib.tli_gemm_skinny_parts(M, n, cfg)
    ssq = torch.full((parts + 2, M), math.nan, device=DEV)
    xw = torch.empty((M, n), dtype=BF, device=DEV)
    r = resid.clone()
    ops._call(ops.lib.tli_gemm_skinny_fused_bf16, x.data_ptr(), tiled.data_ptr(), None, M, n, K, 0, None, 0, 0.0, r.data_ptr(), nw.data_ptr(),
              xw.data_ptr(), ssq.data_ptr(), cfg, 0, 1.0, 0, ops._stream())
    h = resid.double() + x.double() @ w.double().T
    assert torch.allclose(ssq[:parts].sum(0).double(), (h * h).sum(-1), rtol=1e-4)
    assert bool(ssq[parts:].isnan().all())


def test_half_tiles_want_whole_pieces_of_a_residual(ops):
    from tiny_llm_infer_amd.kernels.ops import KernelError
    x, tiled = rnd_dev((2, 128), 1), ops.tile_matrix(rnd_dev((1030, 128), 2))
    r, nw = torch.zeros((2, 1030), device=DEV), torch.ones(1030, device=DEV)
    xw, ssq = torch.empty((2, 1030), dtype=BF, device=DEV), torch.empty((200, 2), device=DEV)
    with pytest.raises(KernelError):
        ops._call(ops.lib.tli_gemm_skinny_fused_bf16, x.data_ptr(), tiled.data_ptr(), None, 2, 1030, 128, 0, None, 0, 0.0, r.data_ptr(),
                  nw.data_ptr(), xw.data_ptr(), ssq.data_ptr(), 8, 0, 1.0, 0, ops._stream())


# (outputs, k): half tiles on either side of their lines (k as long as the outputs are many, 256) and of the rows' way through
# LDS (1,024); a tile a workgroup; two, of eight and of four waves, on either side of k 4,096, ragged ends of k
WAYS = [(256, 256), (264, 256), (1016, 1016), (1024, 1032), (72, 128), (3000, 1024), (3000, 1000), (4096, 2056), (8192, 4096), (8200, 4088),
        (16640, 4104), (16640, 520)]


@pytest.mark.parametrize("nk", WAYS)
def test_a_row_is_the_same_by_either_way_of_its_operands(ops, nk):
    """16 rows, 8, 5 and 1 of them: whether they go through LDS or straight into the operand registers, and by whole tiles or
    half ones, a row's sums are those of one order."""
    from tiny_llm_infer_amd.kernels.ops import NormedRows
    from tiny_llm_infer_amd.parts.base import BuildEnv
    from tiny_llm_infer_amd.parts.linear import GatedMatrix, Matrix
    N, K = nk
    env = BuildEnv(dtype=BF, device=torch.device(DEV), ops=ops, max_model_len=64)
    x, w = rnd_dev((16, K), 1), rnd_dev((N, K), 2, 0.05)
    ssq = torch.rand((4, 16), device=DEV) * K / 4
    m = Matrix(w, env)
    gated = GatedMatrix(w[:N // 32 * 16], w[-(N // 32 * 16):], env)

    def forms(rows):
        normed = NormedRows(x[rows].contiguous(), ssq[:, rows].contiguous(), 1e-5)
        return [ops.linear(x[rows].contiguous(), m), ops.linear(x[rows].contiguous(), m, out_dtype=torch.float32), ops.linear(normed, m),
                ops.linear_swiglu(normed, gated), ops.linear_swiglu(x[rows].contiguous(), gated)]
    want = x.double() @ w.double().T
    all_rows = forms(slice(0, 16))
    assert bool(((all_rows[1].double() - want).abs() <= allowed(x, w)).all())
    for rows in (slice(0, 1), slice(3, 8), slice(8, 16)):
        for a, b in zip(forms(rows), all_rows):
            assert torch.equal(a, b[rows])


def test_short_heads_are_split_later(ops):
    """A key of a head of 64 is half as many bytes: few rows of them go over several workgroups from a reach of 2,048 keys on,
    more rows from 4,096; longer heads from 1,024."""
    if ops.DECODE_WORKGROUPS != 256:
        pytest.skip("the rule's lines are of 256 compute units")
    step, *_ = make_step([600], [1], 16, 45, 5, 2, 64, BF, None)
    for rows, hd, reach, splits in ((1, 64, 1024, 1), (1, 64, 2048, 8), (16, 64, 2048, 8), (17, 64, 2048, 1), (17, 64, 4096, 8), (1, 128, 512, 1),
                                    (1, 128, 1024, 8), (17, 128, 2048, 8), (1, 192, 1024, 8), (1, 256, 1024, 8)):
        assert ops._decode_splits(rows, reach, step.cache.group, 4, 2, hd, None)[0] == splits, (rows, hd, reach)
