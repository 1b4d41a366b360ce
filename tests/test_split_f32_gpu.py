"""float32 products of few rows left as the sums of their ranges of k: what reads them gives, bit for bit, what it gives from the
product itself."""
import pytest
import torch

from test_gemm_f32_gpu import rnd
from test_kernels_gpu import fill_cache, make_step

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
F32 = torch.float32


@pytest.fixture(scope="module")
def ops():
    from tiny_llm_infer_amd.kernels.ops import HipOps
    return HipOps(DEV)


# rows, outputs, k: outputs that are no whole tile, an odd number of tiles; k of less than a step, of fewer steps than ranges, with a
# partial last step, of an odd number of batches; the edges of 16 and 32 rows; the most outputs that are split
SIZES = [(1, 64, 4), (5, 100, 100), (16, 2048, 1024), (17, 48, 260), (32, 1028, 3076), (8, 1020, 1540), (3, 2044, 68)]


@pytest.mark.parametrize("mnk", SIZES)
def test_norm_of_a_product_left_in_ranges(ops, mnk):
    from tiny_llm_infer_amd.kernels.ops import PendingProduct
    M, N, K = mnk
    x, w, resid, weight = rnd((M, K), 1), rnd((N, K), 2, 0.05), rnd((M, N), 3), 1 + rnd((N,), 4, 0.1)
    left = ops.linear(x, w, deferred=True)
    assert isinstance(left, PendingProduct) and torch.equal(ops.resolve(left), ops.linear(x, w))
    for rows in (None, torch.tensor([M - 1, 0], dtype=torch.int32, device=DEV)):
        one, two = resid.clone(), resid.clone()
        got = ops.add_rmsnorm(one, left, weight, 1e-6, F32, rows=rows)
        want = ops.add_rmsnorm(two, ops.linear(x, w), weight, 1e-6, F32, rows=rows)
        assert torch.equal(got, want) and torch.equal(one, two)


@pytest.mark.parametrize("mn", [(33, 64), (5, 2064)])
def test_more_rows_or_outputs_are_not_left(ops, mn):
    x, w = rnd((mn[0], 64), 1), rnd((mn[1], 64), 2)
    assert isinstance(ops.linear(x, w, deferred=True), torch.Tensor)


# heads, kv heads, head size, page, norms, elements rotated, keys of the sequences, rows they bring, window, writes
CASES = [(16, 4, 64, 16, True, 64, [1, 16, 17, 52, 65], None, None, True),
         (4, 2, 64, 4, True, 32, [63, 64, 1], None, 33, True),
         (6, 3, 128, 8, False, 128, [200, 5, 13], None, None, True),
         (2, 1, 192, 16, True, 0, [90, 41], None, None, True),
         (2, 2, 256, 16, True, 256, [300, 16], None, 20, True),
         (4, 2, 64, 16, True, 64, [30, 31], None, None, False),
         (4, 2, 64, 16, True, 64, [30, 45], [3, 1], None, True),
         # many heads of more than 64 elements: their squares in one order of roundings
         (4, 1, 192, 16, True, 192, [9] * 32, None, None, True), (8, 2, 128, 8, True, 128, [20] * 32, None, None, True)]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(str(v) for v in c[:6]) + f"-{len(c[6])}rows-window{c[8]}-writes{c[9]}")
def test_attention_from_projections_left_in_ranges(ops, case):
    """From a pending product, from its ranges' sums and from the product: the output and the cache that the two launches
    (the heads' norms, rotation and cache writes; the attention) leave."""
    heads, kv_heads, hd, page, norms, rd, lens, news, window, writes = case
    news = news or [1] * len(lens)
    pages = sum((n + page - 1) // page for n in lens) + 3
    step, tables, pos, _ = make_step(lens, news, page, pages, 7, kv_heads, hd, F32, window)
    fill_cache(step, tables, lens, kv_heads, hd, F32, 300)
    step.cache.writes = writes
    x, w = rnd((len(pos), 96), 5), rnd(((heads + 2 * kv_heads) * hd, 96), 6, 0.1)
    x[0, :48] *= 1e20                                    # values that overflow: they come into the cache as 0
    w[-hd:, :48] *= 1e22
    qn = (1 + rnd((hd,), 22, 0.2), 1e-5) if norms else None
    kn = (1 + rnd((hd,), 23, 0.2), 3e-6) if norms else None
    rotary = None
    if rd:
        angle = torch.arange(512, dtype=torch.float64)[:, None] * (1e4 ** (-2.0 * torch.arange(rd // 2, dtype=torch.float64) / rd))
        rotary = (torch.cos(angle).float().to(DEV), torch.sin(angle).float().to(DEV), rd)
    k0, v0 = step.cache.k.clone(), step.cache.v.clone()

    def run(qkv, apart):
        step.cache.k.copy_(k0)
        step.cache.v.copy_(v0)
        ops.unfused_decode = apart
        try:
            if qkv is None:
                q = ops.qkv_to_cache(product, step, step.cache, heads, kv_heads, hd, qn, kn, rotary)
                out = ops.paged_attention(q, step, step.cache, heads, kv_heads, hd, hd ** -0.5, window)
            else:
                out = ops.qkv_attention(qkv, step, step.cache, heads, kv_heads, hd, qn, kn, rotary, hd ** -0.5, window)
        finally:
            ops.unfused_decode = False
        return out, step.cache.k.clone(), step.cache.v.clone()
    product = ops.linear(x, w)
    assert not bool(product[0, -hd:].isfinite().any())
    want = run(None, True)
    assert (not torch.equal(want[1], k0)) == writes
    pending = ops.linear(x, w, sums_only=True)
    for qkv in (product, pending, ops._f32_ranges(pending)):
        for apart in (False, True):
            for a, b in zip(run(qkv, apart), want):
                assert torch.equal(a.nan_to_num(7e30), b.nan_to_num(7e30))


def test_the_library_says_which_products_are_left(ops, monkeypatch):
    """Not a setting of the attention kernels: what ``linear`` leaves is what the kernel for the ranges takes."""
    monkeypatch.setattr(ops, "DECODE_WORKGROUPS", 4 * ops.DECODE_WORKGROUPS)
    x, w, weight = rnd((5, 64), 1), rnd((4096, 64), 2), 1 + rnd((4096,), 3, 0.1)
    left = ops.linear(x, w, deferred=True)
    assert isinstance(left, torch.Tensor)
    ops.add_rmsnorm(torch.zeros((5, 4096), device=DEV), left, weight, 1e-6, F32)


# outputs that are no multiple of four (rows of the planes without 16-byte alignment, the norm's element-by-element path) and k of every length
@pytest.mark.parametrize("mnk", SIZES + [(1, 1, 4), (5, 77, 260), (17, 1999, 132), (32, 2047, 1028), (3, 2046, 2304)])
def test_ranges_whatever_their_reader_would_take(ops, mnk):
    from tiny_llm_infer_amd.kernels.ops import PendingProduct
    M, N, K = mnk
    x, w, resid, weight = rnd((M, K), 1), rnd((N, K), 2, 0.05), rnd((M, N), 3), 1 + rnd((N,), 4, 0.1)
    parts, product = ops._f32_ranges(PendingProduct(x, w)), ops.linear(x, w)
    assert torch.equal(ops.resolve(parts), product)
    for rows in (None, torch.tensor([M - 1, 0], dtype=torch.int32, device=DEV)):
        one, two = resid.clone(), resid.clone()
        got = ops.add_rmsnorm(one, parts, weight, 1e-6, F32, rows=rows)
        want = ops.add_rmsnorm(two, product, weight, 1e-6, F32, rows=rows)
        assert torch.equal(got, want) and torch.equal(one, two)


@pytest.mark.parametrize("nk, pay", [((64, 252), False), ((64, 256), True), ((1024, 256), True), ((1026, 1024), False), ((1028, 1020), False),
                                     ((1028, 1024), True), ((2047, 2044), False), ((2047, 2048), True)])
def test_short_products_are_read_whole(ops, nk, pay):
    from tiny_llm_infer_amd.kernels.ops import DeferredSum, PendingProduct
    N, K = nk
    assert isinstance(ops._f32_sums(PendingProduct(rnd((5, K), 1), rnd((N, K), 2))), DeferredSum if pay else torch.Tensor)


@pytest.mark.parametrize("hd", [64, 128, 192, 256])
@pytest.mark.parametrize("window", [None, 17])
def test_own_key_at_the_edges_of_blocks(ops, hd, window):
    """The row's own key first, in the middle and last of a block of 16 keys, alone in one, and in every wave's share."""
    test_attention_from_projections_left_in_ranges(ops, (4, 2, hd, 16, True, hd, [1, 2, 16, 17, 32, 33, 48, 49, 64, 65, 80, 81, 130], None, window, True))


@pytest.mark.parametrize("heads, rows", [(12, 21), (12, 22), (8, 32), (8, 13)])
def test_own_key_of_heads_of_128_on_both_sides_of_a_workgroup_a_compute_unit(ops, heads, rows):
    """Up to one it is handled in the loop over the keys, from there on apart."""
    lens = ([1, 2, 16, 17, 32, 33, 48, 49, 64, 65, 80, 81, 130] * 3)[:rows]
    test_attention_from_projections_left_in_ranges(ops, (heads, 2, 128, 16, True, 128, lens, None, None, True))


def test_a_step_with_many_workgroups_is_two_launches(ops, monkeypatch):
    """By the rule, and the same bits as one launch of it."""
    rows, heads, hd = 300, 16, 192
    step, _, pos, _ = make_step([1 + i % 20 for i in range(rows)], [1] * rows, 16, 2 * rows + 3, 7, 4, hd, F32)
    qkv, outs, given = rnd((rows, (heads + 8) * hd), 5), [], []
    call = ops._call
    monkeypatch.setattr(ops, "_call", lambda fn, *args: (given.append(args[2]) if fn == ops.lib.tli_qkv_attention_f32 else None, call(fn, *args))[1])
    for reach in (step.reach, 256):                      # rows of more keys: one launch
        step.reach = reach
        outs.append(ops.qkv_attention(qkv, step, step.cache, heads, 4, hd, None, None, None, hd ** -0.5, None))
    assert given[0] is not None and given[1] is None and torch.equal(*outs)


@pytest.mark.parametrize("nk, pay", [((848, 392), False), ((848, 384), True), ((800, 640), True), ((512, 392), True), ((250, 256), True), ((322, 256), False),
                                     ((322, 512), True), ((893, 1020), False), ((893, 1024), True)])
def test_uneven_ranges_and_rows_read_element_by_element_are_left_later(ops, nk, pay):
    test_short_products_are_read_whole(ops, nk, pay)
