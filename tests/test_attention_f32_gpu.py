"""The float32 attention with four lanes a key: beside a float64 reference and the plain kernel at the edges of its blocks
(16 keys of four waves in turn), pages of 4 and 12 slots, heads of 192 elements, windows; rows that hold no numbers."""
import dataclasses
import math

import pytest
import torch

from test_kernels_gpu import close, fill_cache, make_step, ref_attention, rnd

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
F32 = torch.float32


@pytest.fixture(scope="module")
def ops():
    from tiny_llm_infer_amd.kernels.ops import HipOps
    return HipOps(DEV)


# heads, kv heads, head size, page, keys of the sequences, rows they bring, window
CASES = [(4, 2, 192, 16, [1, 15, 16, 17], [1, 2, 16, 3], None),
         (4, 1, 64, 4, [63, 64, 65, 129], [1, 1, 65, 2], None),
         (6, 3, 128, 12, [200, 5, 13], [1, 5, 13], None),
         (2, 2, 256, 8, [300, 77], [4, 77], 33),
         (8, 2, 64, 16, [700, 1030], [2, 3], 100),
         (3, 1, 192, 4, [90, 41], [90, 1], 7)]


def setup(case, seed=3):
    heads, kv_heads, hd, page, lens, news, window = case
    num_pages = sum((n + page - 1) // page for n in lens) + 5
    step, tables, pos, seq = make_step(lens, news, page, num_pages, seed, kv_heads, hd, F32, window)
    ks, vs = fill_cache(step, tables, lens, kv_heads, hd, F32, 100)
    q = rnd((len(pos), heads * hd), F32, 50)
    return step, pos, seq, ks, vs, q


def run(ops, case, step, q, plain=False):
    heads, kv_heads, hd, window = case[0], case[1], case[2], case[6]
    ops.force_plain = plain
    try:
        return ops.paged_attention(q.to(DEV), step, step.cache, heads, kv_heads, hd, 1 / math.sqrt(hd), window)
    finally:
        ops.force_plain = False


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"{c[0]}-{c[1]}x{c[2]}-page{c[3]}-window{c[6]}")
def test_values_and_a_row_alone(ops, case):
    """As the reference and the plain kernel have it; a row alone is bit for bit the row among others."""
    step, pos, seq, ks, vs, q = setup(case)
    heads, kv_heads, hd, window = case[0], case[1], case[2], case[6]
    assert ops.lib.tli_attention_f32_takes(hd, case[3])
    want = ref_attention(q, ks, vs, pos, seq, heads, kv_heads, 1 / math.sqrt(hd), window)
    got = run(ops, case, step, q)
    close(got, want, F32, "attention")
    close(run(ops, case, step, q, plain=True), want, F32, "attention of the plain kernel")
    for row in (0, len(pos) // 2, len(pos) - 1):
        alone = dataclasses.replace(step, num_rows=1, positions=step.positions[row:row + 1].clone(),
                                    seq_of_row=step.seq_of_row[row:row + 1].clone())
        assert torch.equal(run(ops, case, alone, q[row:row + 1])[0], got[row]), row


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"{c[0]}-{c[1]}x{c[2]}-page{c[3]}-window{c[6]}")
def test_rows_that_hold_no_numbers(ops, case):
    """A query with a NaN, with an infinity and of NaNs: as from the plain kernel, NaNs where that has them; the other rows are
    bit for bit what they are without them."""
    step, _, _, _, _, q = setup(case)
    hd = case[2]
    want = run(ops, case, step, q)
    bad = q.clone()
    bad[0, :hd] = math.nan
    bad[1, hd + 3] = math.nan
    bad[2, 5] = math.inf
    got, plain = run(ops, case, step, bad), run(ops, case, step, bad, plain=True)
    assert torch.equal(got.isnan(), plain.isnan()) and bool(got[0, :hd].isnan().all()) and bool(got[1, hd:2 * hd].isnan().all())
    assert torch.equal(got[3:], want[3:])


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"{c[0]}-{c[1]}x{c[2]}-page{c[3]}-window{c[6]}")
def test_slots_that_no_row_sees_may_hold_anything(ops, case):
    """NaNs and infinities in pages that nobody holds, in slots behind a sequence's end and before its window."""
    step, pos, seq, ks, vs, q = setup(case)
    want = run(ops, case, step, q)
    page, window = case[3], case[6]
    tables = step.cache.group.tables.cpu().numpy()
    unseen = torch.ones((step.cache.k.shape[0], page), dtype=torch.bool)
    for p, s in zip(pos, seq):
        for t in range(0 if window is None else max(0, p - window + 1), p + 1):
            unseen[int(tables[s, t // page]), t % page] = False
    for fill in (math.nan, math.inf):
        step.cache.k.masked_fill_(unseen.to(DEV)[:, None, :, None], fill)
        step.cache.v.masked_fill_(unseen.to(DEV)[:, None, None, :], fill)
        assert torch.equal(run(ops, case, step, q), want), fill
