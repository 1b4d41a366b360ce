"""The routed experts of few rows in two launches, the shared expert among them, beside float64: tiles of 16 rows and their
edges, more experts than pairs and fewer, k of less than a step of 128 and of more steps than waves, experts that hand
their input on; and a row's independence of the rows beside it."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
BF = torch.bfloat16


@pytest.fixture(scope="module")
def ops():
    from tiny_llm_infer_amd.kernels.ops import HipOps
    return HipOps(DEV)


# (rows, experts, of which identity, top, width, hidden units, hidden units of the shared expert or 0)
SIZES = [(1, 4, 0, 2, 72, 40, 48), (5, 6, 2, 3, 128, 64, 0), (8, 16, 0, 2, 2048, 512, 1024), (16, 40, 0, 2, 264, 200, 96),
         (17, 8, 1, 4, 136, 272, 32), (32, 3, 0, 1, 1000, 2304, 16), (33, 64, 0, 1, 96, 48, 112), (64, 16, 0, 8, 512, 136, 256)]


def make(ops, size, kind):
    from tiny_llm_infer_amd.parts.base import BuildEnv
    from tiny_llm_infer_amd.parts.linear import GatedMatrix, as_matrix, fuse_rows
    T, E, identity, top, D, ff, sff = size
    g = torch.Generator(device=DEV).manual_seed(T + ff)
    env = BuildEnv(dtype=BF, device=torch.device(DEV), ops=ops, max_model_len=64)

    def rnd(*shape, std=1.0):
        return (torch.randn(shape, generator=g, device=DEV) * std).to(BF)
    gated = kind in ("silu", "limited")
    w = {"x": rnd(T, D), "gate": rnd(E, ff, D, std=D ** -0.5), "up": rnd(E, ff, D, std=D ** -0.5), "down": rnd(E, D, ff, std=ff ** -0.5)}
    packed = ops.pack_experts(torch.cat([w["gate"], w["up"]], 1) if gated else w["up"], w["down"], gated=gated)
    scores = torch.rand(T, E + identity, generator=g, device=DEV)
    weights, ids = torch.topk(scores, top, dim=1)
    shared = (None, None, None)
    if sff:
        w["sg"], w["su"], w["sd"] = rnd(sff, D, std=D ** -0.5), rnd(sff, D, std=D ** -0.5), rnd(D, sff, std=sff ** -0.5)
        up = GatedMatrix(w["sg"], w["su"], env) if kind == "silu" else fuse_rows([w["sg"], w["su"]], env) if gated else as_matrix(w["su"], env)
        shared = (up, as_matrix(w["sd"], env), torch.rand(T, generator=g, device=DEV))
    return w, packed, ids.to(torch.int32).contiguous(), weights.contiguous(), shared


def plain(w, ids, weights, gate, E, kind):
    x = w["x"].double()

    def expert(h, wg, wu, wd):
        u = h @ wu.double().T
        if kind == "silu":
            a = torch.nn.functional.silu(h @ wg.double().T) * u
        elif kind == "limited":
            z = torch.clamp(h @ wg.double().T, max=1.5)
            a = z * torch.sigmoid(1.702 * z) * (torch.clamp(u, -1.5, 1.5) + 1)
        else:
            a = torch.relu(u) ** 2
        return a @ wd.double().T
    out = torch.zeros_like(x)
    for t in range(x.shape[0]):
        for j in range(ids.shape[1]):
            e, by = int(ids[t, j]), float(weights[t, j])
            if e >= E:
                out[t] += by * x[t]
            elif kind == "relu2":
                out[t] += expert(by * x[t], None, w["up"][e], w["down"][e])
            else:
                out[t] += by * expert(x[t], w["gate"][e], w["up"][e], w["down"][e])
    if gate is not None:
        out += gate.double()[:, None] * expert(x, w["sg"], w["su"], w["sd"])
    return out


@pytest.mark.parametrize("kind", ["silu", "limited", "relu2"])
@pytest.mark.parametrize("size", SIZES)
def test_experts_of_few_rows(ops, size, kind):
    T, E, identity = size[:3]
    if kind == "relu2" and identity:
        pytest.skip("experts whose weight goes on their input all have matrices")
    w, packed, ids, weights, (up, down, gate) = make(ops, size, kind)
    how = {"silu": {}, "limited": dict(limit=1.5, slope=1.702, shared_limit=1.5), "relu2": dict(activation="relu2", weight_on_input=True)}[kind]

    def few(at):
        return ops.resolve(ops.experts_of_few_rows(w["x"][at].clone(), ids[at].clone(), weights[at].clone(), packed, up, down,
                                                   None if gate is None else gate[at].clone(), handed_on=identity > 0, **how))
    got = few(slice(0, T))
    want = plain(w, ids, weights, gate, E, kind)
    # hidden units and results are rounded to bfloat16 (2^-9 of their size each): the sum over ff rounded units is off by
    # 2^-9 of the root of the sum of their squares, which is the size of the result itself; five times that for the largest
    scale = float(want.square().mean().sqrt())
    assert float((got.double() - want).abs().max()) <= 5 * 2.0 ** -9 * scale + 2.0 ** -8 * float(want.abs().max())
    for at in (slice(0, 1), slice(T - 1, T), slice(T // 2, T)):
        assert torch.equal(few(at), got[at]), "a row's result depends on the rows beside it"


def test_layer_norm_of_unfinished_sums(ops):
    """The layer norm adds up the parts, and rounds their sum, as the reduction of its own does."""
    from tiny_llm_infer_amd.kernels.ops import DeferredSum
    g = torch.Generator(device=DEV).manual_seed(1)
    for rows, n in ((1, 64), (5, 100), (3, 5120), (2, 17000)):
        parts = [DeferredSum(torch.randn((p, rows, n), generator=g, device=DEV), BF) for p in (3, 2)]
        weight = torch.rand(n, generator=g, device=DEV)
        resid = torch.randn((rows, n), generator=g, device=DEV)
        for deltas in (parts[:1], parts, [ops.resolve(parts[0]), parts[1]]):
            mine, want = resid.clone(), resid.clone()
            y = ops.add_layernorm(mine, deltas, (weight,), 1e-5, BF)[0]
            z = ops.add_layernorm(want, [ops.resolve(d) for d in deltas], (weight,), 1e-5, BF)[0]
            assert torch.equal(y, z) and torch.equal(mine, want)


def test_sizes_that_other_kernels_take(ops):
    w, packed, ids, weights, (up, down, gate) = make(ops, (65, 8, 0, 2, 64, 32, 0), "silu")
    assert ops.experts_of_few_rows(w["x"], ids, weights, packed, None, None, None) is None
    w, packed, ids, weights, _ = make(ops, (2, 300, 0, 2, 64, 32, 0), "silu")
    assert ops.experts_of_few_rows(w["x"], ids, weights, packed, None, None, None) is None


# (experts, top, groups, kept groups): more places than lanes share experts; several experts a lane; groups of which some are out
CHOICES = [(16, 2, 1, 1), (64, 8, 1, 1), (40, 3, 4, 2), (130, 32, 1, 1)]


def _diverged(x):
    """Rows that hold no numbers, among others that do: all NaN, one NaN, an infinity of either sign, one past another."""
    x = x.clone()
    x[0], x[1, 3], x[5, 2], x[6, 7], x[11, :2] = math.nan, math.nan, math.inf, -math.inf, math.inf
    x[8], x[9] = math.nan, math.nan
    return x, [2, 3, 4, 7, 10, 12, 13, 14, 15]


@pytest.mark.parametrize("score", ["sigmoid", "softmax"])
@pytest.mark.parametrize("choice", CHOICES)
def test_choice_for_rows_that_hold_no_numbers(ops, choice, score):
    """Whatever a row holds, its choice is of different experts, and the other rows' is what it is without it."""
    E, top, groups, keep = choice
    g = torch.Generator(device=DEV).manual_seed(E)
    x = torch.randn((16, 72), generator=g, device=DEV).to(BF)
    rows = (torch.randn((E + 1, 72), generator=g, device=DEV) * 0.3).to(BF)
    bad, healthy = _diverged(x)
    want = ops.router(x, rows, E, top, groups, keep, 1.0, True, score=score)
    got = ops.router(bad, rows, E, top, groups, keep, 1.0, True, score=score)
    for a, b in zip(got, want):
        assert torch.equal(a[healthy], b[healthy])
    z = torch.randn((3, E + 1), generator=g, device=DEV)
    z[1], z[2, E // 2] = math.nan, math.nan
    from_logits = ops.route_experts(z, E, top, groups, keep, 1.0, True, score=score)[0]
    for ids in (got[0], from_logits):
        assert int(ids.min()) >= 0 and int(ids.max()) < E
        assert bool((ids.sort(dim=1).values.diff(dim=1) > 0).all()), "an expert was chosen twice"
    assert torch.equal(got[0][0], from_logits[1]), "the two kernels choose differently for a row of NaNs"


@pytest.mark.parametrize("sizes", [(16, 4), (64, 8)])
def test_diverged_rows_leave_the_others_alone(ops, sizes):
    """Router and experts of 16 rows, eight of them diverged, some before healthy ones in the step: the healthy rows are bit for
    bit what they are without them.  (The memory that the parts come from holds NaNs beforehand.)"""
    E, top = sizes
    w, packed, _, _, _ = make(ops, (16, E, 0, top, 128, 64, 0), "silu")
    rows = (torch.randn((E, 128), generator=torch.Generator(device=DEV).manual_seed(3), device=DEV) * 0.3).to(BF)
    bad, healthy = _diverged(w["x"])
    bad[12] = math.nan
    healthy.remove(12)

    def run(x):
        ids, weights, _ = ops.router(x, rows, E, top, 1, 1, 1.0, False)
        stale = torch.full((top, 16, 128), math.nan, device=DEV)
        del stale
        return ops.resolve(ops.experts_of_few_rows(x, ids, weights, packed, None, None, None))
    want, got = run(w["x"]), run(bad)
    assert torch.equal(got[healthy], want[healthy])
    assert bool(got[[0, 8, 9, 12]].isnan().all())


@pytest.mark.parametrize("size", [(3, 4, 0, 2, 72, 40, 48), (16, 16, 0, 3, 136, 72, 0), (17, 8, 1, 4, 136, 272, 32), (20, 200, 0, 4, 96, 48, 0),
                                  (64, 5, 0, 8, 128, 64, 16)])
@pytest.mark.parametrize("kind", ["silu", "relu2"])
def test_rows_that_name_an_expert_twice(ops, size, kind):
    """More pairs of an expert than rows: the slots are filled several times, and no part is left as the memory was."""
    T, E, identity, top, D = size[:5]
    if kind == "relu2" and identity:
        pytest.skip("experts whose weight goes on their input all have matrices")
    w, packed, ids, weights, (up, down, gate) = make(ops, (T, max(E, top), identity, top, *size[4:]), kind)
    E = max(E, top)
    g = torch.Generator(device=DEV).manual_seed(T)
    ids = torch.randint(0, 2, (T, top), generator=g, device=DEV, dtype=torch.int32) + E - 2 + identity
    weights = torch.rand((T, top), generator=g, device=DEV)
    how = {"silu": {}, "relu2": dict(activation="relu2", weight_on_input=True)}[kind]
    stale = torch.full((top + 1, T, D), math.nan, device=DEV)
    del stale
    got = ops.resolve(ops.experts_of_few_rows(w["x"], ids, weights, packed, up, down, gate, handed_on=identity > 0, **how))
    want = plain(w, ids, weights, gate, E, kind)
    # as for test_experts_of_few_rows; terms of the same expert add up, by at most the root of their number (8 places: 3 times)
    scale = float(want.square().mean().sqrt())
    assert float((got.double() - want).abs().max()) <= 15 * 2.0 ** -9 * scale + 2.0 ** -8 * float(want.abs().max())


def test_an_infinity_at_the_end_of_k(ops):
    """Rows whose last values are infinite, with k no multiple of 128: the sums are infinite and not NaN, in the hidden units
    and (these being infinite) in the outputs; the other rows are what they are without them."""
    T, E, top, D, ff = 5, 4, 2, 72, 200
    w, packed, ids, weights, _ = make(ops, (T, E, 0, top, D, ff, 0), "relu2")
    down = w["down"].abs().clamp(min=0.01)
    up = w["up"].clone()
    up[:, :, D - 1] = 0.5
    packed = ops.pack_experts(up, down, gated=False)

    def run(x):
        return ops.resolve(ops.experts_of_few_rows(x, ids, weights + 0.1, packed, None, None, None, activation="relu2"))
    x = w["x"].clone()
    x[3, D - 1] = math.inf
    got, without = run(x), run(w["x"])
    assert bool((got[3] == math.inf).all())
    assert torch.equal(got[[0, 1, 2, 4]], without[[0, 1, 2, 4]])


def test_rows_and_experts_of_the_faster_way(ops):
    """Beyond 32 rows only up to 32 experts go to the kernels of few rows; what the part gives is the same either way."""
    from tiny_llm_infer_amd.kernels.ops import DeferredSum
    from tiny_llm_infer_amd.config import PartSpec
    from tiny_llm_infer_amd.parts.base import BuildEnv, build_part
    env = BuildEnv(dtype=BF, device=torch.device(DEV), ops=ops, max_model_len=64)
    g = torch.Generator(device=DEV).manual_seed(4)
    for E, rows, few in ((32, 64, True), (33, 32, True), (33, 33, False), (200, 64, False), (33, 1, True)):
        part = build_part("ffn", PartSpec("routed_experts", {"hidden_size": 64, "experts": E, "top": 2, "intermediate_size": 32},
                                          {"router": "router", "experts": "e{}."}))
        part.load({d.name: (torch.randn(d.shape, generator=g, device=DEV) * d.shape[1] ** -0.5).to(BF) for d in part.tensors()}, env)
        x = torch.randn((rows, 64), generator=g, device=DEV).to(BF)
        y = part.forward(x, None)
        assert isinstance(y, DeferredSum) == few, (E, rows)
        ids, weights, _ = ops.router(x, part.w_router, E, 2, 1, 1, 1.0, False)
        other = ops.apply_experts(x, ids, weights, None, None, part.packed, None, None)
        # hidden units, parts and results are rounded to bfloat16 on the way: a few of its steps at the size of the largest
        assert float((ops.resolve(y).double() - other.double()).abs().max()) <= 2.0 ** -6 * float(other.double().abs().max())
