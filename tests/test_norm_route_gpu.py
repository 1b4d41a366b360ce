"""Norms that choose the routed experts of their rows in the same launch, beside the norm and the router on their own: the same
bits, for every width and number of logits at the edges of what the launch takes, and None past them."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
BF = torch.bfloat16

# (rows, width, experts, shared gate, top, groups, keep, more)
CASES = [(1, 8, 1, False, 1, 1, 1, {}), (8, 2048, 16, True, 2, 4, 4, {}), (3, 2056, 16, False, 3, 1, 1, {"score": "softmax"}),
         (128, 512, 31, True, 8, 1, 1, {"normalize": False}), (5, 4096, 32, False, 4, 8, 3, {"group_score": "max"}),
         (2, 1000, 17, True, 17, 1, 1, {"correction": True}), (16, 4088, 24, True, 2, 6, 2, {"correction": True, "score": "softmax"})]


@pytest.fixture(scope="module")
def ops():
    from tiny_llm_infer_amd.kernels.ops import DeferredSum, HipOps
    out = HipOps(DEV)
    out.deferred = DeferredSum
    return out


def make(case):
    T, n, E, shared, top, groups, keep, more = case
    g = torch.Generator(device=DEV).manual_seed(T * n + E)
    rnd = lambda *shape: torch.randn(*shape, generator=g, device=DEV)
    route = dict(w_rows=(rnd(E + shared, n) * n ** -0.5 * 2).to(BF), experts=E, top=top, groups=groups, keep=keep, scale=1.5, has_shared=shared, **more)
    if more.get("correction"):
        route["correction"] = rnd(E)
    return rnd, route


def same(a, b):
    assert (a is None) == (b is None)
    if a is not None:
        assert a.dtype == b.dtype and torch.equal(a.view(torch.uint8), b.view(torch.uint8))


def deltas_of(ops, kind, rnd, T, n):
    if kind == "none":
        return ()
    if kind == "sums":
        return (rnd(T, n).to(BF), ops.deferred(rnd(3, T, n), BF))
    return tuple(rnd(T, n).to(BF) for _ in range(1 if kind == "one" else 2))


@pytest.mark.parametrize("kind", ["none", "one", "two", "sums"])
@pytest.mark.parametrize("case", CASES)
def test_layer_norms_with_a_router(ops, case, kind):
    T, n = case[:2]
    rnd, route = make(case)
    resid = rnd(T, n) * 3
    if T > 1:
        resid[1, n // 2] = float("nan")                    # (a row that holds no numbers chooses different experts too)
    deltas, weights = deltas_of(ops, kind, rnd, T, n), tuple(rnd(n) + 1 for _ in range(2 if kind != "one" else 1))
    r1, r2 = resid.clone(), resid.clone()
    outs, routed = ops.add_layernorm_route(r1, deltas, weights, 1e-5, BF, route)
    want = ops.add_layernorm(r2, deltas, weights, 1e-5, BF)
    same(r1, r2)
    for a, b in zip(outs, want):
        same(a, b)
    for a, b in zip(routed, ops.router(want[-1], **route)):
        same(a, b)


@pytest.mark.parametrize("kind", ["none", "one", "sums"])
@pytest.mark.parametrize("case", CASES)
def test_norms_behind_a_normed_sum_with_a_router(ops, case, kind):
    T, n = case[:2]
    rnd, route = make(case)
    resid = rnd(T, n) * 3
    if T > 1:
        resid[1, n // 2] = float("nan")
    owed = deltas_of(ops, kind, rnd, T, n)
    y, w_out, w_in = owed[-1] if owed else None, rnd(n) + 1, rnd(n) + 1
    r1, r2 = resid.clone(), resid.clone()
    out, routed = ops.norm_add_norm_route(r1, y, w_out, 1e-6, w_in, 1e-5, BF, route)
    want = ops.norm_add_norm(r2, y, w_out, 1e-6, w_in, 1e-5, BF)
    same(r1, r2)
    same(out, want)
    for a, b in zip(routed, ops.router(want, **route)):
        same(a, b)


@pytest.mark.parametrize("T, n, E, shared", [(129, 64, 4, False), (4, 4104, 4, False), (4, 64, 32, True), (4, 64, 33, False), (4, 60, 4, False)])
def test_what_such_a_norm_leaves_to_the_router(ops, T, n, E, shared):
    rnd, route = make((T, n, E, shared, 2, 1, 1, {}))
    resid = rnd(T, n)
    before = resid.clone()
    assert ops.add_layernorm_route(resid, (rnd(T, n).to(BF),), (rnd(n),), 1e-5, BF, route) is None
    assert ops.norm_add_norm_route(resid, rnd(T, n).to(BF), rnd(n), 1e-5, rnd(n), 1e-5, BF, route) is None
    same(resid, before)
