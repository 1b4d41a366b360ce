"""Steps of one row a sequence of the recurrent layers with the wide and the narrow workgroups, at both sides of the rule that chooses
and at sizes that leave threads idle or bring them back, beside the recurrence for any step."""
import pytest
import torch

from test_kapanex_gpu import _view

pytestmark = pytest.mark.gpu

# (heads, rows, dk, dv): workgroups and elements of a head's state at the rule's edges (512 and 256 workgroups, 2,048 elements, keys of 16)
SIZES = [(64, 8, 16, 16), (32, 8, 17, 120), (43, 6, 17, 120), (32, 16, 64, 32), (27, 19, 64, 32), (33, 16, 33, 300), (57, 9, 128, 16),
         (65, 8, 128, 24), (32, 17, 100, 128), (64, 8, 129, 16), (65, 8, 256, 20)]


@pytest.fixture(scope="module")
def ops():
    from tiny_llm_infer_amd.kernels.ops import HipOps
    return HipOps("cuda:0")


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("kind", ["retention", "mlstm", "wkv"])
@pytest.mark.parametrize("heads, rows, dk, dv", SIZES)
def test_wide_and_narrow_workgroups(ops, monkeypatch, kind, heads, rows, dk, dv, dtype):
    """The state to float32's sums (up to 256 products in another order); the rows to that or to the rounding of bfloat16, of sizes that
    the norm behind them makes about one."""
    g = torch.Generator(device="cuda").manual_seed(heads * rows + dk)
    rnd = lambda *shape: torch.randn(*shape, generator=g, device="cuda")
    view = _view([3 * (i % 5) for i in range(rows)], [1] * rows, list(reversed(range(rows))))          # every fifth sequence is new
    rank, n = 72, 136
    proj = rnd(rows, 2 * heads * (dk + dv)).to(dtype)
    x, w_gates, bias, weight = rnd(rows, n).to(dtype), (rnd(2 * heads, n) * n ** -0.5).to(dtype), rnd(2 * heads), rnd(heads * dv)
    z, w2, w0, u = rnd(rows, rank), (rnd(heads * dk, rank) * rank ** -0.5).to(dtype), rnd(heads * dk) - 2, rnd(heads, dk)
    first = rnd(rows, *(ops.mlstm_state_shape(heads, dk, dv) if kind == "mlstm" else (heads, dv, dk)))
    results = []
    for unfused in (False, True):
        monkeypatch.setattr(ops, "unfused_decode", unfused)
        state, maxima = first.clone(), torch.zeros(rows, heads, device="cuda")
        y = torch.zeros(rows, heads * dv, dtype=dtype, device="cuda")
        if kind == "retention":
            ops.retention(proj, 0, torch.linspace(0.5, 1.0, heads, device="cuda"), state, view, heads, dk, dv, None, dk ** -0.5, 1e-5, 1.0, y, 0)
        elif kind == "mlstm":
            ops.mlstm(proj, 0, x, w_gates, bias, 6.0, state, maxima, view, heads, dk, dv, dk ** -0.5, weight, 1e-5, 1.0, y, 0)
        else:
            y = ops.wkv(proj, z, (rank, 1), w2, w0, u, state, view, heads, dk, dv, weight, 1e-5, dtype)
        results.append((state, maxima, y.double()))
    (s0, m0, y0), (s1, m1, y1) = results
    assert float((s0 - s1).abs().max()) <= 2e-5 * float(s1.abs().max()) and float((m0 - m1).abs().max()) <= 2e-5 * (1 + float(m1.abs().max()))
    assert float((y0 - y1).norm() / y1.norm()) <= (1e-4 if dtype == torch.float32 else 2 ** -8)
