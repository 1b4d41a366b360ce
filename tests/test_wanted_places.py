"""Which places' logits a step hands out: all of its rows in their order, some of them, one of them twice; eagerly and from
recordings, on the CPU with a stand-in for the device's recording."""
import contextlib

import numpy as np
import pytest
import torch

from helpers import TINY

# What the requests of steps of one token each want, step by step: as many places as entries, so that all are recorded steps.
RECORDED = {1: [((0,),), ((0,),), ((0,),)],
            2: [((0,), (0,)), ((0, 0), ()), ((0,), (0,)), ((), (0, 0)), ((0, 0), ()), ((0,), (0,))],
            3: [((0,), (0,), (0,)), ((0, 0), (), (0,)), ((), (0,), (0, 0)), ((0,), (0,), (0,)), ((0, 0, 0), (), ())],
            16: [((0,),) * 16, ((0, 0), ()) * 8, ((0,),) * 16, ((), (0, 0)) * 8]}
# ... and steps that are not recorded: fewer places than entries, and more.
EAGER = {n: [((0,),) * (n - 1) + ((),), ((),) * (n - 1) + ((0, 0),) if n > 2 else ((0, 0),) * n] for n in RECORDED}


def _steps(requests):
    return RECORDED[requests] + EAGER[requests]


def _setup(runner, vocab, requests, seed=3):
    """The requests' prompts are run; returns the tokens of the steps that follow."""
    from tiny_llm_infer_amd.engine.runner import StepEntry
    rng = np.random.default_rng(seed)
    for i in range(requests):
        runner.admit(i)
        runner.step([StepEntry(i, rng.integers(0, vocab, 3 + i).tolist(), [])])
    return rng.integers(0, vocab, (len(_steps(requests)), requests)).tolist()


def _run(runner, tokens, wants):
    from tiny_llm_infer_amd.engine.runner import StepEntry
    y = runner.step([StepEntry(i, [t], w) for i, (t, w) in enumerate(zip(tokens, wants))])
    return None if y is None else y.float().cpu().clone()


def _places(wants):
    return [i for i, w in enumerate(wants) for _ in w]


class Recording:
    """A replay runs the step that was recorded, with the host's values of then and the device's inputs of now."""
    taking, forward = None, None

    def pool(self):
        return None

    def replay(self):
        view, wanted, out = self.taken
        out.copy_(Recording.forward(view, wanted))


@contextlib.contextmanager
def _take(graph, pool=None):
    Recording.taking = graph
    yield
    Recording.taking = None


def _record_on_cpu(runner, monkeypatch):
    plain = Recording.forward = runner.forward

    def forward(view, wanted):
        out = plain(view, wanted)
        if Recording.taking is not None:
            Recording.taking.taken = (view, wanted, out)
        return out

    monkeypatch.setattr(runner, "forward", forward)
    monkeypatch.setattr(torch.cuda, "synchronize", lambda device=None: None)
    monkeypatch.setattr(torch.cuda, "CUDAGraph", Recording)
    monkeypatch.setattr(torch.cuda, "graph", _take)
    runner.use_graphs = True


@pytest.mark.parametrize("requests", sorted(RECORDED))
def test_places_of_recorded_steps(model_folders, monkeypatch, requests):
    """Every step's logits are those of a runner that hands out every row, picked by place, whatever was recorded before."""
    from cpu_ops import CpuOps
    from tiny_llm_infer_amd.engine.loading import load_model
    from tiny_llm_infer_amd.engine.runner import ModelRunner
    model, _ = load_model(model_folders["A"], "float32", "cpu", ops=CpuOps())
    fast, slow = (ModelRunner(model, model.env, page_size=TINY["A"]["page_size"], num_pages=200, max_requests=16, max_batch_tokens=64) for _ in range(2))
    vocab = model.spec.vocab_size
    tokens = _setup(fast, vocab, requests)
    assert tokens == _setup(slow, vocab, requests)
    _record_on_cpu(fast, monkeypatch)
    for step, (row, wants) in enumerate(zip(tokens, _steps(requests))):
        every = _run(slow, row, ((0,),) * requests)
        got, at = _run(fast, row, wants), _places(wants)
        if not at:
            assert got is None
            continue
        # (another number of rows may add up in another order)
        assert got.shape == every[at].shape and float((got - every[at]).abs().max()) <= 2e-5 * float(every.abs().max()), f"step {step}: {wants}"
    assert fast.graph_replays > 0


def test_fewer_places_than_a_step_was_packed_with(model_folders):
    """A packed step's first rows alone: ``forward`` of fewer places than it has."""
    from cpu_ops import CpuOps
    from tiny_llm_infer_amd.engine.loading import load_model
    from tiny_llm_infer_amd.engine.runner import ModelRunner, StepEntry
    model, _ = load_model(model_folders["A"], "float32", "cpu", ops=CpuOps())
    runner = ModelRunner(model, model.env, page_size=TINY["A"]["page_size"], num_pages=200, max_requests=16, max_batch_tokens=64)
    runner.admit(0)
    runner.cache.reserve(0, 4)
    view = runner._pack([StepEntry(0, [1, 2, 3, 4], [0, 1, 2, 3])])
    every = runner.forward(view, 4)
    asked = {}
    view.sample_rows = view.sample_rows[:2]
    close = model.close_residual
    model.close_residual = lambda *args, **how: (asked.update(how), close(*args, **how))[1]
    assert view.all_wanted and torch.allclose(runner.forward(view, 2), every[:2], atol=1e-5) and not asked["all_rows"]


@pytest.mark.gpu
@pytest.mark.parametrize("recorded", [True, False])
@pytest.mark.parametrize("requests", sorted(RECORDED))
@pytest.mark.parametrize("name", ["B", "D"])
def test_places_on_the_device(model_folders, name, requests, recorded):
    """The same with the norms in the products and in launches of their own, on the device: bfloat16 rows that are rounded in other
    places (2^-9 of an element each time, some ten times a layer, three layers at most: a 50th of the largest logit at the outside), and
    places of one row with the same bits."""
    from tiny_llm_infer_amd.engine.loading import load_model
    from tiny_llm_infer_amd.engine.runner import ModelRunner
    model, _ = load_model(model_folders[name], "bfloat16", "cuda:0")
    ops = model.env.ops
    fast, slow = (ModelRunner(model, model.env, page_size=16, num_pages=60, max_requests=16, max_batch_tokens=64) for _ in range(2))
    fast.use_graphs, slow.use_graphs = recorded, False
    vocab = model.spec.vocab_size
    tokens = _setup(fast, vocab, requests)
    assert tokens == _setup(slow, vocab, requests)
    for step, (row, wants) in enumerate(zip(tokens, _steps(requests))):
        got, at = _run(fast, row, wants), _places(wants)
        before, ops.separate_norms = ops.separate_norms, True
        every = _run(slow, row, ((0,),) * requests)
        ops.separate_norms = before
        if not at:
            assert got is None
            continue
        assert got.shape == every[at].shape and float((got - every[at]).abs().max()) <= 0.02 * float(every.abs().max()), f"step {step}: {wants}"
        for i in range(1, len(at)):
            assert at[i] != at[i - 1] or torch.equal(got[i], got[i - 1])
    assert (fast.graph_replays > 0) == recorded
