"""Decode steps of the float32 path, replayed from recordings: the logits of every design equal those of steps run eagerly, with
requests that come and go in between, and are the caller's: later steps leave them as they are."""
import numpy as np
import pytest
import torch

import defosun_helpers
import gimipel_helpers
import kapanex_helpers
import kosusun_helpers
import kunitar_helpers
import sinepel_helpers

pytestmark = pytest.mark.gpu


def _kosusun(folder):
    cfg, _, seed = kosusun_helpers.SMALL["A"]
    return kosusun_helpers.write_folder(folder, cfg, kosusun_helpers.make_weights(cfg, seed))


def _defosun(folder):
    return defosun_helpers.make_folder(folder, "A")


DESIGNS = {"kapanex": lambda f: kapanex_helpers.make_folder(f, "A"), "gimipel": lambda f: gimipel_helpers.make_folder(f, "A"),
           "sinepel": lambda f: sinepel_helpers.make_folder(f, "R"), "kunitar": lambda f: kunitar_helpers.make_folder(f, "A"),
           "kosusun": _kosusun, "defosun": _defosun}


def _folder(design, tmp_path, model_folders):
    if design.startswith("qwen3"):
        return model_folders[design[-1]]
    return DESIGNS[design](str(tmp_path / design))


@pytest.mark.parametrize("design", ["qwen3 A", "qwen3 B", "qwen3 D"] + list(DESIGNS))
def test_recorded_steps_equal_eager_ones_and_stay(tmp_path, model_folders, design):
    from tiny_llm_infer_amd.engine.loading import load_model
    from tiny_llm_infer_amd.engine.runner import ModelRunner, StepEntry
    model, _ = load_model(_folder(design, tmp_path, model_folders), "float32", "cuda:0", max_model_len=256)
    vocab = model.spec.vocab_size
    fast, slow = (ModelRunner(model, model.env, page_size=16, num_pages=40, max_requests=4, max_batch_tokens=128) for _ in range(2))
    assert fast.use_graphs
    slow.use_graphs = False
    rng = np.random.default_rng(5)
    live, kept = {}, []
    for it in range(60):
        if len(live) < 3 and rng.random() < 0.5:
            key, prompt = f"r{it}", rng.integers(0, vocab, int(rng.integers(2, 40))).tolist()
            for r in (fast, slow):
                r.admit(key)
                r.step([StepEntry(key, prompt, [])])
            live[key] = len(prompt)
        if not live:
            continue
        entries = [StepEntry(k, [int(rng.integers(0, vocab))], [0]) for k in live]
        kept.append((fast.step(entries), slow.step(entries).clone()))
        torch.cuda.synchronize()
        for k in list(live):
            live[k] += 1
            if live[k] > 100 or rng.random() < 0.03:
                live.pop(k)
                for r in (fast, slow):
                    r.release(k)
    assert fast.graph_replays > 30
    for i, (a, b) in enumerate(kept):
        # (a step is filled up to a few sizes, and some sums go in another order with the number of rows)
        assert float((a - b).abs().max()) <= 2e-5 * float(b.abs().max()), f"step {i} of {len(kept)}"
