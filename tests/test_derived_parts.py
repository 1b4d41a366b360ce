"""Parts derived from the stock ones with a ``forward`` of their own are run as they were written: what the stock parts' launches take
in besides (a block's opening norm, a norm's rows or its factor, a choice of experts) is theirs alone."""
import types

from tiny_llm_infer_amd.engine.model import Model
from tiny_llm_infer_amd.parts.block import PreNormBlock
from tiny_llm_infer_amd.parts.embedding import LinearHead, TokenEmbedding
from tiny_llm_infer_amd.parts.joined import OneNormParallelBlock
from tiny_llm_infer_amd.parts.moe import RoutedExperts
from tiny_llm_infer_amd.parts.norm import RMSNorm


def derived(cls):
    return type("Own" + cls.__name__, (cls,), {"forward": lambda self, *args: None})


def bare(cls, **attributes):
    part = object.__new__(cls)
    part.__dict__.update(attributes)
    return part


def test_heads_and_experts():
    weight = types.SimpleNamespace(tiled=object())
    assert bare(LinearHead, weight=weight).takes_normed_rows and not bare(derived(LinearHead), weight=weight).takes_normed_rows
    assert not bare(LinearHead).takes_normed_rows and not bare(LinearHead, weight=types.SimpleNamespace(tiled=None)).takes_normed_rows
    assert bare(RoutedExperts).takes_choice and not bare(derived(RoutedExperts)).takes_choice


def test_blocks():
    part = types.SimpleNamespace(replayable=True, load_rows=None, rows=None)
    for cls, norms in ((PreNormBlock, {"mixer": part, "ffn": part}), (OneNormParallelBlock, {"mixer": part})):
        spec = types.SimpleNamespace(params={}, names={}, parts={})
        assert cls(spec, part, part, norms).opening_norm is part and derived(cls)(spec, part, part, norms).opening_norm is None


def test_embeddings():
    ops = types.SimpleNamespace(embed_rmsnorm=lambda *args: "both")
    norm = types.SimpleNamespace(as_rms=lambda: (None, 1e-6))
    own = dict(env=types.SimpleNamespace(ops=ops), pos_table=None, scale=1.0, table=None)
    assert bare(TokenEmbedding, **own).forward_normed(None, 1, norm) == "both"
    assert bare(derived(TokenEmbedding), **own).forward_normed(None, 1, norm) is None
    assert bare(TokenEmbedding, **dict(own, scale=2.0)).forward_normed(None, 1, norm) is None
    assert bare(TokenEmbedding, **own).forward_normed(None, 1, types.SimpleNamespace(as_rms=lambda: None)) is None


def test_norms_at_both_ends_of_a_model():
    """A norm derived from the stock one with a ``forward`` of its own makes its rows itself, as a model's first norm and as its last;
    that ``forward`` takes what ``Norm.forward`` says and no more."""
    def forward(self, resid, delta, rows=None, num_rows=None):
        return "own", rows is None
    own_norm = type("OwnNorm", (RMSNorm,), {"forward": forward})
    ops = types.SimpleNamespace(embed_rmsnorm=lambda *args: ("resid", "normed"), embed=lambda *args: "rows",
                                add_rmsnorm=lambda *args, lazy=False, rows=None, num_rows=None: ("stock", lazy, rows is None))
    env = types.SimpleNamespace(ops=ops, dtype=None)
    embedding = bare(TokenEmbedding, env=env, pos_table=None, scale=1.0, table=None)
    head = bare(LinearHead, weight=types.SimpleNamespace(tiled=object()))
    for norm, opening, closing in ((bare(RMSNorm, env=env, weight=None, eps=1e-6), ("resid", {"normed": "normed"}), ("stock", True, True)),
                                   (bare(own_norm, env=env, weight=None, eps=1e-6), ("rows", {}), ("own", False))):
        block = bare(PreNormBlock, opening_norm=norm)
        model = bare(Model, embedding=embedding, blocks=[block], schedule=[types.SimpleNamespace(block=0)], final_norm=norm, head=head)
        assert model.embed(None, 2, None) == opening
        assert model.close_residual("rows", None, rows=[0, 1], num_rows=2, all_rows=True) == closing
        model.schedule = []
        assert model.close_residual("rows", None, rows=[0, 1], num_rows=2, all_rows=True) == closing
