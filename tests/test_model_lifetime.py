"""A model's lifetime: decoders and captured graphs go with the last reference to it."""
import copy
import gc
import pickle
import weakref

import pytest
import torch

from smlm_hip.model import ModelConfig, Transformer, _FusedDecodeStep, _StepDecoder

MEMORY = dict(mem_layers=[1], mem_n_keys=8, mem_heads=2, mem_knn=2, mem_k_dim=16)


def _model(**over):
    torch.manual_seed(0)
    return Transformer(ModelConfig(vocab_size=64, d_model=32, n_layers=2, n_heads=2, ffn_hidden=32, max_seq_len=32,
                                   **over)).eval()


def _generate(model):
    return model.generate(torch.arange(6).view(2, 3), 4, use_graph=False)


@pytest.fixture
def no_collector():
    gc.collect()
    was = gc.isenabled()
    gc.disable()
    yield
    if was:
        gc.enable()


def test_a_model_that_has_decoded_dies_with_its_last_reference(no_collector):
    """Without the cyclic collector: a decoder that kept its model alive would leave both, with the model's table, the
    caches and the captured graphs, to a collection at some later time."""
    model = _model()
    _generate(model)
    gone = [weakref.ref(model), weakref.ref(model.tok_emb.weight), *map(weakref.ref, model._decoders.values())]
    del model
    assert [r() for r in gone] == [None] * 3


def test_the_fused_step_does_not_keep_its_model(no_collector):
    model = _model(**MEMORY)
    step = _FusedDecodeStep(model)
    assert step.model is model
    gone = weakref.ref(model)
    del model
    assert gone() is None
    with pytest.raises(ReferenceError):
        step.run(torch.zeros(1, 1, dtype=torch.long), torch.zeros((), dtype=torch.long), [], None)


@pytest.mark.parametrize("copied", [copy.deepcopy, lambda m: pickle.loads(pickle.dumps(m))], ids=["deepcopy", "pickle"])
def test_copies_and_pickles_of_a_model_decode_on_their_own(copied):
    model = _model()
    want = _generate(model)
    other = copied(model)
    (dec,) = other._decoders.values()
    assert type(dec) is _StepDecoder and dec.model is other
    assert torch.equal(_generate(other), want)
    assert list(other._decoders.values()) == [dec]


def test_a_shallow_copy_decodes_after_its_model_is_gone(no_collector):
    model = _model()
    want = _generate(model)
    other = copy.copy(model)
    assert torch.equal(_generate(other), want)
    del model
    assert torch.equal(_generate(other), want)
    (dec,) = other._decoders.values()
    assert dec.model is other
