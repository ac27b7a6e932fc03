"""When Mamba.step takes the whole-layer call (redpanda_amd/layer_step.py):
the models that must keep the separate ops, decided on the CPU from the models
alone."""

import pytest
import torch
import torch.nn as nn

from redpanda_amd import layer_step
from redpanda_amd.mamba import Mamba, Mamba3Block, MambaConfig


def _model(**kw):
    return Mamba(MambaConfig(**{**dict(d_model=64, n_layer=2, vocab_size=64, d_state=20,
                                       n_track_state=4, mimo_p=2), **kw})).eval()


def _x(R=4):
    return torch.randn(R, 64)


def _mixer(m):
    return m.layers[1]["mixer"]


def test_plain_models_take_it():
    for kw in ({}, dict(bias=True), dict(use_bcnorm=False), dict(n_track_state=0),
               dict(use_complex=False)):
        assert layer_step.usable(_model(**kw), _x())


@pytest.mark.parametrize("where,n", [
    (lambda m: m.layers[1]["norm"], 1), (lambda m: m.layers[0]["norm"], 68),
    (lambda m: _mixer(m).b_norm, 1), (lambda m: _mixer(m).c_norm, 44)])
def test_norm_weights_of_another_length_are_left_to_the_separate_ops(where, n):
    m = _model()
    where(m).weight = nn.Parameter(torch.ones(n))
    assert not layer_step.usable(m, _x())


@pytest.mark.parametrize("proj", ["in_proj", "x_proj", "dt_proj", "out_proj"])
def test_biases_of_another_length_are_left_to_the_separate_ops(proj):
    m = _model(bias=True)
    getattr(_mixer(m), proj).bias = nn.Parameter(torch.ones(4))
    assert not layer_step.usable(m, _x())


def test_a_skip_of_another_length_is_left_to_the_separate_ops():
    m = _model()
    _mixer(m).D = nn.Parameter(torch.ones(4))
    assert not layer_step.usable(m, _x())


def test_a_layer_is_judged_by_its_own_configuration():
    """A mixer with BCNorm in a model configured without it."""
    m = _model(use_bcnorm=False)
    m.layers[1]["mixer"] = _model().layers[1]["mixer"]
    assert layer_step.usable(m, _x())
    _mixer(m).b_norm.weight = nn.Parameter(torch.ones(4))
    assert not layer_step.usable(m, _x())


class _CountingBlock(Mamba3Block):
    def step(self, *args, **kw):
        return super().step(*args, **kw)


def _subclass(m, monkeypatch):
    _mixer(m).__class__ = _CountingBlock


def _own_step(m, monkeypatch):
    block = _mixer(m)
    block.step = lambda *args, **kw: Mamba3Block.step(block, *args, **kw)


def _class_step(m, monkeypatch):
    step = Mamba3Block.step
    monkeypatch.setattr(Mamba3Block, "step", lambda self, *args, **kw: step(self, *args, **kw))


def _own_forward(m, monkeypatch):
    lin = _mixer(m).dt_proj
    lin.forward = lambda x: nn.Linear.forward(lin, x) * 2


def _class_forward(m, monkeypatch):
    fwd = nn.Linear.forward
    monkeypatch.setattr(nn.Linear, "forward", lambda self, x: fwd(self, x) * 2)


class _Wrapped(torch.Tensor):
    pass


def _tensor_subclass(m, monkeypatch):
    lin = _mixer(m).in_proj
    lin.weight = nn.Parameter(lin.weight.detach().as_subclass(_Wrapped))


def _no_module(m, monkeypatch):
    _mixer(m).x_proj = nn.Sequential(_mixer(m).x_proj)


@pytest.mark.parametrize("change", [_subclass, _own_step, _class_step, _own_forward, _class_forward,
                                    _tensor_subclass, _no_module])
def test_replaced_methods_and_types_keep_the_separate_ops(change, monkeypatch):
    """What ran in the layer's place before the whole-layer call still runs."""
    m = _model()
    change(m, monkeypatch)
    assert not layer_step.usable(m, _x())
    monkeypatch.undo()
    assert layer_step.usable(_model(), _x())


def test_host_tensors_are_refused_as_before():
    """By the separate ops' own check, whether or not a GPU is there."""
    with torch.no_grad(), pytest.raises(ValueError, match="device tensor"):
        _model().step(input_embed=_x())


@pytest.mark.parametrize("d,rows", [(64, 256), (512, 256), (576, 128), (1024, 128), (1280, 51),
                                    (2048, 32)])
def test_the_most_rows_fall_with_the_width(d, rows):
    m = _model(d_model=d, n_layer=1)
    assert layer_step.usable(m, torch.zeros(rows, d))
    assert not layer_step.usable(m, torch.zeros(rows + 1, d))


def test_the_inner_width_counts_too():
    m = _model(d_model=256, expand=8, n_layer=1)  # as wide as d_model 1024
    assert layer_step.usable(m, torch.zeros(128, 256))
    assert not layer_step.usable(m, torch.zeros(129, 256))
