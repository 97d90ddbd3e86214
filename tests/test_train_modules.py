"""The short walk through a model's modules, against the calls that it stands for (host code: no GPU)."""

import pytest
import torch
from torch import nn

from minitrain_amd.train.modules import parameters_of, plain_modules, set_training
from minitrain_amd.train.step import train_step


def _model():
    shared = nn.Linear(3, 3)
    return nn.Sequential(shared, nn.Sequential(nn.Dropout(0.1), shared, nn.ModuleList([nn.Linear(3, 2, bias=False)])), nn.Identity())


def test_modules_and_parameters_are_those_of_the_model():
    model = _model()
    modules = plain_modules(model)
    assert {id(m) for m in modules} == {id(m) for m in model.modules()} and len(modules) == len(list(model.modules()))
    assert {id(p) for p in parameters_of(model, modules)} == {id(p) for p in model.parameters()}
    assert [id(p) for p in parameters_of(model, None)] == [id(p) for p in model.parameters()]


def test_modules_that_are_not_in_training_are_put_there():
    model = _model()
    model[1][0].eval()
    set_training(model, plain_modules(model))
    assert all(m.training for m in model.modules())


@pytest.mark.parametrize("name", ["train", "named_parameters", "children"])
@pytest.mark.parametrize("how", ["class", "instance"])
def test_a_module_with_an_answer_of_its_own_is_asked(name, how):
    calls = []

    def answer(self, *args, **kwargs):
        calls.append(name)
        return getattr(nn.Linear, name)(self, *args, **kwargs)

    model = _model()
    if how == "class":
        model[1].append(type("Own", (nn.Linear,), {name: answer})(3, 3))
    else:
        model[1].append(nn.Linear(3, 3))
        model[1][-1].__dict__[name] = answer.__get__(model[1][-1])
    assert plain_modules(model) is None
    set_training(model, plain_modules(model))
    if name == "train":
        assert calls == ["train"]
    assert {id(p) for p in parameters_of(model, plain_modules(model))} == {id(p) for p in model.parameters()}
    model[1][-1].__dict__.pop(name, None)
    assert torch.is_tensor(model[1][-1].weight)


class _Head(nn.Linear):
    def forward(self, ids, *, targets, use_fused_loss):
        return (super().forward(ids) - targets).square().mean(), None


class _Wrapper:
    """No module, but all that a step calls."""

    def __init__(self, model):
        self.model, self.asked = model, 0

    def train(self):
        self.asked += 1
        return self.model.train()

    def parameters(self):
        return self.model.parameters()

    def __call__(self, *args, **kwargs):
        return self.model(*args, **kwargs)


def test_a_model_that_is_no_module_is_asked():
    model = _Wrapper(_Head(2, 1).eval())
    before = [p.detach().clone() for p in model.parameters()]
    train_step(model, torch.optim.SGD(model.parameters(), lr=0.1), {"input_ids": torch.ones(1, 2), "targets": torch.full((1, 1), 5.0)})
    assert model.asked == 1 and model.model.training
    assert not any(torch.equal(a, b) for a, b in zip(before, model.parameters()))
    assert plain_modules(model) is None and [id(p) for p in parameters_of(model, None)] == [id(p) for p in model.parameters()]


@pytest.mark.parametrize("name", ["train", "parameters", "_named_members"])
def test_a_call_that_was_replaced_on_the_class_of_all_modules_is_made(monkeypatch, name):
    calls, stock = [], getattr(nn.Module, name)

    def answer(self, *args, **kwargs):
        calls.append(name)
        return stock(self, *args, **kwargs)

    model = _model()
    monkeypatch.setattr(nn.Module, name, answer)
    set_training(model, plain_modules(model))
    list(parameters_of(model, plain_modules(model)))
    assert calls


def test_a_class_that_watches_its_mode_is_told():
    told = []

    class Watching(nn.Linear):
        def __setattr__(self, name, value):
            if name == "training":
                told.append(value)
            super().__setattr__(name, value)

    class Property(nn.Linear):
        @property
        def training(self):
            return True

        @training.setter
        def training(self, value):
            told.append(value)

    for cls in (Watching, Property):
        model = nn.Sequential(cls(3, 3))
        told.clear()
        set_training(model, plain_modules(model))
        assert told == [True]
