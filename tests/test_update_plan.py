"""Which optimizers the update in the kernels stands in for (host code: no GPU)."""

import functools

import torch

from minitrain_amd.train import update


def _optimizer():
    return torch.optim.AdamW([torch.nn.Parameter(torch.ones(3))], lr=1e-3)


def test_a_step_replaced_on_the_class_is_called(monkeypatch):
    opt = _optimizer()
    assert update._runs_as_written(opt)
    torch.optim.lr_scheduler.LambdaLR(opt, lambda _: 1.0)
    assert update._runs_as_written(opt)
    known = torch.optim.AdamW.step

    def step(self, closure=None):
        return known(self, closure)

    for replaced in (step, functools.wraps(known)(step)):
        with monkeypatch.context() as m:
            m.setattr(torch.optim.AdamW, "step", replaced)
            fresh = _optimizer()
            assert not update._runs_as_written(fresh) and not update._runs_as_written(opt)
            torch.optim.lr_scheduler.LambdaLR(fresh, lambda _: 1.0)
            assert not update._runs_as_written(fresh)
        assert update._runs_as_written(opt)


def test_decay_by_the_gradient_stays_stock():
    opt = torch.optim.AdamW([torch.nn.Parameter(torch.ones(3))], lr=1e-3)
    group = {**opt.param_groups[0], "fused": True}
    assert update.Update(opt).add_group(group)
    assert not update.Update(opt).add_group({**group, "decoupled_weight_decay": False})


def test_clipping_that_was_replaced_is_called(monkeypatch):
    assert update._clips_as_written()
    known = torch.nn.utils.clip_grad_norm_

    def clip(parameters, max_norm, *args, **kwargs):
        return known(parameters, max_norm, *args, **kwargs)

    for replaced in (clip, functools.wraps(known)(clip), functools.partial(known, norm_type=1.0)):
        with monkeypatch.context() as m:
            m.setattr(torch.nn.utils, "clip_grad_norm_", replaced)
            assert not update._clips_as_written()
    assert update._clips_as_written()


def test_gradients_that_another_zero_grad_may_keep_are_clipped_by_the_stock_calls(monkeypatch):
    opt = _optimizer()
    with monkeypatch.context() as m:
        m.setattr(torch.optim.AdamW, "zero_grad", lambda self, set_to_none=True: None)
        assert not update._runs_as_written(opt)
    assert update._runs_as_written(opt)
    opt.zero_grad = lambda set_to_none=True: None
    assert not update._runs_as_written(opt)
