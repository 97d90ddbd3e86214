"""Clipping and the AdamW update of a training step in the kernels of ``csrc/mts_optim.hip``.

Same results as ``clip_grad_norm_`` and the stock fused ``AdamW.step()``: the state is the optimizer's own, so a state
dict, a scheduler or a later stock step goes on from it.  :func:`plan` says whether an update may be taken so; everything else (other
optimizers and options, hooks that look on, parameters that the optimizer does not own) stays with the stock calls.
"""

import torch
from torch.optim import optimizer as _optimizer

from minitrain_amd import _lib
from minitrain_amd.train.modules import parameters_of, plain_modules


# torch._compile: wraps zero_grad, for the compiler to leave it alone
_TORCH_OWN = ("torch.optim.optimizer", "torch.optim.adam", "torch.optim.adamw", "torch.nn.utils.clip_grad", "torch._compile")


def _is_torch_own(function) -> bool:
    """Whether ``function`` and all that it wraps are written in the modules of torch's AdamW and clipping."""
    while function is not None:
        if getattr(function, "__globals__", {}).get("__name__") not in _TORCH_OWN:
            return False
        function = getattr(function, "__wrapped__", None)
    return True


def _runs_as_written(optimizer) -> bool:
    """Whether ``optimizer.step()`` is AdamW's and nobody looks on."""
    if type(optimizer) is not torch.optim.AdamW or hasattr(optimizer, "grad_scale") or hasattr(optimizer, "found_inf"):
        return False
    if optimizer._optimizer_step_pre_hooks or optimizer._optimizer_step_post_hooks:
        return False
    if _optimizer._global_optimizer_pre_hooks or _optimizer._global_optimizer_post_hooks:
        return False
    if not _is_torch_own(torch.optim.AdamW.step):   # replaced on the class
        return False
    if "zero_grad" in optimizer.__dict__ or not _is_torch_own(torch.optim.AdamW.zero_grad):   # may keep the gradients, which are to be clipped ones then
        return False
    step = optimizer.__dict__.get("step")   # a learning-rate scheduler wraps it to note that it has run
    return step is None or (getattr(step, "_wrapped_by_lr_sched", False) and getattr(step, "__wrapped__", None) is torch.optim.AdamW.step)


def _clips_as_written() -> bool:
    """Whether the clipping that a step calls is torch's: another may stand in its place."""
    return _is_torch_own(torch.nn.utils.clip_grad_norm_)


class Update:
    """The tensors of one update."""

    def __init__(self, optimizer):
        self.optimizer = optimizer
        self.params, self.exp_avgs, self.exp_avg_sqs, self.steps, self.groups, self.settings = [], [], [], [], [], []
        self.clipped = False

    def add_group(self, group) -> bool:
        if not group["fused"] or group["amsgrad"] or group["maximize"] or group["capturable"] or group["differentiable"] or group["foreach"]:
            return False
        if not group.get("decoupled_weight_decay", True):   # Adam's decay, by the gradient
            return False
        numbers = (group["lr"], *group["betas"], group["eps"], group["weight_decay"])
        if any(isinstance(n, torch.Tensor) for n in numbers):
            return False
        for p, defined in zip(group["params"], _lib.host().gradients_defined(group["params"])):
            if not defined:
                continue
            state = self.optimizer.state.get(p)
            if not state:   # the first step makes it
                return False
            self.params.append(p)
            self.exp_avgs.append(state["exp_avg"])
            self.exp_avg_sqs.append(state["exp_avg_sq"])
            self.steps.append(state["step"])
            self.groups.append(len(self.settings))
        self.settings.append(tuple(float(n) for n in numbers))
        return True

    def norm(self, max_norm: float | None, loss: torch.Tensor) -> torch.Tensor:
        """``[norm, clipping coefficient, whether norm or loss are not finite]``"""
        self.clipped = max_norm is not None
        return _lib.host().grad_norm(self.params, -1.0 if max_norm is None else max_norm, loss)

    def apply(self, norm: torch.Tensor, skip_if_not_finite: bool) -> None:
        _lib.host().adamw(self.params, self.exp_avgs, self.exp_avg_sqs, self.steps, self.groups, self.settings, norm, self.clipped,
                           skip_if_not_finite)
        if "step" in self.optimizer.__dict__:
            self.optimizer._opt_called = True

    def drop_gradients(self) -> None:
        """``optimizer.zero_grad(set_to_none=True)``: no other parameter of the optimizer has a gradient"""
        _lib.host().drop_gradients(self.params)


def plan(model: torch.nn.Module, optimizer: torch.optim.Optimizer, loss: torch.Tensor, grad_clip_norm: float | None) -> Update | None:
    """The update that the kernels can take in the place of clipping and ``optimizer.step()``, or None."""
    if not loss.is_cuda or loss.dtype != torch.float32 or loss.numel() != 1 or torch.compiler.is_compiling() or torch.cuda.is_current_stream_capturing():
        return None
    if not _runs_as_written(optimizer) or (grad_clip_norm is not None and not (grad_clip_norm >= 0 and _clips_as_written())):
        return None
    update = Update(optimizer)
    if len(optimizer.param_groups) > _lib.host().ADAM_GROUPS or not all(update.add_group(g) for g in optimizer.param_groups):
        return None
    # clipping looks at the model's gradients, the update at the optimizer's: the same ones
    of_model = parameters_of(model, plain_modules(model))
    if {id(p) for p, defined in zip(of_model, _lib.host().gradients_defined(of_model)) if defined} != {id(p) for p in update.params}:
        return None
    if not _lib.host().adamw_supported(update.params, update.exp_avgs, update.exp_avg_sqs, update.steps) or loss.device != update.params[0].device:
        return None
    return update
