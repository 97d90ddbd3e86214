"""The modules of a model in a short walk, for a training step that would otherwise recurse through them: with 47 modules (four layers)
``train()`` costs the host 160 us and ``parameters()`` 65 us, the walk 20 us.  A step makes two, one in front of the forward pass, which may change the model."""

from operator import attrgetter

from torch import nn

# what ``train()`` and ``parameters()`` go through, of every module on the way
_WALKED = ("train", "parameters", "named_parameters", "_named_members", "named_modules", "children", "named_children", "__setattr__")
_walked = attrgetter(*_WALKED)


def plain_modules(model: nn.Module) -> list[nn.Module] | None:
    """``list(model.modules())``, or None where the model or a module in it answers one of the calls that the walk stands for in a way of its own."""
    if not isinstance(model, nn.Module):   # anything with ``train()`` and ``parameters()``
        return None
    modules, seen = [model], {model}
    for module in modules:   # grows on the way
        for child in module._modules.values():
            if child is not None and child not in seen:
                seen.add(child)
                modules.append(child)
    stock = _walked(nn.Module)
    if any(getattr(call, "__globals__", {}).get("__name__") != nn.Module.__module__ for call in stock):   # replaced for all modules
        return None
    for cls in {type(m) for m in modules}:
        if _walked(cls) != stock or hasattr(cls, "training"):
            return None
    for module in modules:
        own = module.__dict__
        if ("train" in own or "parameters" in own or "named_parameters" in own or "_named_members" in own or "named_modules" in own or "children" in own
                or "named_children" in own):
            return None
    return modules


def set_training(model: nn.Module, modules: list[nn.Module] | None) -> None:
    """``model.train()``, which is nothing where every module is in training already."""
    if modules is None or not all(m.training for m in modules):
        model.train()


def parameters_of(model: nn.Module, modules: list[nn.Module] | None) -> list[nn.Parameter]:
    """``model.parameters()``, one that several modules share as often as they do."""
    if modules is None:
        return list(model.parameters())
    return [p for m in modules for p in m._parameters.values() if p is not None]
