"""The optimizer update in the kernels against stock clipping and fused AdamW, and against fp64."""

import copy

import pytest
import torch

from tests.helpers import hip_backend

pytestmark = pytest.mark.gpu

# a chunk of the update is 4096 elements, one of the norm 16 384, a launch of the update holds 56 tensors and one of the norm 128
SIZES = {
    "edges": [1, 3, 4, 4095, 4096, 4097, 16383, 16384, 16385, 70001],
    "many": [5 + 37 * i for i in range(130)],
    "large": [3_000_003, 1 << 20],
}


class Bag(torch.nn.Module):
    def __init__(self, sizes, offset=0):
        super().__init__()
        g = torch.Generator().manual_seed(len(sizes))
        make = lambda n: torch.randn(n + offset, generator=g).cuda()[offset:]   # offset: off the 16-byte boundaries
        self.p = torch.nn.ParameterList(torch.nn.Parameter(make(n)) for n in sizes)
        self.grads = [torch.randn(n + offset, generator=g).cuda()[offset:] * 3 for n in sizes]


def _optimizer(bag):
    groups = [{"params": list(bag.p)[0::2], "weight_decay": 0.1}, {"params": list(bag.p)[1::2], "weight_decay": 0.0, "lr": 2e-3}]
    return torch.optim.AdamW(groups, lr=1e-3, betas=(0.9, 0.95), eps=1e-8, fused=True)


def _fp64_step(p, g, state, group, coefficient):
    t = state["t"] = state.get("t", 0) + 1
    b1, b2 = group["betas"]
    g = g.double() * coefficient
    state["m"] = b1 * state.get("m", 0) + (1 - b1) * g
    state["v"] = b2 * state.get("v", 0) + (1 - b2) * g * g
    p = p * (1 - group["lr"] * group["weight_decay"])
    return p - group["lr"] / (1 - b1**t) * state["m"] / ((state["v"] / (1 - b2**t)).sqrt() + group["eps"])


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("sizes", list(SIZES))
def test_update_equals_stock_and_fp64(sizes, offset):
    from minitrain_amd.train.update import plan

    ours, stock = Bag(SIZES[sizes], offset), Bag(SIZES[sizes], offset)
    opt_a, opt_b = _optimizer(ours), _optimizer(stock)
    exact, states = [p.detach().double() for p in ours.p], [{} for _ in ours.p]
    loss = torch.ones((), device="cuda")
    for step in range(3):
        for bag in (ours, stock):
            for p, g in zip(bag.p, bag.grads):
                p.grad = (g * (step + 1)).contiguous()
        norm64 = torch.sqrt(sum(p.grad.double().square().sum() for p in ours.p))
        # the third step's gradients are so small that nothing is clipped
        limit = 1.0 if step < 2 else float(norm64) * 2
        coefficient = min(1.0, limit / (float(norm64) + 1e-6))
        index = {id(p): i for i, p in enumerate(ours.p)}
        for group in opt_a.param_groups:
            for p in group["params"]:
                i = index[id(p)]
                exact[i] = _fp64_step(exact[i], p.grad, states[i], group, coefficient)
        held = ours.p[0].grad
        update = plan(ours, opt_a, loss, limit)
        if step == 0:
            assert update is None   # the first step makes the state
            torch.nn.utils.clip_grad_norm_(ours.parameters(), limit)
            opt_a.step()
        else:
            norm = update.norm(limit, loss)
            update.apply(norm, True)
            torch.testing.assert_close(norm[0].double(), norm64, rtol=1e-6, atol=0)
            assert float(norm[2]) == 0
        torch.nn.utils.clip_grad_norm_(stock.parameters(), limit)
        opt_b.step()
        # a gradient that is held outside is left clipped (one rounding of the coefficient, one of the product)
        torch.testing.assert_close(held, stock.p[0].grad, rtol=1e-6, atol=0)
    for i, (a, b) in enumerate(zip(ours.p, stock.p)):
        sa, sb = opt_a.state[a], opt_b.state[b]
        assert float(sa["step"]) == float(sb["step"]) == 3
        # against fp64: no further off than the stock operator (plus one rounding of the result)
        err = lambda x, want: float((x.double() - want).abs().max())
        one = float(exact[i].abs().max()) * 2**-24
        assert err(a.detach(), exact[i]) <= err(b.detach(), exact[i]) + one
        torch.testing.assert_close(sa["exp_avg"], sb["exp_avg"], rtol=1e-6, atol=1e-12)
        torch.testing.assert_close(sa["exp_avg_sq"], sb["exp_avg_sq"], rtol=1e-6, atol=1e-16)


def _model(vocab=61):
    from minitrain_amd.model.config import ModelConfig
    from minitrain_amd.model.decoder import MiniTransformer

    torch.manual_seed(3)
    cfg = ModelConfig(vocab_size=vocab, seq_len=32, n_layers=2, n_heads=2, hidden_size=128, intermediate_size=128, num_experts=4, experts_per_token=2)
    model = MiniTransformer(cfg, hip_backend(), activation_dtype=torch.bfloat16).cuda()
    ids = torch.randint(0, vocab, (4, 33))
    return model, {"input_ids": ids[:, :-1].contiguous(), "targets": ids[:, 1:].contiguous()}


def test_not_finite_leaves_everything_as_it_was():
    from minitrain_amd.train.step import build_optimizer, train_step

    model, batch = _model()
    opt = build_optimizer(model)
    for _ in range(2):
        train_step(model, opt, batch)
    params, state = [p.detach().clone() for p in model.parameters()], copy.deepcopy(opt.state_dict())
    hook = model.norm.weight.register_hook(lambda g: g * float("nan"))
    with pytest.raises(FloatingPointError):
        train_step(model, opt, batch)
    hook.remove()
    assert all(torch.equal(a, b) for a, b in zip(params, model.parameters()))
    for key, want in state["state"].items():
        for name, value in want.items():
            assert torch.equal(opt.state_dict()["state"][key][name], value), name
    assert all(p.grad is None for p in model.parameters())
    train_step(model, opt, batch)


def test_who_looks_on_gets_the_stock_calls(monkeypatch):
    """Hooks, options of another kind and parameters outside the optimizer keep the stock path; a scheduler goes with either."""
    from minitrain_amd.train import update
    from minitrain_amd.train.step import build_optimizer, train_step

    taken = []
    apply = update.Update.apply
    monkeypatch.setattr(update.Update, "apply", lambda self, *a, **k: (taken.append(1), apply(self, *a, **k))[1])

    def steps(prepare):
        model, batch = _model()
        opt = build_optimizer(model)
        train_step(model, opt, batch)
        keep = prepare(model, opt)
        taken.clear()
        train_step(model, opt, batch)
        del keep
        return len(taken)

    assert steps(lambda m, o: None) == 1
    assert steps(lambda m, o: torch.optim.lr_scheduler.LambdaLR(o, lambda _: 0.5)) == 1
    assert steps(lambda m, o: o.register_step_pre_hook(lambda *a: None)) == 0
    assert steps(lambda m, o: o.param_groups[0].update(amsgrad=True) or [s.update(max_exp_avg_sq=torch.zeros_like(s["exp_avg"])) for s in o.state.values()]) == 0
    assert steps(lambda m, o: o.param_groups[0].update(lr=torch.tensor(1e-3, device="cuda"))) == 0
    assert steps(lambda m, o: o.param_groups[1]["params"].pop()) == 0


class _Linear(Bag):
    """A model whose gradients are given numbers, whatever the parameters are."""

    def forward(self, input_ids, *, targets, use_fused_loss):
        return sum((p * g).sum() for p, g in zip(self.p, self.grads)) * input_ids.float().mean(), None


@pytest.mark.parametrize("clip,check,poison", [(None, True, None), (None, True, "inf"), (None, True, "nan"), (1.0, True, None), (1.0, False, None), (1.0, False, "inf"),
                                               (1.0, False, "nan"), (None, False, "nan")])
def test_steps_without_clipping_and_without_the_check(monkeypatch, clip, check, poison):
    """Against the stock calls. Without clipping nobody looks at the norm, so that a gradient that is not finite passes with a finite loss; without
    the check everything passes."""
    from minitrain_amd.train import step, update

    print(f"clip={clip} check={check} poison={poison}", flush=True)
    taken = []
    apply = update.Update.apply
    monkeypatch.setattr(update.Update, "apply", lambda self, *a, **k: (taken.append(1), apply(self, *a, **k))[1])
    batch = {"input_ids": torch.ones(2, 3, dtype=torch.long), "targets": torch.ones(2, 3, dtype=torch.long)}
    sides = []
    for own in (True, False):
        if not own:
            monkeypatch.setattr(step, "plan", lambda *a: None)
        model = _Linear([5, 4097, 20000])
        opt = _optimizer(model)
        for i in range(3):
            hook = model.p[1].register_hook(lambda g: g * float(poison)) if poison and i == 2 else None
            loss = step.train_step(model, opt, batch, autocast_dtype=None, grad_clip_norm=clip, check_finite=check)
            if hook:
                hook.remove()
            assert loss.isfinite()
        sides.append([t for p in model.p for t in (p.detach(), *opt.state[p].values())])
        assert len(taken) == 2   # the first step makes the state
    assert not poison or sides[0][4].isnan().any()
    for a, b in zip(*sides):   # three updates, a few roundings each
        torch.testing.assert_close(a, b, rtol=2e-6, atol=1e-9, equal_nan=True)
