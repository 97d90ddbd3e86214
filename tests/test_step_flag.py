"""The flag of a training step is waited for on the stream that copies it (CPU: a device that is not the current one is played)."""

import pytest
import torch

from minitrain_amd.train import step


class _Flag:
    device = torch.device("cuda", 1)

    def __init__(self, value):
        self.value = value

    def __getitem__(self, index):
        return self

    def copy_(self, source, non_blocking):
        return self

    def __float__(self):
        return self.value


class _Model(torch.nn.Linear):
    def forward(self, ids, *, targets, use_fused_loss):
        return super().forward(ids).sum(), None


@pytest.mark.parametrize("value", [0.0, 1.0])
def test_event_is_recorded_where_the_flag_is_copied(monkeypatch, value):
    calls = []

    class Event:
        def record(self, stream=None):
            calls.append(("record", stream))

        def synchronize(self):
            calls.append("synchronize")

    class Update:
        def norm(self, limit, loss):
            return _Flag(value)

        def apply(self, norm, skip_if_not_finite):
            calls.append("apply")

        def drop_gradients(self):
            calls.append("drop")

    model = _Model(2, 1)
    optimizer = torch.optim.SGD(model.parameters(), lr=0.0)
    batch = {"input_ids": torch.ones(1, 2), "targets": torch.ones(1)}
    monkeypatch.setattr(step, "plan", lambda *a: Update())
    monkeypatch.setattr(torch.cuda, "Event", Event)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: ("stream of", device))
    monkeypatch.setattr(torch, "empty", lambda *a, **k: _Flag(value))
    if value:
        with pytest.raises(FloatingPointError):
            step.train_step(model, optimizer, batch)
    else:
        step.train_step(model, optimizer, batch)
    assert calls == [("record", ("stream of", _Flag.device)), "apply", "synchronize", "drop"]
