"""The served benchmark's operation times: another form of an operation counts as that operation, so that no rate divides by nothing."""
import torch

from qserve_amd.serving import bench


class Event:
    def __init__(self, **_):
        pass

    def record(self):
        pass

    def elapsed_time(self, other):
        return 1.0


class Ops:
    def __getattr__(self, name):
        return lambda *a, **k: name


def test_other_forms_are_timed_as_their_operation(monkeypatch):
    monkeypatch.setattr(torch.cuda, "Event", Event)
    monkeypatch.setattr(torch.cuda, "synchronize", lambda: None)
    for m in bench.OpTimer._linear_users():                  # (the timer wraps these modules' products: put back afterwards)
        for name in ("linear", "float_linear"):
            if hasattr(m, name):
                monkeypatch.setattr(m, name, getattr(m, name))
    ops = Ops()
    timer = bench.OpTimer(ops)
    times, _ = timer.step(lambda: [ops.latent_prompt(), ops.moe_experts_shared(), ops.moe_experts(), ops.hc_read()])
    assert times == {"latent_attention": 1.0, "moe_experts": 2.0, "hc_read": 1.0}
    assert timer.replay("latent_attention", 1) == 1.0 and timer.replay("moe_experts", 1) == 2.0
