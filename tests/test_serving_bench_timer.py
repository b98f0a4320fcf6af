"""The served benchmark's operation times: another form of an operation counts as that operation, so that no rate divides by nothing."""
import pathlib
import re

import pytest
import torch

import qserve_amd.layers
import qserve_amd.models
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


def test_every_operation_of_a_model_is_timed():
    files = [f for pkg in (qserve_amd.layers, qserve_amd.models) for f in pathlib.Path(pkg.__path__[0]).glob("*.py") if f.name != "ops.py"]
    called = {n for f in files for n in re.findall(r"\bops\.([a-z_]+)\(", f.read_text())}
    assert len(files) > 8 and "recurrent_gated" in called
    assert called <= set(bench.OpTimer.NAMES) | set(bench.OpTimer.HOST)
    assert set(bench.OpTimer.FORMS) | set(bench.OpTimer.HAND_OVER) <= set(bench.OpTimer.NAMES)


class Step(Ops):
    """Operations that take their calls in a launch of their own, or hand them over to others."""
    own = True

    def recurrent_gated(self):
        return None if self.own else (self.recurrent_scan(), self.head_rms_gate())

    def hc_write_read(self):
        return None if self.own else (self.hc_write(), self.hc_read())

    def hc_write(self, again=False):
        return None if self.own or again else self.hc_write(True)

    def moe_experts_pending(self):
        return "riding"


@pytest.fixture
def events(monkeypatch):
    monkeypatch.setattr(torch.cuda, "Event", Event)
    monkeypatch.setattr(torch.cuda, "synchronize", lambda: None)


def test_steps_in_launches_of_their_own(events):
    ops = Step()
    timer = bench.OpTimer(ops)
    times, _ = timer.step(lambda: [ops.recurrent_gated(), ops.hc_write_read(), ops.hc_write()])
    assert times == {"recurrent_scan": 1.0, "hc_write_read": 1.0, "hc_write": 1.0}
    assert timer.replays(("recurrent_scan", "head_rms_gate", "hc_write_read"), 2) == {"recurrent_scan": 0.5, "hc_write_read": 0.5}


def test_calls_handed_over_count_once(events):
    ops = Step()
    ops.own = False
    timer = bench.OpTimer(ops)
    times, _ = timer.step(lambda: [ops.recurrent_gated(), ops.hc_write_read(), ops.hc_write()])
    assert times == {"recurrent_scan": 1.0, "head_rms_gate": 1.0, "hc_write": 2.0, "hc_read": 1.0}


def test_experts_do_not_ride_in_a_timed_step(events):
    ops = Step()
    timer = bench.OpTimer(ops)
    seen = []
    timer.step(lambda: seen.append(ops.moe_experts_pending()))
    assert seen == [None] and ops.moe_experts_pending() == "riding"


def test_a_rate_of_nothing_is_none():
    assert bench._rate(4e9, 1e9, {"a": 2.0}, "a", "b") == 2000.0 and bench._rate(1.0, 1.0, {}, "a") is None
    assert bench._of(None, 8.0) is None and bench._of(2.0, 8.0) == 0.25
