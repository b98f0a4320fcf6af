"""A mixture's launches that are left to be made beside others: which of them are made, in which order, and on which stream."""
import pytest

from qserve_amd.layers.ops import PendingExperts


class Ops:
    def __init__(self):
        self.stream, self.launched = 7, []

    def _s(self):
        return self.stream

    def expert_launch(self, job):
        self.launched.append((job, self.stream))


def _pending():
    ops = Ops()
    return ops, PendingExperts(ops, ("up", "down"), [], ["rows"])


@pytest.mark.parametrize("taken, launched", [((), ["up", "down"]), ((0,), ["down"]), ((0, 1), []), ((1,), ["up"]), ((1, 0), ["up"]), ((0, 0), ["down"])])
def test_what_nobody_took_is_made_once(taken, launched):
    ops, p = _pending()
    made = [p.take(i) for i in taken]
    assert p.results() == ["rows"] == p.results()
    assert [j for j, _ in ops.launched] == launched
    assert sorted([j for j in made if j] + launched) == ["down", "up"]


@pytest.mark.parametrize("taken", [(), (0,), (0, 1)])
def test_another_stream(taken):
    ops, p = _pending()
    for i in taken:
        p.take(i)
    ops.stream = 8
    assert p.take(0) is None and p.take(1) is None
    with pytest.raises(RuntimeError, match="another stream"):
        p.results()
    assert not ops.launched
    ops.stream = 7
    assert p.results() == ["rows"] and all(s == 7 for _, s in ops.launched)
