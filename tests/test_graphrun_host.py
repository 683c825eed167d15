"""The commit of a replayed step on CPU tensors, where every copy is made by
torch, one after the other, and the library call is a stub."""
import pytest
import torch

from jaxabm_amd import graphrun


@pytest.fixture
def runner(monkeypatch):
    class Lib:
        def abm_commit_step(self, *args):
            return 0

    monkeypatch.setattr(graphrun, "lib", lambda: Lib())
    monkeypatch.setattr(graphrun, "stream_handle", lambda stream=None: None)
    r = graphrun._Runner.__new__(graphrun._Runner)
    r.n, r.width, r.waiting, r.colls = 4, 1, [], []
    r.row = torch.zeros(1, dtype=torch.int64)
    r.ts = r.done = r.keys = r.table = torch.zeros(1, dtype=torch.int32)
    return r


def test_a_metric_that_is_an_env_slot_is_read_before_the_slot_is_written(runner):
    """env["prev"] = env["cur"], env["cur"] = new and a metric of env["prev"],
    its first element and a Python value that a slot takes."""
    old, new = torch.arange(3.0), torch.arange(3.0) + 10
    r = runner
    r.env = {"prev": torch.zeros(3), "cur": old.clone(), "scale": torch.tensor(2.0)}
    r.hist = {"was": torch.zeros(4, 3), "first": torch.zeros(4), "scale": torch.zeros(4),
              "new": torch.zeros(4, 3)}
    prev, scale = r.env["cur"], r.env["scale"]
    r.commit({}, {"prev": prev, "cur": new, "scale": 5.0},
             {"was": prev, "first": prev[1], "scale": scale, "new": new})
    assert torch.equal(r.env["prev"], old) and torch.equal(r.env["cur"], new)
    assert torch.equal(r.hist["was"][0], old) and torch.equal(r.hist["new"][0], new)
    assert r.hist["first"][0] == 1.0
    assert r.hist["scale"][0] == 2.0 and r.env["scale"] == 5.0
