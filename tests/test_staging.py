"""The buffer that a step's tables pass through: it is not filled while its copy may still run, a step hears what the steps before the last
one have to tell, and a graph that may be running is not dropped."""
from types import SimpleNamespace

import pytest
import torch

from rocml_amd.engine import Engine, StepEntry
from rocml_amd.errors import RocmlError, StepFailedError
from rocml_amd.staging import Staging


@pytest.fixture
def device(monkeypatch):
    """A device that only takes down what it is asked for."""
    said = []

    class Event:
        def record(self, stream):
            said.append("record")

        def synchronize(self):
            said.append("wait")

    empty = torch.empty
    monkeypatch.setattr(torch.cuda, "Event", Event)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: None)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: device.capturing)
    monkeypatch.setattr(torch.cuda, "synchronize", lambda device=None: said.append("all"))
    monkeypatch.setattr(torch, "empty", lambda *a, pin_memory=False, **kw: empty(*a, **kw))
    device = SimpleNamespace(said=said, capturing=False)
    return device


def test_a_buffer_is_filled_when_its_copy_has_ended(device):
    staging, dest = Staging(), torch.zeros(300, dtype=torch.int32)
    for words in (5, 5, 300, 40):
        staged = staging.take(words)
        assert staged.numel() == words and device.said.count("wait") == device.said.count("record")
        staged.fill_(words)
        staging.send(staged, dest[:words])
        assert device.said[-1] == "record" and bool((dest[:words] == words).all())


def test_a_capture_waits_for_nothing(device):
    staging, dest = Staging(), torch.zeros(8, dtype=torch.int32)
    staging.send(staging.take(8), dest)
    before = list(device.said)
    staged = staging.take(8, recorded=True)
    assert staged.data_ptr() == staging.take(8, recorded=True).data_ptr()          # the buffer that a replay will read
    staging.send(staged, dest, recorded=True)
    assert device.said == before


def _engine(device, late):
    engine = Engine.__new__(Engine)
    engine.model = SimpleNamespace(spec=None, device="cuda:0")
    engine.workspace = SimpleNamespace(was_late=lambda: late and "wait" in device.said)
    engine._staging = Staging()
    engine._staging.send(engine._staging.take(4), torch.zeros(4, dtype=torch.int32))
    return engine


def test_a_step_hears_of_all_before_the_last(device):
    """The last step's tables were copied behind the step before it, so when that copy has ended that step's failure is known."""
    with pytest.raises(StepFailedError):
        _engine(device, True).step([StepEntry(0, [1], [])])


def test_a_step_is_refused_under_a_capture_before_anything_is_waited_for(device):
    engine = _engine(device, True)
    device.capturing = True
    with pytest.raises(RocmlError, match="recorded from outside"):
        engine.step([StepEntry(0, [1], [])])
    assert "wait" not in device.said


def test_graphs_are_dropped_when_nothing_runs(device):
    engine = _engine(device, False)
    engine._graphs, engine.max_prompt_graphs = {}, 2
    waits = lambda: device.said.count("all")          # noqa: E731
    engine._remember((3, 3, 1, False), (1, None, None))
    engine._remember((3, 3, 1, False), (1, "graph", "logits"))
    assert waits() == 0                                # nothing that could run was dropped
    engine._remember((3, 3, 1, False), (2, None, None))
    assert waits() == 1                                # a graph of buffers that have moved
    prompts = [(2, "graph of one", "logits"), (2, "graph of another", "logits")]
    for n in range(2):
        engine._remember(("prompt", n), prompts[n])
    assert waits() == 1
    engine._remember(("prompt", 0), prompts[0])
    assert waits() == 1 and list(engine._graphs)[-1] == ("prompt", 0)
    engine._remember(("prompt", 2), (2, None, None))
    assert waits() == 2 and ("prompt", 1) not in engine._graphs
