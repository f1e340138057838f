"""Steps launched one behind the other without waiting: the tables of a step stay what they were when it was launched."""
import pytest
import torch

from tests import helpers

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("use_graphs", [True, False])
@pytest.mark.parametrize("batch,steps", [(1, 13), (3, 9)])
def test_many_steps_in_flight(tmp_path, batch, steps, use_graphs):
    """More steps than the ring of staging buffers holds, behind a kernel that keeps the GPU busy: bit for bit the logits of the
    same steps waited for one by one (no product of this model depends on the batch's history)."""
    from rocml_amd.engine import Engine, StepEntry
    from rocml_amd.weights import load_model
    cfg, seed = helpers.TINY["B"]
    path = helpers.make_model_dir(tmp_path, cfg, seed, torch.float32)
    said = [helpers.random_tokens(70 + 3 * b + steps, cfg["vocab_size"], b) for b in range(batch)]

    def run(waits):
        engine = Engine(load_model(path, dtype="float32", device="cuda:0"), max_tokens=4096, use_graphs=use_graphs)
        slots = [engine.new_sequence() for _ in said]
        engine.step([StepEntry(s, t[:-steps], []) for s, t in zip(slots, said)])
        if not waits:
            torch.cuda._sleep(50_000_000)
        out = []
        for k in range(steps):
            out.append(engine.step([StepEntry(s, [t[len(t) - steps + k]], [0]) for s, t in zip(slots, said)]).clone())
            if waits:
                torch.cuda.synchronize()
        return torch.stack(out).cpu()

    assert torch.equal(run(False), run(True))


def test_parameters_of_draws_in_flight():
    """Draws launched before the ones before them have run: each with its own parameters."""
    from rocml_amd.sampling import SamplingParams
    from rocml_amd.sampling.sampler import DeviceSampler, SequenceSampling
    logits = torch.randn(2, 1000, generator=torch.Generator().manual_seed(3)).cuda()

    def run(waits):
        sampler = DeviceSampler("cuda:0")
        out = []
        if not waits:
            torch.cuda._sleep(50_000_000)
        for k in range(11):
            seqs = [SequenceSampling.start(SamplingParams(temperature=0.5 + 0.1 * k, top_p=0.9, seed=7 + k), i, [k]) for i in range(2)]
            out.append(sampler.sample_start(logits, seqs)[0])
            if waits:
                torch.cuda.synchronize()
        return torch.stack(out).cpu()

    assert torch.equal(run(False), run(True))


def test_a_step_is_not_recorded_from_outside(tmp_path):
    from rocml_amd.engine import Engine, StepEntry
    from rocml_amd.errors import RocmlError
    from rocml_amd.weights import load_model
    cfg, seed = helpers.TINY["A"]
    engine = Engine(load_model(helpers.make_model_dir(tmp_path, cfg, seed, torch.float32), dtype="float32", device="cuda:0"), max_tokens=256)
    slot = engine.new_sequence()
    want = engine.step([StepEntry(slot, [1, 2, 3], [2])]).cpu()
    graph = torch.cuda.CUDAGraph()
    with pytest.raises(RocmlError, match="recorded from outside"):
        with torch.cuda.graph(graph):
            torch.zeros(1, device="cuda:0")
            engine.step([StepEntry(slot, [4], [0])])
    engine.release(slot)
    slot = engine.new_sequence()
    assert torch.equal(engine.step([StepEntry(slot, [1, 2, 3], [2])]).cpu(), want)
