"""Steps launched one behind the other without waiting: the tables of a step stay what they were when it was launched."""
import pytest
import torch

from tests import helpers

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("use_graphs", [True, False])
@pytest.mark.parametrize("batch,steps", [(1, 13), (3, 9)])
def test_many_steps_in_flight(tmp_path, batch, steps, use_graphs):
    """Steps launched while the GPU is busy with something else, so that the copy of every step's tables still waits when the next step
    is prepared: bit for bit the logits of the same steps waited for one by one (no product of this model depends on the batch's history).
    The first two are of the shape but not counted: a shape runs plainly, is recorded and only then replayed."""
    from rocml_amd.engine import Engine, StepEntry
    from rocml_amd.weights import load_model
    cfg, seed = helpers.TINY["B"]
    path = helpers.make_model_dir(tmp_path, cfg, seed, torch.float32)
    said = [helpers.random_tokens(70 + 3 * b + steps, cfg["vocab_size"], b) for b in range(batch)]

    def run(waits):
        engine = Engine(load_model(path, dtype="float32", device="cuda:0"), max_tokens=4096, use_graphs=use_graphs)
        slots = [engine.new_sequence() for _ in said]
        engine.step([StepEntry(s, t[:-steps], []) for s, t in zip(slots, said)])
        out = []
        for k in range(steps):
            if k >= 2 and not waits:
                if k == 2:
                    replayed = [key for key, entry in engine._graphs.items() if key[0] != "prompt" and entry[1] is not None]
                    assert bool(replayed) == use_graphs
                torch.cuda._sleep(3_000_000)
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
        for k in range(11):
            if not waits:
                torch.cuda._sleep(3_000_000)
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


def test_draws_recorded_from_outside():
    """A draw whose buffers are there is recorded as any launch; a replay brings the parameters that lie in the sampler's buffer, those of
    the last draw, and draws between the replays are as they would be without them."""
    from rocml_amd.sampling import SamplingParams
    from rocml_amd.sampling.sampler import DeviceSampler, SequenceSampling
    logits = torch.randn(3, 700, generator=torch.Generator().manual_seed(4)).cuda()

    def seqs(seed):
        return [SequenceSampling.start(SamplingParams(temperature=0.9, top_p=0.95, seed=seed), i, [1]) for i in range(3)]

    sampler, other = DeviceSampler("cuda:0"), DeviceSampler("cuda:0")
    for k in range(5):
        assert sampler.sample(logits, seqs(k)) == other.sample(logits, seqs(k))
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        ids = sampler.sample_start(logits, seqs(17))[0]
    for seed in (17, 18, 19, 20):
        want = other.sample(logits, seqs(seed))
        if seed > 17:
            assert sampler.sample(logits, seqs(seed)) == want
        graph.replay()
        torch.cuda.synchronize()
        assert ids.tolist() == want
