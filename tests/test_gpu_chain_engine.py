"""Decode steps of small layers that run as one launch (``DecoderModel._chains``), through the engine and the generation loop."""
import dataclasses
import functools

import pytest
import torch

pytestmark = pytest.mark.gpu

from rocml_amd import ops  # noqa: E402
from rocml_amd.config import architecture_of  # noqa: E402
from rocml_amd.config.catalog import resolve  # noqa: E402
from rocml_amd.engine import DecoderModel, Engine, EngineBackend, Generator, Request, StepEntry  # noqa: E402
from rocml_amd.errors import StepFailedError  # noqa: E402
from rocml_amd.weights import random_model  # noqa: E402

DEV = "cuda:0"


def _model(n_layers, dtype="bfloat16", **sizes):
    """The smallest layers that the chain takes, unless told otherwise."""
    cfg = dict(resolve("qwen3-0.6b").entry.config, num_hidden_layers=n_layers, vocab_size=512, hidden_size=512, intermediate_size=512,
               num_attention_heads=4, num_key_value_heads=2, **sizes)
    return random_model(cfg, seed=n_layers, dtype=dtype, device=DEV, norm_jitter=True)


def _pair(dtype, n_layers, change=None):
    """The same model twice: one that may run layers in one launch and one that must not.  Matrices of variance 1 / columns, so that
    every layer adds about as much as the stream holds.  ``change(i, layer spec)``: another layer in the place of layer ``i``."""
    cfg = dict(resolve("qwen3-0.6b").entry.config, num_hidden_layers=n_layers, vocab_size=512, hidden_size=512, intermediate_size=512,
               num_attention_heads=4, num_key_value_heads=2)
    arch = architecture_of(cfg)
    spec = arch.to_spec(arch.read_config(cfg))
    if change is not None:
        spec = dataclasses.replace(spec, layers=tuple(change(i, layer) for i, layer in enumerate(spec.layers)))
    models = []
    for _ in range(2):
        model, g = DecoderModel(spec, dtype, device=DEV), torch.Generator(device=DEV).manual_seed(n_layers)
        tensors = {}
        for name, p in model.param_specs().items():
            t = torch.randn(*p.shape, generator=g, device=DEV)
            t = 1.0 + 0.1 * t if p.role == "gain" else t * (1.0 if name.startswith("embed.") else p.shape[-1] ** -0.5)
            tensors[name] = t.to(model.storage_dtype(p))
        model.bind(tensors)
        models.append(model)
    models[1].chain_sizes = [None] * len(models[1].blocks)
    return models


def _compare(engines, prompts, steps, dtype, seed=0):
    """Prompts and ``steps`` decode steps in both engines, the same tokens; the logits of every step.  32-bit: sums in another order,
    some 1e-6 a layer; 2e-5.  bfloat16: either way of 28 such layers ends some 0.006 away from the sums in 64 bits; 0.03 covers two
    of them three times, and a layer that is lost or run twice is off by more than 0.1."""
    slots = [[e.new_sequence() for _ in prompts] for e in engines]
    g = torch.Generator().manual_seed(seed)
    logits = [[e.step([StepEntry(s, p, [len(p) - 1]) for s, p in zip(sl, prompts)]).double().clone()] for e, sl in zip(engines, slots)]
    for _ in range(steps):
        ids = torch.randint(512, (len(prompts),), generator=g).tolist()
        for e, sl, out in zip(engines, slots, logits):
            out.append(e.step([StepEntry(s, [t], [0]) for s, t in zip(sl, ids)]).double().clone())
    for step, (a, b) in enumerate(zip(*logits)):
        assert torch.isfinite(a).all()
        assert float(((a - b).norm(dim=-1) / b.norm(dim=-1)).max()) < (2e-5 if dtype == "float32" else 0.03), step
    for e, sl in zip(engines, slots):
        for s in sl:
            e.release(s)


def _count_launches(monkeypatch):
    launches, whole = [], ops.decode_chain

    def counted(x, xn, layers, *a, **kw):
        launches.append(len(layers))
        whole(x, xn, layers, *a, **kw)
    monkeypatch.setattr(ops, "decode_chain", counted)
    return launches


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("prompts", [[[7]], [[1] * 130], [[3] * 65, [9], [4, 2], [8] * 64]], ids=["1 of 1", "1 of 130", "4"])
def test_more_layers_than_one_launch_takes(monkeypatch, prompts, dtype):
    """34 layers: two launches in a step that share their state, run, recorded and replayed."""
    launches = _count_launches(monkeypatch)
    engines = [Engine(m, max_tokens=2048, max_seqs=4) for m in _pair(dtype, 34)]
    _compare(engines, prompts, 5, dtype)
    assert launches[:2] == [32, 2] and len(launches) % 2 == 0


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("odd", [(0,), (2,), (5,), (0, 2, 4), (1, 2)])
def test_layers_of_another_kind_between(monkeypatch, odd, dtype):
    """Six layers of which some have another activation and run their own kernels before, between and behind the launches: sums
    that are left to the next norm, norms that a product prepares, and a launch of one layer."""
    def change(i, layer):
        return dataclasses.replace(layer, ffn=dataclasses.replace(layer.ffn, activation="relu")) if i in odd else layer
    launches = _count_launches(monkeypatch)
    engines = [Engine(m, max_tokens=2048, max_seqs=4) for m in _pair(dtype, 6, change)]
    _compare(engines, [[3] * 65, [9, 1]], 4, dtype)
    runs = "".join("." if i in odd else "x" for i in range(6)).split(".")
    assert launches[:sum(1 for r in runs if r)] == [len(r) for r in runs if r]


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_layers_of_two_sizes(monkeypatch, dtype):
    """A second launch in a step that needs more state than the first: the state grows in the middle of the step."""
    def change(i, layer):
        return dataclasses.replace(layer, ffn=dataclasses.replace(layer.ffn, intermediate=2048)) if i >= 2 else layer
    launches = _count_launches(monkeypatch)
    engines = [Engine(m, max_tokens=2048, max_seqs=4) for m in _pair(dtype, 5, change)]
    _compare(engines, [[3] * 65, [9, 1]], 4, dtype)
    assert launches[:2] == [2, 3]


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_state_that_grows_while_recorded_steps_exist(dtype):
    """Steps of one sequence are recorded with the state as it is, steps of four long ones then need a larger one: what was recorded is
    recorded again, for the first shape too."""
    engines = [Engine(m, max_tokens=16384, max_seqs=4) for m in _pair(dtype, 3)]
    _compare(engines, [[5] * 10], 4, dtype, seed=1)
    _compare(engines, [[5] * 1500, [6] * 900, [7], [8] * 3], 4, dtype, seed=2)
    _compare(engines, [[9] * 12], 4, dtype, seed=3)
    _compare(engines, [[4] * 30, [2] * 3], 4, dtype, seed=4)


def _generate(engine, prompts, new):
    return [r.tokens for r in Generator(EngineBackend(engine), max_batch=len(prompts)).run([Request(p, new) for p in prompts])]


def test_a_step_whose_wait_ended_is_told(monkeypatch):
    """A launch whose waits are told to end at once: the loop raises where it fetches the tokens, the next step of whoever steps
    the engine itself raises too, both once; slots and pages come back, and the engine then gives what it gave before."""
    model, prompts = _model(2), [[3, 5, 8], [2] * 70]
    engine = Engine(model, max_tokens=2048, max_seqs=4, use_graphs=False)
    want = _generate(engine, prompts, 6)
    whole = ops.decode_chain
    monkeypatch.setattr(ops, "decode_chain", functools.partial(whole, polls=1, patience=0.0))
    with pytest.raises(StepFailedError):
        _generate(engine, prompts, 6)
    slot = engine.new_sequence()
    engine.step([StepEntry(slot, [3, 5, 8], [2])])
    assert torch.isnan(engine.step([StepEntry(slot, [1], [0])])).any()
    torch.cuda.synchronize()
    monkeypatch.setattr(ops, "decode_chain", whole)
    with pytest.raises(StepFailedError):
        engine.step([StepEntry(slot, [1], [0])])
    engine.release(slot)
    engine.check_steps()
    assert _generate(engine, prompts, 6) == want
    engine.cache.check()
    assert not engine.cache.lengths


@pytest.mark.parametrize("lengths,chained", [([4031, 3], True), ([4100, 3], False), ([4100], True)])
def test_long_sequences_run_the_layers_kernels(monkeypatch, lengths, chained):
    """Two sequences share one launch up to 64 pages of keys (a table of 128 is refused), one sequence far beyond that; a sequence that
    grows over the line in the middle goes on."""
    engine = Engine(_model(2), max_tokens=16384, max_seqs=2)
    calls = []
    whole = ops.decode_chain
    monkeypatch.setattr(ops, "decode_chain", lambda *a, **kw: (calls.append(1), whole(*a, **kw)))
    prompts = [[i % 500 for i in range(n)] for n in lengths]
    got = _generate(engine, prompts, 3)
    assert bool(calls) == chained
    again = _generate(engine, [p + g[:2] for p, g in zip(prompts, got)], 1)
    assert [a[0] for a in again] == [g[2] for g in got]
