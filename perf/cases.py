"""The work that the library's speed is measured on: whole requests through the generation loop.

A case is a batch of requests to a model with random weights: ``batch`` prompts of ``shortest`` to ``longest`` random
tokens run in one step, then ``new`` tokens are drawn for each, one decode step after the other, as
``rocml_amd.api.Model.generate`` and ``bench.py`` do it (``Generator`` over ``EngineBackend``); with ``places`` "all" the
texts are scored instead: one step whose logits are wanted at every place.  A pass returns the logits of every step.

Two correct implementations in bfloat16 do not draw the same tokens for long (the best two of 151,936 random logits are
often closer than the rounding), so every sequence goes on with tokens that were laid down beforehand: the sampler runs
as it always does, its draws come back beside the logits in 32-bit models, and the next step takes the scripted tokens.

The models are the catalog's.  The larger ones are cut to their first layers (as ``bench.py --layers`` does), so that
three of them and their inputs are made in a moment; every size inside a layer and the vocabulary stay.
"""
import functools
import math

import torch

from rocml_amd.config import architecture_of
from rocml_amd.config.catalog import QWEN_THINKING_SAMPLING, resolve
from rocml_amd.engine import DecoderModel, Engine, EngineBackend, Generator, Request, StepEntry
from rocml_amd.sampling import SamplingParams
from rocml_amd.sampling.sampler import DeviceSampler
from rocml_amd.weights import random_model, random_tensor

DEVICE = "cuda:0"
SAMPLING = {"greedy": SamplingParams.greedy(),
            "preset": QWEN_THINKING_SAMPLING,
            "penalty": SamplingParams(temperature=0.8, top_p=0.9, repeat_penalty=1.1)}


def _case(name, model, layers, dtype, batch, shortest, longest, new, sampling="greedy", places="last"):
    c = {"model": model, "layers": layers, "dtype": dtype, "batch": batch, "shortest": shortest, "longest": longest,
         "new": new, "sampling": sampling, "places": places}
    return c if name is None else dict(c, name=name)


def listed():
    return [
        # the smallest call: a test model in the 32-bit mode, a few tokens; all launches and host work
        _case("tiny fp32", "tiny-b", 3, "float32", 1, 5, 5, 8),
        # one user chatting with the smallest released model, a short turn, the model's sampling preset
        _case("chat 0.6b", "qwen3-0.6b", 28, "bfloat16", 1, 37, 37, 32, "preset"),
        # evaluation: the logits at every place of a few texts (what bin/trace_run writes)
        _case("score 0.6b", "qwen3-0.6b", 28, "bfloat16", 3, 100, 300, 1, "greedy", "all"),
        # the 32-bit mode, the one whose results are compared with other implementations
        _case("fp32 0.6b", "qwen3-0.6b", 28, "float32", 4, 20, 300, 16, "preset"),
        # one user of the 8B shape
        _case("8b batch 1", "qwen3-8b", 12, "bfloat16", 1, 512, 512, 48),
        # the benchmark's batch: 8 prompts of 2,048 tokens and decoding behind them
        _case("8b batch 8", "qwen3-8b", 12, "bfloat16", 8, 2048, 2048, 48),
        # a full server: 64 short requests of unequal lengths, drawn with the model's preset
        _case("8b batch 64", "qwen3-8b", 12, "bfloat16", 64, 16, 700, 24, "preset"),
        # the benchmark's prompt: 2,048 tokens, the first token of the answer
        _case("8b prompt 2048", "qwen3-8b", 12, "bfloat16", 1, 2048, 2048, 1),
        # a book in the prompt: the longest one the benchmark runs
        _case("8b prompt 32768", "qwen3-8b", 8, "bfloat16", 1, 32768, 32768, 8),
        # the benchmark's unequal batch on the 14B shape
        _case("14b unequal", "qwen3-14b", 8, "bfloat16", 16, 128, 4096, 32),
        # the further designs without routed experts (a choice of experts that flips with a rounding cannot be compared
        # in bfloat16): latent attention and biased block attention ...
        _case("dokulix", "dokulix-2b", 8, "bfloat16", 8, 2048, 2048, 32),
        # ... and latent rows shared between layers, windowed attention with kept positions, a gated recurrence
        _case("kakalorn", "kakalorn-2b", 12, "bfloat16", 5, 300, 2500, 32),
    ]


# model -> the layers a drawn case may have
_DRAWN = {"tiny-a": (2, 2), "tiny-b": (3, 3), "qwen3-0.6b": (8, 28), "qwen3-1.7b": (6, 28), "qwen3-4b": (4, 18),
          "qwen3-8b": (4, 12), "qwen3-14b": (3, 8), "qwen3-32b": (2, 4), "dokulix-2b": (4, 12), "kakalorn-2b": (6, 12)}
# of several draws the shapes that the library is about come most often
_WEIGHTS = {"qwen3-0.6b": 3, "qwen3-4b": 2, "qwen3-8b": 4, "qwen3-14b": 2}


def draw(rng):
    def spread(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    while True:
        model = rng.choice([m for m in _DRAWN for _ in range(_WEIGHTS.get(m, 1))])
        tiny = model.startswith("tiny")
        dtype = "float32" if tiny and rng.random() < 0.5 or model == "qwen3-0.6b" and rng.random() < 0.3 else "bfloat16"
        layers = rng.randint(*_DRAWN[model])
        batch = spread(1, 8 if tiny else 16 if dtype == "float32" else 64)
        most = {"tiny-a": 100, "tiny-b": 400}.get(model, 1000 if dtype == "float32" else 20000 if batch == 1 else 4096)
        longest = spread(2, most)
        shortest = max(1, min(longest, spread(max(1, longest // 16), longest)))
        places = "all" if model.startswith("qwen3") and batch * longest <= 1200 and rng.random() < 0.2 else "last"
        case = _case(None, model, layers, dtype, batch, shortest, longest, 1 if places == "all" else spread(1, 24 if tiny else 48),
                     rng.choice(["greedy", "greedy", "preset", "penalty"]), places)
        if batch * longest > 36000:
            continue
        if _cost(case) <= 0.7 * max(_cost(c) for c in listed()):
            return case


def _cost(case):
    """Seconds that a pass takes at an ordinary rate: to keep drawn cases below the largest listed one."""
    w = work(case)
    return w["bytes"] / 4e12 + w["flops"] / (8e14 if case["dtype"] == "bfloat16" else 1.5e13) + case["new"] * case["layers"] * 5e-5


# -- the model and its inputs ----------------------------------------------------------------------------------

def _config(case):
    raw = resolve(case["model"]).entry.config
    if case["model"].startswith(("dokulix", "kakalorn")):
        return dict(raw, layers=list(raw["layers"][:case["layers"]]))
    return dict(raw, num_hidden_layers=case["layers"])


@functools.lru_cache(maxsize=64)
def _outline(model, layers, dtype):
    """The model without weights: its parameters and their checkpoint names."""
    cfg = _config({"model": model, "layers": layers})
    arch = architecture_of(cfg)
    spec = arch.to_spec(arch.read_config(cfg))
    outline = DecoderModel(spec, dtype, device="meta")
    return outline, arch.checkpoint_names(spec)


def _lengths(case):
    """Prompt lengths, the shortest and the longest among them; the same for every seed, as a pass has one amount of work."""
    lo, hi, n = case["shortest"], case["longest"], case["batch"]
    if n == 1 or lo == hi:
        return [hi] * n
    g = torch.Generator().manual_seed(n * 100003 + lo * 1009 + hi)
    between = torch.exp(torch.rand(n - 2, generator=g, dtype=torch.float64) * math.log(hi / lo)) * lo if n > 2 else []
    return [lo] + [min(hi, max(lo, int(round(float(t))))) for t in between] + [hi]


def _tokens(case, seed):
    """Per sequence its prompt and the tokens that it goes on with."""
    vocab = _outline(case["model"], case["layers"], case["dtype"])[0].spec.vocab
    g = torch.Generator().manual_seed(int(seed))
    return [(torch.randint(vocab, (n,), generator=g).tolist(), torch.randint(vocab, (case["new"],), generator=g).tolist())
            for n in _lengths(case)]


class _Script:
    """The device sampler, but the sequences go on with tokens laid down beforehand."""

    def __init__(self, inner, host, device):
        self.inner, self.host, self.device = inner, host, device
        self.logits, self.drawn = [], []

    def sample_start(self, logits, seqs):
        k = len(self.logits)
        started = self.inner.sample_start(logits, seqs)
        self.logits.append(logits.clone())          # (the engine's buffer holds until its next step)
        self.drawn.append(started[0])
        return self.device[k], started, k

    def finish(self, started):
        self.inner.finish(started[1])
        return self.host[started[2]]

    def sample(self, logits, seqs):
        return self.finish(self.sample_start(logits, seqs))


def prepare(case, seed):
    model = random_model(_config(case), seed=int(seed), dtype=case["dtype"], device=DEVICE, norm_jitter=True)
    said = _tokens(case, seed)
    pages = sum((len(p) + case["new"] + 63) // 64 + 1 for p, _ in said)
    engine = Engine(model, max_tokens=64 * pages, max_seqs=case["batch"])
    host = [[s[k] for _, s in said] for k in range(case["new"])]
    params = SAMPLING[case["sampling"]]
    return {"case": case, "engine": engine, "sampler": DeviceSampler(DEVICE), "host": host,
            "device": torch.tensor(host, dtype=torch.int32, device=DEVICE), "prompts": [p for p, _ in said],
            "requests": [Request(p, case["new"], params) for p, _ in said]}


def run(state):
    engine, case = state["engine"], state["case"]
    if case["places"] == "all":
        entries = [StepEntry(engine.new_sequence(), p, list(range(len(p)))) for p in state["prompts"]]
        logits = engine.step(entries)
        for e in entries:
            engine.release(e.slot)
        return {"logits": logits}
    script = _Script(state["sampler"], state["host"], state["device"])
    Generator(EngineBackend(engine, sampler=script), max_batch=case["batch"]).run(state["requests"])
    out = {"logits": torch.stack(script.logits)}
    if case["dtype"] == "float32":
        out["drawn"] = torch.stack(script.drawn)
    return out


# -- what a pass cannot do without ----------------------------------------------------------------------------

def _numel(specs):
    return sum(math.prod(p.shape) for p in specs.values())


def _layer_costs(cfg, i):
    """Of layer ``i``: (numbers kept per position, operations per query and key, keys a query sees at most, numbers of state)."""
    if "layers" not in cfg:
        d, hq, hk = cfg["head_dim"], cfg["num_attention_heads"], cfg["num_key_value_heads"]
        return 2 * hk * d, 4 * hq * d, 1 << 40, 0
    lay = cfg["layers"][i]
    m = lay["mixer"]
    if lay["type"] == "hgrn2":
        return 0, 0, 0, m["heads"] * m["dim"] * m["vdim"]
    if lay["type"] == "latent_attention":
        per_pair = 2 * m["heads"] * (m["dim"] + m["rot_dim"] + m["vdim"])
        return m["kv_rank"] + m["rot_dim"], per_pair, m.get("mask", {"size": 1 << 40})["size"], 0
    return 2 * m["kv_heads"] * m["dim"], 2 * m["heads"] * (m["dim"] + m["vdim"]), m["mask"]["size"], 0


def work(case):
    outline, _ = _outline(case["model"], case["layers"], case["dtype"])
    cfg = _config(case)
    size = 2 if case["dtype"] == "bfloat16" else 4
    vocab, width = outline.spec.vocab, outline.spec.hidden
    layer_params = [_numel(b.param_specs()) for b in outline.blocks]
    costs = [_layer_costs(cfg, i) for i in range(len(layer_params))]
    lengths, steps = _lengths(case), case["new"]
    wanted = sum(lengths) if case["places"] == "all" else len(lengths)
    total = {"bytes": 0.0, "flops": 0.0}
    for k in range(steps):                          # the prompt step, then a token per sequence and step
        new = lengths if k == 0 else [1] * len(lengths)
        rows = wanted if k == 0 else len(lengths)
        total["bytes"] += (sum(layer_params) + vocab * width) * size + sum(new) * width * size + rows * vocab * 4
        total["flops"] += 2.0 * sum(layer_params) * sum(new) + 2.0 * vocab * width * rows
        for kept, per_pair, sees, state in costs:
            for n, at in zip(new, lengths if k else [0] * len(lengths)):
                first = at + (k - 1 if k else 0)    # positions before this step
                pairs = sum_seen(first, n, sees)
                total["flops"] += per_pair * pairs + 6.0 * state * n
                total["bytes"] += kept * size * (min(first, sees) + n) + 8 * state
    return total


def sum_seen(first, n, sees):
    """Keys that ``n`` queries at the positions from ``first`` on see, all before them and themselves up to ``sees``."""
    full = max(0, min(n, sees - first))             # queries that see everything before them
    return full * first + full * (full + 1) // 2 + (n - full) * min(sees, first + n)


def tolerance(case):
    # bfloat16: the inputs of every product, q, k, v and probabilities carry 8 bits; twelve layers of the 8B shape end 0.019
    # away from the 64-bit result, the others between 0.006 and 0.019.  32-bit: 0.5e-6 to 2e-6 from sums in another order.
    if case["dtype"] == "bfloat16":
        return {"rel": 0.03, "max": 0.3}
    return {"rel": 2e-5, "max": 1e-3, "differ": 0.005}


# -- the same in 64 bits --------------------------------------------------------------------------------------

def _rms(x, w, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w


def _frequencies(dims, base, scaling=None):
    f = torch.tensor([base ** (-2.0 * i / dims) for i in range(dims // 2)], dtype=torch.float64, device=DEVICE)
    if scaling is None:
        return f, 1.0

    def turns(t):
        return dims * math.log(scaling["original"] / (2.0 * math.pi * t)) / (2.0 * math.log(base))
    lo, hi = max(math.floor(turns(scaling["fast"])), 0), min(math.ceil(turns(scaling["slow"])), dims - 1)
    ramp = ((torch.arange(dims // 2, dtype=torch.float64, device=DEVICE) - lo) / max(hi - lo, 0.001)).clamp(0.0, 1.0)
    return f / scaling["factor"] * ramp + f * (1.0 - ramp), 0.1 * math.log(scaling["factor"]) + 1.0


def _rotate(x, pos, dims, base, scaling=None, neighbours=False):
    """``x [T, heads, d]``: the first ``dims`` numbers turn in pairs of halves or of neighbours."""
    f, factor = _frequencies(dims, base, scaling)
    angle = pos[:, None].double() * f[None]
    c, s = (torch.cos(angle) * factor)[:, None], (torch.sin(angle) * factor)[:, None]
    a, b = (slice(0, dims, 2), slice(1, dims, 2)) if neighbours else (slice(0, dims // 2), slice(dims // 2, dims))
    y = x.clone()
    y[..., a] = x[..., a] * c - x[..., b] * s
    y[..., b] = x[..., b] * c + x[..., a] * s
    return y


def _attend(q, k, v, scale, seen=None, sink=None, slopes=None):
    """One sequence: ``q [T, H, d]``, ``k, v [T, G, *]``; ``seen(i, j)`` beside the causal rule, ``sink [H]`` one more term of the
    denominator, ``slopes [H]`` times the distance taken off the scores."""
    T, H, G = q.shape[0], q.shape[1], k.shape[1]
    out = torch.empty(T, H, v.shape[2], dtype=q.dtype, device=q.device)
    rows = max(1, min(T, (1 << 27) // max(T * (H // G), 1)))
    for g in range(G):
        heads = slice(g * (H // G), (g + 1) * (H // G))
        kt, vg = k[:, g].T.contiguous(), v[:, g].contiguous()
        for lo in range(0, T, rows):
            hi = min(T, lo + rows)
            i, j = torch.arange(lo, hi, device=q.device)[:, None], torch.arange(hi, device=q.device)[None]
            s = (q[lo:hi, heads].transpose(0, 1).reshape(-1, q.shape[2]) @ kt[:, :hi]).view(-1, hi - lo, hi) * scale
            if slopes is not None:
                s -= slopes[heads][:, None, None] * (i - j)[None]
            hidden = j > i if seen is None else (j > i) | ~seen(i, j)
            s.masked_fill_(hidden[None], -math.inf)
            top = s.amax(-1, keepdim=True)
            if sink is not None:
                top = torch.maximum(top, sink[heads][:, None, None])
            e = torch.exp(s - top)
            total = e.sum(-1, keepdim=True)
            if sink is not None:
                total = total + torch.exp(sink[heads][:, None, None] - top)
            o = (e.reshape(-1, hi) @ vg[:hi]).view(-1, hi - lo, vg.shape[1]) / total
            out[lo:hi, heads] = o.transpose(0, 1)
    return out


def _by_sequence(cu, f):
    """``f(lo, hi)`` for every sequence's rows, put one under the other."""
    return torch.cat([f(lo, hi) for lo, hi in zip(cu, cu[1:])])


def _qwen_layer(x, t, i, cfg, pos, cu, eps):
    p = f"model.layers.{i}."
    hq, hk, d, n = cfg["num_attention_heads"], cfg["num_key_value_heads"], cfg["head_dim"], x.shape[0]
    h = _rms(x, t(p + "input_layernorm.weight"), eps)
    q, k, v = ((h @ t(p + f"self_attn.{m}_proj.weight").T).view(n, -1, d) for m in "qkv")
    q = _rotate(_rms(q, t(p + "self_attn.q_norm.weight"), eps), pos, d, cfg["rope_theta"])
    k = _rotate(_rms(k, t(p + "self_attn.k_norm.weight"), eps), pos, d, cfg["rope_theta"])
    o = _by_sequence(cu, lambda a, b: _attend(q[a:b], k[a:b], v[a:b], d ** -0.5))
    x = x + o.reshape(n, hq * d) @ t(p + "self_attn.o_proj.weight").T
    h = _rms(x, t(p + "post_attention_layernorm.weight"), eps)
    g = h @ t(p + "mlp.gate_proj.weight").T
    return x + (g * torch.sigmoid(g) * (h @ t(p + "mlp.up_proj.weight").T)) @ t(p + "mlp.down_proj.weight").T


def _latent(h, p, m, pos, cu, eps, kept, neighbours, seen=None):
    """Latent attention's heads, before their gates; ``kept``: the rows of latents and rotated key parts."""
    n, H, d, r = h.shape[0], m["heads"], m["dim"], m["rot_dim"]
    turn = functools.partial(_rotate, pos=pos, dims=m["rot"]["dims"], base=m["rot"]["base"], scaling=m["rot"].get("scaling"),
                             neighbours=neighbours)
    if kept is None:
        z = h @ p("dkv").T
        kept = (_rms(z[:, :m["kv_rank"]], p("dkv.norm"), eps), turn(z[:, None, m["kv_rank"]:]))
    c, kr = kept
    q = (_rms(h @ p("dq").T, p("dq.norm"), eps) @ p("uq").T).view(n, H, d + r)
    q = torch.cat([q[..., :d], turn(q[..., d:])], -1)
    k = torch.cat([(c @ p("uk").T).view(n, H, d), kr.expand(n, H, r)], -1)
    v = (c @ p("uv").T).view(n, H, -1)
    return _by_sequence(cu, lambda a, b: _attend(q[a:b], k[a:b], v[a:b], m["scale"], seen)), kept


def _dokulix_layer(x, t, i, cfg, pos, cu, eps):
    lay, n = cfg["layers"][i], x.shape[0]
    m, size = lay["mixer"], lay["mixer"]["mask"]["size"]
    p = lambda name: t(f"l{i}.mix.{name}")                                      # noqa: E731
    h = _rms(x, 1.0 + t(f"l{i}.norm1"), eps)
    if lay["type"] == "latent_attention":
        o, _ = _latent(h, p, m, pos, cu, eps, None, False, lambda a, b: a - b < size)
        x = x + (o.reshape(n, -1) * torch.sigmoid(h @ p("g").T)) @ p("o").T
    else:
        H = m["heads"]
        q, k, v = ((h @ p(c).T + p(c + ".b")).view(n, -1, m["dim"]) for c in "qkv")
        q, k = _rms(q, p("q.norm"), eps), _rms(k, p("k.norm"), eps)
        slopes = torch.tensor([2.0 ** (-8.0 * (a + 1) / H) for a in range(H)], dtype=torch.float64, device=DEVICE)
        o = _by_sequence(cu, lambda a, b: _attend(q[a:b], k[a:b], v[a:b], m["scale"], lambda u, w: u // size == w // size,
                                                  torch.zeros_like(slopes), slopes))
        x = x + o.reshape(n, -1) @ p("o").T + p("o.b")
    h = _rms(x, 1.0 + t(f"l{i}.norm2"), eps)
    return x + (torch.relu(h @ t(f"l{i}.mlp.gate").T) * (h @ t(f"l{i}.mlp.up").T)) @ t(f"l{i}.mlp.down").T


def _recurrence(q, f, v):
    state = torch.zeros(q.shape[1], q.shape[2], v.shape[2], dtype=q.dtype, device=q.device)
    out = torch.empty(q.shape[0], q.shape[1], v.shape[2], dtype=q.dtype, device=q.device)
    for s in range(q.shape[0]):
        state = torch.addcmul(f[s][:, :, None] * state, (1.0 - f[s])[:, :, None], v[s][:, None, :])
        torch.matmul(q[s][:, None, :], state, out=out[s][:, None, :])
    return out


def _kakalorn_layer(x, t, i, cfg, pos, cu, eps, kept):
    lay, n = cfg["layers"][i], x.shape[0]
    m = lay["mixer"]
    p = lambda name: t(f"l{i}.mix.{name}")                                      # noqa: E731
    u, taps = _rms(x, t(f"l{i}.norm1"), eps), t(f"l{i}.canon1")

    def convolved(a, b):
        y = u[a:b].clone()
        for j in range(taps.shape[1]):
            back = taps.shape[1] - 1 - j
            if back < b - a:
                y[back:] += taps[:, j] * u[a:b - back]
        return y
    h = _by_sequence(cu, convolved)
    if lay["type"] == "attention":
        d, size, first = m["dim"], m["mask"]["size"], m["mask"]["keep_first"]
        q, v = ((h @ p(c).T + p(c + ".b")).view(n, -1, d) for c in "qk")
        q, k = (_rotate(_rms(z, p(c + ".norm"), eps), pos, m["rot"]["dims"], m["rot"]["base"]) for z, c in ((q, "q"), (v, "k")))
        o = _by_sequence(cu, lambda a, b: _attend(q[a:b], k[a:b], v[a:b], m["scale"], lambda r, w: (r - w < size) | (w < first), p("sink")))
    elif lay["type"] == "hgrn2":
        shape = (n, m["heads"], -1)
        q, low = h @ p("q").T, p("lower")
        q = (q * torch.sigmoid(q)).view(shape)
        f = (low + (1.0 - low) * torch.sigmoid(h @ p("f").T + p("f.b"))).view(shape)
        v = (h @ p("v").T).view(shape)
        o = _rms(_by_sequence(cu, lambda a, b: _recurrence(q[a:b], f[a:b], v[a:b])), p("norm"), eps)
    else:
        src = m.get("kv_from")
        o, rows = _latent(h, p, m, pos, cu, eps, None if src is None else kept[src], True)
        kept.setdefault(i, rows)
        o = o * torch.sigmoid(h @ p("g").T)[:, :, None]
    x = x + _rms(o.reshape(n, -1) @ p("o").T, t(f"l{i}.norm1b"), eps)
    z = torch.relu(_rms(x, t(f"l{i}.norm2"), eps) @ t(f"l{i}.mlp.up").T)
    return x + _rms((z * z) @ t(f"l{i}.mlp.down").T, t(f"l{i}.norm2b"), eps)


def exact(case, seed):
    cfg = _config(case)
    outline, names = _outline(case["model"], case["layers"], case["dtype"])
    specs = {names[k]: p for k, p in outline.param_specs().items()}

    def t(name):                                    # the weight of that checkpoint name, as the model holds it
        p = specs[name]
        return random_tensor(name, p, int(seed), outline.storage_dtype(p), True, device=DEVICE).double()

    said = _tokens(case, seed)
    whole = [p + s[:case["new"] - 1] for p, s in said]
    cu = [0]
    for w in whole:
        cu.append(cu[-1] + len(w))
    ids = torch.tensor([i for w in whole for i in w], device=DEVICE)
    pos = torch.cat([torch.arange(len(w), device=DEVICE) for w in whole])
    design = "layers" in cfg
    eps = cfg["norm"]["eps"] if design else cfg["rms_norm_eps"]
    x = t("embed" if design else "model.embed_tokens.weight")[ids]
    kept = {}
    for i in range(case["layers"]):
        if case["model"].startswith("kakalorn"):
            x = _kakalorn_layer(x, t, i, cfg, pos, cu, eps, kept)
        else:
            x = (_dokulix_layer if design else _qwen_layer)(x, t, i, cfg, pos, cu, eps)
    if case["places"] != "all":                     # the last place of every prompt and the scripted ones: [step, sequence]
        rows = torch.tensor([[cu[b] + len(said[b][0]) - 1 + k for b in range(len(said))] for k in range(case["new"])], device=DEVICE)
        x = x[rows]
    gain = t("final.norm" if design else "model.norm.weight")
    x = _rms(x, 1.0 + gain if case["model"].startswith("dokulix") else gain, eps)
    head = t("head" if design else "lm_head.weight" if "lm_head.weight" in specs else "model.embed_tokens.weight")
    out = {"logits": torch.cat([r @ head.T for r in x.view(-1, x.shape[-1]).split(256)]).view(x.shape[:-1] + (-1,))}
    if case["dtype"] == "float32" and case["places"] != "all":
        out["drawn"] = None
    return out
