"""Decode attention of batches whose blocks are shared out by the sequences' lengths: against plain softmax attention, at the edges of the
rule that chooses it, with lengths that need most of the blocks for one sequence, and in a recorded launch whose sequences grow."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu

from rocml_amd import ops  # noqa: E402
from tests.test_gpu_attention import MFMA, PAGE, PLAIN, _build, _check, _fused_case, _reference  # noqa: E402

# (Hq, Hkv, D, lengths): on 256 CUs 8 kv heads share from 5 sequences on; 17 and more where the table has room for 32 pages
SHARED = [(16, 8, 128, [1, 64, 65, 300, 2100]), (16, 8, 64, [1, 1, 1, 1, 1, 4000]), (8, 8, 128, [130] * 7), (32, 8, 128, [63, 64, 65, 127, 128, 129] * 2),
          (40, 8, 128, [700, 1, 2, 3, 64, 128, 192, 256, 320, 1500, 30, 31, 32, 33, 34, 35]), (16, 2, 128, list(range(50, 1700, 50))),
          (6, 3, 96, [5, 900, 17, 64, 200, 1, 33, 450, 128, 70, 1100, 12]), (4, 1, 32, [1 + 37 * i for i in range(40)]),
          (8, 8, 128, [1 + 13 * i for i in range(23)] + [2049]), (8, 8, 128, [2000 + i for i in range(17)]), (8, 4, 64, [40 * i + 1 for i in range(63)] + [2050])]


@pytest.mark.parametrize("hq,hkv,d,lengths", SHARED)
def test_unequal_lengths(hq, hkv, d, lengths):
    _check([(n, 1) for n in lengths], hq, hkv, d, torch.bfloat16, MFMA, n_splits=ops.decode_splits(len(lengths) * hkv, 256, 64), seed=5, unequal=True)
    if d != 96 and d != 32:
        _fused_case([(n, 1) for n in lengths], hq, hkv, d, 2, ops.decode_splits(len(lengths) * hkv, 256, 64), None, seed=7, unequal=True)


def _options(name, hq):
    g = torch.Generator().manual_seed(41)
    return {"slopes": dict(slopes=0.02 * torch.rand(hq, generator=g)), "sink": dict(sink=True),
            "sinks": dict(sink=True, sinks=3.0 * torch.randn(hq, generator=g)), "softcap": dict(softcap=1.5),
            "all": dict(slopes=0.02 * torch.rand(hq, generator=g), sink=True, sinks=3.0 * torch.randn(hq, generator=g), softcap=2.0)}[name]


def _exact(q, k, v, scale, slopes=None, sink=False, sinks=None, softcap=None):
    """The last position's query ``[Hq, D]`` over keys and values ``[L, Hkv, D]``, 64 bits."""
    out = torch.zeros(q.shape, dtype=torch.float64)
    for h in range(q.shape[0]):
        kv = h // (q.shape[0] // k.shape[1])
        s = (k[:, kv].double() @ q[h].double()) * scale
        if softcap is not None:
            s = softcap * torch.tanh(s / softcap)
        if slopes is not None:
            s = s - float(slopes[h]) * torch.arange(len(s) - 1, -1, -1)
        if sink:
            s = torch.cat([s, torch.tensor([0.0 if sinks is None else float(sinks[h])], dtype=torch.float64)])
        out[h] = torch.softmax(s, 0)[:k.shape[0]] @ v[:, kv].double()
    return out


WITH_OPTIONS = [(16, 8, 128, [1, 64, 65, 300, 2100, 7, 900]), (8, 8, 64, [1 + 23 * i for i in range(23)] + [2300]), (12, 4, 96, [3, 1500, 64, 100, 9, 77, 128, 5, 33])]


@pytest.mark.parametrize("option", ["slopes", "sink", "sinks", "softcap", "all"])
@pytest.mark.parametrize("hq,hkv,d,lengths", WITH_OPTIONS)
def test_unequal_lengths_with_options(hq, hkv, d, lengths, option):
    dev, ks, vs, qs = _build([(n, 1) for n in lengths], hq, hkv, d, torch.bfloat16, 12)
    options, scale = _options(option, hq), 2.0 / math.sqrt(d)
    cuda = {k: v.cuda() if torch.is_tensor(v) else v for k, v in options.items()}
    ws = torch.full((32 << 20,), 0xff, dtype=torch.uint8, device="cuda")         # (what no split has written is NaN)
    out = torch.full_like(dev["q"], float("nan"))
    ops.attention(dev["q"], out, dev["kc"], dev["vc"], dev["table"], dev["tok_seq"], dev["tok_pos"], hq, hkv, d, scale, None, algo=MFMA,
                  workspace=ws, cu_seqlens=dev["cu"], max_new=1, q_counts=[1] * len(lengths), max_len=max(lengths),
                  n_splits=ops.decode_splits(len(lengths) * hkv, 256, 64), unequal=True, **cuda)
    for b in range(len(lengths)):
        want = _exact(qs[b][0], ks[b], vs[b], scale, **options)
        assert float((out[b].cpu().double().view(hq, d) - want).abs().max()) < 1.5e-2, lengths[b]


@pytest.mark.parametrize("rot,values_are_keys,with_bias", [(1.0, False, True), (0.5, False, False), (0.5, True, True), (1.0, True, False)])
@pytest.mark.parametrize("hq,hkv,d,lengths", WITH_OPTIONS[:2])
def test_fused_unequal_lengths_with_options(hq, hkv, d, lengths, rot, values_are_keys, with_bias):
    """Biases, a rotation of a part of the head, values that are the projected keys, slopes and sinks in the kernel that reads the
    projection, against the norm-and-rotation kernel and the plain attention kernel: the same cache rows and, within rounding, output."""
    n, rot, g = len(lengths), int(d * rot), torch.Generator().manual_seed(43)
    draw = lambda *s: torch.randn(*s, generator=g).cuda()          # noqa: E731
    dev, *_ = _build([(length, 1) for length in lengths], hq, hkv, d, torch.bfloat16, 13)
    rows = (hq + (1 if values_are_keys else 2) * hkv) * d
    qkv, bias = draw(n, rows), 0.5 * draw(rows) if with_bias else None
    q_gain, k_gain = 1 + 0.3 * draw(d), 1 + 0.3 * draw(d)
    angle = 6.28 * torch.rand(n, rot // 2, generator=g)
    cos, sin = angle.cos().cuda(), angle.sin().cuda()
    slopes, sinks, scale = (0.02 * torch.rand(hq, generator=g)).cuda(), 2 * draw(hq), 1 / math.sqrt(d)
    ws = torch.full((32 << 20,), 0xff, dtype=torch.uint8, device="cuda")
    kc, vc = dev["kc"].clone(), dev["vc"].clone()
    q = torch.empty(n, hq * d, dtype=torch.bfloat16, device="cuda")
    want, got = torch.full_like(q, float("nan")), torch.full_like(q, float("nan"))
    ops.qk_norm_rope_append(qkv, hq, hkv, d, q_gain, k_gain, 1e-5, cos, sin, rot, q, kc, vc, dev["table"], dev["tok_seq"], dev["tok_pos"],
                            bias=bias, values_are_keys=values_are_keys)
    ops.attention(q, want, kc, vc, dev["table"], dev["tok_seq"], dev["tok_pos"], hq, hkv, d, scale, None, algo=PLAIN, slopes=slopes,
                  sink=True, sinks=sinks)
    ops.attention_decode_fused(qkv, got, dev["kc"], dev["vc"], dev["table"], None, dev["tok_pos"], hq, hkv, d, scale, q_gain, k_gain, 1e-5,
                               cos, sin, workspace=ws, max_len=max(lengths), n_splits=ops.decode_splits(n * hkv, 256, 64), bias=bias,
                               slopes=slopes, sink=True, sinks=sinks, values_are_keys=values_are_keys, unequal=True)
    for a, b in ((dev["kc"], kc), (dev["vc"], vc)):
        assert float(((a.float() - b.float()).abs() / b.float().abs().clamp_min(1e-3)).max()) < 1e-2
    assert float((got.float() - want.float()).abs().max()) < 2e-2


@pytest.mark.parametrize("room", [1, 2, 5])
def test_little_workspace(room):
    """A workspace that holds so many splits of every token: no more are made, with one none."""
    lengths, hq, hkv, d = [10, 2500, 64, 300, 1, 129, 600], 16, 8, 128
    dev, ks, vs, qs = _build([(n, 1) for n in lengths], hq, hkv, d, torch.bfloat16, 3)
    size = len(lengths) * hq * (d + 2) * 4 * room
    ws = torch.full((size + 4096,), 0x7f, dtype=torch.uint8, device="cuda")
    out = torch.full_like(dev["q"], float("nan"))
    ops.attention(dev["q"], out, dev["kc"], dev["vc"], dev["table"], dev["tok_seq"], dev["tok_pos"], hq, hkv, d, d ** -0.5, None, algo=MFMA,
                  workspace=ws[:size], cu_seqlens=dev["cu"], max_new=1, q_counts=[1] * len(lengths), max_len=max(lengths), n_splits=0, unequal=True)
    assert bool((ws[size:] == 0x7f).all())
    for b, n in enumerate(lengths):
        want = _reference(qs[b], ks[b], vs[b], [n - 1], d ** -0.5, None)
        assert float((out[b].cpu().double().view(1, hq, d) - want).abs().max()) < 1.5e-2


def test_recorded_while_lengths_change():
    """A recorded launch follows the positions it finds at each replay."""
    lengths, hq, hkv, d = [1000, 64, 700, 65, 1400, 300, 2], 16, 8, 128
    dev, ks, vs, qs = _build([(n, 1) for n in lengths], hq, hkv, d, torch.bfloat16, 9)
    ws = torch.empty(16 << 20, dtype=torch.uint8, device="cuda")
    out = torch.empty_like(dev["q"])

    def step():
        ops.attention(dev["q"], out, dev["kc"], dev["vc"], dev["table"], dev["tok_seq"], dev["tok_pos"], hq, hkv, d, d ** -0.5, None, algo=MFMA,
                      workspace=ws, cu_seqlens=dev["cu"], max_new=1, q_counts=[1] * len(lengths), max_len=max(lengths), n_splits=5, unequal=True)
    step()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        step()
    for sub in (0, 1, 63, 900):
        now = [max(1, n - sub) if n != 1400 else n for n in lengths]
        dev["tok_pos"].copy_(torch.tensor(now, dtype=torch.int32) - 1)
        ws.fill_(0xff)                              # what is left from before is NaN
        graph.replay()
        torch.cuda.synchronize()
        replayed = out.clone()
        step()
        torch.cuda.synchronize()
        assert torch.equal(out, replayed)
        for b, n in enumerate(now):
            want = _reference(qs[b], ks[b][:n], vs[b][:n], [n - 1], 1.0 / math.sqrt(d), None)
            assert float((replayed[b].cpu().double().view(1, hq, d) - want).abs().max()) < 1.5e-2, (sub, n, PAGE)


@pytest.mark.parametrize("hq,hkv,d,n,length", [(16, 8, 128, 8, 2070), (8, 8, 128, 24, 700), (16, 8, 64, 6, 130)])
def test_as_many_splits_as_asked_for(hq, hkv, d, n, length):
    """Without ``unequal`` every token has ``n_splits`` splits, with one no merge: the workspace stays as it is."""
    dev, ks, vs, qs = _build([(length - i, 1) for i in range(n)], hq, hkv, d, torch.bfloat16, 4)
    for splits in (1, 3):
        ws = torch.full((32 << 20,), 0x7f, dtype=torch.uint8, device="cuda")
        out = torch.full_like(dev["q"], float("nan"))
        ops.attention(dev["q"], out, dev["kc"], dev["vc"], dev["table"], dev["tok_seq"], dev["tok_pos"], hq, hkv, d, d ** -0.5, None, algo=MFMA,
                      workspace=ws, cu_seqlens=dev["cu"], max_new=1, q_counts=[1] * n, max_len=length, n_splits=splits)
        used = n * hq * (d + 2) * 4 * splits if splits > 1 else 0
        assert bool((ws[used:] == 0x7f).all()) and (used == 0 or not bool((ws[used - 4096:used] == 0x7f).all()))
        for b in range(0, n, 5):
            want = _reference(qs[b], ks[b], vs[b], [length - b - 1], d ** -0.5, None)
            assert float((out[b].cpu().double().view(1, hq, d) - want).abs().max()) < 1.5e-2


def test_engine_batches_that_become_alike(tmp_path):
    """Steps of a batch whose lengths differ by much and less and less run, and are recorded, as one launch and then the other; steps of
    one length only as the other.  Bit for bit the logits of steps that are not recorded."""
    from rocml_amd.engine import Engine, StepEntry
    from rocml_amd.weights import load_model
    from tests import helpers
    cfg = dict(helpers.TINY_H, hidden_size=128, num_attention_heads=8, num_key_value_heads=8, head_dim=64)
    path = helpers.make_model_dir(tmp_path, cfg, 31, torch.bfloat16)

    def run(lengths, steps, use_graphs):
        engine = Engine(load_model(path, dtype="bfloat16", device="cuda:0"), max_tokens=4096, use_graphs=use_graphs)
        texts = [helpers.random_tokens(n + steps, cfg["vocab_size"], 3 + i) for i, n in enumerate(lengths)]
        slots = [engine.new_sequence() for _ in lengths]
        engine.step([StepEntry(s, t[:n], []) for s, t, n in zip(slots, texts, lengths)])
        out = []
        for k in range(steps):
            out.append(engine.step([StepEntry(s, [t[n + k]], [0]) for s, t, n in zip(slots, texts, lengths)]).cpu())
        return torch.stack(out), {key[3] for key, entry in engine._graphs.items() if key[0] != "prompt" and entry[1] is not None}

    got, sides = run([10, 10, 11, 12, 100, 10], 160, True)
    want, none = run([10, 10, 11, 12, 100, 10], 160, False)
    assert torch.equal(got, want) and sides == {True, False} and not none
    assert run([70] * 6, 5, True)[1] == {False}
