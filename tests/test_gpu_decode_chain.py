"""The layers of a decode step in one launch (``ops.decode_chain``) against the same layers in 64 bits written here: the
smallest sizes it takes, one, several and all of a wave's weights asked for at once, odd positions around page edges, one and
many splits of the keys, one to four sequences; the state kept over calls of other sizes, and a recorded launch replayed.

Bound: the operands of every product, q, k, v and probabilities carry 8 bits (a rounding error of up to 2^-9, 0.0011 root mean
square), and a layer's result passes about eight such roundings, 0.0032; two layers and what the second makes of the first's
error stay below 0.01 in the 2-norm of what the layers added, row by row.  32-bit: sums of up to 6,144 products in runs, about 1e-6; 1e-5."""
import pytest
import torch

pytestmark = pytest.mark.gpu

from rocml_amd import ops  # noqa: E402

D, PAGE, EPS = 128, 64, 1e-6
DEV = "cuda:0"


class _Position:
    spec = "the test's"


def _model(hidden, hq, hkv, inter, n_layers, lens, width, seed, dtype=torch.bfloat16):
    g = torch.Generator(device=DEV).manual_seed(seed)

    def rand(*shape, scale=1.0):
        return torch.randn(*shape, generator=g, device=DEV) * scale
    n_pages = sum((n + PAGE) // PAGE for n in lens) + 3
    order = torch.randperm(n_pages, generator=torch.Generator().manual_seed(seed)).tolist()
    table = torch.full((len(lens), width), -1, dtype=torch.int32)
    for b, n in enumerate(lens):
        for i in range(n // PAGE + 1):
            table[b, i] = order.pop()
    table = table.to(DEV)
    layers = []
    for _ in range(n_layers):
        w = [rand(r, c, scale=c ** -0.5).to(dtype) for r, c in (((hq + 2 * hkv) * D, hidden), (hidden, hq * D), (2 * inter, hidden), (hidden, inter))]
        gains = [1.0 + rand(n, scale=0.1) for n in (D, D, hidden, hidden)]
        k, v = rand(n_pages, hkv, PAGE, D).to(dtype), rand(n_pages, hkv, D, PAGE).to(dtype)
        layers.append(ops.ChainLayer(*w, *gains, k, v, table, hq, hkv, D ** -0.5, EPS, EPS, EPS, _Position()))
    x = rand(len(lens), hidden)
    inv = 1e4 ** (-torch.arange(0, D, 2, device=DEV, dtype=torch.float64) / D)
    angle = torch.tensor(lens, device=DEV, dtype=torch.float64)[:, None] * inv
    return layers, x, angle.cos().float(), angle.sin().float(), torch.tensor(lens, dtype=torch.int32, device=DEV)


def _rms(x, gain):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * gain.double()


def _plain(layers, x, cos, sin, lens):
    """The layers in 64 bits; the stream and each layer's new keys and values."""
    x, kept = x.double(), []
    for c in layers:
        hq, hkv, n = c.n_heads, c.n_kv_heads, x.shape[0]
        y = (_rms(x, c.mix_gain) @ c.w_qkv.double().T).view(n, hq + 2 * hkv, D)
        q, k, v = _rms(y[:, :hq], c.q_gain), _rms(y[:, hq:hq + hkv], c.k_gain), y[:, hq + hkv:]

        def turn(z):
            a, b, co, si = z[..., :D // 2], z[..., D // 2:], cos.double()[:, None], sin.double()[:, None]
            return torch.cat([a * co - b * si, a * si + b * co], -1)
        q, k = turn(q), turn(k)
        kept.append((k, v))
        o = torch.empty(n, hq, D, dtype=torch.float64, device=DEV)
        for b, ln in enumerate(lens):
            pages = c.block_table[b, :ln // PAGE + 1].long()
            ks = c.k_cache[pages].double().permute(0, 2, 1, 3).reshape(-1, hkv, D)[:ln]
            vs = c.v_cache[pages].double().permute(0, 3, 1, 2).reshape(-1, hkv, D)[:ln]
            ks, vs = torch.cat([ks, k[b:b + 1]]), torch.cat([vs, v[b:b + 1]])
            for h in range(hq):
                p = torch.softmax(ks[:, h * hkv // hq] @ q[b, h] * c.scale, 0)
                o[b, h] = p @ vs[:, h * hkv // hq]
        x = x + o.reshape(n, -1) @ c.w_o.double().T
        gu = _rms(x, c.ffn_gain) @ c.w_gate_up.double().T
        gate, up = gu[:, 0::2], gu[:, 1::2]
        x = x + (gate * torch.sigmoid(gate) * up) @ c.w_down.double().T
    return x, kept


def _run(layers, x, cos, sin, pos, state, **how):
    xn = torch.empty(x.shape, dtype=layers[0].w_qkv.dtype, device=DEV)
    ops.rmsnorm(x, layers[0].mix_gain, EPS, xn)
    ops.decode_chain(x, xn, layers, pos, cos, sin, state, **how)


def _check(layers, x0, x, cos, sin, lens):
    want, kept = _plain(layers, x0, cos, sin, lens)
    added = want - x0.double()
    bound = 0.01 if layers[0].w_qkv.dtype == torch.bfloat16 else 1e-5
    assert torch.isfinite(x).all()
    assert float(((x.double() - want).norm(dim=-1) / added.norm(dim=-1)).max()) < bound
    for c, (k, v) in zip(layers, kept):
        for b, ln in enumerate(lens):
            page, at = int(c.block_table[b, ln // PAGE]), ln % PAGE
            assert float((c.k_cache[page, :, at].double() - k[b]).norm() / k[b].norm()) < bound
            assert float((c.v_cache[page, :, :, at].double() - v[b]).norm() / v[b].norm()) < bound


CASES = [
    # hidden, query heads, kv heads, intermediate, layers, positions, pages a table has room for
    (512, 4, 4, 512, 1, [0], 1),                            # the smallest: one group of steps a wave, no key but the step's own
    (512, 8, 1, 1024, 2, [63, 64], 2),                      # a group of eight heads; the last row of a page and the first of the next
    (1024, 16, 8, 3072, 2, [37], 1),                        # three tiles an item
    (1024, 16, 8, 3072, 2, [255, 0, 128], 4),               # as many pages as one split takes
    (1024, 16, 8, 3072, 2, [256, 700, 1, 1023], 16),        # several splits, some without a page
    (1536, 12, 4, 2560, 2, [300], 5),                       # three groups of steps, an odd number of pages
    (2048, 16, 8, 6144, 2, [1000, 65], 64),                 # longer than the ring of weights; a split a page and more
    (2560, 32, 8, 9728, 1, [129], 4),
    (1024, 16, 8, 3072, 2, [9000], 256),                    # the most splits, several pages each
]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=["bf16", "f32"])
@pytest.mark.parametrize("case", CASES, ids=[f"{c[0]}-{c[1]}-{c[3]}-{c[5]}" for c in CASES])
def test_layers_in_one_launch(case, dtype):
    hidden, hq, hkv, inter, n_layers, lens, width = case
    layers, x0, cos, sin, pos = _model(hidden, hq, hkv, inter, n_layers, lens, width, hidden + len(lens), dtype)
    words = ops.decode_chain_words(layers[0], len(lens), n_layers)
    assert words > 0
    state = torch.zeros(words, dtype=torch.int64, device=DEV)
    x = x0.clone()
    _run(layers, x, cos, sin, pos, state)
    _check(layers, x0, x, cos, sin, lens)
    # the state is as good for the next launch, and the sums do not depend on timing
    for _ in range(3):
        again = x0.clone()
        _run(layers, again, cos, sin, pos, state)
        assert torch.equal(again, x)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=["bf16", "f32"])
@pytest.mark.parametrize("case", CASES, ids=[f"{c[0]}-{c[1]}-{c[3]}-{c[5]}" for c in CASES])
def test_every_key_counts_once(case, dtype):
    """A layer whose feed-forward adds nothing, so that what is added is attention's alone: the output of ``n`` keys with random
    scores changes by the root of ``m / n`` when ``m`` of them are lost or taken twice, 0.06 for a piece of 32 among 9,000 (0.04 for 16 in
    32-bit), which the bounds above do not let pass; beside the feed-forward's sums it would be hidden."""
    hidden, hq, hkv, inter, _, lens, width = case
    layers, x0, cos, sin, pos = _model(hidden, hq, hkv, inter, 1, lens, width, hidden + 7, dtype)
    layers[0].w_down.zero_()
    state = torch.zeros(ops.decode_chain_words(layers[0], len(lens), 1), dtype=torch.int64, device=DEV)
    x = x0.clone()
    _run(layers, x, cos, sin, pos, state)
    _check(layers, x0, x, cos, sin, lens)


def test_one_state_for_launches_of_other_sizes():
    small = _model(1024, 16, 8, 3072, 2, [70], 2, seed=1)
    large = _model(1024, 16, 8, 3072, 3, [90, 500], 16, seed=2)
    state = torch.zeros(max(ops.decode_chain_words(m[0][0], m[1].shape[0], len(m[0])) for m in (small, large)), dtype=torch.int64, device=DEV)
    for layers, x0, cos, sin, pos in (small, large, small, large):
        x = x0.clone()
        _run(layers, x, cos, sin, pos, state)
        _check(layers, x0, x, cos, sin, pos.tolist())


def test_recorded_launch_replayed_with_other_inputs():
    layers, x0, cos, sin, pos = _model(1024, 16, 8, 3072, 2, [130, 77], 4, seed=3)
    state = torch.zeros(ops.decode_chain_words(layers[0], 2, 2), dtype=torch.int64, device=DEV)
    x = x0.clone()
    _run(layers, x, cos, sin, pos, state)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        _run(layers, x, cos, sin, pos, state)
    for i in range(4):
        fresh = x0 * (1.0 + 0.25 * i)
        x.copy_(fresh)
        graph.replay()
        got = x.clone()
        eager = fresh.clone()
        _run(layers, eager, cos, sin, pos, state)
        torch.cuda.synchronize()
        assert torch.equal(got, eager)


@pytest.mark.parametrize("case", [CASES[0], CASES[4], CASES[6]], ids=["smallest", "splits", "wide"])
def test_as_few_blocks_as_there_may_be(case):
    """Eight blocks, which each have a counter to themselves, give the same bits, and the state is as good for the next launch."""
    hidden, hq, hkv, inter, n_layers, lens, width = case
    layers, x0, cos, sin, pos = _model(hidden, hq, hkv, inter, n_layers, lens, width, 7)
    state = torch.zeros(ops.decode_chain_words(layers[0], len(lens), n_layers), dtype=torch.int64, device=DEV)
    x = x0.clone()
    _run(layers, x, cos, sin, pos, state)
    _check(layers, x0, x, cos, sin, lens)
    for blocks in (8, 0, 24, 104, 8, 0):
        again = x0.clone()
        _run(layers, again, cos, sin, pos, state, blocks=blocks)
        assert torch.equal(again, x), blocks


def test_two_launches_side_by_side():
    """Launches on two streams, which may each have some of the dies first."""
    models = [_model(1024, 16, 8, 3072, 3, lens, 16, seed=len(lens)) for lens in ([700, 90], [800])]
    states = [torch.zeros(ops.decode_chain_words(m[0][0], m[1].shape[0], 3), dtype=torch.int64, device=DEV) for m in models]
    want = []
    for (layers, x0, cos, sin, pos), state in zip(models, states):
        x = x0.clone()
        _run(layers, x, cos, sin, pos, state)
        _check(layers, x0, x, cos, sin, pos.tolist())
        want.append(x)
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in models]
    got = [[], []]
    for _ in range(20):
        for i, (layers, x0, cos, sin, pos) in enumerate(models):
            with torch.cuda.stream(streams[i]):
                x = x0.clone()
                _run(layers, x, cos, sin, pos, states[i])
                got[i].append(x)
    torch.cuda.synchronize()
    assert all(torch.equal(x, w) for xs, w in zip(got, want) for x in xs)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=["bf16", "f32"])
def test_a_wait_that_ended_concerns_its_own_launch_only(dtype):
    """A launch whose waits are told to end at once (every wait still ends by itself, the launch runs through) gives NaN and leaves
    none in the cache; the next one on the same state, whose waits look for a mark at every turn, gives what a fresh state gives."""
    layers, x0, cos, sin, pos = _model(1024, 16, 8, 3072, 2, [70, 300], 5, seed=5, dtype=dtype)
    state = torch.zeros(ops.decode_chain_words(layers[0], 2, 2), dtype=torch.int64, device=DEV)
    x = x0.clone()
    _run(layers, x, cos, sin, pos, state, polls=1, patience=0.0)
    assert torch.isnan(x).any()
    assert all(torch.isfinite(t).all() for c in layers for t in (c.k_cache, c.v_cache))
    for _ in range(3):
        x = x0.clone()
        _run(layers, x, cos, sin, pos, state, polls=1)
        _check(layers, x0, x, cos, sin, pos.tolist())


@pytest.mark.parametrize("dtype,rows,hidden,inter,most", [
    (torch.bfloat16, 1, 1024, 3072, 512), (torch.bfloat16, 2, 1024, 3072, 64), (torch.bfloat16, 3, 1024, 3072, 42), (torch.bfloat16, 4, 2048, 6144, 32),
    (torch.float32, 4, 1024, 3072, 1 << 20), (torch.float32, 1, 2048, 6144, 1 << 20), (torch.float32, 2, 2048, 6144, 0), (torch.bfloat16, 1, 4096, 12288, 0)])
def test_up_to_how_many_pages_it_pays(dtype, rows, hidden, inter, most):
    hq = 2 * hidden // D
    layer = _model(hidden, hq, 8, inter, 1, [5] * rows, 1, seed=9, dtype=dtype)[0][0]
    for pages in (1, max(most, 1), most + 1):
        layer.block_table = torch.zeros(rows, pages, dtype=torch.int32, device=DEV)
        assert ops.decode_chain_pays(layer, rows) == (0 < pages <= most or most == 1 << 20), pages


def test_what_the_chain_does_not_take():
    layers, x0, cos, sin, pos = _model(512, 4, 4, 512, 1, [5], 1, seed=4)
    state = torch.zeros(ops.decode_chain_words(layers[0], 1, 1), dtype=torch.int64, device=DEV)
    xn = x0.bfloat16()
    with pytest.raises(ops.KernelError):                    # a state that is too short
        ops.decode_chain(x0, xn, layers, pos, cos, sin, state[:-16])
    with pytest.raises(ops.KernelError):                    # more rows than it knows
        many = _model(512, 4, 4, 512, 1, [5] * 5, 1, seed=4)
        ops.decode_chain(many[1], many[1].bfloat16(), many[0], many[4], many[2], many[3], state)
    assert ops.decode_chain_words(layers[0], 5, 1) == 0
    layer = layers[0]                                       # operands that the layer's own kernels take and the chain's loads do not
    assert ops.decode_chain_pays(layer, 1)
    w = layer.w_o
    layer.w_o = torch.empty(w.shape[0], w.shape[1] + 8, dtype=w.dtype, device=DEV)[:, :w.shape[1]]
    assert not ops.decode_chain_pays(layer, 1)
    layer.w_o = torch.empty(w.numel() + 1, dtype=w.dtype, device=DEV)[1:].view(w.shape)
    assert not ops.decode_chain_pays(layer, 1)
    with pytest.raises(ops.KernelError):
        ops.decode_chain(x0, xn, [layer], pos, cos, sin, state)
    odd = _model(768, 6, 2, 768, 1, [5], 1, seed=4)[0][0]    # no whole groups of steps in a wave's share of K
    assert ops.decode_chain_words(odd, 1, 1) == 0 and not ops.decode_chain_pays(odd, 1)
