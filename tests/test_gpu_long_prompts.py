"""The attention kernel for long prompts (64 query rows a wave) against softmax attention in 64 bits: edges of its tiles and pages, cut
prompts, several sequences, queries from the projection, references that rows leave behind, numbers that are not finite."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu

from rocml_amd import ops  # noqa: E402
from tests.test_gpu_attention import PAGE, _build, _run  # noqa: E402

D = 128
SCALE = D ** -0.5


def _exact(q, k, v, first, scale=SCALE):
    """q [n, Hq, D] at the positions from ``first`` on, k, v [L, Hkv, D]: 64 bits, on the GPU."""
    q, k, v = q.cuda().double(), k.cuda().double(), v.cuda().double()
    n, hq, _ = q.shape
    out = torch.empty_like(q)
    hidden = torch.arange(k.shape[0], device="cuda")[None] > torch.arange(first, first + n, device="cuda")[:, None]
    for h in range(hq):
        s = (q[:, h] @ k[:, h // (hq // k.shape[1])].T.contiguous()) * scale
        s.masked_fill_(hidden, -math.inf)
        out[:, h] = torch.softmax(s, -1) @ v[:, h // (hq // k.shape[1])].contiguous()
    return out.cpu()


def _check(got, want):
    """Probabilities and results carry 8 bits (2^-9 of a value at most, each): a row's error is below twice that of its own norm, a
    value's below 2^-7 of the row's largest."""
    error = (got.double() - want).norm(dim=-1) / want.norm(dim=-1)
    assert float(error.max()) < 2 ** -7, float(error.max())
    assert float(((got.double() - want).abs().amax(-1) / want.abs().amax(-1)).max()) < 2 ** -6


@pytest.mark.parametrize("hq,hkv", [(2, 1), (5, 5), (8, 2), (16, 4)])
@pytest.mark.parametrize("seqs", [
    [(2, 2)], [(64, 64)], [(65, 65)], [(63, 63), (3, 2)], [(256, 256), (257, 257)], [(300, 300), (129, 2), (64, 63), (1, 1)],
    [(1000, 31), (641, 449)], [(1024, 512), (190, 97), (1100, 1100)]])
def test_tiles_pages_and_cuts(seqs, hq, hkv):
    dev, ks, vs, qs = _build(seqs, hq, hkv, D, torch.bfloat16, seed=len(seqs) * 31 + hq)
    got = _run(dev, seqs, hq, hkv, D, SCALE, None, ops.ATTN_PROMPT).view(-1, hq, D)
    at = 0
    for (length, n), k, v, q in zip(seqs, ks, vs, qs):
        _check(got[at:at + n], _exact(q, k, v, length - n))
        at += n


@pytest.mark.parametrize("algo", [ops.ATTN_MFMA, ops.ATTN_PROMPT])
@pytest.mark.parametrize("n_seqs,longer", [(16, {0: 300, 15: 513}), (17, {0: 513, 15: 129, 16: 257}), (64, {15: 257, 16: 300, 63: 513}),
                                           (65, {0: 130, 63: 300, 64: 600}), (70, {16: 129, 62: 257, 64: 300, 69: 513})])
def test_many_sequences_of_more_than_a_tile(n_seqs, longer, algo):
    """A tile's sequence and place in it are found in a walk up to 16 sequences and 64 at a time beyond: sequences of several tiles first,
    last and at the edges of those groups, beside some of one token."""
    counts = [longer.get(i, 1 + 5 * i % 97) for i in range(n_seqs)]
    seqs = [(n + (0 if i % 3 else 40), n) for i, n in enumerate(counts)]
    dev, ks, vs, qs = _build(seqs, 2, 1, D, torch.bfloat16, seed=n_seqs)
    got = _run(dev, seqs, 2, 1, D, SCALE, None, algo).view(-1, 2, D)
    at = 0
    for (length, n), k, v, q in zip(seqs, ks, vs, qs):
        _check(got[at:at + n], _exact(q, k, v, length - n))
        at += n


def test_the_rule_takes_it_and_both_ways_agree():
    """A prompt that the library's own rule gives to this kernel (its bits are those of the forced one, not of the other kernel)."""
    seqs = [(3100, 3100)]
    dev, ks, vs, qs = _build(seqs, 16, 4, D, torch.bfloat16, seed=5)
    chosen, forced, other = (_run(dev, seqs, 16, 4, D, SCALE, None, a) for a in (ops.ATTN_AUTO, ops.ATTN_PROMPT, ops.ATTN_MFMA))
    assert torch.equal(chosen, forced) and not torch.equal(chosen, other)
    want = _exact(qs[0], ks[0], vs[0], 0)
    _check(chosen.view(-1, 16, D), want)
    assert float((chosen.view(-1, 16, D).double() - want).norm()) <= 1.05 * float((other.view(-1, 16, D).double() - want).norm())


@pytest.mark.parametrize("normed", [False, True])
def test_queries_from_the_projection(normed):
    """Norm, rotation and rounding of the queries inside the kernel, at a size that the rule gives to it."""
    n, hq, hkv = 3100, 16, 4
    seqs = [(n, n)]
    dev, ks, vs, qs = _build(seqs, hq, hkv, D, torch.bfloat16, seed=6)
    g = torch.Generator().manual_seed(7)
    qkv = torch.randn(n, (hq + 2 * hkv) * D, generator=g)
    rows = qkv[:, :hq * D].view(n, hq, D).double()
    gain = cos = sin = None
    if normed:
        gain = 1.0 + 0.1 * torch.randn(D, generator=g)
        angle = torch.arange(n)[:, None].double() * (1e4 ** (-torch.arange(D // 2).double() / (D // 2)))[None]
        cos, sin = angle.cos().float().cuda(), angle.sin().float().cuda()
        rows = rows / torch.sqrt((rows * rows).mean(-1, keepdim=True) + 1e-6) * gain.double()
        c, s, a, b = angle.cos()[:, None], angle.sin()[:, None], rows[..., :D // 2], rows[..., D // 2:]
        rows = torch.cat([a * c - b * s, a * s + b * c], -1)
        gain = gain.cuda()
    out = torch.full((n, hq * D), float("nan"), dtype=torch.bfloat16, device="cuda")
    ops.attention_prefill_fused(qkv.cuda(), out, dev["kc"], dev["vc"], dev["table"], dev["tok_pos"], hq, hkv, D, SCALE, gain, 1e-6, cos, sin,
                                None, dev["cu"], [n])
    _check(out.cpu().view(n, hq, D), _exact(rows.to(torch.bfloat16), ks[0], vs[0], 0))


@pytest.mark.parametrize("jump", [40.0, 3000.0, -3000.0])
def test_references_that_are_left_behind(jump):
    """Scores that grow (or fall) by far more than the exponents' range behind the first page."""
    seqs = [(700, 700)]
    dev, ks, vs, qs = _build(seqs, 4, 2, D, torch.bfloat16, seed=8)
    q, k = qs[0], ks[0]
    q[..., 0] = 8.0
    k[..., 0] = 0.0
    k[400:, :, 0] = jump / 8.0
    k[:64, :, 0] -= jump / 16.0
    dev["q"].copy_(q.view(700, -1))
    for page in range((700 + PAGE - 1) // PAGE):
        rows = k[page * PAGE:(page + 1) * PAGE]
        dev["kc"][int(dev["table"][0, page]), :, :rows.shape[0]] = rows.transpose(0, 1).cuda()
    got = _run(dev, seqs, 4, 2, D, 1.0, None, ops.ATTN_PROMPT).view(-1, 4, D)
    # (with a scale of 1 two scores differ by tens: a probability's exponent carries the 32-bit score's error, at most 2^-24 of 3000 x 1.45)
    _check(got, _exact(q, k, vs[0], 0, 1.0))


@pytest.mark.parametrize("a_page", [3.0, 25.0, 55.0])
def test_references_that_stay_or_follow(a_page):
    """Scores that climb by so much a page (in all by 4 to 76, and by 47 to 860), for some rows and heads, and fall or stay for the others:
    up to some 80 the first page's reference does, beyond it the rows are done again, beside rows that keep theirs."""
    seqs = [(1000, 1000)]
    dev, ks, vs, qs = _build(seqs, 4, 2, D, torch.bfloat16, seed=10)
    q, k = qs[0], ks[0]
    q[..., 0] = 8.0
    q[::3, :, 0] = 0.0
    q[1::7, :, 0] = -8.0
    q[:, 3, 0] = 1.0
    k[:, 0, 0] = torch.arange(1000) // 16 * (a_page / 4.0 / 8.0)
    dev["q"].copy_(q.view(1000, -1))
    for page in range((1000 + PAGE - 1) // PAGE):
        rows = k[page * PAGE:(page + 1) * PAGE]
        dev["kc"][int(dev["table"][0, page]), :, :rows.shape[0]] = rows.transpose(0, 1).cuda()
    got = _run(dev, seqs, 4, 2, D, SCALE, None, ops.ATTN_PROMPT).view(-1, 4, D)
    _check(got, _exact(q, k, vs[0], 0))
    got = _run(dev, seqs, 4, 2, D, 1.0, None, ops.ATTN_PROMPT).view(-1, 4, D)
    _check(got, _exact(q, k, vs[0], 0, 1.0))


@pytest.mark.parametrize("value", [float("inf"), float("nan")])
@pytest.mark.parametrize("where", ["key", "value"])
def test_numbers_that_are_not_finite_stay_with_the_rows_that_see_them(where, value):
    seqs = [(600, 600)]
    at = 330                                        # (a row before the 32 keys that hold it sees nothing of it)
    dev, ks, vs, qs = _build(seqs, 4, 2, D, torch.bfloat16, seed=9)
    page, row = int(dev["table"][0, at // PAGE]), at % PAGE
    if where == "key":
        dev["kc"][page, 1, row, 5] = value
    else:
        dev["vc"][page, 1, 5, row] = value
    got = _run(dev, seqs, 4, 2, D, SCALE, None, ops.ATTN_PROMPT).view(-1, 4, D)
    want = _exact(qs[0], ks[0], vs[0], 0)
    _check(got[:, :2], want[:, :2])
    _check(got[:at // 32 * 32], want[:at // 32 * 32])
    other = _run(dev, seqs, 4, 2, D, SCALE, None, ops.ATTN_MFMA).view(-1, 4, D)
    assert torch.equal(torch.isfinite(got), torch.isfinite(other))


def test_what_it_does_not_take_is_refused():
    from rocml_amd.errors import KernelError
    for d, window, counts in ((64, None, [(70, 70)]), (D, 32, [(70, 70)]), (D, None, [(70, 1)])):
        dev, *_ = _build(counts, 4, 2, d, torch.bfloat16, seed=1)
        with pytest.raises(KernelError, match="long prompts"):
            _run(dev, counts, 4, 2, d, SCALE, window, ops.ATTN_PROMPT)
