"""The prompt forms of the row kernels (wide loads, several rows a wave, values in the same launch) against the general forms that
take the same work in pieces or from an address that allows no wide loads."""
import pytest
import torch

pytestmark = pytest.mark.gpu

from rocml_amd import ops  # noqa: E402

DEV = "cuda:0"


def _tables(n, half, g):
    angle = torch.rand(n, half, generator=g, dtype=torch.float64) * 6.0
    return torch.cos(angle).float().to(DEV), torch.sin(angle).float().to(DEV)


# one set of rows a wave and four (65,536 rows and more); a last wave with less; no norm, no rotation, a bias, a stretch, factors of
# a whole-row norm; keys and values without queries; bfloat16 rows
@pytest.mark.parametrize("tokens,hq,hkv,d,form", [
    (64, 4, 2, 128, "plain"), (65, 16, 8, 128, "plain"), (2800, 16, 8, 128, "plain"), (670, 3, 1, 256, "plain"), (9363, 6, 1, 256, "plain"),
    (130, 4, 2, 128, "bias"), (130, 4, 2, 128, "stretch"), (130, 4, 2, 128, "span"), (130, 4, 2, 128, "no rotation"),
    (130, 4, 2, 128, "keys only"), (300, 4, 2, 128, "bfloat16 rows"), (200, 0, 3, 192, "moved"), (200, 2, 3, 64, "moved"), (64, 0, 2, 48, "moved")])
def test_prompt_rows_match_few_rows(tokens, hq, hkv, d, form):
    g = torch.Generator().manual_seed(tokens + d)
    in_dtype = torch.bfloat16 if form in ("bfloat16 rows", "moved") else torch.float32
    out_dtype = torch.bfloat16 if in_dtype == torch.bfloat16 else torch.float32
    qkv = torch.randn(tokens, (hq + 2 * hkv) * d, generator=g).to(DEV, in_dtype)
    gains = [None, None] if form == "moved" else [(1 + 0.1 * torch.randn(d, generator=g)).to(DEV) for _ in range(2)]
    kw = {}
    if form == "bias":
        kw["bias"] = torch.randn(qkv.shape[1], generator=g).to(DEV)
    if form == "stretch":
        kw["q_temp"] = (0.1, 16)
    if form == "span":
        gains = [(1 + 0.1 * torch.randn(h * d, generator=g)).to(DEV) for h in (hq, hkv)]
        kw["span_inv"] = (0.5 + torch.rand(tokens, 2, generator=g)).to(DEV)
    cos, sin = (None, None) if form in ("no rotation", "moved") else _tables(tokens, d // 2, g)
    seq = (torch.arange(tokens) // 100).to(torch.int32).to(DEV)               # sequences of 100 tokens, pages in disorder
    pos = (torch.arange(tokens) % 100 + 7).to(torch.int32).to(DEV)
    pages = 2 * ((tokens + 99) // 100)
    table = torch.randperm(pages, generator=g).to(torch.int32).view(-1, 2)
    table[-1, 1] = -1                                                           # a page that is not there
    table = table.to(DEV)
    with_q = hq > 0 and form != "keys only"
    outs = []
    for step in (tokens, 63):
        q = torch.zeros(tokens, hq * d, dtype=out_dtype, device=DEV) if with_q else None
        k = torch.zeros(pages, hkv, 64, d, dtype=out_dtype, device=DEV)
        v = torch.zeros(pages, hkv, d, 64, dtype=out_dtype, device=DEV)
        for lo in range(0, tokens, step):
            part = slice(lo, min(tokens, lo + step))
            kp = dict(kw, span_inv=kw["span_inv"][part].contiguous()) if "span_inv" in kw else kw
            ops.qk_norm_rope_append(qkv[part], hq, hkv, d, gains[0], gains[1], 1e-6, None if cos is None else cos[part],
                                    None if sin is None else sin[part], 0 if cos is None else d, None if q is None else q[part], k, v, table,
                                    seq[part], pos[part], **kp)
        outs.append([t for t in (q, k, v) if t is not None])
    for a, b in zip(*outs):
        assert torch.equal(a, b)         # a token's q, k and v do not depend on how many tokens its step has
        assert float(a.float().abs().max()) > 0


@pytest.mark.parametrize("pairing", ["halves", "neighbours"])
@pytest.mark.parametrize("tokens,heads,lead,part,dims", [(1, 1, 0, 8, 0), (3, 2, 0, 16, 16), (5, 3, 128, 64, 64), (70, 16, 128, 64, 32), (9, 4, 8, 24, 16)])
def test_rotated_heads_eight_numbers_a_thread(tokens, heads, lead, part, dims, pairing):
    g = torch.Generator().manual_seed(part + dims)
    stride = lead + part + 8
    q = torch.randn(tokens, heads * stride, generator=g).to(DEV)
    cos, sin = _tables(tokens, dims // 2, g) if dims else (None, None)
    whole = [torch.zeros(tokens, heads * (lead + part + 16), dtype=torch.float32, device=DEV) for _ in range(2)]
    ops.rope_heads(q, heads, stride, lead, part, dims, cos, sin, whole[0], lead + part + 16, 8, lead=lead, pairing=pairing)
    # the general form: the same rows behind one number
    shifted = torch.empty(q.numel() + 1, device=DEV)[1:].view_as(q)
    shifted.copy_(q)
    ops.rope_heads(shifted, heads, stride, lead, part, dims, cos, sin, whole[1], lead + part + 16, 8, lead=lead, pairing=pairing)
    assert float((whole[0] - whole[1]).abs().max()) <= 1e-6 and float(whole[0].abs().max()) > 0       # (a product rounded before the sum or not)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("gate", ["none", "head", "value"])
@pytest.mark.parametrize("rows,heads,n,stride", [(1, 1, 8, 8), (33, 3, 24, 40), (100, 16, 128, 192)])
def test_gated_heads_eight_numbers_a_thread(rows, heads, n, stride, gate, dtype):
    g = torch.Generator().manual_seed(n)
    x = torch.randn(rows, heads * stride, generator=g).to(DEV, dtype)
    wide = torch.randn(rows, heads * n + 4, generator=g).to(DEV)
    gates = None if gate == "none" else wide[:, 4:4 + (heads if gate == "head" else heads * n)]
    outs = []
    for shift in (0, 1):
        flat = torch.empty(x.numel() + shift, dtype=dtype, device=DEV)[shift:].view_as(x)
        flat.copy_(x)
        out = torch.empty(rows, heads * n, dtype=dtype, device=DEV)
        ops.gate_heads(flat, stride, gates, out, heads, n)
        outs.append(out)
    assert torch.equal(outs[0], outs[1])


@pytest.mark.parametrize("rows,n", [(1, 4), (37, 2048), (3, 1000), (5, 7)])
def test_row_vector_four_numbers_a_thread(rows, n):
    g = torch.Generator().manual_seed(n)
    x, b = torch.randn(rows, n, generator=g).to(DEV), torch.randn(n, generator=g).to(DEV)
    want = x + b
    ops.add_row_vector(x, b)
    assert torch.equal(x, want)
