"""A decode step's latent attention: sequences of up to 16 rows of work (one block a sequence and split), its queries in one launch, its
latents in one trip."""
import pytest
import torch

pytestmark = pytest.mark.gpu

from rocml_amd import ops  # noqa: E402

DEV = "cuda:0"
PAGE = 64


def _i32(v):
    return torch.tensor(v, dtype=torch.int32, device=DEV)


# sequences of one key, of less than a piece of 32, of many pieces beside them (splits without a key), two tokens a sequence; sizes of every
# instantiation, whole tiles and padded ones; few and many splits by the room for partial results
@pytest.mark.parametrize("H,DK,DV", [(16, 576, 512), (5, 96, 64), (16, 48, 40), (3, 192, 128), (7, 320, 256), (1, 568, 504)])
@pytest.mark.parametrize("lens,tokens,window", [([1, 31, 700, 64], 1, None), ([33, 1500], 1, 100), ([5, 90], 2, None), ([2000], 1, 1024)])
@pytest.mark.parametrize("splits", [1, 3, 64])
def test_decode_step_of_unequal_sequences(H, DK, DV, lens, tokens, window, splits):
    if tokens * H > 16:
        pytest.skip("more than 16 rows of work")
    gen = torch.Generator().manual_seed(H + DK + sum(lens))
    n, pages = tokens * len(lens), [(t + PAGE - 1) // PAGE for t in lens]
    perm = torch.randperm(sum(pages) + 2, generator=gen)
    table = torch.full((len(lens), max(pages)), -1, dtype=torch.int32)
    cache = torch.zeros(len(perm), PAGE, DK, dtype=torch.bfloat16)
    q = torch.randn(n, H, DK, generator=gen).to(torch.bfloat16)
    want, at = [], 0
    for b, T in enumerate(lens):
        mine = perm[at:at + pages[b]]
        at += pages[b]
        table[b, :pages[b]] = mine.to(torch.int32)
        k = torch.randn(T, DK, generator=gen).to(torch.bfloat16)
        flat = torch.zeros(pages[b] * PAGE, DK, dtype=torch.bfloat16)
        flat[:T] = k
        cache[mine] = flat.view(-1, PAGE, DK)
        for i in range(tokens):
            pos = T - tokens + i
            lo = 0 if window is None else max(0, pos - window + 1)
            seen = k[lo:pos + 1].double()
            p = torch.softmax(q[b * tokens + i].double() @ seen.T * DK ** -0.5, -1)
            want.append(p @ seen[:, :DV])
    want = torch.stack(want)
    out = torch.full((n, H * DV), float("nan"), dtype=torch.bfloat16, device=DEV)
    ws = torch.full((splits * n * H * (DV + 2) * 4,), 0xff, dtype=torch.uint8, device=DEV)          # NaN where nothing is written
    positions = [T - tokens + i for T in lens for i in range(tokens)]
    ops.attention(q.reshape(n, -1).to(DEV), out, cache.to(DEV).unsqueeze(1), None, table.to(DEV), _i32([b for b in range(len(lens)) for _ in range(tokens)]),
                  _i32(positions), H, 1, DK, DK ** -0.5, window, algo=ops.ATTN_MFMA, workspace=ws,
                  cu_seqlens=_i32([tokens * b for b in range(len(lens) + 1)]), max_new=tokens, q_counts=[tokens] * len(lens), max_len=max(lens),
                  v_head_dim=DV, values_in_keys=True)
    # (probabilities and outputs of 8 bits: 2^-8 of the largest each)
    assert float((out.double().cpu().view(n, H, DV) - want).abs().max()) < 2.0 ** -6 * float(want.abs().max())


@pytest.mark.parametrize("pairing", ["halves", "neighbours"])
@pytest.mark.parametrize("rows,H,N,K,part,dims", [(1, 16, 512, 128, 64, 64), (8, 16, 512, 128, 64, 64), (16, 3, 40, 24, 20, 8), (5, 2, 32, 8, 0, 0)])
def test_latent_queries_are_the_two_kernels(rows, H, N, K, part, dims, pairing):
    g = torch.Generator().manual_seed(rows + N)
    stride, width = K + part, N + part
    q = torch.randn(rows, H * stride, generator=g).to(DEV)
    w = (torch.randn(H, N, K, generator=g) * K ** -0.5).to(DEV, torch.bfloat16)
    angle = torch.rand(rows, dims // 2, generator=g) * 6
    cos, sin = (torch.cos(angle).to(DEV), torch.sin(angle).to(DEV)) if dims else (None, None)
    one, two = (torch.full((rows, H * width), float("nan"), dtype=torch.bfloat16, device=DEV) for _ in range(2))
    ops.latent_queries(q, stride, w, one, width, K, part, dims, cos, sin, pairing=pairing)
    ops.gemm_batched(q, stride, w, two, width)
    if part:
        ops.rope_heads(q, H, stride, K, part, dims, cos, sin, two, width, N, pairing=pairing)
    assert float((one.float() - two.float()).abs().max()) <= 2.0 ** -8 * float(two.float().abs().max())       # (a rounding at most)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("pairing", ["halves", "neighbours"])
@pytest.mark.parametrize("rows,q_rank,kv_rank,part,dims,own", [(3, 768, 512, 64, 64, True), (9, 1024, 1024, 1024, 32, True), (2, 4, 8, 0, 0, True), (5, 100, 36, 12, 8, False)])
def test_latents_in_one_trip_match_the_general_kernel(rows, q_rank, kv_rank, part, dims, own, pairing, dtype):
    g = torch.Generator().manual_seed(q_rank)
    proj = torch.randn(rows, q_rank + kv_rank + part + 8, generator=g).to(DEV)
    gains = [(1 + 0.1 * torch.randn(n, generator=g)).to(DEV) for n in (q_rank, kv_rank)]
    angle = torch.rand(rows, dims // 2, generator=g) * 6
    cos, sin = (torch.cos(angle).to(DEV), torch.sin(angle).to(DEV)) if dims else (None, None)
    table = _i32([[2, -1], [0, 1]])
    seq, pos = _i32([i % 2 for i in range(rows)]), _i32([3 + 40 * (i // 2) for i in range(rows)])
    got = []
    for shift in (0, 1):                                # one number further on no wide load is possible
        flat = torch.empty(proj.numel() + shift, device=DEV)[shift:].view_as(proj)
        flat.copy_(proj)
        cq = torch.zeros(rows, q_rank, dtype=dtype, device=DEV)
        cache = torch.zeros(3, 64, kv_rank + part, dtype=dtype, device=DEV)
        ops.latent_prepare(flat, q_rank, kv_rank, part, dims, gains[0], gains[1], 1e-6, cos, sin, cq, cache, table, seq, pos, write_cache=own, pairing=pairing)
        got.append((cq.float(), cache.float()))
    for a, b in zip(*got):
        assert float((a - b).abs().max()) <= (2.0 ** -7 if dtype == torch.bfloat16 else 2e-6) * max(1.0, float(b.abs().max()))
    assert float(got[0][0].abs().max()) > 0 and (float(got[0][1].abs().max()) > 0) == own
