"""The matrix product kernels alone against a plain 32-bit product of the same operands,
at sizes other than the engine's: sizes that are no multiple of a tile, single rows,
every algorithm and epilogue."""
import pytest
import torch

pytestmark = pytest.mark.gpu

from rocml_amd import ops  # noqa: E402
from rocml_amd.errors import KernelError  # noqa: E402

PLAIN, TILE, SKINNY, KPAR, TILE256, TILE256X192, TILE128X192, TILE256X128, TILE64X128 = 1, 2, 3, 4, 5, 6, 7, 8, 9


def _operands(m, n, k, dtype, seed):
    g = torch.Generator(device="cpu").manual_seed(seed)
    x = torch.randn(m, k, generator=g).to(dtype).cuda()
    w = (torch.randn(n, k, generator=g) * 0.05).to(dtype).cuda()
    return x, w


def _ref(x, w):
    return (x.double() @ w.double().t())


@pytest.mark.parametrize("m,n,k", [(1, 7, 5), (3, 64, 16), (65, 130, 33), (200, 96, 257), (17, 384, 96)])
def test_plain_float32(m, n, k):
    x, w = _operands(m, n, k, torch.float32, 1)
    out = torch.empty(m, n, dtype=torch.float32, device="cuda")
    ops.gemm(x, w, out, algo=PLAIN)
    ref = _ref(x, w)
    assert float((out.double() - ref).abs().max()) < 1e-5 * max(1.0, float(ref.abs().max()))
    base = torch.randn(m, n, device="cuda")
    acc = base.clone()
    ops.gemm(x, w, acc, accumulate=True, algo=PLAIN)
    assert float((acc.double() - (ref + base.double())).abs().max()) < 1e-5 * max(1.0, float(ref.abs().max()))


SHAPES = [(1, 64, 64), (5, 200, 72), (16, 130, 512), (17, 96, 264), (33, 4096, 1024), (48, 1000, 776), (64, 257, 4096),
          (8, 1000, 2056), (128, 128, 64), (129, 300, 200), (300, 515, 72), (2048, 512, 1024),
          (1409, 300, 128), (2561, 200, 64)]       # 12 and 21 tile rows of 128, 6 and 11 of 256: whole bands of eight and a rest


@pytest.mark.parametrize("algo", [PLAIN, TILE, SKINNY, KPAR, TILE256, TILE256X192, TILE128X192, TILE256X128, TILE64X128])
@pytest.mark.parametrize("m,n,k", SHAPES)
def test_bfloat16_algorithms(m, n, k, algo):
    if (algo == SKINNY and m > 64) or (algo == KPAR and m > 16):
        pytest.skip("the few-rows kernels take at most 64 and 16 rows")
    x, w = _operands(m, n, k, torch.bfloat16, 2)
    ref = _ref(x, w)
    scale = max(1.0, float(ref.abs().max()))
    ws = torch.empty(64 << 20, dtype=torch.uint8, device="cuda")
    out = torch.full((m, n), float("nan"), dtype=torch.float32, device="cuda")
    ops.gemm(x, w, out, algo=algo, workspace=ws)
    assert float((out.double() - ref).abs().max()) < 2e-5 * scale, "32-bit output"
    out16 = torch.empty(m, n, dtype=torch.bfloat16, device="cuda")
    ops.gemm(x, w, out16, algo=algo, workspace=ws)
    assert float((out16.double() - ref).abs().max()) < 5e-3 * scale, "bfloat16 output"
    base = torch.randn(m, n, device="cuda")
    acc = base.clone()
    ops.gemm(x, w, acc, accumulate=True, algo=algo, workspace=ws)
    assert float((acc.double() - (ref + base.double())).abs().max()) < 2e-5 * scale, "accumulating"


# one chunk of 256 a wave, one and a rest, K in pieces of 1024 with a rest; N that is no tile; rows to either side of the rule's limits
@pytest.mark.parametrize("m,n,k", [(1, 40, 8), (3, 1000, 1024), (8, 2047, 1032), (9, 2048, 2048), (16, 520, 3080), (8, 4096, 2048), (2, 70, 264),
                                   (1, 1536, 4096), (2, 1552, 4096), (1, 4096, 3072), (2, 4112, 4096),
                                   (1, 8208, 3080), (12, 4112, 640), (16, 2560, 1408), (4, 4112, 1280), (3, 4112, 256), (8, 4112, 1800)])
def test_few_rows_in_one_trip(m, n, k):
    """The operands are column ranges of wider matrices that hold NaN beside them; whole sums, deferred pieces and the gated
    activation, by the library's own choice of kernel."""
    x, w = _operands(m, n, k, torch.bfloat16, 9)
    wide_x, wide_w = torch.full((m, k + 16), float("nan"), dtype=torch.bfloat16, device="cuda"), torch.full(
        (n, k + 8), float("nan"), dtype=torch.bfloat16, device="cuda")
    wide_x[:, 8:8 + k], wide_w[:, :k] = x, w
    x, w = wide_x[:, 8:8 + k], wide_w[:, :k]
    ref = _ref(x, w)
    scale = max(1.0, float(ref.abs().max()))
    ws = torch.empty(16 << 20, dtype=torch.uint8, device="cuda")
    for defer in (False, True):
        acc = torch.ones(m, n, device="cuda")
        pieces = ops.gemm(x, w, acc, accumulate=True, workspace=ws, defer=defer)
        if pieces:
            acc += ws[:pieces * m * n * 4].view(torch.float32).view(pieces, m, n).sum(0)
        assert float((acc.double() - 1 - ref).abs().max()) < 2e-5 * scale, (defer, pieces)
    if n % 2 == 0:
        h = torch.empty(m, n // 2, dtype=torch.bfloat16, device="cuda")
        ops.gemm(x, w, h, workspace=ws, epilogue="swiglu")
        want = torch.nn.functional.silu(ref[:, 0::2]) * ref[:, 1::2]
        assert float((h.double() - want).abs().max()) < 5e-3 * max(1.0, float(want.abs().max()))


# rows around 16 and 32 (the few-rows kernel's tiles) and beyond; K of a run of 64, less, and runs with a rest; N that is no tile;
# products cut along K (narrow, deep) and whole
@pytest.mark.parametrize("m,n,k", [(1, 5, 4), (2, 384, 96), (16, 300, 1028), (17, 51, 640), (32, 4112, 260), (33, 70, 68), (64, 64, 32),
                                   (130, 1000, 4100), (700, 130, 2052), (5, 20000, 64), (3, 100, 2052), (20, 1024, 3076)])
def test_float32_matrix_cores(m, n, k):
    x, w = _operands(m, n, k, torch.float32, 5)
    wide = torch.full((m, k + 8), float("nan"), device="cuda")
    wide[:, 4:4 + k] = x
    ref = _ref(x, w)
    scale = max(1.0, float(ref.abs().max()))
    ws = torch.empty(64 << 20, dtype=torch.uint8, device="cuda")
    out = torch.full((m, n), float("nan"), device="cuda")
    ops.gemm(wide[:, 4:4 + k], w, out, workspace=ws)
    assert float((out.double() - ref).abs().max()) < 1e-5 * scale
    base = torch.randn(m, n, device="cuda")
    acc = base.clone()
    ops.gemm(x, w, acc, accumulate=True, workspace=ws)
    assert float((acc.double() - (ref + base.double())).abs().max()) < 1e-5 * scale
    acc = base.clone()
    pieces = ops.gemm(x, w, acc, accumulate=True, workspace=ws, defer=True)
    if pieces:
        acc += ws[:pieces * m * n * 4].view(torch.float32).view(pieces, m, n).sum(0)
    assert float((acc.double() - (ref + base.double())).abs().max()) < 1e-5 * scale, pieces
    if n % 2 == 0:
        for epilogue, act in (("swiglu", torch.nn.functional.silu), ("relu_glu", torch.relu)):
            h = torch.full((m, n // 2), float("nan"), device="cuda")
            ops.gemm(x, w, h, workspace=ws, epilogue=epilogue)
            want = act(ref[:, 0::2]) * ref[:, 1::2]
            assert float((h.double() - want).abs().max()) < 2e-5 * max(1.0, float(want.abs().max())), epilogue


@pytest.mark.parametrize("m,n,k", [(4200, 4400, 72), (4100, 4609, 8), (2305, 8200, 200)])
@pytest.mark.parametrize("epilogue", [None, "swiglu", "relu2"])
def test_more_tiles_than_compute_units(m, n, k, epilogue):
    """256x256 tiles of which a block walks through several (306, 323 and 330 of them), the rest of K not a whole stage; the
    operands are column ranges of wider matrices that hold NaN beside them."""
    n -= n % 2 if epilogue == "swiglu" else 0
    x, w = _operands(m, n, k, torch.bfloat16, 7)
    wide_x, wide_w = torch.full((m, k + 64), float("nan"), dtype=torch.bfloat16, device="cuda"), torch.full(
        (n, k + 72), float("nan"), dtype=torch.bfloat16, device="cuda")
    wide_x[:, 8:8 + k], wide_w[:, 16:16 + k] = x, w
    ref = _ref(x, w)
    if epilogue == "swiglu":
        ref = torch.nn.functional.silu(ref[:, 0::2]) * ref[:, 1::2]
    elif epilogue == "relu2":
        ref = ref.clamp(min=0) ** 2
    out = torch.empty(ref.shape, dtype=torch.float32 if epilogue is None else torch.bfloat16, device="cuda")
    ops.gemm(wide_x[:, 8:8 + k], wide_w[:, 16:16 + k], out, algo=TILE256, epilogue=epilogue)
    # 32-bit sums of at most 200 products; a bfloat16 result is rounded to 8 bits
    assert float((out.double() - ref).abs().max()) < (2e-5 if epilogue is None else 5e-3) * max(1.0, float(ref.abs().max()))


@pytest.mark.parametrize("m,n,k", [(4200, 4400, 72), (4100, 4609, 200)])
def test_more_tiles_than_compute_units_into_the_stream(m, n, k):
    """The same with the sums added to what is there, which reads memory while the next tile's operands are on their way, and
    with a plain bfloat16 result."""
    x, w = _operands(m, n, k, torch.bfloat16, 7)
    ref = _ref(x, w)
    base = torch.randn(m, n, device="cuda")
    acc = base.clone()
    ops.gemm(x, w, acc, accumulate=True, algo=TILE256)
    assert float((acc.double() - (ref + base.double())).abs().max()) < 2e-5 * max(1.0, float(ref.abs().max()))
    out16 = torch.empty(m, n, dtype=torch.bfloat16, device="cuda")
    ops.gemm(x, w, out16, algo=TILE256)
    assert float((out16.double() - ref).abs().max()) < 5e-3 * max(1.0, float(ref.abs().max()))


def test_strided_rows_and_refusals():
    from rocml_amd.errors import KernelError
    big = torch.randn(40, 200, device="cuda").to(torch.bfloat16)
    x = big[:, 8:72]                       # row stride 200, 64 columns
    w = (torch.randn(48, 64, device="cuda") * 0.1).to(torch.bfloat16)
    out = torch.empty(40, 48, dtype=torch.float32, device="cuda")
    ops.gemm(x, w, out)
    assert float((out.double() - _ref(x, w)).abs().max()) < 1e-4
    odd = torch.randn(4, 36, device="cuda").to(torch.bfloat16)   # K = 36 is no multiple of 8
    w2 = torch.randn(8, 36, device="cuda").to(torch.bfloat16)
    out2 = torch.empty(4, 8, dtype=torch.float32, device="cuda")
    ops.gemm(odd, w2, out2)                # falls back to the plain kernel
    assert float((out2.double() - _ref(odd, w2)).abs().max()) < 1e-3
    with pytest.raises(KernelError):
        ops.gemm(odd, w2, out2, algo=TILE)
    with pytest.raises(KernelError):
        ops.gemm(x.cpu(), w, out)


@pytest.fixture(scope="module")
def sixteen_far_rows():
    """Room for 16 rows that lie 2^27 numbers apart, more than 31 bits of bytes in all."""
    return torch.empty(15 * (1 << 27) + 4096, dtype=torch.bfloat16, device="cuda")


def _far(t, room):
    wide = room[:(t.shape[0] - 1) * (1 << 27) + t.shape[1]].as_strided(t.shape, (1 << 27, 1))
    wide.copy_(t)
    return wide


@pytest.mark.parametrize("m,n,k,which", [(16, 40, 264, "x"), (3, 16, 1032, "w"), (9, 70, 64, "x"), (1, 13, 3080, "w")])
def test_few_rows_far_apart(m, n, k, which, sixteen_far_rows):
    """The K-parallel kernel with operand rows beyond each other's 31-bit reach: whole sums, K pieces, the gated activation."""
    x, w = _operands(m, n, k, torch.bfloat16, 14)
    ref = _ref(x, w)
    tol = 2e-5 * max(1.0, float(ref.abs().max()))
    if which == "x":
        x = _far(x, sixteen_far_rows)
    else:
        w = _far(w, sixteen_far_rows)
    ws = torch.empty(1 << 20, dtype=torch.uint8, device="cuda")
    for algo in ([0, KPAR] if which == "x" else [KPAR]):
        out = torch.full((m, n), float("nan"), device="cuda")
        ops.gemm(x, w, out, algo=algo, workspace=ws)
        assert float((out.double() - ref).abs().max()) < tol
        pieces = ops.gemm(x, w, out, algo=algo, workspace=ws, defer=True)
        got = ws[:pieces * m * n * 4].view(torch.float32).view(pieces, m, n).sum(0) if pieces else out
        assert float((got.double() - ref).abs().max()) < tol, pieces
    if n % 2 == 0:
        h = torch.empty(m, n // 2, dtype=torch.bfloat16, device="cuda")
        ops.gemm(x, w, h, algo=KPAR, workspace=ws, epilogue="swiglu")
        want = torch.nn.functional.silu(ref[:, 0::2]) * ref[:, 1::2]
        assert float((h.double() - want).abs().max()) < 5e-3 * max(1.0, float(want.abs().max()))


@pytest.mark.parametrize("algo", [PLAIN, TILE, SKINNY, KPAR, TILE256, TILE256X192, TILE128X192, TILE256X128, TILE64X128])
@pytest.mark.parametrize("m,n,k", [(1, 64, 64), (7, 448, 96), (25, 300, 520), (41, 130, 1032), (64, 1000, 264), (130, 256, 128), (300, 2048, 512)])
def test_gated_epilogue(m, n, k, algo):
    """Rows of the weight are (gate, up) pairs; the output is silu(gate) * up, formed from
    the 32-bit sums."""
    if (algo == SKINNY and m > 64) or (algo == KPAR and m > 16):
        pytest.skip("the few-rows kernels take at most 64 and 16 rows")
    x, w = _operands(m, n, k, torch.bfloat16, 3)
    full = _ref(x, w)
    gate, up = full[:, 0::2], full[:, 1::2]
    ref = gate / (1 + torch.exp(-gate)) * up
    ws = torch.empty(16 << 20, dtype=torch.uint8, device="cuda")
    out = torch.empty(m, n // 2, dtype=torch.bfloat16, device="cuda")
    ops.gemm(x, w, out, algo=algo, workspace=ws, epilogue="swiglu")
    assert float((out.double().cpu() - ref.cpu()).abs().max()) < 5e-3 * max(1.0, float(ref.abs().max()))
    if algo == PLAIN:
        x32, w32 = x.float(), w.float()
        out32 = torch.empty(m, n // 2, dtype=torch.float32, device="cuda")
        ops.gemm(x32, w32, out32, workspace=ws, epilogue="swiglu")
        assert float((out32.double().cpu() - ref.cpu()).abs().max()) < 2e-5 * max(1.0, float(ref.abs().max()))


@pytest.mark.parametrize("m,n,k,algo", [(1, 64, 64, PLAIN), (25, 300, 520, PLAIN), (130, 256, 30, 0), (7, 70, 33, 0)])
def test_float32_gated_by_the_plain_kernel(m, n, k, algo):
    """Asked for by number, and where K is no multiple of 4."""
    x, w = _operands(m, n, k, torch.float32, 3)
    full = _ref(x, w)
    ws = torch.empty(1 << 20, dtype=torch.uint8, device="cuda")
    for epilogue, act in (("swiglu", torch.nn.functional.silu), ("relu_glu", torch.relu)):
        out = torch.empty(m, n // 2, device="cuda")
        ops.gemm(x, w, out, algo=algo, workspace=ws, epilogue=epilogue)
        ref = act(full[:, 0::2]) * full[:, 1::2]
        assert float((out.double() - ref).abs().max()) < 2e-5 * max(1.0, float(ref.abs().max())), epilogue


@pytest.mark.parametrize("m,algo", [(1, KPAR), (8, SKINNY), (40, SKINNY), (130, TILE), (130, TILE64X128), (130, TILE256X192), (300, TILE256)])
def test_gated_results_are_the_exact_ones_rounded_once(m, algo):
    """silu(gate) * up over the whole range in which exp(-gate) is finite, formed in 32-bit: the stored bfloat16 is the rounding of
    a number within four units in the last place (exponential, sum, division and product) of the exact one."""
    half = 1 << 16
    g = torch.Generator().manual_seed(31)
    gate = torch.rand(half, generator=g) * 118 - 88              # [-88, 30)
    parts, rest = [], gate
    for _ in range(3):                                           # a 32-bit number is the sum of three of 8 bits
        parts.append(rest.bfloat16())
        rest = rest - parts[-1].float()
    assert not rest.any()
    w = torch.zeros(half, 2, 8, dtype=torch.bfloat16)
    w[:, 0, :3] = torch.stack(parts, -1)
    w[:, 1, 3] = 2.0 ** 60                                       # (what a gate of -88 leaves of it is an ordinary number)
    x = torch.zeros(m, 8, dtype=torch.bfloat16)
    x[:, :4] = 1.0
    out = torch.empty(m, half, dtype=torch.bfloat16, device="cuda")
    ops.gemm(x.cuda(), w.view(2 * half, 8).cuda(), out, algo=algo, epilogue="swiglu")
    exact = gate.double() / (1 + torch.exp(-gate.double())) * 2.0 ** 60
    exact = exact.cuda()
    step = torch.exp2(torch.floor(torch.log2(exact.abs().clamp_min(1e-300))) - 8)      # half a bfloat16 step
    off = (out.double() - exact).abs() - step - 4 * 2.0 ** -23 * exact.abs()
    assert float((off / exact.abs().clamp_min(1e-300)).max()) <= 0


def test_deferred_split_sums():
    """A product split along K may leave its partial sums to the caller; adding them in split
    order gives the product."""
    x, w = _operands(8, 256, 4096, torch.bfloat16, 4)
    ref = _ref(x, w)
    ws = torch.empty(16 << 20, dtype=torch.uint8, device="cuda")
    base = torch.randn(8, 256, device="cuda")
    out = base.clone()
    splits = ops.gemm(x, w, out, accumulate=True, workspace=ws, defer=True)
    assert splits > 1 and torch.equal(out, base)              # nothing was added yet
    partials = ws[:splits * 8 * 256 * 4].view(torch.float32).view(splits, 8, 256)
    assert float((partials.double().sum(0) - ref).abs().max()) < 2e-5 * float(ref.abs().max())
    ops.splitk_reduce(partials, out, accumulate=True)
    assert float((out.double() - (ref + base.double())).abs().max()) < 2e-5 * float(ref.abs().max())
    assert ops.gemm(x, w, out, workspace=None, defer=True) == 0   # no workspace: no split, complete result
    assert float((out.double() - ref).abs().max()) < 2e-5 * float(ref.abs().max())


@pytest.mark.parametrize("m,n,k", [(512, 768, 4096), (300, 515, 2056), (1000, 256, 2048), (100, 384, 1544)])
def test_many_rows_with_k_cut_in_pieces(m, n, k):
    """Few tiles and a long K: the tile kernel gives each piece of K to a block of its own and
    adds the pieces in order, or leaves them to the caller."""
    x, w = _operands(m, n, k, torch.bfloat16, 5)
    ref = _ref(x, w)
    scale = max(1.0, float(ref.abs().max()))
    ws = torch.empty(32 << 20, dtype=torch.uint8, device="cuda")
    out = torch.full((m, n), float("nan"), dtype=torch.float32, device="cuda")
    assert ops.gemm(x, w, out, workspace=ws) == 0
    assert float((out.double() - ref).abs().max()) < 2e-5 * scale
    base = torch.randn(m, n, device="cuda")
    acc = base.clone()
    splits = ops.gemm(x, w, acc, accumulate=True, workspace=ws, defer=True)
    assert 2 <= splits <= 8 and torch.equal(acc, base)
    partials = ws[:splits * m * n * 4].view(torch.float32).view(splits, m, n)
    ops.splitk_reduce(partials, acc, accumulate=True)
    assert float((acc.double() - (ref + base.double())).abs().max()) < 2e-5 * scale
    # without room for the pieces the product is done in one
    small = torch.empty(m * n * 4, dtype=torch.uint8, device="cuda")
    out16 = torch.empty(m, n, dtype=torch.bfloat16, device="cuda")
    assert ops.gemm(x, w, out16, workspace=small, defer=True) == 0
    assert float((out16.double() - ref).abs().max()) < 5e-3 * scale


# sizes at which the library cuts K and takes 256x256 tiles, with remainders in M, N and K and a short last piece; the last has
# more tiles and pieces than compute units, so that a block goes from one K piece to another
@pytest.mark.parametrize("m,n,k,pieces", [(1051, 2749, 5320, 4), (402, 4046, 9328, 7), (546, 3295, 7280, 6), (1309, 5576, 8816, 3)])
def test_256x256_tiles_with_k_cut_in_pieces(m, n, k, pieces):
    """Every piece holds the sums of its own range of K, the same bits as that range's product alone; added they are the product.
    The operands are column ranges of wider matrices that hold NaN beside them."""
    x, w = _operands(m, n, k, torch.bfloat16, 8)
    wide_x, wide_w = torch.full((m, k + 64), float("nan"), dtype=torch.bfloat16, device="cuda"), torch.full(
        (n, k + 72), float("nan"), dtype=torch.bfloat16, device="cuda")
    wide_x[:, 8:8 + k], wide_w[:, 16:16 + k] = x, w
    x, w = wide_x[:, 8:8 + k], wide_w[:, 16:16 + k]
    ref = _ref(x, w)
    scale = max(1.0, float(ref.abs().max()))
    ws = torch.full((pieces * m * n,), float("nan"), device="cuda")
    base = torch.randn(m, n, device="cuda")
    acc = base.clone()
    assert ops.gemm(x, w, acc, accumulate=True, workspace=ws, defer=True) == pieces and torch.equal(acc, base)
    step = (-(-k // pieces) + 63) // 64 * 64
    alone = torch.empty(m, n, device="cuda")
    for p, sums in enumerate(ws.view(pieces, m, n)):
        ops.gemm(x[:, p * step:(p + 1) * step], w[:, p * step:(p + 1) * step], alone, algo=TILE256)
        assert torch.equal(sums, alone), p
    ops.splitk_reduce(ws.view(pieces, m, n), acc, accumulate=True)
    whole = base.clone()
    assert ops.gemm(x, w, whole, accumulate=True, workspace=ws) == 0
    assert torch.equal(whole, acc)
    assert float((acc.double() - (ref + base.double())).abs().max()) < 2e-5 * scale
    out16 = torch.empty(m, n, dtype=torch.bfloat16, device="cuda")
    ops.gemm(x, w, out16, workspace=ws)
    assert float((out16.double() - ref).abs().max()) < 5e-3 * scale


@pytest.mark.parametrize("waves", [0, 4, 8, 12, 16])
@pytest.mark.parametrize("m,n,k", [(1, 64, 64), (3, 100, 72), (8, 4096, 1032), (16, 130, 4096), (7, 515, 264), (2, 88, 12288)])
def test_residual_sum_that_prepares_the_next_norm(m, n, k, waves):
    """resid += x W^T with whole sums, xg = bfloat16(resid * gain), and per 16 columns the sum of
    squares of the new residual row, from which the consumer forms the norm's scale."""
    x, w = _operands(m, n, k, torch.bfloat16, 5)
    g = torch.Generator().manual_seed(6)
    base = torch.randn(m, n, generator=g)
    gain = 1 + 0.2 * torch.randn(n, generator=g)
    resid = base.cuda()
    xg = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device="cuda")
    tiles = (n + ops.PRESCALE_TILE - 1) // ops.PRESCALE_TILE
    ssq = torch.full((m, tiles), float("nan"), device="cuda")
    assert ops.gemm_residual_prescale_fits(x, w)
    ops.gemm_residual_prescale(x, w, resid, gain.cuda(), xg, ssq, waves=waves)
    want = base.double() + _ref(x, w).cpu()
    scale = max(1.0, float(want.abs().max()))
    assert float((resid.double().cpu() - want).abs().max()) < 2e-5 * scale
    assert float((xg.double().cpu() - want * gain.double()).abs().max()) < 5e-3 * float((want * gain.double()).abs().max())
    padded = torch.zeros(m, tiles * 16, dtype=torch.float64)
    padded[:, :n] = want ** 2
    assert float((ssq.double().cpu() - padded.view(m, tiles, 16).sum(-1)).abs().max()) < 1e-5 * float(padded.max()) * 16
    # the norm's output, put together the way a consumer does
    eps = 1e-5
    inv = 1.0 / torch.sqrt(ssq.double().cpu().sum(-1, keepdim=True) / n + eps)
    normed = want / torch.sqrt((want ** 2).mean(-1, keepdim=True) + eps) * gain.double()
    assert float((xg.double().cpu() * inv - normed).abs().max()) < 5e-3 * float(normed.abs().max())
    with pytest.raises(KernelError):
        ops.gemm_residual_prescale(torch.zeros(17, k, dtype=torch.bfloat16, device="cuda"), w,
                                   torch.zeros(17, n, device="cuda"), gain.cuda(),
                                   torch.zeros(17, n, dtype=torch.bfloat16, device="cuda"), torch.zeros(17, tiles, device="cuda"))


@pytest.mark.parametrize("m,n,k", [(1, 64, 64), (3, 102, 72), (8, 4096, 1032), (16, 130, 4096)])
def test_residual_sum_with_a_bias(m, n, k):
    """The bias is added to the stream in 32 bits before the product's sums: rows and columns in whole tiles and not (the
    element-by-element end), against the sum in 64 bits."""
    x, w = _operands(m, n, k, torch.bfloat16, 7)
    g = torch.Generator().manual_seed(8)
    base, bias = torch.randn(m, n, generator=g), torch.randn(n, generator=g)
    gain = 1 + 0.2 * torch.randn(n, generator=g)
    resid = base.cuda()
    xg = torch.empty(m, n, dtype=torch.bfloat16, device="cuda")
    ssq = torch.empty(m, (n + 15) // 16, device="cuda")
    ops.gemm_residual_prescale(x, w, resid, gain.cuda(), xg, ssq, bias=bias.cuda())
    want = base.double() + bias.double() + _ref(x, w).cpu()
    assert float((resid.double().cpu() - want).abs().max()) < 2e-5 * max(1.0, float(want.abs().max()))
    assert float((ssq.double().sum(-1).cpu() - (want ** 2).sum(-1)).abs().max()) < 1e-5 * float((want ** 2).sum(-1).max())
    with pytest.raises(KernelError):
        ops.gemm_residual_prescale(x, w, resid, gain.cuda(), xg, ssq, bias=torch.zeros(n + 1, device="cuda"))


@pytest.mark.parametrize("m,n,k,pays", [(1, 2048, 4096, True), (4, 2048, 6144, True), (1, 2048, 6152, False), (4, 2560, 8192, False),
                                        (4, 3072, 8192, True), (5, 3072, 8192, False), (8, 4096, 12288, True), (1, 4112, 4096, False)])
def test_when_the_prepared_norm_pays(m, n, k, pays):
    """The rule's lines for 256 compute units, from both ways' measured times."""
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the lines are those of 256 compute units")
    x, w = torch.empty(m, k, dtype=torch.bfloat16, device="cuda"), torch.empty(n, k, dtype=torch.bfloat16, device="cuda")
    assert ops.gemm_residual_prescale_pays(x, w) == pays


@pytest.mark.parametrize("m,n,k,which", [(16, 40, 264, "x"), (3, 16, 1032, "w"), (11, 130, 4096, "x")])
def test_residual_sum_of_rows_far_apart(m, n, k, which, sixteen_far_rows):
    """The same with operand rows beyond each other's 31-bit reach."""
    x, w = _operands(m, n, k, torch.bfloat16, 15)
    want = 1.0 + _ref(x, w)
    if which == "x":
        x = _far(x, sixteen_far_rows)
    else:
        w = _far(w, sixteen_far_rows)
    tiles = (n + 15) // 16
    resid, gain = torch.ones(m, n, device="cuda"), torch.linspace(0.5, 1.5, n, device="cuda")
    xg, ssq = torch.empty(m, n, dtype=torch.bfloat16, device="cuda"), torch.empty(m, tiles, device="cuda")
    for waves in (0, 8):
        resid.fill_(1.0)
        ops.gemm_residual_prescale(x, w, resid, gain, xg, ssq, waves=waves)
        assert float((resid.double() - want).abs().max()) < 2e-5 * max(1.0, float(want.abs().max()))
        assert float((xg.double() - want * gain.double()).abs().max()) < 5e-3 * float((want * gain.double()).abs().max())
        squares = torch.nn.functional.pad(want ** 2, (0, tiles * 16 - n)).view(m, tiles, 16).sum(-1)
        assert float((ssq.double() - squares).abs().max()) < 1e-4 * float(squares.max())


@pytest.mark.parametrize("algo", [0, SKINNY, KPAR])
@pytest.mark.parametrize("m,n,k,parts", [(1, 64, 64, 4), (2, 24576, 4096, 256), (8, 448, 96, 6), (16, 1000, 264, 17), (13, 300, 1032, 64)])
def test_gated_epilogue_applies_a_row_scale(m, n, k, parts, algo):
    """The operand lacks its norm's scale; the gated epilogue multiplies the sums of a row by
    1 / sqrt(sum of the row's parts / K + eps) before the activation."""
    x, w = _operands(m, n, k, torch.bfloat16, 7)
    g = torch.Generator().manual_seed(8)
    ssq = (torch.rand(m, parts, generator=g) * 3 * k / parts).cuda()
    eps = 1e-5
    inv = 1.0 / torch.sqrt(ssq.double().sum(-1, keepdim=True) / k + eps)
    full = _ref(x, w) * inv
    gate, up = full[:, 0::2], full[:, 1::2]
    ref = gate / (1 + torch.exp(-gate)) * up
    ws = torch.empty(16 << 20, dtype=torch.uint8, device="cuda")
    out = torch.empty(m, n // 2, dtype=torch.bfloat16, device="cuda")
    ops.gemm(x, w, out, algo=algo, workspace=ws, epilogue="swiglu", row_scale=ops.RowScale(ssq, eps, k))
    assert float((out.double() - ref).abs().max()) < 5e-3 * max(1.0, float(ref.abs().max()))
    with pytest.raises(KernelError):                       # not without the gated epilogue, not for more rows
        ops.gemm(x, w, torch.empty(m, n, device="cuda"), workspace=ws, row_scale=ops.RowScale(ssq, eps, k))
    with pytest.raises(KernelError):
        ops.gemm(torch.zeros(17, k, dtype=torch.bfloat16, device="cuda"), w, torch.empty(17, n // 2, dtype=torch.bfloat16, device="cuda"),
                 workspace=ws, epilogue="swiglu", row_scale=ops.RowScale(torch.ones(17, parts, device="cuda"), eps, k))


@pytest.mark.parametrize("m", [3, 16, 20, 40, 64])
@pytest.mark.parametrize("n,k", [(34816, 264), (51200, 512), (65568, 256), (90, 2056)])
def test_wide_gated_products_take_blocks_of_many_waves(m, n, k):
    """The gated product runs on blocks of as many waves as make one round over the chip: nine at
    34816 columns, thirteen (sixteen at 49 to 64 rows) at 51200, and beyond one round of sixteen
    waves the count that leaves the busiest CU the fewest columns; with and without a row scale."""
    x, w = _operands(m, n, k, torch.bfloat16, 11)
    full = _ref(x, w)
    ws = torch.empty(16 << 20, dtype=torch.uint8, device="cuda")
    out = torch.empty(m, n // 2, dtype=torch.bfloat16, device="cuda")
    for scaled in (False, True):
        if scaled and m > ops.ROW_SCALE_MAX_ROWS:
            continue
        inv = 1.0
        scale = None
        if scaled:
            ssq = (torch.rand(m, 5, generator=torch.Generator().manual_seed(12)) * k).cuda()
            inv = 1.0 / torch.sqrt(ssq.double().sum(-1, keepdim=True) / k + 1e-6)
            scale = ops.RowScale(ssq, 1e-6, k)
        gate, up = (full * inv)[:, 0::2], (full * inv)[:, 1::2]
        ref = gate / (1 + torch.exp(-gate)) * up
        out.fill_(float("nan"))
        ops.gemm(x, w, out, workspace=ws, epilogue="swiglu", row_scale=scale)
        assert float((out.double() - ref).abs().max()) < 5e-3 * max(1.0, float(ref.abs().max()))


@pytest.mark.parametrize("m", [5, 16, 24, 32])
@pytest.mark.parametrize("n,k", [(6144, 4096), (7168, 5120), (5120, 5120), (1000, 3080), (4096, 4096)])
def test_few_rows_products_with_chosen_blocks(m, n, k):
    """A product cut along K whose waves a block and K pieces are chosen for the busiest CU (six
    waves and four pieces at 6144 x 4096, seven at 7168 x 5120, five at 5120 x 5120), complete or
    with its partial sums left to the caller."""
    x, w = _operands(m, n, k, torch.bfloat16, 13)
    ref = _ref(x, w)
    tol = 2e-5 * max(1.0, float(ref.abs().max()))
    ws = torch.empty(32 << 20, dtype=torch.uint8, device="cuda")
    base = torch.randn(m, n, device="cuda")
    out = base.clone()
    ops.gemm(x, w, out, accumulate=True, workspace=ws)
    assert float((out.double() - (ref + base.double())).abs().max()) < tol
    splits = ops.gemm(x, w, out, workspace=ws, defer=True)
    if splits:
        partials = ws[:splits * m * n * 4].view(torch.float32).view(splits, m, n)
        assert float((partials.double().sum(0) - ref).abs().max()) < tol
    else:
        assert float((out.double() - ref).abs().max()) < tol


# tiles of the ring kernel (rows x columns) by the algorithm that asks for them
RING = {TILE: (128, 128), TILE128X192: (128, 192), TILE256X128: (256, 128), TILE64X128: (64, 128), 10: (64, 64), 11: (128, 64), 12: (128, 256)}


@pytest.mark.parametrize("algo", sorted(RING))
@pytest.mark.parametrize("k", [8, 64, 72, 192, 392, 904])       # less than a stage, whole ones, a rest; fewer stages than the ring and more
@pytest.mark.parametrize("dm,dn", [(-1, 1), (0, 0), (1, -1)])
def test_ring_tiles(algo, k, dm, dn):
    """Around one tile and two, of operands with NaN beside them: whole sums and the gated activation."""
    m, n = RING[algo][0] + dm, 2 * RING[algo][1] + 2 * dn
    x, w = _operands(m, n, k, torch.bfloat16, 11)
    wide_x, wide_w = torch.full((m, k + 16), float("nan"), dtype=torch.bfloat16, device="cuda"), torch.full(
        (n, k + 8), float("nan"), dtype=torch.bfloat16, device="cuda")
    wide_x[:, 8:8 + k], wide_w[:, :k] = x, w
    x, w = wide_x[:, 8:8 + k], wide_w[:, :k]
    ref = _ref(x, w)
    out = torch.full((m, n), float("nan"), device="cuda")
    ops.gemm(x, w, out, algo=algo)
    assert float((out.double() - ref).abs().max()) < 2e-5 * max(1.0, float(ref.abs().max()))
    h = torch.empty(m, n // 2, dtype=torch.bfloat16, device="cuda")
    ops.gemm(x, w, h, algo=algo, epilogue="swiglu")
    want = torch.nn.functional.silu(ref[:, 0::2]) * ref[:, 1::2]
    assert float((h.double() - want).abs().max()) < 5e-3 * max(1.0, float(want.abs().max()))


# runs of 512 of K and a rest, with and without pieces; both 32-bit tiles
@pytest.mark.parametrize("m,n,k", [(33, 64, 508), (65, 130, 512), (200, 4100, 1028), (64, 6144, 1540), (574, 1024, 3072), (1000, 2048, 520)])
def test_float32_sums_in_runs(m, n, k):
    x, w = _operands(m, n, k, torch.float32, 12)
    ref = _ref(x, w)
    out = torch.full((m, n), float("nan"), device="cuda")
    ops.gemm(x, w, out)
    # a run's 512 products are added up with an error of a few times sqrt(512) * 2^-24 of their size at most: 2e-6 of the largest sum
    assert float((out.double() - ref).abs().max()) < 2e-6 * max(1.0, float(ref.abs().max()))
    ws = torch.empty(64 << 20, dtype=torch.uint8, device="cuda")
    acc = torch.zeros(m, n, device="cuda")
    pieces = ops.gemm(x, w, acc, accumulate=True, workspace=ws, defer=True)
    if pieces:
        acc += ws[:pieces * m * n * 4].view(torch.float32).view(pieces, m, n).sum(0)
    assert float((acc.double() - ref).abs().max()) < 2e-6 * max(1.0, float(ref.abs().max())), pieces
