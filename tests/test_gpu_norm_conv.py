"""The norm on a sublayer's output with the next layer's input convolution in one kernel, against the two kernels one after the other: the
same bits, at the edges of the rows it takes, for steps that follow each other."""
import pytest
import torch

pytestmark = pytest.mark.gpu

from rocml_amd import ops  # noqa: E402
from rocml_amd.errors import KernelError  # noqa: E402


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows,n,taps,pieces,replace", [(1, 4, 2, 0, False), (5, 2048, 4, 4, True), (3, 1020, 3, 1, False), (64, 1024, 4, 2, True),
                                                        (2, 1028, 2, 9, False), (7, 260, 4, 0, False)])
def test_same_bits_as_both_kernels(rows, n, taps, pieces, replace, dtype):
    g = torch.Generator().manual_seed(rows * 7 + n)
    draw = lambda *s: torch.randn(*s, generator=g).cuda()          # noqa: E731
    x, y, gain, next_gain, w = draw(rows, n), draw(rows, n), draw(n), draw(n), draw(taps, n)
    partials = draw(pieces, rows, n) if pieces else None
    slots = torch.randperm(rows + 3, generator=g)[:rows].int().cuda()
    state = draw(rows + 3, taps - 1, n).to(dtype)
    assert ops.norm_add_conv_fits(n, taps)
    x2, state2, cu = x.clone(), state.clone(), torch.arange(rows + 1, dtype=torch.int32).cuda()
    for _ in range(taps + 1):                       # until every kept row is one of these steps
        args = dict(layer=False, partials=partials, replace=replace, next_gain=next_gain, next_eps=1e-5)
        got, normed, want = (torch.full((rows, n), float("nan"), dtype=dtype, device="cuda") for _ in range(3))
        ops.norm_add(x, y, gain, None, 1e-6, copy=got, conv=(w, state, slots), **args)
        ops.norm_add(x2, y, gain, None, 1e-6, copy=normed, **args)
        ops.added_conv(normed, w, state2, cu, slots, [1] * rows, want)
        assert torch.equal(x, x2) and torch.equal(got, want) and torch.equal(state, state2)


def test_what_it_does_not_take():
    assert not any(ops.norm_add_conv_fits(n, taps) for n, taps in ((2048, 1), (2048, 5), (2052, 4), (1022, 4)))
    x, gain = torch.zeros(2, 64, device="cuda"), torch.ones(64, device="cuda")
    out, slots = torch.empty(2, 64, device="cuda"), torch.zeros(2, dtype=torch.int32, device="cuda")
    for state in (torch.zeros(2, 2, 64, device="cuda"), torch.zeros(2, 3, 64, dtype=torch.bfloat16, device="cuda")):
        with pytest.raises(KernelError):
            ops.norm_add(x, x, gain, None, 1e-6, False, copy=out, next_gain=gain, next_eps=1e-6, conv=(torch.zeros(4, 64, device="cuda"), state, slots))


@pytest.mark.parametrize("n,taps,slots_held", [(100, 4, 3), (1028, 2, 1), (2044, 4, 5)])
def test_kept_rows_of_a_second_line(n, taps, slots_held):
    """The kept rows of a cache's odd lines start 8 bytes off in bfloat16 where a row is 4 values more than a multiple of 8."""
    g = torch.Generator().manual_seed(n)
    draw = lambda *s: torch.randn(*s, generator=g).cuda()          # noqa: E731
    x, y, gain, next_gain, w = draw(1, n), draw(1, n), draw(n), draw(n), draw(taps, n)
    lines = draw(2, slots_held, taps - 1, n).bfloat16()
    slots, cu = torch.tensor([slots_held - 1], dtype=torch.int32).cuda(), torch.tensor([0, 1], dtype=torch.int32).cuda()
    assert lines[1].data_ptr() % 16 == 8
    x2, lines2 = x.clone(), lines.clone()
    got, normed, want = (torch.full((1, n), float("nan"), dtype=torch.bfloat16, device="cuda") for _ in range(3))
    assert ops.norm_add_conv_takes(x, y, gain, got, None, next_gain, w, lines[1])
    for _ in range(taps):
        ops.norm_add(x, y, gain, None, 1e-6, layer=False, next_gain=next_gain, next_eps=1e-5, copy=got, conv=(w, lines[1], slots))
        ops.norm_add(x2, y, gain, None, 1e-6, layer=False, next_gain=next_gain, next_eps=1e-5, copy=normed)
        ops.added_conv(normed, w, lines2[1], cu, slots, [1], want)
        assert torch.equal(x, x2) and torch.equal(got, want) and torch.equal(lines, lines2)


@pytest.mark.parametrize("bound_off", [False, True])
@pytest.mark.parametrize("max_seqs", [1, 3])
def test_models_whose_rows_start_anywhere(tmp_path, max_seqs, bound_off):
    """A width of 100 in bfloat16 (odd lines of kept rows 8 bytes off), and gains that a program bound as parts of larger tensors, which
    the kernel cannot read: one token at a time gives what the whole prompt gives."""
    from rocml_amd.engine import Engine
    from rocml_amd.weights import load_model
    from tests import helpers
    from tests import kakalorn_models as km
    layer = km.hgrn2(2, 16, 24, km.dense(64))
    cfg = km.config(120, 100, 4, [layer, layer, km.attention(2, 1, 32, 0.2, 40, 2, (1000.0, 32), km.dense(48)), layer])
    model = load_model(km.write_model(str(tmp_path), cfg, km.random_tensors(cfg, 5)), dtype="bfloat16", device="cuda:0")
    if bound_off:
        for block in model.blocks:
            for norm in (block.children["mixer_norm"], block.children["mixer_out_norm"]):
                norm.gain = torch.cat([norm.gain[:1], norm.gain])[1:]
                assert norm.gain.data_ptr() % 16 == 4
    engine = Engine(model, max_tokens=512, max_seqs=max_seqs)
    tokens = helpers.random_tokens(24, cfg["vocab"], 9)
    whole, tail = helpers.run_whole(engine, tokens).double(), helpers.run_tail_by_one(engine, tokens, 14).double()
    # (two orders of the recurrences' sums over bfloat16 operands: as tests/test_gpu_kakalorn.py holds its runs against each other)
    errors = (tail - whole).abs().amax(-1) / whole.abs().amax(-1)
    assert float(torch.quantile(errors, 0.9)) < 6e-2, errors
