"""The row norm's variants: widths at the edges of a thread's vectors, few rows and many, K pieces at the edges of a group of loads."""
import pytest
import torch

from rocml_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [4, 1024, 1028, 2048, 2052, 3072, 3076, 4096, 4100, 5120, 5124, 8192])
@pytest.mark.parametrize("rows", [1, 512, 513])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_rows_and_pieces(n, rows, dtype):
    g = torch.Generator().manual_seed(n + rows)
    x = torch.randn(rows, n, generator=g)
    gain = torch.randn(n, generator=g)
    for splits in (0, 1, 2, 3, 4, 5, 8, 9):
        p = torch.randn(splits, rows, n, generator=g) if splits else None
        got_x, out = x.cuda(), torch.empty(rows, n, dtype=dtype, device="cuda")
        ops.rmsnorm(got_x, gain.cuda(), 1e-6, out, None, partials=None if p is None else p.cuda())
        want_x = x.clone()                                      # in the order of the pieces, in 32-bit: the same bits
        for i in range(splits):
            want_x += p[i]
        assert torch.equal(got_x.cpu(), want_x), splits
        wide = want_x.double()
        want = wide / (wide.square().mean(-1, keepdim=True) + 1e-6).sqrt() * gain.double()
        # a sum of squares of positive terms in a chain of at most 32 values a thread, 6 lanes and 16 waves is off by at most
        # 54 roundings, its root by half of that; the factor and the two products add 5; a bfloat16 result (8 bits) rounds by at most 2^-8
        bound = (27 + 5) * 2.0 ** -24 + (2.0 ** -8 if dtype == torch.bfloat16 else 0.0)
        assert ((out.cpu().double() - want).abs() <= bound * want.abs() + 1e-30).all(), splits
        picks = torch.tensor([rows - 1, 0], dtype=torch.int32)  # gathered rows: the stream is not written
        got_x, some = x.cuda(), torch.empty(2, n, dtype=dtype, device="cuda")
        ops.rmsnorm(got_x, gain.cuda(), 1e-6, some, picks.cuda(), partials=None if p is None else p.cuda())
        assert torch.equal(got_x.cpu(), x)
        assert ((some.cpu().double() - want[picks.long()]).abs() <= bound * want[picks.long()].abs() + 1e-30).all(), splits
