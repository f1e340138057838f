"""The convolution on a mixer's input in steps of one token: the same bits as over the whole sequence at once."""
import pytest
import torch

from rocml_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("taps", [1, 2, 3, 4, 16])
@pytest.mark.parametrize("n,dtype", [(8, torch.bfloat16), (2056, torch.bfloat16), (37, torch.bfloat16), (1028, torch.float32), (5, torch.float32)])
def test_steps_of_one_token(taps, n, dtype):
    g = torch.Generator().manual_seed(taps * 100 + n)
    total, slots = 21, torch.tensor([2, 0, 1], dtype=torch.int32, device="cuda")
    h = torch.randn(3, total, n, generator=g).to(dtype).cuda()
    w = torch.randn(taps, n, generator=g).cuda()

    def run(state, parts):
        """One step: parts[i] = (from, to) of sequence i."""
        counts = [b - a for a, b in parts]
        cu = torch.tensor([0, counts[0], counts[0] + counts[1], sum(counts)], dtype=torch.int32, device="cuda")
        rows = torch.cat([h[i, a:b] for i, (a, b) in enumerate(parts)]).contiguous()
        out = torch.empty_like(rows)
        ops.added_conv(rows, w, state, cu, slots, counts, out)
        return list(out.split(counts))

    kept = [torch.zeros(3, taps - 1, n, dtype=dtype, device="cuda") if taps > 1 else None for _ in range(2)]
    whole = run(kept[0], [(0, total)] * 3)
    # one token each; one token beside a run that fills more than one of the kernel's 16 tokens; one token each again
    at, got = [0, 0, 0], [[], [], []]
    steps = [(1, 1, 1)] * 2 + [(1, 18, 1)] + [(1, 1, 1)]
    for counts in steps:
        outs = run(kept[1], [(at[i], at[i] + counts[i]) for i in range(3)])
        for i in range(3):
            got[i].append(outs[i])
            at[i] += counts[i]
    assert at[1] == total
    for i in range(3):
        assert torch.equal(torch.cat(got[i]), whole[i][:at[i]])
    if taps > 1:
        for i in range(3):
            past = torch.cat([torch.zeros(taps - 1, n, dtype=dtype, device="cuda"), h[i, :at[i]]])[-(taps - 1):]
            assert torch.equal(kept[1][int(slots[i])], past)
