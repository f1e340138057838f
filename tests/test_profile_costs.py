"""What the profiler prices calls with."""
import torch

from rocml_amd.profile import _COSTS


def test_a_convolution_inside_the_norms_kernel_is_priced():
    rows, n, taps = 5, 64, 4
    x, y, gain = torch.zeros(rows, n), torch.zeros(rows, n), torch.ones(n)
    copy, partials = torch.zeros(rows, n, dtype=torch.bfloat16), torch.zeros(3, rows, n)
    w, state, slots = torch.zeros(taps, n), torch.zeros(9, taps - 1, n, dtype=torch.bfloat16), torch.zeros(rows, dtype=torch.int32)
    label, cost = _COSTS["norm_add"]
    args, kw = (x, y, gain, None, 1e-5), dict(layer=False, copy=copy, partials=partials, replace=True, next_gain=gain, next_eps=1e-5)
    bytes_, flops = cost(*args, **kw)
    assert (bytes_, flops) == (2 * rows * n * 4 + rows * n * 2 + 3 * rows * n * 4, 8 * rows * n)
    with_conv = cost(*args, **kw, conv=(w, state, slots))
    alone = _COSTS["added_conv"][1](copy, w, state, None, slots, [1] * rows, copy)
    # what the convolution costs by itself, without writing and reading its rows in between
    assert with_conv == (bytes_ + alone[0] - 2 * rows * n * 2, flops + alone[1])
    assert alone == (2 * rows * n * 2 + taps * n * 4 + 2 * rows * (taps - 1) * n * 2, 2 * taps * rows * n)
    assert len({label(*args), label(*args, **kw), label(*args, **kw, conv=(w, state, slots))}) == 3
