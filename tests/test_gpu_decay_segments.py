"""The walk of a recurrence in segments against the walk of whole sequences and against 64 bits, every form of the decays."""
import pytest
import torch

pytestmark = pytest.mark.gpu

from rocml_amd import ops  # noqa: E402

DEV = "cuda:0"


def _case(lens, H, dk, dv, form, seed=0):
    g = torch.Generator().manual_seed(seed)
    T = sum(lens)
    cu = torch.tensor([0] + [sum(lens[:i + 1]) for i in range(len(lens))], dtype=torch.int32)
    proj = torch.randn(T, 2 * H * dk + H * dv + 4, generator=g)
    kw = {"head": {"head_decay": 0.9 + 0.1 * torch.rand(H, generator=g)},
          "token": {"decay": 0.3 + 0.7 * torch.rand(T, H * dk, generator=g)},
          "bonus": {"decay": torch.randn(T, H * dk, generator=g) - 3, "bonus": torch.randn(H * dk, generator=g),
                    "decay_offset": 0.3 * torch.randn(H * dk, generator=g)},
          "gate": {"gate_lower": torch.rand(H * dk, generator=g), "gate_bias": torch.randn(H * dk, generator=g)}}[form]
    state = torch.randn(len(lens) + 1, H, dv, dk, generator=g)
    slots = torch.randperm(len(lens) + 1, generator=g)[:len(lens)].to(torch.int32)
    return proj, cu, kw, state, slots


def _run(lens, H, dk, dv, form, case, **kw):
    proj, cu, extra, state, slots = case
    p, st = proj.to(DEV), state.to(DEV)
    out = torch.full((sum(lens), H * dv), float("nan"), device=DEV)
    ops.decay_scan(p, 0, p, H * dk, p, 2 * H * dk, st, cu.to(DEV), slots.to(DEV), out, H, dk, dv,
                   **{k: v.to(DEV) for k, v in extra.items()}, out_scale=0.5, **kw)
    return out.double().cpu(), st.double().cpu()


def _exact(lens, H, dk, dv, form, case):
    proj, cu, kw, state, slots = case
    x = proj.double()
    q, k, v = (t.view(len(x), H, -1) for t in (x[:, :H * dk], x[:, H * dk:2 * H * dk], x[:, 2 * H * dk:2 * H * dk + H * dv]))
    kw = {n: t.double() for n, t in kw.items()}
    out, st = torch.empty(len(x), H, dv, dtype=torch.float64), state.double().clone()
    for b, slot in enumerate(slots.tolist()):
        S = st[slot].transpose(1, 2).clone()                                       # [H, dk, dv]
        for t in range(int(cu[b]), int(cu[b + 1])):
            kk, qq, u = k[t], q[t], None
            if form == "head":
                w = kw["head_decay"].view(H, 1).expand(H, dk)
            elif form == "gate":
                low = kw["gate_lower"].view(H, dk)
                w = low + (1 - low) * torch.sigmoid(kk + kw["gate_bias"].view(H, dk))
                kk, qq = 1 - w, qq * torch.sigmoid(qq)
            elif form == "bonus":
                w, u = torch.exp(-torch.exp(kw["decay"][t].view(H, dk) + kw["decay_offset"].view(H, dk))), kw["bonus"].view(H, dk)
            else:
                w = kw["decay"][t].view(H, dk)
            kv = kk[:, :, None] * v[t][:, None, :]
            read = S + u[:, :, None] * kv if u is not None else None
            S = w[:, :, None] * S + kv
            out[t] = torch.einsum("hk,hkv->hv", qq, S if read is None else read)
        st[slot] = S.transpose(1, 2)
    return 0.5 * out.view(len(x), -1), st


# segments of 16 and 64: whole ones, a last one of one token, sequences of one token and of none, of a segment and of fewer, 70 sequences;
# key sizes of either kernel that takes them, columns that are no whole tile
@pytest.mark.parametrize("form", ["head", "token", "bonus", "gate"])
@pytest.mark.parametrize("lens,H,dk,dv,segment", [([64], 1, 64, 32, 16), ([33, 1, 0, 16, 50], 2, 128, 40, 16), ([200, 65, 129], 2, 100, 32, 64),
                                                  ([3] * 69 + [40], 1, 64, 16, 16)])
def test_walk_in_segments(lens, H, dk, dv, segment, form):
    case = _case(lens, H, dk, dv, form)
    ws = torch.full((32 << 20,), 0x7f, dtype=torch.uint8, device=DEV)
    out, st = _run(lens, H, dk, dv, form, case, workspace=ws, segment=segment)
    whole, st_whole = _run(lens, H, dk, dv, form, case, workspace=ws, segment=-1)
    want, st_want = _exact(lens, H, dk, dv, form, case)
    # a segment's start is the state of a walk with one rounding more: as far from 64 bits as the whole walk, within a tenth and 1e-7
    for got, plain, exact in ((out, whole, want), (st, st_whole, st_want)):
        far, plain_far = float((got - exact).norm() / exact.norm()), float((plain - exact).norm() / exact.norm())
        assert far < 1.1 * plain_far + 1e-7 and far < 2e-6, (far, plain_far)


def test_segments_fit_the_memory():
    """Less memory than the segments wanted: longer ones, and without room for two the whole walk."""
    lens, H, dk, dv = [2000, 100], 2, 64, 32
    case = _case(lens, H, dk, dv, "token")
    want = _run(lens, H, dk, dv, "token", case)
    for room in (1 << 24, 8 * H * (dv + 1) * dk * 4, 2 * H * (dv + 1) * dk * 4, 16):
        ws = torch.empty(room + 4096, dtype=torch.uint8, device=DEV)
        ws[room:] = 7
        got = _run(lens, H, dk, dv, "token", case, workspace=ws[:room], longest=2000, segment=16)
        assert torch.all(ws[room:] == 7)
        for a, b in zip(got, want):
            assert float((a - b).norm() / b.norm()) < 1e-6


@pytest.mark.parametrize("lens,H,segment", [([16 * 64 + 1], 32, 16), ([1, 40, 16, 0, 33], 2, 16)])
def test_first_segments_start_from_the_state_before_the_step(lens, H, segment):
    """The last segment's block may have written a sequence's new state before the first segment's block starts: many more blocks than
    the chip holds, last segments of one token.  A first segment reads a copy, in the place that the last segment leaves free."""
    dk, dv = 128, 128
    case = _case(lens, H, dk, dv, "token")
    _, cu, _, state, slots = case
    numbers = [0]
    for n in lens:
        numbers.append(numbers[-1] + -(-n // segment))
    count = sum(lens) // segment + len(lens)
    ws = torch.full((count * H * (dv + 1) * dk * 4,), 0x7f, dtype=torch.uint8, device=DEV)
    out, st = _run(lens, H, dk, dv, "token", case, workspace=ws, segment=segment)
    whole, st_whole = _run(lens, H, dk, dv, "token", case, segment=-1)
    places = ws[:count * H * dv * dk * 4].view(torch.float32).view(count, H, dv, dk).cpu()
    for b, n in enumerate(lens):
        if n > segment:
            assert torch.equal(places[numbers[b + 1] - 1], state[slots[b]]), "the state before the step"
        got, want = out[cu[b]:cu[b] + min(n, segment)], whole[cu[b]:cu[b] + min(n, segment)]
        # the same walk from the same state: sums of 128 products at most in another order
        assert n == 0 or float((got - want).norm() / want.norm()) < 2e-6
    assert float((out - whole).norm() / whole.norm()) < 2e-6 and float((st - st_whole).norm() / st_whole.norm()) < 2e-6
