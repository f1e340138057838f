"""What a block may prepare for the one behind it: the norm that the next block names, with that block's input convolution where it rides
along, and nothing where the stream changes between the two."""
from types import SimpleNamespace

import pytest
import torch

from rocml_amd.engine import DecoderModel
from rocml_amd.config import architecture_of
from rocml_amd.parts.block import SandwichNormBlock
from tests import kakalorn_models as km


def _model(taps=3, width=72, layers=3):
    cfg = km.config(60, width, taps, [km.hgrn2(2, 8, 12, km.dense(40)) for _ in range(layers)])
    arch = architecture_of(cfg)
    model = DecoderModel(arch.to_spec(arch.read_config(cfg)), "bfloat16", device="meta")
    for block in model.blocks:
        for child in block.children.values():
            if hasattr(child, "gain"):
                child.gain = torch.ones(width)
        block.input_conv.w = torch.zeros(taps, width)
    return model


class _Cache:
    """Views with kept rows of their own for every entry."""
    def has_line(self, i):
        return True

    def view(self, i, step):
        return SimpleNamespace(parts=("mixer", SimpleNamespace(state=torch.full((1, 2, 72), float(i)))))


ONE_EACH = SimpleNamespace(max_new=1, n_tokens=3, n_seqs=3)
PROMPT = SimpleNamespace(max_new=4, n_tokens=6, n_seqs=3)


def test_the_convolution_rides_in_steps_of_one_token():
    model = _model()
    hint = model.next_hint(0, _Cache(), ONE_EACH)
    assert hint.gain is model.blocks[1].children["mixer_norm"].gain and hint.width == 72
    assert hint.conv[0] is model.blocks[1].input_conv.w and float(hint.conv[1][0, 0, 0]) == 1.0
    assert model.next_hint(0, _Cache(), PROMPT).conv is None
    assert model.next_hint(2, _Cache(), ONE_EACH) is None               # nothing behind the last


@pytest.mark.parametrize("taps,width", [(1, 72), (5, 72), (3, 70), (3, 2052)])
def test_sizes_that_do_not_ride(taps, width):
    assert _model(taps, width).next_hint(0, _Cache(), ONE_EACH).conv is None


def test_blocks_with_a_hint_of_their_own():
    """``entry_hint`` takes the step alone, also in a block that derives from this one."""
    class Derived(SandwichNormBlock):
        def entry_hint(self, step):
            return super().entry_hint(step) if step.max_new > 1 else None

    model = _model()
    model.blocks[1].__class__ = Derived
    assert model.next_hint(0, _Cache(), ONE_EACH) is None
    assert model.next_hint(0, _Cache(), PROMPT) is not None
