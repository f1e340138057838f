"""When a decode step's attention blocks go by the sequences' lengths."""
from rocml_amd.ops import lengths_differ, may_share


def test_lengths_that_differ():
    assert not lengths_differ([]) and not lengths_differ([7]) and not lengths_differ([2048] * 8)
    assert not lengths_differ([2070 - i for i in range(24)]) and not lengths_differ([100, 140])
    assert lengths_differ([100, 300]) and lengths_differ([200, 300, 700, 4000])
    assert lengths_differ([1, 1, 2]) and not lengths_differ([1, 1])


def test_a_batch_changes_sides_once_at_most():
    for lengths in ([10, 10, 11, 12, 150, 10], [128, 4096, 700, 900], [5, 6], [1, 64, 64]):
        sides = [lengths_differ([n + k for n in lengths]) for k in range(9000)]
        assert sides == sorted(sides, reverse=True)


def test_steps_that_may_share():
    assert not may_share(4, 8, 256) and may_share(5, 8, 256) and may_share(64, 8, 256) and not may_share(65, 8, 256)
    assert not may_share(1, 64, 256) and may_share(2, 32, 256) and not may_share(8, 0, 256) and not may_share(64, 8, 0)
