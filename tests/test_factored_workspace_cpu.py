"""Workspace sizes of the factored step: what is said for one group holds for every larger one,
and what is said for a tensor holds in any group."""
import pytest


@pytest.mark.parametrize("shape", [(1, 32, 8), (1, 300, 5000), (3, 1100, 2050), (1, 33000, 36), (1, 16384, 16384),
                                   (1, 17000, 17000)])
def test_group_workspace_covers_larger_groups(shape):
    from adafactor8bit import _native as nat
    L = nat.lib()
    B, R, C = shape
    own = B * R * C
    totals = sorted({own, own + 1, 1 << 27, 234_881_024, 234_881_025, 1 << 28, (1 << 28) + 1, 1 << 31, 1 << 40})
    sizes = [L.a8_factored_group_workspace_floats(B, R, C, t) for t in totals if t >= own]
    assert sizes == sorted(sizes, reverse=True)
    assert L.a8_factored_workspace_floats(B, R, C) == sizes[0]
    assert sizes[0] >= 2 * (B * R + B * C)
