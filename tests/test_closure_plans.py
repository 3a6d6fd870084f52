"""Scratch sizes of the closure's weight gradient (host only)."""

import pytest

from oracle import closure_oracle as co


@pytest.mark.parametrize("shape", [(1, 1, 16), (8, 8, 16), (128, 64, 64), (2, 1101, 16), (1, 65536, 16), (3, 9, 64)])
def test_weight_gradient_scratch_is_bounded(shape):
    """One row of sums a block and at most 512 blocks, however wide the grid."""
    from projecticy_amd import _native_closure as nc

    size = int(nc.lib().icyc_wgrad_partials_size(*shape))
    assert size % co.LAYER_PARAMS == 0
    assert co.LAYER_PARAMS <= size <= 512 * co.LAYER_PARAMS
