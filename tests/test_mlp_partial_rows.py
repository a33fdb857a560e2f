"""CPU: the partial-gradient buffer that a training step asks for holds one row
(6,663 gradients and the loss) per workgroup of the gradient kernel: a tile of
32 regions each, at most 512 workgroups, for every number of regions."""

from __future__ import annotations

import pytest

import cujpegxl_amd as cj

ROW = 64 * 96 + 64 + 7 * 64 + 7 + 1


@pytest.mark.parametrize("n,rows", [(0, 0), (1, 1), (32, 1), (33, 2), (4096, 128), (512 * 32 - 1, 512),
                                    (512 * 32, 512), (512 * 32 + 1, 512), (2_000_000, 512), (2**32 - 32, 512),
                                    (2**32 - 31, 512), (2**32 - 1, 512)])
def test_a_row_per_workgroup(n, rows):
    assert cj.stages_lib().cjx_mlp_partial_floats(n) == rows * ROW
