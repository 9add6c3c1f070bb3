"""Workspace sizes of the C ABI, on the host (no device needed)."""

import pytest

from prospective_rqf_amd import _lib


@pytest.mark.parametrize("rows", [16, 48, 256, 520, 1024, 4096, 8192])
@pytest.mark.parametrize("ac,bc", [(1, 1), (0, 0), (1, 0), (0, 1)])
def test_weight_gradients_do_not_grow_with_the_columns(rows, ac, bc):
    """256 MB, or the real rows' products once in fp32 (tiles of up to 128 rows), and 16
    bytes per output element."""
    size = _lib.load().rqf_weight_grad_workspace
    m, k = (-(-rows * (1 + c) // 128) * 128 for c in (ac, bc))
    bound = max(256 << 20, 4 * m * k) + 16 * m * k
    sizes = [size(rows, ac, rows, bc, n) for n in (1, 4096, 262144, 1 << 20, 1 << 24, 1 << 30)]
    assert 0 < min(sizes) and max(sizes) <= bound
