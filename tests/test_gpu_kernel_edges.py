"""Kernels at the sizes where their tiling changes: remainders, group edges,
the smallest sizes and the hand-over between variants."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


def relerr(a, b):
    return float(np.abs(a - b).max() / max(np.abs(b).max(), 1e-300))


@pytest.mark.parametrize("shape", [
    (1, 1, 1), (2, 3, 4), (17, 16, 15), (18, 33, 31), (3, 25, 26), (5, 32, 65),
    # 32 lines a block up to 253 samples on the axis, then 16, 8, ... and from
    # 8190 one thread per line in global memory
    (2, 253, 3), (2, 254, 3), (3, 509, 2), (3, 510, 2), (510, 2, 35), (2, 2, 1022),
    (2, 8189, 1), (1, 8190, 2), (2, 1, 8190), (8190, 1, 2)])
def test_prefilter_line_groups(shape):
    """Against the oracle's recursion; the two differ by the contraction of a
    few operations, each within an ulp of coefficients of order one (the
    recursion damps earlier errors by 0.27 a step), so 1e-13 holds with room."""
    from numbacs_amd import _lib
    from numbacs_amd.flows import prefilter3_device

    U = np.random.default_rng(sum(shape)).standard_normal(shape)
    C = _lib.to_host(prefilter3_device(U))
    assert C.shape == tuple(n + 2 for n in shape)
    assert relerr(C, oracle.prefilter3(U)) < 1e-13
