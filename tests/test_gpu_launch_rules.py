"""Which launch a call takes, and what it may ask of the device around it:
requested launch shapes are the ones that run, default ones take no memory
that a caller cannot spare, and sizes past 32-bit launch or index limits give
the results of the smaller ones."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

RELAXED, GLOBAL = 2, 0  # hipStreamCaptureMode


@pytest.fixture(scope="module")
def lib():
    from numbacs_amd import _lib

    _lib.torch()
    return _lib


@pytest.fixture
def configs(lib):
    from numbacs_amd import autotune

    saved = {(k, p): autotune.get(k, p) for k in range(4) for p in (0, 1)}
    orders = {p: autotune.get_order(p) for p in (0, 1)}
    yield autotune
    for (k, p), cfg in saved.items():
        autotune.set_config(k, p, cfg)
    for p, o in orders.items():
        autotune.set_order(p, o)


@pytest.mark.parametrize("shape", [(1, 23170, 23170), (23171, 23171, 1)])
def test_prefilter_of_more_lines_than_one_launch_holds(lib, shape):
    """Axes of one sample with 2^29 lines and more across them (8 threads of the
    line-group kernels each): a coefficient of such an axis equals its sample,
    and along the others the coefficients interpolate it."""
    from numbacs_amd.flows import prefilter3_device

    torch = lib.torch()
    gen = torch.Generator(device="cuda").manual_seed(5)
    U = torch.rand(shape, generator=gen, dtype=torch.float64, device="cuda") - 0.5
    C = prefilter3_device(U)
    one = shape.index(1)
    planes = [C.select(one, k) for k in range(3)]
    assert torch.equal(planes[0], planes[1]) and torch.equal(planes[2], planes[1])
    # (c[i-1] + 4 c[i] + c[i+1]) / 6 along both long axes
    c = planes[1][-4001:, -4001:]
    for axis in (0, 1):
        m = c.shape[axis] - 2
        c = (c.narrow(axis, 0, m) + 4 * c.narrow(axis, 1, m) + c.narrow(axis, 2, m)) / 6
    u = U.select(one, 0)[-c.shape[0]:, -c.shape[1]:]
    # rounding of coefficients up to 9 times the samples, and of the check's sums
    assert float((c - u).abs().max()) < 64 * 2.0 ** -52 * 4.5
    del U, C, planes, c, u
    torch.cuda.empty_cache()
