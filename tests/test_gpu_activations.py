"""The surrogate's short forms of GELU, sine and cosine (csrc/activations.h):
where they say that their rounding to bf16 is decided, it is the library
function's."""
import ctypes
import os

import numpy as np
import pytest

from conftest import ROOT

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def check():
    from numbacs_amd import _lib

    _lib.torch()
    path = os.path.join(ROOT, "tests", "native", "libactivation_check.so")
    assert os.path.exists(path), f"{path} is not built: run __graft_entry__.build()"
    lib = ctypes.CDLL(path)
    lib.activation_check.argtypes = [ctypes.c_int, ctypes.c_void_p, ctypes.c_void_p]
    lib.activation_gelu.argtypes = [ctypes.c_void_p, ctypes.c_int64, ctypes.c_void_p,
                                    ctypes.c_void_p]
    return lib


@pytest.mark.parametrize("which", ["gelu", "sine", "cosine"])
def test_every_float(check, which):
    """All 2^32 bit patterns, infinities and NaN among them."""
    import torch

    from numbacs_amd import _lib

    counts = torch.zeros(2, dtype=torch.int64, device="cuda")
    assert check.activation_check(("gelu", "sine", "cosine").index(which), _lib.ptr(counts),
                                  _lib.stream_ptr()) == 0
    wrong, undecided = counts.tolist()
    assert wrong == 0
    # (most patterns of the sine are too near zero or beyond 10^4 revolutions, where
    # the short form leaves the rounding open)
    assert 0 < undecided < 2 ** 32


@pytest.mark.parametrize("scale", [1e-30, 1e-3, 1.0, 4.0, 30.0, 1e30])
def test_gemm_rounds_as_the_library_form(check, scale):
    """The forward GEMM's epilogue with zero products: each pre-activation is
    the bias, of both signs and all magnitudes up to scale, and each output the
    library form's bf16 value."""
    import torch

    from numbacs_amd import _lib

    M, N, K = 64, 1 << 18, 32
    rng = np.random.default_rng(int(scale * 8) % 1000 + 1)
    bias = torch.tensor((rng.uniform(-1, 1, N) * scale).astype(np.float32), device="cuda")
    A = torch.zeros((M, K), dtype=torch.bfloat16, device="cuda")
    B = torch.zeros((K, N), dtype=torch.bfloat16, device="cuda")
    out = torch.empty((M, N), dtype=torch.bfloat16, device="cuda")
    want = torch.empty(N, dtype=torch.bfloat16, device="cuda")
    s = _lib.stream_ptr()
    _lib.check(_lib.load().nbx_mlp_gemm(0, _lib.ptr(A), _lib.ptr(B), M, N, K, None, _lib.ptr(out),
                                        _lib.ptr(bias), None, s))
    assert check.activation_gelu(_lib.ptr(bias), N, _lib.ptr(want), s) == 0
    assert torch.equal(out.view(torch.int16), want.view(torch.int16).expand(M, N))
