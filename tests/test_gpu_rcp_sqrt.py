"""Exhaustive device check of the fan backprojection's distance weight: rcp_sqrt_fast (estimate,
Goldschmidt step, exact residuals) equals the correctly rounded 1.0f / sqrtf(t) for every float
of its range [2^-100, 2^100]."""
import ctypes
import os

import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

KIT = os.path.join(os.path.dirname(__file__), "native", "libpyronn_testkit.so")


def test_rcp_sqrt_fast_matches_ieee_for_every_float_of_its_range():
    if not os.path.exists(KIT):
        pytest.fail("tests/native/libpyronn_testkit.so missing: run pyro-nn-layers_amd/build.py")
    check = ctypes.CDLL(KIT).pyronn_testkit_rcp_sqrt_check
    check.argtypes, check.restype = [ctypes.c_void_p, ctypes.c_void_p], ctypes.c_int
    counts = torch.full((1 << 24,), 0xFFFF, dtype=torch.int32, device="cuda")
    assert check(counts.data_ptr(), torch.cuda.current_stream().cuda_stream) == 0
    torch.cuda.synchronize()
    assert int(counts.sum().item()) == 0
