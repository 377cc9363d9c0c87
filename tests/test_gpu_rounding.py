"""The kernels' fp32 -> bf16 rounding (one packed convert) against the integer construction it stands for: every
fp32 pattern, and the double -> float -> bf16 chains of the exact kernels where one rounding and two differ."""

import ctypes

import pytest
import torch

from mini_infra_qwen3_amd import build

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def check():
    lib = ctypes.CDLL(str(build.CALIB_LIBRARY_PATH))
    lib.calib_round_patterns.argtypes = [ctypes.c_uint64, ctypes.c_uint64, ctypes.c_void_p, ctypes.c_void_p]
    lib.calib_round_doubles.argtypes = [ctypes.c_void_p, ctypes.c_uint64, ctypes.c_void_p, ctypes.c_void_p]
    return lib


def test_every_fp32_pattern(check, device):
    bad = torch.zeros(1, dtype=torch.int64, device=device)
    assert check.calib_round_patterns(0, 1 << 32, bad.data_ptr(), torch.cuda.current_stream().cuda_stream) == 0
    assert bad.item() == 0
    assert check.calib_round_patterns(1, 1 << 32, bad.data_ptr(), None) == -1  # past the last pattern


def test_doubles_round_to_float_first(check, device):
    """Doubles a little above and below every bf16 tie: their float is the tie, which rounds to even; one rounding would
    take them to the nearer side.  With subnormals, infinities, NaN and values past the largest float."""
    ties = ((torch.arange(1 << 16, dtype=torch.int64) << 16) | 0x8000).to(torch.int32).view(torch.float32).double()
    values = torch.cat([ties * (1 + s * 2.0 ** -e) for s in (-1, 1) for e in (26, 30, 40, 50)]
                       + [ties, torch.tensor([float("inf"), -float("inf"), float("nan"), 3.5e38, -3.4028236e38, 1e-46, 0.0])])
    bad = torch.zeros(1, dtype=torch.int64, device=device)
    values = values.to(device)
    assert check.calib_round_doubles(values.data_ptr(), values.numel(), bad.data_ptr(),
                                     torch.cuda.current_stream().cuda_stream) == 0
    assert bad.item() == 0
