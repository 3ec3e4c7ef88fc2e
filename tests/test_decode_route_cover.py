"""The decode parity lists against the dispatch (host code: no device): which of their cases
run on the 16-row MFMA GEMV."""
import ctypes

import pytest

import dyninfer_amd as d
import test_gpu_parity as parity


class _Problem(ctypes.Structure):
    _fields_ = [("w", ctypes.c_void_p), ("sc", ctypes.c_void_p), ("bi", ctypes.c_void_p), ("y", ctypes.c_void_p),
                ("n", ctypes.c_uint32)]


@pytest.fixture(scope="module")
def applies():
    # dmx::gemv_mfma_applies(enc, probs, nprob, batch, K, y_bf16, group), kernels.hpp
    f = d.library()["_ZN3dmx17gemv_mfma_appliesEjPKNS_11GemvProblemEijjbj"]
    f.restype = ctypes.c_bool
    f.argtypes = [ctypes.c_uint32, ctypes.c_void_p, ctypes.c_int, ctypes.c_uint32, ctypes.c_uint32, ctypes.c_bool,
                  ctypes.c_uint32]
    return lambda enc, n, k, batch, ybf16, group=0: f(enc, (_Problem * 1)(_Problem(n=n)), 1, batch, k, ybf16, group)


def test_mfma_cases_run_on_the_16_row_kernels(applies):
    on = [c for c in parity.MFMA_CASES + parity.MFMA_NOT_CASES if applies(parity.ENC[c[0]], *c[1:5])]
    assert on == parity.MFMA_CASES
    assert {(c[3] > 4) + (c[3] > 8) for c in on} == {0, 1, 2}
    on = [c for c in parity.MLX_MFMA_CASES + parity.MLX_MFMA_NOT_CASES
          if applies(d.ENC_MLX_U4, c[0], c[1], c[4], c[5], c[2])]
    assert on == parity.MLX_MFMA_CASES
    assert all(applies(parity.ENC[c[0]], *c[1:5]) for c in parity.PRESTAGE_CASES)
