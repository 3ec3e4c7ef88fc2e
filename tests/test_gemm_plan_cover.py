"""The shapes of the prefill GEMM's parity tests against its planner (host code: no device):
they pick every configuration that any shape of a wide sweep picks, for each encoding."""
import ctypes
import random

import pytest

import dyninfer_amd as d
from test_gpu_gemm_plans import BLOCKS, ODD_SHAPES, SHAPES, SUPER


class _Plan(ctypes.Structure):
    _fields_ = [(f, ctypes.c_uint32) for f in ("tm", "nb", "s", "wn", "wm", "mt", "nt")]


@pytest.fixture(scope="module")
def plan():
    f = d.library()["_ZN3dmx9gemm_planEjPKjijj"]  # dmx::gemm_plan(enc, N, count, K, M), kernels.hpp
    f.restype = _Plan
    f.argtypes = [ctypes.c_uint32, ctypes.c_void_p, ctypes.c_int, ctypes.c_uint32, ctypes.c_uint32]

    def call(kind, m, ns, k):
        p = f(getattr(d, "ENC_" + kind.upper()), (ctypes.c_uint32 * len(ns))(*ns), len(ns), k, m)
        assert p.tm and p.mt == -(-(-(-m // 32)) // (p.tm * p.wm))
        assert p.nt == sum(-(-n // (32 * p.nb * p.wn)) for n in ns)
        return p.tm, p.nb, p.s, p.wn, p.wm

    return call


@pytest.mark.parametrize("kind", BLOCKS + SUPER)
def test_shapes_cover_the_planner(plan, kind):
    shapes = SHAPES + (ODD_SHAPES if kind in BLOCKS else [])
    covered = {plan(kind, m, ns, k) for m, ns, k in shapes}
    rng = random.Random(kind)
    picked = set()
    for _ in range(20000):
        k = rng.choice([64, 128, 192, 256, 320, 512, 768, 1024, 1280, 1536, 2048, 3072, 4096, 8192, 12288, 16384])
        if kind in SUPER and k % 256:
            continue
        m, n = int(17 * 241 ** rng.random()), int(32 * 5000 ** rng.random())
        picked.add(plan(kind, m, [n], k))
    assert picked <= covered, sorted(picked - covered)
