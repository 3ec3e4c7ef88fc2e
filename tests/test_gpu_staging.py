"""GPU parity for every route of the prefill activation staging (xprep.hip), through
qlinear against the CPU oracle: a row split over 1..16 waves, eight rows per workgroup
whole or in parts, ragged last slots, padding rows, each fragment layout.  Each row's
largest activation (1e6 times the others, at a different place in every row) sets its
scale: a wave or part whose maximum were lost would overflow f16.

Tolerance, as max over outputs of |y - y64| / sum_k |w||x|: 2^-10 + 2e-5 (one f16
rounding of each weight and each activation, plus f32 accumulation)."""
import numpy as np
import pytest
import torch

import dyninfer_amd as d
import oracle

pytestmark = pytest.mark.gpu

TOL = 2.0 ** -10 + 2e-5


def weight(layout, n, k):
    if layout == "word":
        packed, sc, bi = oracle.synth_mlx_u4(n, k, 64, oracle.D_BF16, seed=k)
        dev = [torch.from_numpy(a).cuda() for a in (packed, sc, bi)]
        return (d.QWeight(d.ENC_MLX_U4, n, k, *dev, 64, d.DTYPE_BF16),
                oracle.dequant_mlx_u4(packed, sc, bi, oracle.D_BF16, n, k, 64))
    g, e = (oracle.Q4_0, d.ENC_Q4_0) if layout == "nib" else (oracle.Q8_0, d.ENC_Q8_0)
    data = oracle.synth_gguf(g, n, k, seed=k)
    return d.QWeight(e, n, k, torch.from_numpy(data).cuda()), oracle.dequant_gguf(g, data, n, k)


@pytest.mark.parametrize("layout", ["nib", "byte", "word"])
@pytest.mark.parametrize("rows,k", [
    (33, 64), (40, 576), (45, 4096), (45, 8192), (45, 12352), (61, 20480),      # one slot a lane: 1..16 waves a row
    (250, 1088), (700, 2112), (255, 4160), (1000, 1024),
    (640, 4096), (630, 5120), (300, 4160), (390, 5120), (20, 33024),  # several slots a lane (f32)
    (2052, 2112), (2100, 4096),                                     # eight rows, whole, a wave each (f32)
    (256, 4096), (257, 4160), (700, 8256), (500, 12288), (300, 20480),  # eight rows a workgroup, in parts
    (1024, 64), (1025, 512), (1030, 1088), (1024, 4160), (1050, 8256), (1024, 12288),  # eight rows, whole
    (1024, 12352),                                                  # too long to hold whole: parts again
])
@pytest.mark.parametrize("xbf16", [False, True], ids=["xf32", "xbf16"])
def test_staging_routes(ctx, layout, rows, k, xbf16):
    n = 64
    w, wf = weight(layout, n, k)
    x = oracle.randn(rows * k, seed=rows + k).reshape(rows, k)
    r = np.arange(rows)
    x[r, (r * 2654435761 + k - 1) % k] *= 1e6
    x[0, k - 1], x[rows - 1, 0], x[rows - 1, k - 1] = 3e6, -3e6, 1e-3
    xt = torch.from_numpy(x)
    if xbf16:
        xt = xt.bfloat16()
        x = xt.float().numpy()
    y = ctx.qlinear(w, xt.cuda()).cpu().numpy()
    pick = np.unique(np.concatenate([r[:9], r[-9:], r[::37]]))  # first and last groups of rows, and between
    y64, absdot = oracle.linear_f64(x[pick], wf)
    assert float((np.abs(y[pick].astype(np.float64) - y64) / absdot).max()) <= TOL
