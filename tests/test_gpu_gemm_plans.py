"""GPU parity for every configuration the prefill GEMM's planner picks (tile, K split,
shared or own activation fragments), each encoding, against the CPU oracle: ragged rows
and columns, several weights in one launch, K slices that differ by a chunk (K = 320,
1088, 1280), slices of one chunk.

Tolerances, as max over outputs of |y - y64| / sum_k |w||x|: 2^-10 + 2e-5 (one f16
rounding of each weight and activation, plus f32 accumulation); Q6_K and IQ4_XS weights
round twice (+ 2^-11); Q4_K and Q5_K weights are RNE_f16(q RNE_f16(d sc) -
RNE_f16(dmin m)), three roundings of terms that may nearly cancel, bounded through
sum_k |dmin m||x|."""
import numpy as np
import pytest
import torch

import dyninfer_amd as d
import oracle

pytestmark = pytest.mark.gpu

BLOCKS = ["q4_0", "q4_1", "q8_0", "mlx_u4"]
SUPER = ["q6_k", "q4_k", "q5_k", "iq4_xs"]


def weight(kind, n, k, seed):
    """(QWeight, dequantised weights, |min| of each weight) of synthetic blocks."""
    if kind == "mlx_u4":
        packed, sc, bi = oracle.synth_mlx_u4(n, k, 64, oracle.D_BF16, seed=seed)
        t = [torch.from_numpy(a).cuda() for a in (packed, sc, bi)]
        return (d.QWeight(d.ENC_MLX_U4, n, k, *t, 64, d.DTYPE_BF16),
                oracle.dequant_mlx_u4(packed, sc, bi, oracle.D_BF16, n, k, 64), None)
    g = getattr(oracle, kind.upper())
    data = oracle.synth_gguf(g, n, k, seed)
    w = d.QWeight(getattr(d, "ENC_" + kind.upper()), n, k, torch.from_numpy(data).cuda())
    wf = oracle.dequant_gguf(g, data, n, k)
    if kind not in ("q4_k", "q5_k"):
        return w, wf, None
    zero = data.reshape(-1, 144 if kind == "q4_k" else 176).copy()
    zero[:, 16:] = 0  # every code 0: the weights are -dmin m
    return w, wf, np.abs(oracle.dequant_gguf(g, zero.reshape(-1), n, k))


def check(ctx, kind, m, ns, k):
    made = [weight(kind, n, k, seed=m + n + k) for n in ns]
    x = oracle.randn(m * k, seed=m + k).reshape(m, k)
    xd = torch.from_numpy(x).cuda()
    ys = ctx.qlinear_multi([w for w, _, _ in made], xd) if len(ns) > 1 else [ctx.qlinear(made[0][0], xd)]
    pick = np.unique(np.concatenate([np.arange(min(m, 3)), np.arange(max(m - 3, 0), m), np.arange(0, m, 61)]))
    for y, (_, wf, mins) in zip(ys, made):
        y64, absdot = oracle.linear_f64(x[pick], wf)
        tol = 2.0 ** -10 + 2e-5 + (2.0 ** -11 if kind in SUPER else 0.0)
        bound = tol * absdot
        if mins is not None:
            bound = bound + 2.0 ** -10 * (np.abs(x[pick]).astype(np.float64) @ mins.T.astype(np.float64))
        err = np.abs(y.cpu().numpy()[pick].astype(np.float64) - y64)
        assert (err <= bound).all(), float((err / absdot).max())


# (rows, weight rows, K): the configuration (TM, NB, S, WN, WM) the planner picks for most encodings
SHAPES = [
    (33, [97], 256),            # 1 1 4 1 1, a chunk per slice
    (45, [131, 62], 1280),      # 1 1 8 1 1, slices of 2 and 3 chunks
    (33, [4000, 101], 256),     # 2 1 4 1 1
    (50, [9001], 512),          # 2 2 4 1 1
    (75, [8000, 900, 103], 256),  # 2 3 4 1 1
    (70, [14001], 512),         # 4 2 4 1 1
    (97, [19000, 1001], 768),   # 4 3 4 1 1
    (131, [13000, 1003], 768),  # 8 2 4 1 1, blocks of 32: 2 2 1 4 1
    (150, [12601], 1024),       # 8 2 4 1 1
    (131, [9001], 256),         # 2 2 1 4 1
    (257, [14002], 256),        # 4 2 1 4 1, Q6_K 4 2 1 2 2
    (68, [35081], 256),         # 4 2 1 4 1
    (645, [10781], 256),        # 4 2 1 2 2
    (3206, [867], 1024),        # 4 2 2 2 1, more copies a window: 8 2 4 1 1
    (400, [20001], 256),        # 8 2 1 4 1
    (400, [20001], 1024),       # the two above over a ring's worth of chunks
    (513, [6000, 3001], 1280),
]
ODD_SHAPES = [(40, [97], 64), (41, [260, 30], 192), (70, [513], 320), (90, [1000], 1088), (300, [20000], 64)]


@pytest.mark.parametrize("kind", BLOCKS + SUPER)
@pytest.mark.parametrize("m,ns,k", SHAPES, ids=[f"{m}-{'+'.join(map(str, ns))}-{k}" for m, ns, k in SHAPES])
def test_gemm_plans(ctx, kind, m, ns, k):
    check(ctx, kind, m, ns, k)


@pytest.mark.parametrize("kind", BLOCKS)
@pytest.mark.parametrize("m,ns,k", ODD_SHAPES)
def test_gemm_plans_odd_chunks(ctx, kind, m, ns, k):
    check(ctx, kind, m, ns, k)


@pytest.mark.parametrize("n", [33, 260])
def test_gemm_activations_past_4gib(ctx, n):
    """rows·K just below the limit of 2^31: rounded up to 32 rows the staged activations pass
    4 GiB, and the last rows' fragments lie beyond a 32-bit offset."""
    k, tail = 20480, 57
    m = (2**31 - 1) // k
    w, wf, _ = weight("q8_0", n, k, seed=5)
    x = torch.zeros(m, k, dtype=torch.bfloat16, device="cuda")
    x[-tail:] = torch.from_numpy(oracle.randn(tail * k, seed=6).reshape(tail, k)).cuda().bfloat16()
    y = ctx.qlinear(w, x)
    assert not y[:-tail].any()
    xt = x[-tail:].float().cpu().numpy()
    y64, absdot = oracle.linear_f64(xt, wf)
    err = np.abs(y[-tail:].cpu().numpy().astype(np.float64) - y64)
    assert (err <= (2.0 ** -10 + 2e-5) * absdot).all(), float((err / absdot).max())


def _shifted(a, off):
    """a on the device, its first byte `off` bytes past a 4-byte boundary."""
    t = torch.zeros(a.nbytes + 4, dtype=torch.uint8, device="cuda")
    t[off:off + a.nbytes] = torch.from_numpy(a.view(np.uint8).reshape(-1)).cuda()
    return t[off:off + a.nbytes]


@pytest.mark.parametrize("sdtype,off", [(oracle.D_BF16, 0), (oracle.D_BF16, 2), (oracle.D_F16, 2), (oracle.D_F32, 0)])
@pytest.mark.parametrize("group,m,ns,k", [
    (96, 40, [97], 192),      # 2 2 1 4 1
    (96, 41, [97, 60], 384),  # 1 1 4 1 1
    (160, 45, [131], 960),    # 1 1 8 1 1
    (96, 45, [131], 960),
    (160, 20, [1000], 320),   # fewer rows than a row block
    (96, 257, [14002], 192),  # 4 2 1 4 1
    (96, 682, [10865], 192),  # 4 2 1 2 2: one of the two waves of a window copies the scales, one the biases
    (160, 260, [14002], 320),
])
def test_gemm_mlx_groups_across_chunks(ctx, sdtype, off, group, m, ns, k):
    """Group sizes that are multiples of 32 and not of 64: a group may end in the middle of a
    64-k chunk, whose halves then take scales and biases of two groups.

    f32 scales and biases are rounded to f16 first: 2^-11 (|q s| + |b|) |x| besides, and
    |q s| <= |w| + |b|."""
    ws, refs = [], []
    for n in ns:
        packed, sc, bi = oracle.synth_mlx_u4(n, k, group, sdtype, seed=n + k + group)
        ws.append(d.QWeight(d.ENC_MLX_U4, n, k, torch.from_numpy(packed).cuda(), _shifted(sc, off), _shifted(bi, off),
                            group, sdtype))
        wf = oracle.dequant_mlx_u4(packed, sc, bi, sdtype, n, k, group)
        b = np.repeat(np.abs(bi.astype(np.float64)).reshape(n, -1), group, axis=1) if sdtype == oracle.D_F32 else None
        refs.append((wf, b))
    x = oracle.randn(m * k, seed=m + k).reshape(m, k)
    ys = ctx.qlinear_multi(ws, torch.from_numpy(x).cuda())
    for y, (wf, b) in zip(ys, refs):
        y64, absdot = oracle.linear_f64(x, wf)
        bound = (2.0 ** -10 + 2e-5) * absdot
        if b is not None:
            bound = bound + 2.0 ** -11 * (absdot + 2.0 * (np.abs(x).astype(np.float64) @ b.T))
        err = np.abs(y.cpu().numpy().astype(np.float64) - y64)
        assert (err <= bound).all(), float((err / absdot).max())
