"""GPU parity for 3..8 activation rows on the 4x4 MFMA kernels, each way a launch splits
its work, every encoding, against the CPU oracle: weight rows that are no multiple of
four, fewer chunks than a row block's sixteen lanes, row counts below the register
batch (whose spare rows restage row 0), two passes (9..16 rows of Q8_0 and Q4_1),
several weights in one launch, bf16 activations and outputs.

Tolerance, as |y - y64| <= tol sum_k |w||x|: 2^-11 + 2e-5 (each activation rounds to f16
once, codes are exact, f32 accumulation), plus 2^-8 |y| for a bf16 output."""
import numpy as np
import pytest
import torch

import dyninfer_amd as d
import oracle

pytestmark = pytest.mark.gpu

KINDS = ["q4_0", "q4_1", "q8_0", "mlx_u4", "q6_k", "q4_k", "q5_k", "iq4_xs"]


def weight(kind, n, k, seed):
    if kind == "mlx_u4":
        packed, sc, bi = oracle.synth_mlx_u4(n, k, 64, oracle.D_BF16, seed=seed)
        t = [torch.from_numpy(a).cuda() for a in (packed, sc, bi)]
        return (d.QWeight(d.ENC_MLX_U4, n, k, *t, 64, d.DTYPE_BF16),
                oracle.dequant_mlx_u4(packed, sc, bi, oracle.D_BF16, n, k, 64))
    g = getattr(oracle, kind.upper())
    data = oracle.synth_gguf(g, n, k, seed)
    return (d.QWeight(getattr(d, "ENC_" + kind.upper()), n, k, torch.from_numpy(data).cuda()),
            oracle.dequant_gguf(g, data, n, k))


def check(ctx, kind, m, ns, k, bf16=False):
    made = [weight(kind, n, k, seed=m + n + k) for n in ns]
    x = torch.from_numpy(oracle.randn(m * k, seed=m + k).reshape(m, k))
    if bf16:
        x = x.bfloat16()
    dt = torch.bfloat16 if bf16 else torch.float32
    ys = [torch.empty(m, n, dtype=dt, device="cuda") for n in ns]
    ctx.qlinear_multi([w for w, _ in made], x.cuda(), ys)
    x = x.float().numpy()
    for y, (_, wf) in zip(ys, made):
        y64, absdot = oracle.linear_f64(x, wf)
        bound = (2.0 ** -11 + 2e-5) * absdot + (2.0 ** -8 * np.abs(y64) if bf16 else 0.0)
        err = np.abs(y.float().cpu().numpy().astype(np.float64) - y64)
        assert (err <= bound).all(), float((err / absdot).max())


SHAPES = [
    (3, [5], 256),                # four waves per row block, chunks for a few lanes only
    (4, [1023], 2048),            # ... of two to a workgroup, a ragged row block
    (5, [997], 3072),
    (8, [1001, 254], 4096),       # ... weights in one launch
    (4, [8190], 512),             # a wave per row block, a chunk per lane or less
    (7, [2051, 64], 1024),        # ... two
    (6, [3001], 1792),            # ... four, some lanes with fewer
    (8, [2077], 3840),            # ... eight of 32 weights
    (4, [4090], 12288),           # four row blocks to a workgroup, one per CU
    (3, [2050], 8448),
    (4, [2051], 14336),           # ... seven chunks a lane, or the pipeline
    (4, [1030, 250], 7936),       # ... four
    (4, [1500], 14336),           # four waves per row block, up to eight chunks a lane
    (3, [1026], 6144),
    (4, [1501], 10240),           # ... three and five
    (3, [1030], 14592),           # ... and eight, where the tile fits
    (4, [2043], 14080),           # ... seven
    (3, [1027, 900], 512),        # a wave each, one chunk a lane
    (5, [997], 4352),             # eight rows, four waves per row block, three chunks a lane
    (7, [2047], 6656),            # ... four
    (4, [2500], 5120),            # three row blocks to a workgroup, three chunks a lane
    (3, [3333], 4352),            # ... four
    (4, [2100], 8192),            # three, four chunks a lane
    (3, [2501], 10240),           # ... five
    (4, [3070], 12288),           # ... six
    (4, [2053], 13312),           # ... seven
    (3, [3075], 10240),           # four, five chunks a lane
    (4, [4095], 8192),            # ... four
    (8, [2101], 5120),            # eight rows: three, three chunks a lane
    (6, [2103], 6656),            # ... four
    (8, [3333], 6144),            # four row blocks, three chunks a lane (of Q8_0 and Q4_1)
    (8, [4001], 6656),
    (4, [3071], 2560),            # 64-weight chunks: the pipeline
    (3, [2301], 7168),
    (4, [3333], 9216),
    (8, [2500], 2560),            # 64-weight chunks: the 16-row kernels
    (4, [8200], 7680),            # one workgroup to a CU, more row blocks than they take at once
    (8, [2100, 2200], 5120),      # the pipeline, one workgroup to a CU
    (4, [33001], 256),
    (7, [16901], 2560),           # the pipeline, one row a lane group
    (8, [8197, 8197], 768),
    (16, [517], 1280),            # two passes, or the 16-row kernels
    (11, [4100], 1024),
]


@pytest.mark.parametrize("kind", KINDS)
def test_shapes(kind):
    ctx = d.Context(0)
    for m, ns, k in SHAPES:
        print(kind, m, ns, k, flush=True)
        check(ctx, kind, m, ns, k)


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("m,n,k", [(4, 1030, 2048), (5, 4099, 1024), (4, 2049, 12288), (4, 3077, 8192), (3, 2053, 5120)])
def test_bf16(kind, m, n, k):
    check(d.Context(0), kind, m, [n], k, bf16=True)
