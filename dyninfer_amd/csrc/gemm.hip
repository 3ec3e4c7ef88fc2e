// Prefill GEMM: launch planning and dispatch (host side).  The kernels are in
// gemm_impl.hpp, instantiated per encoding in gemm_<enc>.hip.
#include "gemm_impl.hpp"

#include <algorithm>

namespace dmx {
namespace gemm {

extern template hipError_t launch_plan<ENC_Q4_0>(const GemmArgs&, const GemmPlan&, hipStream_t);
extern template hipError_t launch_plan<ENC_Q4_1>(const GemmArgs&, const GemmPlan&, hipStream_t);
extern template hipError_t launch_plan<ENC_Q8_0>(const GemmArgs&, const GemmPlan&, hipStream_t);
extern template hipError_t launch_plan<ENC_Q6_K>(const GemmArgs&, const GemmPlan&, hipStream_t);
extern template hipError_t launch_plan<ENC_Q4_K>(const GemmArgs&, const GemmPlan&, hipStream_t);
extern template hipError_t launch_plan<ENC_Q5_K>(const GemmArgs&, const GemmPlan&, hipStream_t);
extern template hipError_t launch_plan<ENC_IQ4_XS>(const GemmArgs&, const GemmPlan&, hipStream_t);
extern template hipError_t launch_plan<ENC_MLX_U4>(const GemmArgs&, const GemmPlan&, hipStream_t);

namespace {

bool fits_enc(uint32_t enc, uint32_t tm, uint32_t nb, uint32_t s, uint32_t wn, uint32_t wm) {
    switch (enc) {
        case ENC_Q4_0: return fits<ENC_Q4_0>(tm, nb, s, wn, wm);
        case ENC_Q4_1: return fits<ENC_Q4_1>(tm, nb, s, wn, wm);
        case ENC_Q8_0: return fits<ENC_Q8_0>(tm, nb, s, wn, wm);
        case ENC_Q6_K: return fits<ENC_Q6_K>(tm, nb, s, wn, wm);
        case ENC_Q4_K: return fits<ENC_Q4_K>(tm, nb, s, wn, wm);
        case ENC_Q5_K: return fits<ENC_Q5_K>(tm, nb, s, wn, wm);
        case ENC_IQ4_XS: return fits<ENC_IQ4_XS>(tm, nb, s, wn, wm);
        case ENC_MLX_U4: return fits<ENC_MLX_U4>(tm, nb, s, wn, wm);
        default: return false;
    }
}

}  // namespace
}  // namespace gemm

using gemm::GemmArgs;

uint32_t gemm_layout(uint32_t enc) {
    switch (enc) {
        case ENC_Q4_0:
        case ENC_Q4_1: return XFRAG_NIB;
        case ENC_Q8_0: return XFRAG_BYTE;
        case ENC_Q6_K: return XFRAG_Q6K;
        case ENC_Q4_K:
        case ENC_Q5_K: return XFRAG_QK;
        case ENC_IQ4_XS: return XFRAG_NIB;  // a sub-block laid out as a Q4_0 block
        case ENC_MLX_U4: return XFRAG_WORD;
        default: return ~0u;
    }
}

bool gemm_supported(uint32_t enc, uint32_t N, uint32_t K, uint32_t M) {
    return gemm_layout(enc) != ~0u && N > 0 && M > 0 && K >= 64u &&
           K % (enc == ENC_Q6_K || enc == ENC_Q4_K || enc == ENC_Q5_K || enc == ENC_IQ4_XS ? 256u : 64u) == 0;
}

// Launch plan from a cost model fitted to graph-replayed launches of every
// configuration on 86 shapes of each of six encodings (M 20..2048, N 1024..24576, K
// 768..12288; Q4_0, Q6_K, Q5_K, Q8_0, IQ4_XS, MLX U4), in us:
//   t = 0.86 + wg·(1 + r·(rounds - 1)),
//   wg = 1.04 + 0.101·TM·NB·S' + nc·(0.00165·V + 0.0673·TM·NB + 0.38)·(1 + 0.37·(w - 1)),
// with rounds = ceil(workgroups / 256), nc the 64-k chunks per wave, V the decode and
// scale VALU of a chunk, w waves per SIMD, S' = S (the epilogue's LDS round trip of
// the partial tiles), r = 0.75 where several workgroups fit a CU (small tiles of four
// waves), otherwise 1.  128x256 tiles of four waves (4, 2, 1, 4, 1), which take the
// fewest bytes from L2 per MFMA beside the 256x256 ones, cost f = 0.84 + 0.0173 for each
// copy of their four weight windows above 12 of that: timed over 1704 shapes (eight
// encodings, M 17..4096) a planner without them took 8% longer on 72 and on none
// less (Q4_0 1536 x 4096 x 4096 84 -> 68 us, 2048 x 4096 x 4096 90 -> 79, 1024 x 24576 x
// 4096 230 -> 207, Q4_K 3000 x 2560 x 2560 69 -> 59); with Q6_K's eight copies a wave, of
// scattered dwords, the 256x128 tiles that share windows stay (2048 x 3072 x 1024 33 us
// against 41).  The configuration it picks takes 1.1% longer on average than the best of
// them (8% at the 95th percentile, 31% at worst).
GemmPlan gemm_plan(uint32_t enc, const uint32_t* N, int count, uint32_t K, uint32_t M) {
    const uint32_t mb = (M + 31u) / 32u, nchk = K / 64u;
    const double valu = 4.0 * gemm::decode_valu(enc) + gemm::scale_valu(enc);
    GemmPlan best{};
    double best_t = 1e300;
    auto consider = [&](uint32_t tm, uint32_t nb, uint32_t s, uint32_t wn, uint32_t wm) {
        if (s == 2u) return;  // below
        // slices that share slots are equal; a slice holds at least one chunk
        if (!gemm::fits_enc(enc, tm, nb, s, wn, wm) || (wn * wm > 1u ? nchk % s != 0 : nchk < s)) return;
        // half the rows would do (but up to 32 rows two row blocks cost nothing more to copy,
        // and wider tiles fewer rounds: Q8_0 17 x 24576 x 4096 43 -> 37 us)
        if (nchk >= 4u && tm * wm > 1u && tm * wm / 2u >= mb && !(mb == 1u && tm * wm == 2u)) return;
        uint32_t nt = 0;
        for (int i = 0; i < count; i++) nt += (N[i] + 32u * nb * wn - 1u) / (32u * nb * wn);
        const uint32_t mt = (mb + tm * wm - 1u) / (tm * wm);
        const double nc = (double)((nchk + s - 1u) / s), rounds = (double)(((uint64_t)mt * nt + 255u) / 256u);
        const double w = s * wn * wm / 4.0, tiles = tm * nb;
        const double wg = 1.04 + 0.101 * tiles * s +
                          nc * (0.00165 * nb * valu + 0.0673 * tiles + 0.38) * (1.0 + 0.37 * (w - 1.0));
        const double f = tm == 4u && wn == 4u ? 0.84 + 0.0173 * (4.0 * gemm::window_copies(enc) - 12.0) : 1.0;
        const double t = f * (0.86 + wg * (1.0 + (tiles <= 4.0 && tm <= 2u && w == 1.0 ? 0.75 : 1.0) * (rounds - 1.0)));
        if (t < best_t * 0.999) {
            best_t = t;
            best = {tm, nb, s, wn, wm, mt, nt};
        }
    };
#define X(TM, NB, S, WN, WM) consider(TM, NB, S, WN, WM);
    DMX_GEMM_CONFIGS(X)
#undef X
    // Rows from three quarters of the columns in one round of 256x64 tiles: 128x128 tiles, of
    // the same area, in two K slices load fewer bytes of X (Q4_0 3000 x 1024 x 3072 49.2 ->
    // 46.4 us, 1536 x 2048 x 2048 32.5 -> 30.4, Q4_K 3000 x 1024 x 4096 64.5 -> 60.5; of eight
    // shapes each of Q4_0, Q4_1, Q4_K and IQ4_XS none slower; fewer rows, 768 x 4096 x 1024, up
    // to 6% slower, and so are the windows of more copies: MLX 3%, Q5_K 5%, Q6_K 18%).
    uint64_t cols = 0;
    for (int i = 0; i < count; i++) cols += N[i];
    if (best.tm == 8u && best.s == 4u && 4ull * M >= 3ull * cols && nchk % 2u == 0 && gemm::fits_enc(enc, 4, 2, 2, 2, 1)) {
        uint32_t nt = 0;
        for (int i = 0; i < count; i++) nt += (N[i] + 127u) / 128u;
        const uint32_t mt = (mb + 3u) / 4u;
        if (best.mt * best.nt <= 256u && mt * nt <= 256u) best = {4, 2, 2, 2, 1, mt, nt};
    }
    return best;
}

hipError_t gemm_launch(const GemmWeight* wts, int count, uint32_t K, const uint16_t* xh, const float* rs, uint32_t M,
                       bool y_bf16, hipStream_t st) {
    if (count < 1 || count > kMaxProblems) return hipErrorInvalidValue;
    const GemmWeight& w0 = wts[0];
    const uint32_t enc = w0.enc;
    uint32_t N[kMaxProblems];
    uint64_t ntotal = 0;
    for (int i = 0; i < count; i++) {
        const GemmWeight& wt = wts[i];
        if (wt.enc != enc || !gemm_supported(enc, wt.N, K, M)) return hipErrorInvalidValue;
        if (enc == ENC_MLX_U4 && (wt.group == 0 || wt.group % 32u || K % wt.group || wt.group != w0.group ||
                                  wt.sdtype != w0.sdtype || wt.sdtype > DT_BF16 || !wt.sc || !wt.bi))
            return hipErrorInvalidValue;
        N[i] = wt.N;
        ntotal += wt.N;
    }
    const GemmPlan p = gemm_plan(enc, N, count, K, M);
    if (p.tm == 0) return hipErrorInvalidConfiguration;
    GemmArgs a{};
    a.xh = xh;
    a.rs = rs;
    a.M = M;
    a.K = K;
    a.mt = p.mt;
    a.nt = p.nt;
    a.y_bf16 = y_bf16 ? 1u : 0u;
    a.group = w0.group;
    a.gmagic = group_magic(w0.group);
    a.sdtype = w0.sdtype;
    a.np = (uint32_t)count;
    for (int i = 0, nt0 = 0; i < count; i++) {
        a.p[i] = {wts[i].w, wts[i].sc, wts[i].bi, wts[i].y, wts[i].N, (uint32_t)nt0};
        nt0 += (int)((wts[i].N + 32u * p.nb * p.wn - 1u) / (32u * p.nb * p.wn));
    }
    switch (enc) {
        case ENC_Q4_0: a.rowbytes = (uint64_t)(K / 32u) * 18u; break;
        case ENC_Q4_1: a.rowbytes = (uint64_t)(K / 32u) * 20u; break;
        case ENC_Q8_0: a.rowbytes = (uint64_t)(K / 32u) * 34u; break;
        case ENC_Q6_K: a.rowbytes = (uint64_t)(K / 256u) * 210u; break;
        case ENC_Q4_K: a.rowbytes = (uint64_t)(K / 256u) * 144u; break;
        case ENC_Q5_K: a.rowbytes = (uint64_t)(K / 256u) * 176u; break;
        case ENC_IQ4_XS: a.rowbytes = (uint64_t)(K / 256u) * 136u; break;
        default: a.rowbytes = (uint64_t)K / 2u; break;  // MLX packed words (scales and biases besides)
    }
    // M-major tile order when the staged activations (2 bytes per element)
    // outweigh the weights (M2048 N3072 K1024: 34.3 against 35.9 us per call)
    a.mmajor = (uint64_t)M * K * 2u > ntotal * a.rowbytes ? 1u : 0u;
    switch (enc) {
        case ENC_Q4_0: return gemm::launch_plan<ENC_Q4_0>(a, p, st);
        case ENC_Q4_1: return gemm::launch_plan<ENC_Q4_1>(a, p, st);
        case ENC_Q8_0: return gemm::launch_plan<ENC_Q8_0>(a, p, st);
        case ENC_Q6_K: return gemm::launch_plan<ENC_Q6_K>(a, p, st);
        case ENC_Q4_K: return gemm::launch_plan<ENC_Q4_K>(a, p, st);
        case ENC_Q5_K: return gemm::launch_plan<ENC_Q5_K>(a, p, st);
        case ENC_IQ4_XS: return gemm::launch_plan<ENC_IQ4_XS>(a, p, st);
        case ENC_MLX_U4: return gemm::launch_plan<ENC_MLX_U4>(a, p, st);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace dmx
