// Prefill GEMM on gfx950 MFMA for the GGUF encodings Q4_0, Q4_1, Q8_0, Q6_K,
// Q4_K, Q5_K and IQ4_XS and for MLX affine U4: Y[M, N] = X[M, K] · Wᵀ with f32
// accumulation.  Kernel templates; gemm.hip plans a launch, and gemm_<enc>.hip
// instantiate the kernels of one encoding each (so they compile in parallel).
//
// Reference semantics: the same `emit_linear` contraction as decode
// (gguf_codegen.rs:268-314, dequantisations :412-472 Q4_0, :382-410 Q8_0,
// :474-526 Q6_K, q4.rs Q4_1; mlx_affine.rs:557-626 `emit_linear_u4`) with
// rows = the prefill window/chunk (512 when paged,
// parameter.rs:107-121, dense_decoder.rs:53-56).
//
// Data path.  W is read as GGUF blocks straight from HBM (no repack); X
// arrives staged by xprep.hip as f16 fragments of the MFMA operand, each row
// scaled by a power of two that rs[m] undoes.
//   * One launch serves up to four weights that share X (q/k/v, gate/up).
//   * A workgroup of S·WN·WM waves owns a (32·TM·WM) x (32·NB·WN) tile of one
//     weight's Y: each wave a (32·TM) x (32·NB) tile (TM x NB blocks of
//     v_mfma_f32_32x32x16_f16), the waves split over S K slices, WN column and WM
//     row subtiles.
//   * K advances in chunks of two weight blocks (64 k, four MFMA k steps).  Weight
//     bytes go to an LDS ring by buffer loads into LDS (16 or 4 bytes per lane,
//     counted by vmcnt, no registers held), each wave's window of the chunk;
//     activation fragments (1 KiB each, contiguous in HBM) the same way where waves
//     share them, straight to registers a chunk ahead where a slice is one wave's.
//   * What bounds it: one wave issues at most one VALU instruction per 8 cycles (two
//     waves on a SIMD together one per 4), an MFMA takes 33, so up to 4 VALU
//     instructions per MFMA and wave are free and the decode, NB·(16..30) per TM·NB
//     MFMAs, wants TM >= 4; an activation fragment read from LDS feeds NB MFMAs, so
//     NB = 1 over shared fragments is bound by LDS (1 KiB per MFMA, 128 B/clk); small
//     M and short K are bound by the first copies' latency and the epilogue, so
//     those take many small tiles with K split over the waves (gemm_plan).
//     Measured (kernel trace, median and least of the launches in a stream of calls,
//     against the same tile shapes with a two-slot ring shared by four waves, one
//     launch per weight): Q4_0 2048 x 24576 x 4096 507 (464 at least) -> 405 us (352,
//     1.17 PFLOP/s), Q6_K 2048 x 4096 x 12288 417 (410) -> 290 (277), 512 x 4096 x
//     12288 189 (186) -> 103 (101), Q5_K 45 x 24576 x 4096 51.3 (50.0) -> 35.3 (34.7),
//     Q4_0 512 x 4096 x 1024 in three weights 23.4 (22.4) -> 10.9 (10.8).
//   * Every lane decodes 32 weights of one row per N-block straight into A
//     operands: lane l takes weight row l % 32 of a 32-row block and its half
//     h = l / 32 of the chunk (the block h, for blocks of 32), so an MFMA k step
//     pairs 8 k of half 0 (lanes 0..31) with 8 k of half 1 (lanes 32..63), and
//     xprep stages the activations in that order.  A code at mantissa bits 0.. under the
//     f16 exponent of 1024 is 1024 + c, one at bits 4.. under that of 64 is
//     64 + c (one v_and_or_b32 per two codes, both exact); a packed add removes
//     the offset (exact) and a packed multiply by the block scale rounds once
//     (Q4_0 RNE_f16((q-8)·d), Q8_0 RNE_f16(q·d)); Q4_1 a packed fma,
//     RNE_f16(q·d + m); Q6_K RNE_f16((q-32)·RNE_f16(d·sc)) (WinQ6K); MLX U4
//     RNE_f16(q·s + b) (WinMlx); Q4_K RNE_f16(q·RNE_f16(d·sc) - RNE_f16(dmin·m))
//     (WinQK); IQ4_XS RNE_f16(kv·RNE_f16(d·(ls - 32))) (WinIQ4XS).
//   * The weights are the MFMA's A operand and the activations its B, so each
//     lane ends with 4 consecutive output columns of one row per block.  K
//     slices meet in LDS after the loop, summed in slice order
//     (deterministic); then the rows are scaled by rs[m] and stored as whole
//     16-byte (f32) or 8-byte (bf16) column groups.
// Accuracy: |y - y_exact| <= 2^-10·Σ|w||x| (one f16 rounding of each weight and
// of each activation; Q6_K's weights round twice: (2^-10 + 2^-11)·Σ|w||x|;
// Q4_K's scale and offset round once each, adding 2^-11·Σ(|q·d·sc| + |dmin·m|)|x|) +
// f32 accumulation error, inside the 2e-3 normalised tolerance.  Weights must
// be finite in f16 (|w| <= 65504: |d| <= 8188 for Q4_0, |d·sc| <= 2047 for
// Q6_K).
#pragma once
#include "device_common.hpp"
#include "kernels.hpp"

#include <type_traits>

namespace dmx {
namespace gemm {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

constexpr uint32_t kLdsMax = 160u * 1024u;

// One weight of a grouped launch: its column tiles are nt0 .. nt0 + its own.
struct GemmProb {
    const uint8_t* w;
    const uint8_t* sc;  // MLX U4: scales and biases [N, K/group] of dtype sdtype
    const uint8_t* bi;
    void* y;
    uint32_t N, nt0;
};

struct GemmArgs {
    const uint16_t* xh;
    const float* rs;
    uint64_t rowbytes;
    uint32_t M, K;
    uint32_t mt, nt;  // workgroup tiles along M and (every weight's) along N
    uint32_t y_bf16;
    uint32_t mmajor;  // tile order: 1 = M-major (consecutive tiles share activation rows)
    uint32_t group, sdtype;
    uint32_t gmagic;  // group_magic(group)
    uint32_t np;
    GemmProb p[kMaxProblems];
};

// A constant the compiler keeps in a scalar (vector) register and does not see
// through, so that (a & mask) | magic stays one v_and_or_b32 (a VOP3 op takes no
// literal and one scalar operand on gfx9).
__device__ __forceinline__ uint32_t in_sgpr(uint32_t v) {
    asm("" : "+s"(v));
    return v;
}
__device__ __forceinline__ uint32_t in_vgpr(uint32_t v) {
    asm("" : "+v"(v));
    return v;
}
__device__ __forceinline__ uint32_t and_or(uint32_t a, uint32_t m, uint32_t b) { return (a & m) | b; }
__device__ __forceinline__ h2 as_h2(uint32_t v) { return __builtin_bit_cast(h2, v); }
__device__ __forceinline__ uint32_t as_u(h2 v) { return __builtin_bit_cast(uint32_t, v); }
__device__ __forceinline__ h8 as_h8(uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
    return __builtin_bit_cast(h8, u32x4{a, b, c, d});
}


// Copies into LDS through a buffer descriptor: 16 (4) bytes per lane from base +
// voff + soff into dst + 16·lane (4·lane), counted by vmcnt.  The chunk's offset is
// scalar and the lane's constant, so a copy takes no vector instruction (the
// global form added a 64-bit address per lane and copy).
struct Src {
    __amdgpu_buffer_rsrc_t r;
    __device__ __forceinline__ void set(const void* p) {
        r = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, -1, 0x00027000);
    }
    __device__ __forceinline__ h8 load16(uint32_t voff, uint32_t soff) const {
        return __builtin_bit_cast(h8, __builtin_amdgcn_raw_buffer_load_b128(r, (int)voff, (int)soff, 0));
    }
    __device__ __forceinline__ void dma16(uint32_t voff, uint32_t soff, void* dst) const {
        __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)dst, 16, (int)voff, (int)soff,
                                                 0, 0);
    }
    __device__ __forceinline__ void dma4(uint32_t voff, uint32_t soff, void* dst) const {
        __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)dst, 4, (int)voff, (int)soff, 0,
                                                 0);
    }
};

// ring_barrier<BASE + k·PER>() (ring_wait when !SYNC) for a wave-uniform k in
// [0, KMAX]: the copies of the k newest chunks, and BASE newer register
// loads, may stay in flight.
template <uint32_t PER, uint32_t KMAX, uint32_t BASE = 0, bool SYNC = true>
__device__ __forceinline__ void ring_barrier_k(uint32_t k) {
    if constexpr (KMAX == 0) {
        if constexpr (SYNC) ring_barrier<BASE>();
        else ring_wait<BASE>();
    } else {
        if (k >= KMAX) {
            if constexpr (SYNC) ring_barrier<BASE + KMAX * PER>();
            else ring_wait<BASE + KMAX * PER>();
        } else {
            ring_barrier_k<PER, KMAX - 1, BASE, SYNC>(k);
        }
    }
}

// Per-encoding block geometry and decode.  A lane reads kDw dwords from the
// 4-byte-aligned dword holding its block's first byte (sh = the block start's
// offset in that dword, 0 or 2); scale() takes the block's f16 scale(s) from
// them and step(t) decodes the MFMA operand of the chunk's k step t: 8 k of
// the block, as 4 packed f16 pairs.
template <uint32_t ENC>
struct Blk;

template <>
struct Blk<ENC_Q4_0> {
    // d (2 B) then 16 code bytes; byte j: k = j (low nibble), k = j + 16 (high).
    // Step t: code bytes 4t..4t+3 -> k = 4t+(0,2), 4t+(1,3), 16+4t+(0,2), 16+4t+(1,3).
    static constexpr uint32_t kBytes = 18, kDw = 5, kLayout = XFRAG_NIB;
    struct Scale {
        h2 d;
        uint32_t sel;
    };
    __device__ static Scale scale(const uint32_t* r, uint32_t sh) {
        return {as_h2(__builtin_amdgcn_perm(r[0], r[0], 0x01000100u + 0x01010101u * sh)),
                0x05040302u + 0x01010101u * sh};  // block bytes 2+4t..5+4t from dwords t, t+1
    }
    __device__ static h8 step(const uint32_t* r, const Scale& s, int t) {
        const h2 ol = {(_Float16)-1032.0f, (_Float16)-1032.0f}, oh = {(_Float16)-72.0f, (_Float16)-72.0f};
        const uint32_t ml = in_vgpr(0x64006400u), mh = in_vgpr(0x54005400u);
        const uint32_t kl = in_sgpr(0x000F000Fu), kh = in_sgpr(0x00F000F0u);
        auto lo = [&](uint32_t v) { return as_u((as_h2(and_or(v, kl, ml)) + ol) * s.d); };
        auto hi = [&](uint32_t v) { return as_u((as_h2(and_or(v, kh, mh)) + oh) * s.d); };
        const uint32_t q = __builtin_amdgcn_perm(r[t + 1], r[t], s.sel), q8 = q >> 8;
        return as_h8(lo(q), lo(q8), hi(q), hi(q8));
    }
};

template <>
struct Blk<ENC_Q4_1> {
    // d, m (2 B each) then 16 code bytes (4-byte-aligned blocks): w = q·d + m;
    // k order as Q4_0.
    static constexpr uint32_t kBytes = 20, kDw = 5, kLayout = XFRAG_NIB;
    struct Scale {
        h2 d, m;
    };
    __device__ static Scale scale(const uint32_t* r, uint32_t) {
        return {as_h2(__builtin_amdgcn_perm(r[0], r[0], 0x01000100u)),
                as_h2(__builtin_amdgcn_perm(r[0], r[0], 0x03020302u))};
    }
    __device__ static h8 step(const uint32_t* r, const Scale& s, int t) {
        const h2 ol = {(_Float16)-1024.0f, (_Float16)-1024.0f}, oh = {(_Float16)-64.0f, (_Float16)-64.0f};
        const uint32_t ml = in_vgpr(0x64006400u), mh = in_vgpr(0x54005400u);
        const uint32_t kl = in_sgpr(0x000F000Fu), kh = in_sgpr(0x00F000F0u);
        auto lo = [&](uint32_t v) {
            return as_u(__builtin_elementwise_fma(as_h2(and_or(v, kl, ml)) + ol, s.d, s.m));
        };
        auto hi = [&](uint32_t v) {
            return as_u(__builtin_elementwise_fma(as_h2(and_or(v, kh, mh)) + oh, s.d, s.m));
        };
        const uint32_t q = r[t + 1], q8 = q >> 8;
        return as_h8(lo(q), lo(q8), hi(q), hi(q8));
    }
};

template <>
struct Blk<ENC_Q8_0> {
    // d (2 B) then 32 int8 codes; step t: codes 8t..8t+7 in the order
    // (0,2) (1,3) (4,6) (5,7): a code c as (c ^ 0x80) under the exponent of 1024
    // is 1152 + c.
    static constexpr uint32_t kBytes = 34, kDw = 9, kLayout = XFRAG_BYTE;
    struct Scale {
        h2 d;
        uint32_t sel;
    };
    __device__ static Scale scale(const uint32_t* r, uint32_t sh) {
        return {as_h2(__builtin_amdgcn_perm(r[0], r[0], 0x01000100u + 0x01010101u * sh)),
                0x05040302u + 0x01010101u * sh};
    }
    __device__ static h8 step(const uint32_t* r, const Scale& s, int t) {
        const h2 o = {(_Float16)-1152.0f, (_Float16)-1152.0f};
        const uint32_t ml = in_vgpr(0x64006400u), kb = in_sgpr(0x00FF00FFu);
        auto p = [&](uint32_t v) { return as_u((as_h2(and_or(v, kb, ml)) + o) * s.d); };
        const uint32_t c0 = __builtin_amdgcn_perm(r[2 * t + 1], r[2 * t], s.sel) ^ 0x80808080u;
        const uint32_t c1 = __builtin_amdgcn_perm(r[2 * t + 2], r[2 * t + 1], s.sel) ^ 0x80808080u;
        return as_h8(p(c0), p(c0 >> 8), p(c1), p(c1 >> 8));
    }
};

// Copy q of a wave that makes part `part` of PARTS of a window's ALL copies.
template <uint32_t PARTS, uint32_t ALL>
__device__ __forceinline__ uint32_t copy_index(uint32_t q, uint32_t part) {
    if constexpr (PARTS == 1) return q;
    const uint32_t qq = q * PARTS + part;
    return qq < ALL ? qq : ALL - 1u;
}

// A wave's weight window: the bytes of its 32·NB weight rows for one 64-k
// chunk, copied into LDS by global_load_lds (16 or 4 bytes per lane, the
// lane's LDS slot at dst + 16·lane or 4·lane), then read and decoded by each
// lane: row 32j + l % 32 of N-block j (j < NB), block (or half-step) h = l / 32
// of the chunk.  A copy instruction whose lanes run past the window's pieces
// re-copies its last valid piece into the window's unread tail, so every
// instruction has the same lanes active and the ring's wait counts hold.
//
// GGUF blocks of 32 weights: a row's two blocks of the chunk are contiguous;
// they are copied from their 4-byte-aligned start as NP 16-byte pieces
// (consecutive lanes on consecutive pieces of a row), the last piece moved
// back so that no read passes the blocks' last dword.
//
// PARTS waves share a window (the waves of an M split): each copies
// every PARTS-th copy instruction (the count rounded up: the last one may be
// copied twice, the same bytes to the same place).
template <uint32_t ENC, int NB, uint32_t PARTS>
struct WinBlocks {
    using B = Blk<ENC>;
    using Scale = typename B::Scale;
    static constexpr uint32_t kRows = 32u * NB;
    static constexpr uint32_t kSpanMax = (2u * B::kBytes + 2u + 3u) & ~3u;  // a row's two blocks, aligned
    static constexpr uint32_t NP = (kSpanMax + 15u) / 16u;                   // 16-byte pieces per row
    static constexpr uint32_t kAll = (kRows * NP + 63u) / 64u;                // copy instructions per chunk
    static constexpr uint32_t kCopies = (kAll + PARTS - 1u) / PARTS;           // ... of one wave
    static constexpr uint32_t kBytes = kAll * 1024u;
    static constexpr uint32_t kDw = B::kDw, kReads = B::kDw;  // (LDS reads of a window per N-block)
    Src base;                       // from the dword holding the weight's first byte
    uint32_t src[kCopies];          // copy lane's piece for the slice's first chunk, from base
    uint32_t dst[kCopies];          // its copy's place in the window
    uint32_t off[NB][kDw], sh[NB];  // this lane's block dwords in the window, its block's start offset

    __device__ void init(const GemmArgs& a, const GemmProb& pr, uint32_t n0, uint32_t lane, uint32_t c0, uint32_t part) {
        const uint32_t b0 = (uint32_t)((uintptr_t)pr.w & 3u);
        base.set(pr.w - b0);
        // offset of row r's blocks from base (a weight is below 4 GiB)
        auto start_of = [&](uint32_t r) {
            const uint32_t n = n0 + r < pr.N ? n0 + r : pr.N - 1u;  // past N: re-read the last row (never stored)
            return b0 + n * (uint32_t)a.rowbytes + B::kBytes * 2u * c0;
        };
#pragma unroll
        for (uint32_t q = 0; q < kCopies; q++) {
            const uint32_t qq = copy_index<PARTS, kAll>(q, part);
            dst[q] = 1024u * qq;
            uint32_t li = 64u * qq + lane;
            li = li < kRows * NP ? li : kRows * NP - 1u;
            const uint32_t r = li / NP, p = li % NP;
            const uint32_t start = start_of(r), al = start & ~3u;
            const uint32_t span = ((start + 2u * B::kBytes + 3u) & ~3u) - al;
            src[q] = al + (p + 1u < NP ? 16u * p : span - 16u);
        }
        // dword k of the lane's block (from its aligned start) at window offset
        // off[j][k]: span bytes past the first NP - 1 pieces sit in the last
        // piece, moved back by span - 16·NP
        const uint32_t h = lane >> 5;
#pragma unroll
        for (int j = 0; j < NB; j++) {
            const uint32_t r = 32u * j + (lane & 31u);
            const uint32_t s0 = start_of(r) & 3u;
            const uint32_t span = (2u * B::kBytes + s0 + 3u) & ~3u;
            const uint32_t bstart = s0 + B::kBytes * h;
            sh[j] = bstart & 3u;
#pragma unroll
            for (uint32_t k = 0; k < kDw; k++) {
                const uint32_t o = (bstart & ~3u) + 4u * k;
                off[j][k] = r * NP * 16u + (o < 16u * (NP - 1u) ? o : o - span + 16u * NP);
            }
        }
    }
    __device__ void issue(uint32_t c, uint8_t* win) const {
#pragma unroll
        for (uint32_t q = 0; q < kCopies; q++) base.dma16(src[q], c * 2u * B::kBytes, win + dst[q]);
    }
    __device__ void read(uint32_t, const uint8_t* win, uint32_t* raw) const {
#pragma unroll
        for (int j = 0; j < NB; j++)
#pragma unroll
            for (uint32_t k = 0; k < kDw; k++) raw[j * kDw + k] = *reinterpret_cast<const uint32_t*>(win + off[j][k]);
    }
    __device__ Scale scale(uint32_t, int j, const uint32_t* r) const { return B::scale(r, sh[j]); }
    __device__ h8 step(const uint32_t* r, const Scale& s, int t) const { return B::step(r, s, t); }
};

// GGUF Q6_K (super-blocks of 256 weights, 210 bytes: ql[128], qh[64], int8
// scales[16], f16 d; gguf_codegen.rs:474-526).  Weight 128·n + 32·j + l of a
// super-block (j = 0..3, l = 0..31) is the (j / 2) nibble of ql[64·n + 32·(j%2) + l]
// under bits 2j of qh[32·n + l], scaled by d·scales[8·n + 2j + l/16].  Chunk g of a
// row takes the 64 weights n = (g / 2) % 2, l = 16·m + 0..15 (m = g % 2), all j:
// both nibbles and all four bit pairs of the bytes it loads, so no byte is loaded
// for two chunks (a chunk of 64 consecutive weights used half of each, 116 bytes
// a row instead of 80).  Lane half h holds the ql bytes of j = h and h + 2: k steps
// 0, 1 are its low nibbles (j = h), 2, 3 its high ones (j = h + 2), 8 weights each,
// pairs (l, l+2) as Q8_0's (XFRAG_Q6K).  The window per row: three 16-byte pieces
// (ql of h = 0, of h = 1, qh), 16 bytes with the chunk's scales, and four dwords:
// the one past each piece (a super-block starting 2 bytes into its dword) and d's.
// Every copy lies within the super-block's dwords.
template <int NB, uint32_t PARTS>
struct WinQ6K {
    static constexpr uint32_t kRows = 32u * NB;
    static constexpr uint32_t kP16 = (kRows * 3u + 63u) / 64u, kT16 = (kRows + 63u) / 64u, kAll16 = kP16 + kT16;
    static constexpr uint32_t kAll4 = kRows * 4u / 64u;
    static constexpr uint32_t kN16 = (kAll16 + PARTS - 1u) / PARTS, kN4 = (kAll4 + PARTS - 1u) / PARTS;
    static constexpr uint32_t kCopies = kN16 + kN4;
    static constexpr uint32_t kOffT = 1024u * kP16, kOff4 = 1024u * kAll16;
    static constexpr uint32_t kBytes = kOff4 + 256u * kAll4;
    static constexpr uint32_t kDw = 13, kReads = 7;  // ql 5, qh 5, two scales, d
    struct Scale {
        uint32_t c[4], c8[4], eL[4], eR[4];  // code bytes, qh bits under the nibbles; the odd bytes' moved down
        h2 ds0, ds1;
    };
    // A copy lane's piece lies at ((row + 210·sb) & ~3) + offset: 210·sb is 2 mod 4
    // for odd sb, so that is a per-lane constant, a per-lane step for odd sb, one
    // for n = 1, and a scalar.
    Src base;  // from the dword holding the weight's first byte
    uint32_t v16[kN16], u16[kN16], h16[kN16], m16[kN16], d16[kN16], v4[kN4], u4[kN4], h4[kN4], m4[kN4], d4[kN4];
    uint32_t row[NB];  // this lane's rows' start mod 4
    uint32_t c0, h, lane;

    __device__ void init(const GemmArgs& a, const GemmProb& pr, uint32_t n0, uint32_t lane_, uint32_t c0_, uint32_t part) {
        lane = lane_;
        c0 = c0_;
        h = lane >> 5;
        const uint32_t b0 = (uint32_t)((uintptr_t)pr.w & 3u);
        base.set(pr.w - b0);
        auto rowp = [&](uint32_t r) {
            const uint32_t n = n0 + r < pr.N ? n0 + r : pr.N - 1u;  // past N: re-read the last row (never stored)
            return b0 + n * (uint32_t)a.rowbytes;  // a weight is below 4 GiB
        };
#pragma unroll
        for (uint32_t q = 0; q < kN16; q++) {
            const uint32_t qq = copy_index<PARTS, kAll16>(q, part);
            d16[q] = 1024u * qq;
            const bool sc = qq >= kP16;  // a copy of scales: one piece a row
            uint32_t li = 64u * (sc ? qq - kP16 : qq) + lane;
            li = li < kRows * (sc ? 1u : 3u) ? li : kRows * (sc ? 1u : 3u) - 1u;
            const uint32_t p = sc ? 3u : li % 3u, rb = rowp(sc ? li : li / 3u);
            v16[q] = (rb & ~3u) + (p == 3u ? 192u : p == 2u ? 128u : 32u * p);
            u16[q] = (rb & 2u) * 2u;  // odd sb: 210·sb - 2, plus 4 in rows starting 2 bytes into a dword
            h16[q] = p == 3u ? 4u : p == 2u ? 32u : 64u;
            m16[q] = p == 3u ? 0u : 16u;
        }
#pragma unroll
        for (uint32_t q = 0; q < kN4; q++) {
            const uint32_t qq = copy_index<PARTS, kAll4>(q, part);
            d4[q] = kOff4 + 256u * qq;
            const uint32_t li = 64u * qq + lane, p = li % 4u, rb = rowp(li / 4u);
            v4[q] = (rb & ~3u) + (p == 3u ? 208u : p == 2u ? 144u : 16u + 32u * p);
            u4[q] = (rb & 2u) * 2u;
            h4[q] = p == 3u ? 0u : p == 2u ? 32u : 64u;
            m4[q] = p == 3u ? 0u : 16u;
        }
#pragma unroll
        for (int j = 0; j < NB; j++) row[j] = rowp(32u * j + (lane & 31u)) & 3u;
    }
    __device__ void issue(uint32_t c, uint8_t* win) const {
        const uint32_t g = c0 + c, sb = g >> 2, n = (g >> 1) & 1u, m = g & 1u;
        const uint32_t odd = sb & 1u, at = 210u * sb - 2u * odd;
#pragma unroll
        for (uint32_t q = 0; q < kN16; q++)
            base.dma16(v16[q] + __umul24(u16[q], odd) + __umul24(h16[q], n) + __umul24(m16[q], m), at, win + d16[q]);
#pragma unroll
        for (uint32_t q = 0; q < kN4; q++)
            base.dma4(v4[q] + __umul24(u4[q], odd) + __umul24(h4[q], n) + __umul24(m4[q], m), at, win + d4[q]);
    }
    __device__ uint32_t shift_of(uint32_t c, int j) const { return (row[j] + 210u * ((c0 + c) >> 2)) & 3u; }
    // (16-byte reads at a pitch of 48 bytes: eight lanes on distinct banks)
    __device__ void read(uint32_t c, const uint8_t* win, uint32_t* raw) const {
        const uint32_t n = ((c0 + c) >> 1) & 1u, m = (c0 + c) & 1u;
#pragma unroll
        for (int j = 0; j < NB; j++) {
            const uint32_t r = 32u * j + (lane & 31u), sh = shift_of(c, j);
            const uint8_t *w = win + 48u * r, *x = win + kOff4 + 16u * r;
            const int8_t* s = reinterpret_cast<const int8_t*>(win + kOffT + 16u * r + 4u * n + m + 2u * h + sh);
            uint32_t* o = raw + j * kDw;
            const u32x4 l = *reinterpret_cast<const u32x4*>(w + 16u * h);
            const u32x4 q = *reinterpret_cast<const u32x4*>(w + 32u);
            o[0] = l.x, o[1] = l.y, o[2] = l.z, o[3] = l.w;
            o[4] = *reinterpret_cast<const uint32_t*>(x + 4u * h);
            o[5] = q.x, o[6] = q.y, o[7] = q.z, o[8] = q.w;
            o[9] = *reinterpret_cast<const uint32_t*>(x + 8u);
            o[10] = (uint32_t)(int32_t)s[0];
            o[11] = (uint32_t)(int32_t)s[4];
            o[12] = *reinterpret_cast<const uint16_t*>(x + 12u + sh);
        }
    }
    __device__ Scale scale(uint32_t c, int j, const uint32_t* r) const {
        const uint32_t sel = 0x03020100u + 0x01010101u * shift_of(c, j);
        const float d = f16_bits_to_f32(r[12]);
        const _Float16 d0 = (_Float16)(d * (float)(int32_t)r[10]);  // exact f32 product, one rounding
        const _Float16 d1 = (_Float16)(d * (float)(int32_t)r[11]);
        Scale s;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            s.c[i] = __builtin_amdgcn_perm(r[i + 1], r[i], sel);
            s.c8[i] = s.c[i] >> 8;
            const uint32_t e = __builtin_amdgcn_perm(r[6 + i], r[5 + i], sel);
            s.eL[i] = e << (4u - 2u * h);  // bits 2h (2h + 4) of bytes 0 and 2 to bit 4 (8)
            s.eR[i] = e >> (4u + 2u * h);  // ... of bytes 1 and 3
        }
        s.ds0 = h2{d0, d0};
        s.ds1 = h2{d1, d1};
        return s;
    }
    __device__ h8 step(const uint32_t*, const Scale& s, int t) const {
        // code bits under the exponent of 1024 (low nibbles) or 64
        const uint32_t mN = in_sgpr(t < 2 ? 0x000F000Fu : 0x00F000F0u), mH = in_sgpr(t < 2 ? 0x00300030u : 0x03000300u);
        const uint32_t magic = in_vgpr(t < 2 ? 0x64006400u : 0x54005400u);
        const _Float16 o = t < 2 ? (_Float16)-1056.0f : (_Float16)-96.0f;
        const h2 off = {o, o}, ds = t < 2 ? s.ds0 : s.ds1;
        auto f = [&](uint32_t cv, uint32_t ev) {
            return as_u((as_h2(and_or(ev, mH, and_or(cv, mN, magic))) + off) * ds);
        };
        const int i = 2 * (t & 1);
        return as_h8(f(s.c[i], s.eL[i]), f(s.c8[i], s.eR[i]), f(s.c[i + 1], s.eL[i + 1]), f(s.c8[i + 1], s.eR[i + 1]));
    }
};

// MLX affine U4 (mlx_affine.rs:557-626; packed u32 [N, K/8], nibble i of a
// word = k offset i, fixture.rs:307-311): a row's chunk is 8 words (32 bytes,
// 4-byte-aligned rows of K/2 bytes) copied as two 16-byte pieces, plus, per
// row, the dwords holding the scale and the bias of the chunk's two 32-k
// halves (always the same group only where 64 divides the group size: a chunk of
// groups of 96 may start in one group and end in the next).  Lane l decodes row 32j + l % 32
// of each N-block j, words 4h .. 4h+3 (h = l / 32): k step t takes word
// 4h + t, nibbles (0,4) (1,5) (2,6) (3,7) as packed pairs (XFRAG_WORD), code q
// exact in f16 and w = RNE_f16(q·s + b) by one packed fma, s and b taken to
// f16 first (bf16 and f16 values exact in f16's normal range; f32 rounded).
template <int NB, uint32_t PARTS>
struct WinMlx {
    static constexpr uint32_t kRows = 32u * NB;
    static constexpr uint32_t kPieces = kRows * 2u / 64u;        // 16-byte copies of the code words
    static constexpr uint32_t kMine = (kPieces + PARTS - 1u) / PARTS;
    static constexpr uint32_t kAuxQ = (kRows + 63u) / 64u;       // 4-byte copies per scale or bias array
    // the scales and biases of one group (PARTS 2: one wave copies the scales, the
    // other the biases); a second copy of each, not counted, where halves differ
    static constexpr uint32_t kCopies = kMine + 2u / PARTS * kAuxQ;
    static constexpr uint32_t kAuxOff = kPieces * 1024u;         // the aux dwords after every row's pieces
    static constexpr uint32_t kAuxPitch = 256u * kAuxQ;          // bytes per aux array: s0, s1, b0, b1
    static constexpr uint32_t kBytes = kAuxOff + 4u * kAuxPitch;
    static constexpr uint32_t kDw = 6, kReads = 3;  // 4 code words, scale dword, bias dword
    struct Scale {
        h2 s, b;
    };
    Src base, sbase, bbase;                  // the words; the dwords holding the first scale and bias
    uint32_t src[kMine], dst[kMine];         // copy lane's piece of the slice's first chunk, from base; its place
    uint32_t srow[kAuxQ], brow[kAuxQ];       // copy lane's row of scales and biases, from sbase and bbase
    uint32_t ssh[NB], bsh[NB];               // this lane's rows' scale and bias row starts mod 4 (per N-block j)
    uint32_t c0, es, gmagic, m32, m16, lane, mine, two;  // (m32, m16: all ones for f32, f16 scales; two: halves' groups differ)

    __device__ void init(const GemmArgs& a, const GemmProb& pr, uint32_t n0, uint32_t lane_, uint32_t c0_, uint32_t part) {
        lane = lane_;
        c0 = c0_;
        mine = part;
        two = a.group % 64u ? 1u : 0u;
        gmagic = a.gmagic;
        m32 = a.sdtype == DT_F32 ? ~0u : 0u;
        m16 = a.sdtype == DT_F16 ? ~0u : 0u;
        es = a.sdtype == DT_F32 ? 4u : 2u;
        const uint32_t rbytes = a.K / 2u, sbytes = a.K / a.group * es;
        auto rowc = [&](uint32_t r) { return n0 + r < pr.N ? n0 + r : pr.N - 1u; };  // past N: re-read the last row
        const uint32_t s0 = (uint32_t)((uintptr_t)pr.sc & 3u), b0 = (uint32_t)((uintptr_t)pr.bi & 3u);
        base.set(pr.w);
        sbase.set(pr.sc - s0);
        bbase.set(pr.bi - b0);
#pragma unroll
        for (uint32_t q = 0; q < kMine; q++) {
            const uint32_t qq = copy_index<PARTS, kPieces>(q, part), li = 64u * qq + lane;
            dst[q] = 1024u * qq;
            src[q] = rowc(li / 2u) * rbytes + 32u * c0 + 16u * (li % 2u);  // a component is below 4 GiB
        }
#pragma unroll
        for (uint32_t q = 0; q < kAuxQ; q++) {
            const uint32_t r = 64u * q + lane < kRows ? 64u * q + lane : kRows - 1u;
            srow[q] = s0 + rowc(r) * sbytes;
            brow[q] = b0 + rowc(r) * sbytes;
        }
#pragma unroll
        for (int j = 0; j < NB; j++) {
            const uint32_t o = rowc(32u * j + (lane & 31u)) * sbytes;
            ssh[j] = (s0 + o) & 3u;
            bsh[j] = (b0 + o) & 3u;
        }
    }
    // byte offset in a scale row of the group of the chunk's 32-k half hh
    __device__ uint32_t goff(uint32_t c, uint32_t hh) const { return div_magic(64u * (c0 + c) + 32u * hh, gmagic) * es; }
    __device__ void issue(uint32_t c, uint8_t* win) const {
        auto aux = [&](uint32_t hh) {
            const uint32_t o = goff(c, hh);
#pragma unroll
            for (uint32_t q = 0; q < kAuxQ; q++) {
                if (PARTS == 1 || mine == 0u)
                    sbase.dma4((srow[q] + o) & ~3u, 0u, win + kAuxOff + kAuxPitch * hh + 256u * q);
                if (PARTS == 1 || mine != 0u)
                    bbase.dma4((brow[q] + o) & ~3u, 0u, win + kAuxOff + kAuxPitch * (2u + hh) + 256u * q);
            }
        };
        if (two) aux(1);  // more copies than the waits count: they wait for older ones than they must
#pragma unroll
        for (uint32_t q = 0; q < kMine; q++) base.dma16(src[q], c * 32u, win + dst[q]);
        aux(0);
    }
    __device__ void read(uint32_t, const uint8_t* win, uint32_t* raw) const {
        const uint32_t h = lane >> 5;
#pragma unroll
        for (int j = 0; j < NB; j++) {
            const uint32_t r = 32u * j + (lane & 31u);
            const u32x4 q = *reinterpret_cast<const u32x4*>(win + 32u * r + 16u * h);
            uint32_t* o = raw + j * kDw;
            o[0] = q.x;
            o[1] = q.y;
            o[2] = q.z;
            o[3] = q.w;
            o[4] = *reinterpret_cast<const uint32_t*>(win + kAuxOff + kAuxPitch * (h * two) + 4u * r);
            o[5] = *reinterpret_cast<const uint32_t*>(win + kAuxOff + kAuxPitch * (2u + h * two) + 4u * r);
        }
    }
    __device__ Scale scale(uint32_t c, int j, const uint32_t* r) const {
        // 16-bit values may sit 2 bytes into their dword
        const uint32_t go = goff(c, lane >> 5);
        // (the three dtypes' conversions formed, one selected: no branch per value)
        const uint32_t is32 = in_vgpr(m32), is16 = in_vgpr(m16);
        auto f16of = [&](uint32_t bits, uint32_t base_mod4) -> _Float16 {
            const uint32_t v = bits >> (8u * ((base_mod4 + go) & 3u));
            const uint32_t wide = (bits & is32) | ((v << 16) & ~is32);  // f32, or bf16 widened
            const uint32_t h = __builtin_bit_cast(uint16_t, (_Float16)__uint_as_float(wide));
            return __builtin_bit_cast(_Float16, (uint16_t)((v & is16) | (h & ~is16)));
        };
        const _Float16 sv = f16of(r[4], ssh[j]), bv = f16of(r[5], bsh[j]);
        return {h2{sv, sv}, h2{bv, bv}};
    }
    __device__ h8 step(const uint32_t* r, const Scale& s, int t) const {
        const h2 ol = {(_Float16)-1024.0f, (_Float16)-1024.0f}, oh = {(_Float16)-64.0f, (_Float16)-64.0f};
        const uint32_t ml = in_vgpr(0x64006400u), mh = in_vgpr(0x54005400u);
        const uint32_t kl = in_sgpr(0x000F000Fu), kh = in_sgpr(0x00F000F0u);
        auto lo = [&](uint32_t v) { return as_u(__builtin_elementwise_fma(as_h2(and_or(v, kl, ml)) + ol, s.s, s.b)); };
        auto hi = [&](uint32_t v) { return as_u(__builtin_elementwise_fma(as_h2(and_or(v, kh, mh)) + oh, s.s, s.b)); };
        const uint32_t w = r[t], w8 = w >> 8;
        return as_h8(lo(w), hi(w), lo(w8), hi(w8));
    }
};

// GGUF Q4_K (GGML block_q4_K, 144-byte super-blocks of 256 weights; the
// reference's schema gguf_block.rs:183-316): chunk g of a row is step
// i = g % 4 of super-block g / 4, weights 64i + 0..63: the low and high nibbles of
// qs[32i .. 32i+32) are sub-blocks 2i and 2i + 1.  Lane half h holds bytes
// 16h .. 16h+15 of the 32: k steps 0, 1 are its low nibbles (weights 64i + 16h + ..),
// 2, 3 its high ones (64i + 32 + 16h + ..), 8 weights each, pairs (l, l+2) as
// Q8_0's (XFRAG_QK).  The window per row: the super-block's 16-byte header (d,
// dmin, the 12 scale bytes) and the step's 32 code bytes, three 16-byte pieces
// (super-blocks are 4-byte aligned: 144 = 36 dwords).  w = RNE_f16(q·RNE_f16(d·sc)
// - RNE_f16(dmin·m)) by one packed fma (d·sc and dmin·m exact in f32).
// Q5_K (block_q5_K, 176 bytes): the window adds qh (bytes 16..48, two more
// pieces, kept before the codes); the fifth bit of weight 64i + 32s + l is bit
// 2i + s of qh[l], moved under the nibble.
template <bool Q5, int NB, uint32_t PARTS>
struct WinQK {
    static constexpr uint32_t kRows = 32u * NB;
    static constexpr uint32_t NP = Q5 ? 5u : 3u, kAll = (kRows * NP + 63u) / 64u, kCopies = (kAll + PARTS - 1u) / PARTS;
    static constexpr uint32_t kPitch = 16u * NP;
    static constexpr uint32_t kBytes = kAll * 1024u;
    static constexpr uint32_t SB = Q5 ? 176u : 144u;  // super-block bytes
    static constexpr uint32_t kReads = Q5 ? 3u : 2u, kDw = 4u * kReads;  // d|dmin, three scale dwords, 4 code, [4 qh] dwords
    struct Scale {
        h2 ds[2], ndm[2];
        uint32_t i2;
    };
    Src base;
    uint32_t rb[kCopies];  // piece of each copy lane in its row's first super-block, from base (the weight)
    uint32_t st[kCopies];  // its step per chunk of a super-block: 32 code bytes, or none (header, qh)
    uint32_t dst[kCopies];
    uint32_t c0, lane;

    __device__ void init(const GemmArgs& a, const GemmProb& pr, uint32_t n0, uint32_t lane_, uint32_t c0_, uint32_t part) {
        lane = lane_;
        c0 = c0_;
        base.set(pr.w);
#pragma unroll
        for (uint32_t q = 0; q < kCopies; q++) {
            const uint32_t qq = copy_index<PARTS, kAll>(q, part);
            dst[q] = 1024u * qq;
            uint32_t li = 64u * qq + lane;
            li = li < kRows * NP ? li : kRows * NP - 1u;
            const uint32_t r = li / NP;
            const uint32_t n = n0 + r < pr.N ? n0 + r : pr.N - 1u;  // past N: re-read the last row (never stored)
            // pieces: header, [qh, qh,] the step's two code pieces (at 16·p for step 0)
            const uint32_t p = li % NP;
            rb[q] = n * (uint32_t)a.rowbytes + 16u * p;  // below 4 GiB
            st[q] = p + 2u < NP ? 0u : 32u;
        }
    }
    __device__ void issue(uint32_t c, uint8_t* win) const {
        const uint32_t g = c0 + c, sb = g >> 2, i = g & 3u;
#pragma unroll
        for (uint32_t q = 0; q < kCopies; q++) base.dma16(rb[q] + __umul24(st[q], i), sb * SB, win + dst[q]);
    }
    __device__ void read(uint32_t, const uint8_t* win, uint32_t* raw) const {
        const uint32_t h = lane >> 5;
#pragma unroll
        for (int j = 0; j < NB; j++) {
            const uint8_t* w = win + (32u * j + (lane & 31u)) * kPitch;
            uint32_t* o = raw + j * kDw;
#pragma unroll
            for (uint32_t v = 0; v < kReads; v++) {
                const u32x4 x = *reinterpret_cast<const u32x4*>(
                    w + (v == 0 ? 0u : v == 1 ? 16u * (NP - 2u) + 16u * h : 16u + 16u * h));
                o[4 * v] = x.x;
                o[4 * v + 1] = x.y;
                o[4 * v + 2] = x.z;
                o[4 * v + 3] = x.w;
            }
        }
    }
    __device__ Scale scale(uint32_t c, int, const uint32_t* r) const {
        // q4k_scale_min_pair without its branches on the (uniform) step: all four
        // scales and mins of this half of the super-block, then the step's pair
        const uint32_t i = (c0 + c) & 3u, hi = in_sgpr(0u - (i >> 1)), at = 16u * (i & 1u);
        const uint32_t k6 = in_sgpr(0x3F3F3F3Fu), k4 = in_sgpr(0x0F0F0F0Fu), k2 = in_sgpr(0x30303030u);
        const uint32_t sx = and_or(r[1] >> 2, k2, r[3] & k4), mx = and_or(r[2] >> 2, k2, (r[3] >> 4) & k4);
        const uint32_t sv = ((sx & hi) | (r[1] & k6 & ~hi)) >> at, mv = ((mx & hi) | (r[2] & k6 & ~hi)) >> at;
        const float d = f16_bits_to_f32(r[0]), dmin = f16_bits_to_f32(r[0] >> 16);
        Scale s;
#pragma unroll
        for (int b = 0; b < 2; b++) {
            const _Float16 ds = (_Float16)(d * (b ? ubyte_f32<1>(sv) : ubyte_f32<0>(sv)));  // exact f32 product, one rounding
            const _Float16 dm = (_Float16)(-(dmin * (b ? ubyte_f32<1>(mv) : ubyte_f32<0>(mv))));
            s.ds[b] = h2{ds, ds};
            s.ndm[b] = h2{dm, dm};
        }
        s.i2 = 2u * i;
        return s;
    }
    __device__ h8 step(const uint32_t* r, const Scale& s, int t) const {
        const int b = t >> 1, k = 2 * (t & 1);
        // code bits under the exponent of 1024 (low nibbles) or 64
        const uint32_t mask = in_sgpr(b ? 0x00F000F0u : 0x000F000Fu), mh = in_sgpr(b ? 0x01000100u : 0x00100010u);
        const uint32_t magic = in_vgpr(b ? 0x54005400u : 0x64006400u);
        const _Float16 o = b ? (_Float16)-64.0f : (_Float16)-1024.0f;
        const h2 off = {o, o}, ds = s.ds[b], ndm = s.ndm[b];
        auto f = [&](uint32_t v, uint32_t e) {
            uint32_t m = magic;
            if constexpr (Q5) m = and_or(e, mh, m);
            return as_u(__builtin_elementwise_fma(as_h2(and_or(v, mask, m)) + off, ds, ndm));
        };
        uint32_t e[4] = {0, 0, 0, 0};  // bit 2i + b of the qh bytes moved to bit 4 (8): even bytes, odd bytes
        if constexpr (Q5) {
#pragma unroll
            for (int q = 0; q < 2; q++) {
                const uint32_t v = r[8 + k + q] >> s.i2;
                e[2 * q] = b ? v << 7 : v << 4;
                e[2 * q + 1] = b ? v >> 1 : v >> 4;
            }
        }
        const uint32_t c = r[4 + k], c2 = r[5 + k];
        return as_h8(f(c, e[0]), f(c >> 8, e[1]), f(c2, e[2]), f(c2 >> 8, e[3]));
    }
};

// GGUF IQ4_XS (GGML block_iq4_xs, 136-byte super-blocks of 256 weights; the
// reference's schema gguf_block.rs:183-316): chunk g of a row covers
// sub-blocks 2i and 2i + 1 (i = g % 4) of super-block g / 4; lane half h
// decodes sub-block 2i + h, laid out as a Q4_0 block (XFRAG_NIB order), each
// nibble looked up in the codebook (iq4nl_lookup) and decoded as Q8_0's codes:
// w = RNE_f16(kv·RNE_f16(d·(ls - 32))).  The window per row: the 16 bytes
// from the super-block's start (d, scales_h, scales_l) and the chunk's 32
// code bytes, three 16-byte pieces within the super-block.
template <int NB, uint32_t PARTS>
struct WinIQ4XS {
    static constexpr uint32_t kRows = 32u * NB;
    static constexpr uint32_t NP = 3, kAll = (kRows * NP + 63u) / 64u, kCopies = (kAll + PARTS - 1u) / PARTS;
    static constexpr uint32_t kPitch = 16u * NP;
    static constexpr uint32_t kBytes = kAll * 1024u;
    static constexpr uint32_t kDw = 6, kReads = 2;  // d|scales_h, scales_l, 4 code dwords
    struct Scale {
        h2 ds;
    };
    Src base;
    uint32_t rb[kCopies];  // piece of each copy lane in its row's first super-block, from base (the weight)
    uint32_t st[kCopies];  // its step per chunk of a super-block: 32 code bytes, or none (header)
    uint32_t dst[kCopies];
    uint32_t c0, lane;

    __device__ void init(const GemmArgs& a, const GemmProb& pr, uint32_t n0, uint32_t lane_, uint32_t c0_, uint32_t part) {
        lane = lane_;
        c0 = c0_;
        base.set(pr.w);
#pragma unroll
        for (uint32_t q = 0; q < kCopies; q++) {
            const uint32_t qq = copy_index<PARTS, kAll>(q, part);
            dst[q] = 1024u * qq;
            uint32_t li = 64u * qq + lane;
            li = li < kRows * NP ? li : kRows * NP - 1u;
            const uint32_t r = li / NP;
            const uint32_t n = n0 + r < pr.N ? n0 + r : pr.N - 1u;  // past N: re-read the last row (never stored)
            const uint32_t p = li % NP;
            rb[q] = n * (uint32_t)a.rowbytes + (p == 0u ? 0u : 8u + 16u * (p - 1u));  // below 4 GiB
            st[q] = p == 0u ? 0u : 32u;
        }
    }
    __device__ void issue(uint32_t c, uint8_t* win) const {
        const uint32_t g = c0 + c, sb = g >> 2, i = g & 3u;
#pragma unroll
        for (uint32_t q = 0; q < kCopies; q++) base.dma16(rb[q] + __umul24(st[q], i), sb * 136u, win + dst[q]);
    }
    __device__ void read(uint32_t, const uint8_t* win, uint32_t* raw) const {
        const uint32_t h = lane >> 5;
#pragma unroll
        for (int j = 0; j < NB; j++) {
            const uint8_t* w = win + (32u * j + (lane & 31u)) * kPitch;
            uint32_t* o = raw + j * kDw;
            const u32x2 hd = *reinterpret_cast<const u32x2*>(w);
            const u32x4 x = *reinterpret_cast<const u32x4*>(w + 16u + 16u * h);
            o[0] = hd.x, o[1] = hd.y;
            o[2] = x.x, o[3] = x.y, o[4] = x.z, o[5] = x.w;
        }
    }
    __device__ Scale scale(uint32_t c, int, const uint32_t* r) const {
        const uint32_t h = lane >> 5, ib = 2u * ((c0 + c) & 3u) + h;
        const float dl = f16_bits_to_f32(r[0]) * (float)((int)iq4xs_scale(r[0] >> 16, r[1], ib) - 32);  // exact
        const _Float16 ds = (_Float16)dl;
        return {h2{ds, ds}};
    }
    __device__ h8 step(const uint32_t* r, const Scale& s, int t) const {
        const h2 o = {(_Float16)-1152.0f, (_Float16)-1152.0f};
        const uint32_t ml = in_vgpr(0x64006400u), kb = in_sgpr(0x00FF00FFu);
        auto f = [&](uint32_t v) { return as_u((as_h2(and_or(v, kb, ml)) + o) * s.ds); };
        const uint32_t q = r[2 + t];
        const uint32_t L = iq4nl_lookup(q & 0x0F0F0F0Fu), H = iq4nl_lookup((q >> 4) & 0x0F0F0F0Fu);
        return as_h8(f(L), f(L >> 8), f(H), f(H >> 8));
    }
};

template <uint32_t ENC, int NB, uint32_t PARTS>
struct WinOf {
    using type = WinBlocks<ENC, NB, PARTS>;
};
template <int NB, uint32_t PARTS>
struct WinOf<ENC_IQ4_XS, NB, PARTS> {
    using type = WinIQ4XS<NB, PARTS>;
};
template <int NB, uint32_t PARTS>
struct WinOf<ENC_Q4_K, NB, PARTS> {
    using type = WinQK<false, NB, PARTS>;
};
template <int NB, uint32_t PARTS>
struct WinOf<ENC_Q5_K, NB, PARTS> {
    using type = WinQK<true, NB, PARTS>;
};
template <int NB, uint32_t PARTS>
struct WinOf<ENC_MLX_U4, NB, PARTS> {
    using type = WinMlx<NB, PARTS>;
};
template <int NB, uint32_t PARTS>
struct WinOf<ENC_Q6_K, NB, PARTS> {
    using type = WinQ6K<NB, PARTS>;
};

// Decode VALU instructions per (N-block, k step) per lane, from the kernels' ISA:
// the share of them issued after each MFMA, and the encoding's term in the cost
// model of the launch plan.
constexpr int decode_valu(uint32_t enc) {
    return enc == ENC_Q8_0 ? 18 : enc == ENC_Q4_K ? 22 : enc == ENC_Q6_K ? 18
         : enc == ENC_Q5_K ? 28 : enc == ENC_IQ4_XS ? 30 : 16;  // Q4_0, Q4_1, MLX U4
}

// ... and of a chunk's scales (and Q6_K's code realignment) per N-block.
constexpr int scale_valu(uint32_t enc) {
    return enc == ENC_Q6_K || enc == ENC_Q4_K || enc == ENC_Q5_K ? 32 : enc == ENC_MLX_U4 ? 20 : enc == ENC_IQ4_XS ? 12 : 4;
}

// Copy instructions of a wave's window of two weight blocks (see WinOf).
constexpr uint32_t window_copies(uint32_t enc) {
    return enc == ENC_Q6_K ? 8u : enc == ENC_Q8_0 || enc == ENC_Q5_K ? 5u : enc == ENC_MLX_U4 ? 4u : 3u;
}

// LDS geometry of one kernel configuration: a wave multiplies TM activation
// row blocks by NB weight row blocks (32 rows each); the workgroup's S·WN·WM waves
// split into S K slices x WN column subtiles x WM row subtiles.
template <uint32_t ENC, int TM, int NB, int S, int WN, int WM>
struct Geo {
    using W = typename WinOf<ENC, NB, (uint32_t)WM>::type;
    static constexpr uint32_t kWaves = S * WN * WM;
    static constexpr uint32_t kCols = 32u * NB;                          // a wave's output columns
    // A slice of one wave (XR) loads its activation fragments into registers, a
    // chunk ahead: no other wave would read them from LDS.
    static constexpr bool XR = WN * WM == 1;
    static constexpr uint32_t kXBytes = XR ? 0u : (uint32_t)S * 4u * TM * WM * 1024u;  // a chunk's activation fragments
    static constexpr uint32_t kWBytes = S * WN * W::kBytes;              // a chunk's weight windows
    static constexpr uint32_t kRs = 32u * TM * WM * 4u;                  // the tile's row factors
    static constexpr uint32_t kEpiPitch = kCols + 4u;                    // floats per output row in LDS
    static constexpr uint32_t kEpiBlock = kWaves * 32u * kEpiPitch * 4u;  // every wave's partial row block
    static constexpr uint32_t kRoom = kLdsMax - kRs;
    static constexpr uint32_t kDmaX = XR ? 0u : 4u * TM / WN;  // activation copies per wave per chunk
    static constexpr uint32_t kDma = kDmaX + W::kCopies;  // all copies per wave per chunk
    // Ring slots: R of activations, R - 1 of weight windows (a wave's own, read
    // whole into registers a step ahead; R where an M split shares them): R - 2
    // chunks of copies in flight across a step.
    static constexpr uint32_t w_slots(uint32_t r) { return WM > 1 ? r : r - 1u; }
    static constexpr uint32_t ring_bytes(uint32_t r) { return r * kXBytes + w_slots(r) * kWBytes; }
    static constexpr uint32_t R = ring_bytes(4u) <= kRoom && 2u * kDma < 64u ? 4u : 3u;
    // Vector memory operations newer than chunk c + 1's copies at step c's wait (at
    // least; XR: the activation loads of half a step besides the copies).
    static constexpr uint32_t kNewer = XR ? (R - 3u) * (4u * TM + kDma) + 2u * TM : (R - 3u) * kDma;
    static constexpr bool kFits = (S != 2 || window_copies(ENC) == 3u) &&  // (gemm_plan's only use of two slices)
                                  ring_bytes(R) <= kRoom && kEpiBlock <= kRoom && (R - 2u) * kDma < 64u && kNewer < 64u;
    // the epilogue reuses the ring: row blocks of the tile per pass
    static constexpr uint32_t kEpiPer = S == 1 ? 1u
                                      : TM % 4 == 0 && 4u * kEpiBlock <= ring_bytes(R) ? 4u
                                      : TM % 2 == 0 && 2u * kEpiBlock <= ring_bytes(R) ? 2u : 1u;
    static constexpr uint32_t kEpi = kEpiPer * kEpiBlock;
    static constexpr uint32_t kRing = ring_bytes(R) > kEpi ? ring_bytes(R) : kEpi;
    static constexpr uint32_t kLds = kRing + kRs;
    static_assert((4u * TM) % WN == 0, "activation fragments split evenly over the slice's waves");
    static_assert(WinOf<ENC, 2, 1>::type::kCopies == window_copies(ENC), "the launch plan's window copies");
};

// Issue order of a k step of MF MFMAs: one MFMA, then a share of the copies, the
// DS reads and the decode's VALU instructions, and so on, evenly (left alone, the
// scheduler moves each read next to the MFMA that needs it and the decode into
// one run: 8x2 tiles of Q4_0 over 2048x24576x4096 took 457 us, 402 in this order).
template <int M, int MF, int VM, int DS, int VALU>
__device__ __forceinline__ void interleave_from() {
    if constexpr (M < MF) {
        constexpr int vm = (M + 1) * VM / MF - M * VM / MF, ds = (M + 1) * DS / MF - M * DS / MF,
                      va = (M + 1) * VALU / MF - M * VALU / MF;
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                         // MFMA
        if constexpr (vm > 0) __builtin_amdgcn_sched_group_barrier(0x020, vm, 0);  // vector memory reads
        if constexpr (ds > 0) __builtin_amdgcn_sched_group_barrier(0x100, ds, 0);  // DS reads
        if constexpr (va > 0) __builtin_amdgcn_sched_group_barrier(0x002, va, 0);  // VALU
        interleave_from<M + 1, MF, VM, DS, VALU>();
    }
}
template <int MF, int VM, int DS, int VALU>
__device__ __forceinline__ void interleave() {
    interleave_from<0, MF, VM, DS, VALU>();
    __builtin_amdgcn_sched_barrier(0);
}

// One workgroup of S·WN waves computes a (32·TM) x (32·NB·WN) tile of one
// weight's Y.  Chunks of 64 k stream through a ring of R LDS slots, every
// operand by global_load_lds with explicit vmcnt waits (the compiler then never
// needs a full drain): per chunk and K slice, the slice's 4·TM activation
// fragments (copied once, shared by the slice's WN waves) and each wave's weight
// window.  Per k step of chunk c: the MFMAs of the step, with the activation
// reads and the weight decode of the next step between them.  Before the last
// step: wait for chunk c + 1 (a barrier when slots are shared: every wave's
// copies landed, every wave past chunk c - 1), copy chunk c + R - 1 into chunk
// c - 1's slot, and read chunk c + 1's weights (past the last chunk a stale slot
// is read and decoded, never multiplied).
//
// Epilogue, kEpiPer row blocks at a time: every wave's partial tile goes to LDS;
// the S waves of a column subtile each take a share of the rows, add the S
// partials in slice order (a fixed order: results do not depend on timing),
// scale by rs[m] and store.
template <uint32_t ENC, int TM, int NB, int S, int WN, int WM>
__global__ __launch_bounds__(S * WN * WM * 64)
__attribute__((amdgpu_waves_per_eu((S * WN * WM + 3) / 4, (S * WN * WM + 3) / 4)))
void gemm_kernel(const GemmArgs a) {
    using G = Geo<ENC, TM, NB, S, WN, WM>;
    using W = typename G::W;
    constexpr uint32_t R = G::R;
    constexpr int kDecodeValu = decode_valu(ENC), kScaleValu = scale_valu(ENC), MF = TM * NB;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];

    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t ks = wave % (uint32_t)S, ns = wave / (uint32_t)S % (uint32_t)WN, wm = wave / (uint32_t)(S * WN);

    // XCD-aware order: consecutive tile indices on the workgroups that land on
    // one XCD (workgroup i on XCD i % 8), so one XCD's L2 holds a band of the
    // larger operand and all of the smaller: tiles sharing weight columns
    // (N-major) when the weights are the larger operand, tiles sharing
    // activation rows (M-major) when the staged activations are.
    const uint32_t T = a.mt * a.nt;
    const uint32_t q8 = T / 8u, r8 = T % 8u, xcd = blockIdx.x % 8u;
    const uint32_t tile = (xcd < r8 ? xcd * (q8 + 1u) : r8 * (q8 + 1u) + (xcd - r8) * q8) + blockIdx.x / 8u;
    const uint32_t mtile = a.mmajor ? tile / a.nt : tile % a.mt, ntile = a.mmajor ? tile % a.nt : tile / a.mt;
    GemmProb pr = a.p[0];
#pragma unroll
    for (uint32_t i = 1; i < (uint32_t)kMaxProblems; i++)
        if (i < a.np && ntile >= a.p[i].nt0) pr = a.p[i];
    const uint32_t n0 = ((ntile - pr.nt0) * WN + ns) * G::kCols;  // this wave's first column
    const uint32_t mb0 = mtile * (uint32_t)(TM * WM);             // first 32-row block
    const uint32_t mbs = (a.M + 31u) / 32u;

    // this wave's K slice: chunks [c0, c0 + nc) of 64 k, nc > 0; where waves share
    // slots S divides the chunk count (every wave runs the same steps), otherwise
    // slices may differ by a chunk
    const uint32_t nchk = a.K / 64u, ksteps = a.K / 16u;
    const uint32_t c0 = nchk * ks / (uint32_t)S, nc = nchk * (ks + 1u) / (uint32_t)S - c0;

    // Activation copies: this wave copies every WN·WM-th fragment f of its
    // slice's 4·TM·WM per chunk (f = 4·i + t: row block i, k step t).
    constexpr bool XR = G::XR;
    constexpr uint32_t NX = XR ? TM : G::kDmaX;
    Src xbase;  // the tile's first row block: the rows rounded up to 32 may pass 4 GiB in all
    xbase.set(a.xh + (size_t)mb0 * ksteps * 512u);
    uint32_t xsrc[NX], xdst[NX];
    if constexpr (XR) {  // row block q's fragments of the slice
#pragma unroll
        for (uint32_t q = 0; q < NX; q++)
            xsrc[q] = ((mb0 + q < mbs ? q : mbs - 1u - mb0) * ksteps + 4u * c0) * 1024u;
    }
#pragma unroll
    for (uint32_t q = 0; !XR && q < NX; q++) {
        const uint32_t f = ns + WN * wm + q * (uint32_t)(WN * WM), i = f / 4u, t = f % 4u;
        const uint32_t mb = mb0 + i < mbs ? i : mbs - 1u - mb0;  // past M: re-read the last block (never stored)
        xsrc[q] = (mb * ksteps + 4u * c0 + t) * 1024u;
        xdst[q] = (ks * 4u * TM * WM + f) * 1024u;
    }
    W win;
    win.init(a, pr, n0, lane, c0, wm);
    auto slot_x = [&](uint32_t slot) { return lds + slot * G::kXBytes; };
    auto slot_w = [&](uint32_t slot) { return lds + R * G::kXBytes + slot * G::kWBytes + (ks + S * ns) * W::kBytes; };
    // chunk c of the range (c < nc) into a slot of each ring
    auto issue = [&](uint32_t c, uint32_t sx, uint32_t sw) {
#pragma unroll
        for (uint32_t q = 0; !XR && q < NX; q++) xbase.dma16(16u * lane, xsrc[q] + c * 4096u, slot_x(sx) + xdst[q]);
        win.issue(c, slot_w(sw));
    };

    // Row factors of the tile's 32·TM rows, copied into LDS ahead of the ring
    // (the oldest copy in flight, so the first ring wait covers it).
    float* rs_lds = reinterpret_cast<float*>(lds + G::kRing);
    if (wave == 0 && lane < 8u * TM * WM) dma16(a.rs + (size_t)mb0 * 32u + 4u * lane, rs_lds);

    constexpr int XA = XR ? 4 : 2;  // activation fragments of this k step and the next (XR: three)
    h8 xa[XA][TM];
    h8 wf[2][NB];               // decoded weights of this k step and the next
    uint32_t raw[W::kDw * NB], rawn[W::kDw * NB];  // raw weights of this chunk and the next
    typename W::Scale sc[NB];
    auto load_x = [&](uint32_t c, int t) {  // XR: k step t of chunk c
#pragma unroll
        for (int i = 0; i < TM; i++) xa[t % XA][i] = xbase.load16(16u * lane, xsrc[i] + c * 4096u + 1024u * t);
    };
    auto read_x = [&](uint32_t slot, int t, int p) {
        const uint8_t* sx = slot_x(slot) + (ks * 4u * TM * WM + wm * 4u * TM) * 1024u + lane * 16u;
#pragma unroll
        for (int i = 0; i < TM; i++) xa[p][i] = *reinterpret_cast<const h8*>(sx + (4u * i + t) * 1024u);
    };
    auto decode = [&](const uint32_t (&rw)[W::kDw * NB], int t, int p) {
#pragma unroll
        for (int j = 0; j < NB; j++) wf[p][j] = win.step(rw + j * W::kDw, sc[j], t);
    };
    f32x16 acc[TM][NB];
    auto mfmas = [&](int t) {
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < NB; j++)
                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(wf[t & 1][j], xa[t % XA][i], acc[i][j], 0, 0, 0);
    };

#pragma unroll
    for (uint32_t c = 0; c < R - 1u; c++)
        if (c < nc) issue(c, c, c);
    if constexpr (XR) {
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int t = 0; t < 4; t++) load_x(0, t);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < TM; i++)  // (under the first copies' latency)
#pragma unroll
        for (int j = 0; j < NB; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] = 0.0f;
    if constexpr (XR) {
        ring_wait<4u * TM>();
    } else {
        // chunk 0 landed (for every wave)
        ring_barrier_k<G::kDma, R - 2u>((nc < R - 1u ? nc : R - 1u) - 1u);
        read_x(0, 0, 0);
    }
    win.read(0, slot_w(0), raw);
#pragma unroll
    for (int j = 0; j < NB; j++) sc[j] = win.scale(0, j, raw + j * W::kDw);
    decode(raw, 0, 0);
    uint32_t cur = 0, nxt = 1, old = R - 1u;  // activation slots of chunks c, c + 1 and c - 1 (c + R - 1)
    // window slots of chunk c + 1 and of chunk c + R - 1 (the one of chunk c, already
    // read; of c - 1 where an M split shares it)
    constexpr uint32_t WR = G::w_slots(R);
    uint32_t wnxt = 1u % WR, wnew = (R - 1u) % WR;
    // the four k steps of chunk c: IN copies a further chunk, LAST has no next chunk
    auto steps = [&](uint32_t c, auto in, auto last) {
        constexpr bool IN = decltype(in)::value, LAST = decltype(last)::value;
        constexpr int D = NB * kDecodeValu, RD = NB * (int)W::kReads;
        constexpr int XV = XR && !LAST ? TM : 0, XD = XR ? 0 : TM;  // activation loads, reads per k step
#pragma unroll
        for (int t = 0; t < 2; t++) {
            if constexpr (!XR) read_x(cur, t + 1, (t + 1) & 1);
            mfmas(t);
            if constexpr (XV > 0) load_x(c + 1u, t);
            decode(raw, t + 1, (t + 1) & 1);
            interleave<MF, XV, XD, D>();
        }
        if constexpr (!LAST) {
            if constexpr (XR) ring_wait<IN ? G::kNewer : 2u * TM>();
            else if constexpr (IN) ring_barrier<G::kNewer>();
            // copies issued so far: chunks up to min(c + R - 2, nc - 1)
            else ring_barrier_k<G::kDma, R - 3u>((c + R - 2u < nc - 1u ? c + R - 2u : nc - 1u) - c - 1u);
            if constexpr (IN) issue(c + R - 1u, old, wnew);
            win.read(c + 1u, slot_w(wnxt), rawn);
        }
        if constexpr (!XR) read_x(cur, 3, 1);
        mfmas(2);
        if constexpr (XV > 0) load_x(c + 1u, 2);
        decode(raw, 3, 1);
        interleave<MF, XV + (IN ? (int)G::kDma : 0), XD + (LAST ? 0 : RD), D + (LAST ? 0 : RD)>();
        if constexpr (!LAST) {
            if constexpr (!XR) read_x(nxt, 0, 0);
#pragma unroll
            for (int j = 0; j < NB; j++) sc[j] = win.scale(c + 1u, j, rawn + j * W::kDw);
        }
        mfmas(3);
        if constexpr (!LAST) {
            if constexpr (XV > 0) load_x(c + 1u, 3);
            decode(rawn, 0, 0);
            interleave<MF, XV, XD, D + NB * kScaleValu>();
#pragma unroll
            for (uint32_t k = 0; k < W::kDw * NB; k++) raw[k] = rawn[k];
            old = cur;
            cur = nxt;
            nxt = nxt + 1u == R ? 0u : nxt + 1u;
            wnxt = wnxt + 1u == WR ? 0u : wnxt + 1u;
            wnew = wnew + 1u == WR ? 0u : wnew + 1u;
        }
    };
    uint32_t c = 0;
    for (; c + R - 1u < nc; c++) steps(c, std::true_type{}, std::false_type{});
    for (; c + 1u < nc; c++) steps(c, std::false_type{}, std::false_type{});
    steps(c, std::false_type{}, std::true_type{});
    wait_vmcnt<0>();
    __syncthreads();  // every wave past its last chunk: the ring is free

    // Epilogue.  D = W-block x X-block: lane l holds activation row l % 32 of
    // the row block and, for r = 0..15, column 8·(r/4) + 4·(l/32) + r%4 of the
    // weight block.
    float* epi = reinterpret_cast<float*>(lds);
    constexpr uint32_t P = G::kEpiPitch, EB = G::kEpiPer;
    constexpr uint32_t RPT = 32u * EB / S, C4 = G::kCols / 4u, NG = RPT * C4, NI = (NG + 63u) / 64u;
    const bool vec_ok = (pr.N & 3u) == 0 && ((uintptr_t)pr.y & (a.y_bf16 ? 7u : 15u)) == 0;
#pragma unroll
    for (int i0 = 0; i0 < TM; i0 += (int)EB) {
        if (S > 1 && i0 > 0) __syncthreads();  // the previous pass has been read
        float* mine = epi + wave * 32u * EB * P;
#pragma unroll
        for (int i = 0; i < (int)EB; i++)
#pragma unroll
            for (int j = 0; j < NB; j++)
#pragma unroll
                for (int q = 0; q < 4; q++)
                    *reinterpret_cast<f32x4*>(mine + (32u * i + (lane & 31u)) * P + 32u * j + 8u * q + 4u * (lane >> 5)) =
                        f32x4{acc[i0 + i][j][4 * q], acc[i0 + i][j][4 * q + 1], acc[i0 + i][j][4 * q + 2],
                              acc[i0 + i][j][4 * q + 3]};
        if constexpr (S > 1) __syncthreads();
        // the S waves of column subtile ns take RPT rows each; lane and step s
        // cover group idx = lane + 64s: row idx / C4, columns 4·(idx % C4) .. +3
        f32x4 v[NI];
#pragma unroll
        for (uint32_t s = 0; s < NI; s++) {
            const uint32_t idx = lane + 64u * s, ml = ks * RPT + idx / C4, c4 = idx % C4;
            v[s] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            if (NG % 64u != 0 && idx >= NG) continue;
#pragma unroll
            for (int k = 0; k < S; k++)  // slice order, the same for every output
                v[s] += *reinterpret_cast<const f32x4*>(epi + (((wm * WN + ns) * S + k) * 32u * EB + ml) * P + 4u * c4);
        }
        // scale by rs[m] and store whole 4-column groups (16-byte f32 or 8-byte
        // bf16 stores, consecutive lanes on consecutive groups of a row),
        // non-temporal: streamed out during the kernel instead of left dirty in L2
        const uint32_t ml0 = 32u * (wm * TM + i0) + ks * RPT, mrow = mb0 * 32u + ml0;
        const bool whole = vec_ok && mrow + RPT <= a.M && n0 + G::kCols <= pr.N;
#pragma unroll
        for (uint32_t s = 0; s < NI; s++) {
            const uint32_t idx = lane + 64u * s, r = idx / C4, n = n0 + 4u * (idx % C4), m = mrow + r;
            if (NG % 64u != 0 && idx >= NG) continue;
            const f32x4 o = v[s] * rs_lds[ml0 + r];
            if (whole) {
                const size_t at = (size_t)m * pr.N + n;
                if (a.y_bf16)
                    __builtin_nontemporal_store(
                        u32x2{f32x2_to_bf16x2_bits(o[0], o[1]), f32x2_to_bf16x2_bits(o[2], o[3])},
                        gptr_mut<u32x2>(static_cast<uint16_t*>(pr.y) + at));
                else
                    __builtin_nontemporal_store(o, gptr_mut<f32x4>(static_cast<float*>(pr.y) + at));
            } else if (m < a.M) {
                const size_t at = (size_t)m * pr.N + n;
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    if (n + (uint32_t)e >= pr.N) break;
                    if (a.y_bf16) gptr_mut<uint16_t>(pr.y)[at + e] = f32_to_bf16_bits(o[e]);
                    else gptr_mut<float>(pr.y)[at + e] = o[e];
                }
            }
        }
    }
}

template <uint32_t ENC, int TM, int NB, int S, int WN, int WM>
hipError_t launch(const GemmArgs& a, hipStream_t st) {
    if constexpr (Geo<ENC, TM, NB, S, WN, WM>::kFits) {
        auto kernel = gemm_kernel<ENC, TM, NB, S, WN, WM>;
        constexpr uint32_t lds = Geo<ENC, TM, NB, S, WN, WM>::kLds;
        if constexpr (lds > 64u * 1024u) {
            static hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                                         hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
            if (attr != hipSuccess) return attr;
        }
        hipLaunchKernelGGL(kernel, dim3(a.mt * a.nt), dim3(S * WN * WM * 64), lds, st, a);
        return hipGetLastError();
    } else {
        return hipErrorInvalidConfiguration;
    }
}

// The configurations built: X(TM, NB, S, WN, WM).
#define DMX_GEMM_CONFIGS(X) \
    X(8, 2, 1, 4, 1) X(4, 2, 1, 4, 1) X(4, 2, 1, 2, 2) X(2, 2, 1, 4, 1) X(4, 2, 2, 2, 1) \
    X(8, 2, 4, 1, 1) X(4, 3, 4, 1, 1) X(4, 2, 4, 1, 1) X(2, 3, 4, 1, 1) X(2, 2, 4, 1, 1) X(2, 1, 4, 1, 1) \
    X(1, 1, 4, 1, 1) X(1, 1, 8, 1, 1)

template <uint32_t ENC>
hipError_t launch_plan(const GemmArgs& a, const GemmPlan& p, hipStream_t st) {
#define X(TM, NB, S, WN, WM) \
    if (p.tm == TM && p.nb == NB && p.s == S && p.wn == WN && p.wm == WM) return launch<ENC, TM, NB, S, WN, WM>(a, st);
    DMX_GEMM_CONFIGS(X)
#undef X
    return hipErrorInvalidConfiguration;
}

// Whether a configuration of encoding ENC fits one workgroup's LDS.
template <uint32_t ENC>
bool fits(uint32_t tm, uint32_t nb, uint32_t s, uint32_t wn, uint32_t wm) {
#define X(TM, NB, S, WN, WM) \
    if (tm == TM && nb == NB && s == S && wn == WN && wm == WM) return Geo<ENC, TM, NB, S, WN, WM>::kFits;
    DMX_GEMM_CONFIGS(X)
#undef X
    return false;
}

}  // namespace gemm
}  // namespace dmx
