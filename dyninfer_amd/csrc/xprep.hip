// Prefill activation staging for the MFMA GEMM: X [M, K] (f32 or bf16) to f16
// once per call, laid out as the GEMM's MFMA operands.
//
//   xh value of (m, k) = RNE_f16(x[m, k] · 2^(15 - e_m)),   rs[m] = 2^(e_m - 15),
//
// e_m the binary exponent of the row's largest magnitude (max |x| < 2^e_m),
// so every scaled value is below 2^15 (no f16 overflow) and the row's large
// values keep f16's full 11-bit precision.  The scaling is exact (a power of
// two); the one rounding is RNE to f16, relative 2^-11 for scaled magnitudes
// in f16's normal range.  A value more than 2^29 below its row's largest
// lands among f16's subnormals (absolute error <= 2^-25 scaled, i.e.
// 2^-40·max|x| per activation).  The GEMM accumulates x_h·w in f32 and
// multiplies each output row by rs[m].
//
// Layout: fragments of a v_mfma_f32_32x32x16_f16 operand, 1 KiB each:
//   fragment (mb, ks) = rows 32·mb .. 32·mb+31, k step ks (16 k), at element
//   offset ((mb·K/16 + ks)·64 + lane)·8; lane l holds row 32·mb + l % 32 and
//   8 k for lane half h = l / 32.
// The GEMM advances K in chunks of 64 (k steps 4c .. 4c+3), lane half h
// decoding the chunk's weight block h, so half h of step 4c+t holds 8 k of
// k = 64c + 32h .. 64c + 32h + 31, in the order the block's decode produces:
//   XFRAG_NIB  (Q4_0, Q4_1: code byte j holds k = j and k = j + 16):
//              4t, 4t+2, 4t+1, 4t+3, 16+4t, 18+4t, 17+4t, 19+4t
//   XFRAG_BYTE (Q8_0: one code byte per k):
//              8t, 8t+2, 8t+1, 8t+3, 8t+4, 8t+6, 8t+5, 8t+7
//              (pairs (j, j+2) of a dword decode together)
//   XFRAG_WORD (MLX U4: packed word t of the block holds k = 8t .. 8t+7, LSB
//              first): 8t, 8t+4, 8t+1, 8t+5, 8t+2, 8t+6, 8t+3, 8t+7
//              (nibbles j and j+4 of a word decode together)
// and for the super-block encodings, whose lane half takes both nibbles of 16
// code bytes (runs of 8 k in XFRAG_BYTE's order, k0 their first):
//   XFRAG_QK   (Q4_K, Q5_K): k0 = 64c + 16h + 32·(t / 2) + 8·(t % 2)
//   XFRAG_Q6K  (Q6_K): k0 = 256·(c / 4) + 128·(c / 2 % 2) + 16·(c % 2) + 32h +
//              64·(t / 2) + 8·(t % 2).  Rows M .. roundup(M, 32) - 1
// are written as zeros, so the GEMM reads whole fragments.
//
// Mapping: a row is shared by WPR waves, each lane taking up to NR output slots
// of 8 elements (slot 8c + 2t + h: chunk c, step t, half h) that it holds in
// registers between the max pass and the conversion; the waves' maxima meet in
// LDS.  Bound: HBM / L2 traffic for many rows, one memory round trip for few, so
// what counts is loads in flight: WPR grows until a lane has one slot or the launch
// enough waves (launch_xprep).  With one wave per row, which reread rows longer
// than 12288, 45 f32 rows of 12288 took 18.2 us, now 5.3; 512 bf16 rows of 12288
// 27.8 -> 11.7; 2048 f32 rows of 12288 113 -> 29.6 us (5.1 TB/s of reads and
// writes); 45 rows of 4096 6.6 -> 4.8.
// From kXprepWholeMinRows rows (there are enough of them), and from
// kXprepPartsMinRows of longer rows, eight rows share a workgroup and
// their slots leave as whole 128-byte lines; otherwise each lane stores its own
// 16-byte slots, four rows or fewer to a workgroup (512 rows of K = 12288 13.7 us
// against 12.5 by lines).
// NaN and inf: the row's scale is taken as 2^15 and the non-finite values
// propagate to the row's outputs.
#include "device_common.hpp"
#include "kernels.hpp"

namespace dmx {

namespace {

typedef _Float16 xh2 __attribute__((ext_vector_type(2)));
typedef float xf2 __attribute__((ext_vector_type(2)));
typedef float xf4 __attribute__((ext_vector_type(4)));

// The 8 activations of output slot `slot` of a row: two runs of 4 k, at
// k0 and k0 + RUN2 (NIB: 16, the others 4, i.e. one run of 8).
template <uint32_t LAYOUT>
__device__ __forceinline__ uint32_t slot_k0(uint32_t slot) {
    const uint32_t c = slot >> 3, t = (slot >> 1) & 3u, h = slot & 1u;
    if (LAYOUT == XFRAG_QK) return 64u * c + 16u * h + 32u * (t >> 1) + 8u * (t & 1u);
    if (LAYOUT == XFRAG_Q6K)
        return 256u * (c >> 2) + 128u * ((c >> 1) & 1u) + 16u * (c & 1u) + 32u * h + 64u * (t >> 1) + 8u * (t & 1u);
    return 64u * c + 32u * h + (LAYOUT == XFRAG_NIB ? 4u * t : 8u * t);
}
template <bool XBF16, uint32_t LAYOUT>
__device__ __forceinline__ void load8(const void* x, size_t row, uint32_t slot, float (&v)[8]) {
    constexpr uint32_t RUN2 = LAYOUT == XFRAG_NIB ? 16u : 4u;
    const size_t k0 = row + slot_k0<LAYOUT>(slot);
    if constexpr (XBF16) {
        typedef uint32_t u32x2_a4 __attribute__((ext_vector_type(2), aligned(4)));
        const u32x2_a4 p = *gptr<u32x2_a4>(static_cast<const uint16_t*>(x) + k0);
        const u32x2_a4 q = *gptr<u32x2_a4>(static_cast<const uint16_t*>(x) + k0 + RUN2);
        const uint32_t w[4] = {p.x, p.y, q.x, q.y};
#pragma unroll
        for (int i = 0; i < 4; i++) {
            v[2 * i] = __uint_as_float(w[i] << 16);
            v[2 * i + 1] = __uint_as_float(w[i] & 0xFFFF0000u);
        }
    } else {
        const xf4 a = *gptr<xf4>(static_cast<const float*>(x) + k0);
        const xf4 b = *gptr<xf4>(static_cast<const float*>(x) + k0 + RUN2);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            v[i] = a[i];
            v[4 + i] = b[i];
        }
    }
}

__device__ __forceinline__ uint32_t absbits_max8(const float (&v)[8], uint32_t m) {
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const uint32_t b = __float_as_uint(v[i]) & 0x7FFFFFFFu;  // |x| bits order as unsigned integers
        m = b > m ? b : m;
    }
    return m;
}

__device__ __forceinline__ uint32_t pk(float a, float b, int sh) {
    const xf2 f = {ldexpf(a, sh), ldexpf(b, sh)};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f, xh2));  // RNE
}

// Element offset in xh of row m's output slot (chunk c, step t, half h).
__device__ __forceinline__ size_t frag_offset(uint32_t m, uint32_t slot, uint32_t ksteps) {
    const uint32_t c = slot >> 3, t = (slot >> 1) & 3u, h = slot & 1u;
    return (((size_t)(m >> 5) * ksteps + 4u * c + t) * 64u + (m & 31u) + 32u * h) * 8u;
}

// All but WORD pair (v0, v2), (v1, v3), (v4, v6), (v5, v7); WORD pairs (v0, v4),
// (v1, v5), (v2, v6), (v3, v7).
typedef uint32_t xu4 __attribute__((ext_vector_type(4)));
template <uint32_t LAYOUT>
__device__ __forceinline__ xu4 pack8(const float (&v)[8], int sh) {
    return LAYOUT == XFRAG_WORD ? xu4{pk(v[0], v[4], sh), pk(v[1], v[5], sh), pk(v[2], v[6], sh), pk(v[3], v[7], sh)}
                                : xu4{pk(v[0], v[2], sh), pk(v[1], v[3], sh), pk(v[4], v[6], sh), pk(v[5], v[7], sh)};
}
// Plain stores: a slot is an eighth of its 128-byte line, and L2 merges the
// rows' slots (non-temporal stores of the pieces took 20.1 us against 13.3 for
// 512 rows of 12288).  Whole lines (xprep_lines_kernel) do leave non-temporally:
// the next kernel reads them, and streaming them out beats leaving dirty lines
// for the end of the kernel (7.3 -> 6.1 us at M = 2048, K = 1024).
template <uint32_t LAYOUT>
__device__ __forceinline__ void store8(uint16_t* xh, size_t off, const float (&v)[8], int sh) {
    *gptr_mut<xu4>(xh + off) = pack8<LAYOUT>(v, sh);
}

// Maximum over the wave (unsigned), every lane receiving it.
__device__ __forceinline__ uint32_t wave_umax(uint32_t v) {
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
        const uint32_t u = (uint32_t)__shfl_xor((int)v, o, 64);
        v = u > v ? u : v;
    }
    return v;
}

// Scale of a row whose largest |x| has the bits mx: binary exponent e of the
// largest magnitude (|x| < 2^e): biased exponent - 126 for normal values; zero
// and subnormal rows clamp to -110 (so 2^(15 - e) stays a normal f32); inf /
// NaN rows take e = 0.
__device__ __forceinline__ int row_exponent(uint32_t mx) {
    const int e = mx >= 0x7F800000u ? 0 : (int)(mx >> 23) - 126;
    return e < -110 ? -110 : e;
}

// The maximum of a row's WPR waves (wave wr of row r), every lane receiving it.
// Every wave of the workgroup calls it.
template <uint32_t WPR>
__device__ __forceinline__ uint32_t row_umax(uint32_t v, uint32_t r, uint32_t wr, uint32_t lane, uint32_t* part) {
    v = wave_umax(v);
    if constexpr (WPR > 1) {
        if (lane == 0) part[r * WPR + wr] = v;
        __syncthreads();
        v = 0;
#pragma unroll
        for (uint32_t i = 0; i < WPR; i++) {
            const uint32_t u = part[r * WPR + i];
            v = u > v ? u : v;
        }
    }
    return v;
}

// Workgroup of R = max(1, 4 / WPR) rows; K <= 512·WPR·NR.
template <bool XBF16, uint32_t LAYOUT, int NR, uint32_t WPR>
__global__ __launch_bounds__((WPR > 4u ? WPR : 4u) * 64u) void xprep_kernel(const void* __restrict__ x, uint32_t M,
                                                                           uint32_t K, uint16_t* __restrict__ xh,
                                                                           float* __restrict__ rs) {
    constexpr uint32_t R = WPR > 4u ? 1u : 4u / WPR;
    __shared__ uint32_t part[R * WPR];
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const uint32_t r = wave / WPR, wr = wave % WPR;
    const uint32_t m = blockIdx.x * R + r;  // below M rounded up to 32: R divides 32
    const uint32_t slots = K / 8u, ksteps = K / 16u;
    const bool real = m < M;  // rows M .. roundup(M, 32) - 1 are zeros
    const size_t row = real ? (size_t)m * K : 0u;
    uint32_t mx = 0;
    float v[NR][8];
#pragma unroll
    for (int i = 0; i < NR; i++) {
        const uint32_t g = 64u * (wr + WPR * (uint32_t)i) + lane;
        if (g < slots) load8<XBF16, LAYOUT>(x, row, g, v[i]);
    }
#pragma unroll
    for (int i = 0; i < NR; i++) {
        const uint32_t g = 64u * (wr + WPR * (uint32_t)i) + lane;
        if (g < slots) {
#pragma unroll
            for (int q = 0; q < 8; q++) v[i][q] = real ? v[i][q] : 0.0f;
            mx = absbits_max8(v[i], mx);
        }
    }
    const int e = row_exponent(row_umax<WPR>(mx, r, wr, lane, part));
#pragma unroll
    for (int i = 0; i < NR; i++) {
        const uint32_t g = 64u * (wr + WPR * (uint32_t)i) + lane;
        if (g < slots) store8<LAYOUT>(xh, frag_offset(m, g, ksteps), v[i], 15 - e);
    }
    if (lane == 0 && wr == 0) gptr_mut<float>(rs)[m] = real ? ldexpf(1.0f, e - 15) : 0.0f;
}

// Eight rows per workgroup of 8·WPR waves, the rows' 16-byte slots gathered in
// LDS so that the eight rows' slots of one (k step, half), consecutive in the
// fragment, leave as one 128-byte line: a store instruction writes 8 whole
// lines instead of 64 pieces of 64 lines.  Workgroup (., p) converts slots
// [p·CAP, (p + 1)·CAP) of the rows, CAP = 64·WPR·NR (held in registers), and
// reads the others for the maximum only, so fewer rows than CUs·8 still fill
// the chip (PARTS; otherwise one workgroup holds the rows whole).  The LDS tile holds SEG slots per lane, so a long part passes
// through it in NR / SEG turns.
constexpr uint32_t kXprepLinesRows = 8, kXprepWholeMinRows = 1024, kXprepPartsMinRows = 256;
template <bool XBF16, uint32_t LAYOUT, int NR, int SEG, uint32_t WPR, bool PARTS>
__global__ __launch_bounds__(kXprepLinesRows * WPR * 64) void xprep_lines_kernel(const void* __restrict__ x, uint32_t M,
                                                                                uint32_t K, uint16_t* __restrict__ xh,
                                                                                float* __restrict__ rs) {
    static_assert(NR % SEG == 0, "whole turns");
    constexpr uint32_t T = kXprepLinesRows * WPR * 64u, kStep = 64u * WPR, kCap = kStep * NR;
    extern __shared__ xu4 tile[];  // [slot of the turn][row of the eight]
    __shared__ uint32_t part[kXprepLinesRows * WPR];
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const uint32_t r = wave / WPR, wr = wave % WPR;
    const uint32_t m0 = blockIdx.x * kXprepLinesRows, m = m0 + r;  // rows rounded up to 32: a multiple of 8
    const uint32_t slots = K / 8u, ksteps = K / 16u, s0 = PARTS ? blockIdx.y * kCap : 0u;
    const bool real = m < M;  // rows M .. roundup(M, 32) - 1 are zeros
    const size_t row = real ? (size_t)m * K : 0u;
    const uint32_t l0 = 64u * wr + lane;
    uint32_t mx = 0;
    float v[NR][8];
#pragma unroll
    for (int i = 0; i < NR; i++) {
        const uint32_t g = s0 + l0 + kStep * (uint32_t)i;
        if (g < slots) load8<XBF16, LAYOUT>(x, row, g, v[i]);
    }
    for (uint32_t b = 0; PARTS && b < slots; b += kCap) {  // the other workgroups' parts
        if (b == s0) continue;
        constexpr int U = NR < 4 ? NR : 4;
#pragma unroll
        for (int i0 = 0; i0 < NR; i0 += U) {
            float o[U][8];
#pragma unroll
            for (int i = 0; i < U; i++) {
                const uint32_t g = b + l0 + kStep * (uint32_t)(i0 + i);
                load8<XBF16, LAYOUT>(x, row, g < slots ? g : 0u, o[i]);
            }
#pragma unroll
            for (int i = 0; i < U; i++) mx = absbits_max8(o[i], mx);
        }
    }
#pragma unroll
    for (int i = 0; i < NR; i++) {
        if (s0 + l0 + kStep * (uint32_t)i < slots) mx = absbits_max8(v[i], mx);
    }
    const int e = row_exponent(row_umax<WPR>(mx, r, wr, lane, part));
    if (lane == 0 && wr == 0 && s0 == 0) gptr_mut<float>(rs)[m] = real ? ldexpf(1.0f, e - 15) : 0.0f;
#pragma unroll
    for (int s = 0; s < NR / SEG; s++) {
        const uint32_t t0 = s0 + kStep * (uint32_t)(SEG * s);  // the turn's first slot
        if (s > 0) __syncthreads();
#pragma unroll
        for (int i = 0; i < SEG; i++) {
            const uint32_t g = l0 + kStep * (uint32_t)i;
            if (t0 + g < slots) {
                const xu4 h = pack8<LAYOUT>(v[SEG * s + i], 15 - e);
                tile[g * kXprepLinesRows + r] = real ? h : xu4{0, 0, 0, 0};
            }
        }
        __syncthreads();
        // piece p = (slot g, row r') of the eight rows: line g at frag_offset(m0, g)
        const uint32_t n = t0 >= slots ? 0u : (slots - t0 < kStep * SEG ? slots - t0 : kStep * SEG);
        for (uint32_t p = threadIdx.x; p < n * kXprepLinesRows; p += T) {
            const uint32_t g = t0 + p / kXprepLinesRows, rr = p % kXprepLinesRows;
            __builtin_nontemporal_store(tile[p], gptr_mut<xu4>(xh + frag_offset(m0 + rr, g, ksteps)));
        }
    }
}

template <bool XBF16, uint32_t LAYOUT, int NR, uint32_t WPR>
hipError_t launch_rows(const void* x, uint32_t M, uint32_t Mp, uint32_t K, uint16_t* xh, float* rs, hipStream_t st) {
    constexpr uint32_t R = WPR > 4u ? 1u : 4u / WPR;
    hipLaunchKernelGGL((xprep_kernel<XBF16, LAYOUT, NR, WPR>), dim3(Mp / R), dim3(R * WPR * 64u), 0, st, x, M, K, xh, rs);
    return hipGetLastError();
}
template <bool XBF16, uint32_t LAYOUT, uint32_t WPR>
hipError_t launch_rows(const void* x, uint32_t M, uint32_t Mp, uint32_t K, uint16_t* xh, float* rs, hipStream_t st) {
    const uint32_t nr = (K / 8u + 64u * WPR - 1u) / (64u * WPR);  // slots per lane
    constexpr int most = WPR < 4u ? 1 : WPR == 4u ? 4 : WPR == 8u ? 2 : 8;  // (launch_xprep's rule meets no more)
    if (nr <= 1u) return launch_rows<XBF16, LAYOUT, 1, WPR>(x, M, Mp, K, xh, rs, st);
    if constexpr (most >= 2)
        if (nr <= 2u) return launch_rows<XBF16, LAYOUT, 2, WPR>(x, M, Mp, K, xh, rs, st);
    if constexpr (most >= 4)
        if (nr <= 4u) return launch_rows<XBF16, LAYOUT, 4, WPR>(x, M, Mp, K, xh, rs, st);
    if constexpr (most >= 8)
        if (nr <= 8u) return launch_rows<XBF16, LAYOUT, 8, WPR>(x, M, Mp, K, xh, rs, st);
    return hipErrorInvalidValue;
}
template <bool XBF16, uint32_t LAYOUT, int NR, int SEG, uint32_t WPR, bool PARTS>
hipError_t launch_lines(const void* x, uint32_t M, uint32_t Mp, uint32_t K, uint16_t* xh, float* rs, hipStream_t st) {
    constexpr uint32_t cap = 64u * WPR * NR, turn = 64u * WPR * SEG;
    const uint32_t slots = K / 8u;
    const size_t lds = (size_t)(slots < turn ? slots : turn) * kXprepLinesRows * 16u;  // 64 KiB at most
    hipLaunchKernelGGL((xprep_lines_kernel<XBF16, LAYOUT, NR, SEG, WPR, PARTS>),
                       dim3(Mp / kXprepLinesRows, (slots + cap - 1u) / cap), dim3(kXprepLinesRows * WPR * 64u), lds, st,
                       x, M, K, xh, rs);
    return hipGetLastError();
}

template <bool XBF16, uint32_t LAYOUT>
hipError_t launch_xprep(const void* x, uint32_t M, uint32_t K, uint16_t* xh, float* rs, hipStream_t st) {
    const uint32_t Mp = (M + 31u) & ~31u, slots = K / 8u;
    if (Mp >= kXprepWholeMinRows && slots <= 1536u) {
        if (slots <= 64u) return launch_lines<XBF16, LAYOUT, 1, 1, 1, false>(x, M, Mp, K, xh, rs, st);
        if (slots <= 128u) return launch_lines<XBF16, LAYOUT, 1, 1, 2, false>(x, M, Mp, K, xh, rs, st);
        if (slots <= 256u) return launch_lines<XBF16, LAYOUT, 2, 2, 2, false>(x, M, Mp, K, xh, rs, st);
        // many f32 rows fill the chip with one wave to a row, and more of them share a CU (3000
        // rows of 3072: two waves 15.2 us, one 10.2; 4096 of 4096 19.8, 16.2; 2048 rows 11.7
        // by one, 10.9; 3000 bf16 rows alike)
        if (!XBF16 && Mp > 2048u && slots > 256u && slots <= 512u)
            return launch_lines<XBF16, LAYOUT, 8, 8, 1, false>(x, M, Mp, K, xh, rs, st);
        if (slots <= 512u) return launch_lines<XBF16, LAYOUT, 4, 4, 2, false>(x, M, Mp, K, xh, rs, st);
        if (slots <= 1024u) return launch_lines<XBF16, LAYOUT, 8, 4, 2, false>(x, M, Mp, K, xh, rs, st);
        return launch_lines<XBF16, LAYOUT, 12, 4, 2, false>(x, M, Mp, K, xh, rs, st);
    }
    // (f32 rows up to 5120 from 641 of them: fewer are faster below, the whole call of 512
    // rows of Q4_0 1024 x 4096 21.0 us in parts, 18.3 below, 1024 x 5120 25.3 and 21.3, Q8_0
    // 400 x 1024 x 4096 22.6 and 19.5; 768 rows stage in 7.2 us in parts, 7.6 below, and
    // 512 bf16 rows of 4096 in 5.3 and 5.8)
    if (Mp >= kXprepPartsMinRows && K >= 4096u && (XBF16 || Mp > 640u || K > 5120u)) {
        // slots per workgroup so that the launch has about 256 of them
        const uint64_t want = ((uint64_t)slots * (Mp / kXprepLinesRows) + 255u) / 256u;
        if (want <= 64u) return launch_lines<XBF16, LAYOUT, 1, 1, 1, true>(x, M, Mp, K, xh, rs, st);
        if (want <= 128u) return launch_lines<XBF16, LAYOUT, 1, 1, 2, true>(x, M, Mp, K, xh, rs, st);
        if (want <= 256u) return launch_lines<XBF16, LAYOUT, 2, 2, 2, true>(x, M, Mp, K, xh, rs, st);
        return launch_lines<XBF16, LAYOUT, 4, 4, 2, true>(x, M, Mp, K, xh, rs, st);
    }
    // waves per row: 4096 waves in all (16 per CU), at least one slot per lane, at most
    // eight; 2500 for the f32 rows above, whose lanes then load two slots or four
    const uint32_t full = (K + 511u) / 512u;  // waves with one slot per lane
    const uint32_t waves = K < 4096u ? 4096u : 2500u;
    uint32_t wpr = 1u;
    while (wpr < 16u && ((wpr < full && wpr * Mp < waves) || 8u * wpr < full)) wpr *= 2u;
    switch (wpr) {
        case 1: return launch_rows<XBF16, LAYOUT, 1>(x, M, Mp, K, xh, rs, st);
        case 2: return launch_rows<XBF16, LAYOUT, 2>(x, M, Mp, K, xh, rs, st);
        case 4: return launch_rows<XBF16, LAYOUT, 4>(x, M, Mp, K, xh, rs, st);
        case 8: return launch_rows<XBF16, LAYOUT, 8>(x, M, Mp, K, xh, rs, st);
        default: return launch_rows<XBF16, LAYOUT, 16>(x, M, Mp, K, xh, rs, st);
    }
}

template <uint32_t LAYOUT>
hipError_t launch_xprep(const void* x, bool x_bf16, uint32_t M, uint32_t K, uint16_t* xh, float* rs, hipStream_t st) {
    return x_bf16 ? launch_xprep<true, LAYOUT>(x, M, K, xh, rs, st) : launch_xprep<false, LAYOUT>(x, M, K, xh, rs, st);
}

}  // namespace

hipError_t xprep_launch(const void* x, bool x_bf16, uint32_t M, uint32_t K, uint32_t layout, uint16_t* xh, float* rs,
                        hipStream_t st) {
    if (M == 0 || K == 0 || K % 64u) return hipErrorInvalidValue;
    switch (layout) {
        case XFRAG_NIB: return launch_xprep<XFRAG_NIB>(x, x_bf16, M, K, xh, rs, st);
        case XFRAG_BYTE: return launch_xprep<XFRAG_BYTE>(x, x_bf16, M, K, xh, rs, st);
        case XFRAG_WORD: return launch_xprep<XFRAG_WORD>(x, x_bf16, M, K, xh, rs, st);
        case XFRAG_QK: return launch_xprep<XFRAG_QK>(x, x_bf16, M, K, xh, rs, st);
        case XFRAG_Q6K: return launch_xprep<XFRAG_Q6K>(x, x_bf16, M, K, xh, rs, st);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace dmx
