// Prefill GEMM: y[m, n] = sum_k x[m, k] * w[n, k], x bf16, y fp32, on bf16 MFMA.
//
// Replaces, per prefill call of linear_gemm() (openmini-server/src/model/inference/
// model.rs:1060-1064), the f32 GEMM over weights dequantized at load
// (gemm_engine.rs:69-71).  Numerics: each code is exact in bf16 (Q4_0 as
// (q-8)/16, Q8_0 as q), bf16 x bf16 products are exact in fp32, and one
// v_mfma_f32_16x16x32_bf16 covers exactly one 32-element block, so every block's
// partial sum is scaled by its fp32 scale and added to an fp32 accumulator:
//   y[m, n] = sum_b d[n, b] * (sum_{k in b} x[m, k] * q[n, k]).
// Weights are never rounded (no bf16 q*d), activations are not requantized.  The
// per-block rescale costs 4 VALU FMAs per MFMA, about as many VALU cycles as the
// MFMA takes, so the kernel keeps both busy: two waves per SIMD, MFMA results in
// VGPRs, and each MFMA issued before the FMAs of the previous one.
// K-quant weights (the reference's reading, quant.rs:338-410 and :515-600) use their
// 32-element sub-blocks as the blocks.  Q4_K: codes as Q4_0, block factor
// 16 * d * scale (exact).  Q6_K: its scale changes every 16 elements, inside one
// MFMA's 32, so q * scale (an exact integer of at most 13 bits) enters as bf16
// hi + lo (two chained MFMAs, both exact), and the row's d is the block factor.
//
// Tiling: a workgroup of eight waves (four in two shapes) computes a kBM x (16 kWT kNW) tile
// of y with kNW column slices x kKS K parts of waves (choose_gemm_shape picks one of eight
// shapes, 128 x 192 to 64 x 32, by problem size).  A wave owns kBM rows x 16 kWT columns
// (kBM/16 x kWT MFMA subtiles of fp32 accumulators) over one K part, and the parts are added
// through LDS at the end (fixed order).  A K step is two blocks (64 elements):
//   * x: each K part's kBM x 64 bf16 slab is copied HBM -> LDS by buffer loads with
//     an LDS destination (no registers) two steps ahead, rows XOR-swizzled in 16-byte
//     segments so the A-fragment reads are bank-conflict free (counted: 0); the fragments
//     of a half step are read while the half before it computes;
//   * weights: each wave loads its kWT tiles' chunks straight into registers a group (4
//     blocks) ahead, one wide load per tile, transposes them to the MFMA lanes by row
//     swaps and converts its own B fragments (its columns are its own, so nothing is
//     converted twice).
// What bounds it: VALU issue.  Per half step and wave of the 128 x 192 shape, 24 MFMAs,
// 96 rescale FMAs, 36 conversions and about 14 others are some 680 issue cycles, 51 us at
// 512 rows of 11008 x 4096 and the 1.7 GHz the part holds under this load; with the copies,
// weight loads and LDS reads it takes 65 us, VALU issuing in 69% of the SIMDs' cycles and MFMAs
// running in 34% (from 72 us: until the stages were arrays of
// their own, the compiler waited for every load just issued before each step's first
// LDS read, so nothing was in flight across a step).  28672 x 8192 at 1024 rows: 638 ->
// 575 us; few-row and fp32 shapes, where one workgroup has its CU alone and nothing else
// hid those waits, gained most: Q8_0 4096 x 11008 at 100 fp32 rows 92 -> 40 us (with the
// 64 x 32 shape, which fills the chip there).
#include "qmm_device.hpp"
#include "qmm_gemm_shape.hpp"

#include <type_traits>

namespace qmm {
namespace {

constexpr int kBMMax = 128;  // most x rows per workgroup
constexpr int kCeilWT = 3;   // weight tiles per wave of the launch shapes the ceiling yardstick mirrors

__device__ __forceinline__ uint32_t pack_hi16(float lo, float hi) {
    // bf16 of exactly-representable values = high halves of their fp32 bits.
    return __builtin_amdgcn_perm(__float_as_uint(hi), __float_as_uint(lo), 0x07060302u);
}

// 8 Q4_0 nibbles (one code word of two's-complement q - 8, elements in order) ->
// 8 bf16 (q-8)/16.
__device__ __forceinline__ bf16x8 cvt_q4(uint32_t w) {
    uint32_t h = w >> 4;
    asm("" : "+v"(h));  // keep the shift: 1 shift + 4 SDWA converts, not 4 bit-field extracts
    const float a0 = __builtin_amdgcn_cvt_off_f32_i4(w & 0xFFu);
    const float a1 = __builtin_amdgcn_cvt_off_f32_i4((w >> 8) & 0xFFu);
    const float a2 = __builtin_amdgcn_cvt_off_f32_i4((w >> 16) & 0xFFu);
    const float a3 = __builtin_amdgcn_cvt_off_f32_i4(w >> 24);
    const float b0 = __builtin_amdgcn_cvt_off_f32_i4(h & 0xFFu);
    const float b1 = __builtin_amdgcn_cvt_off_f32_i4((h >> 8) & 0xFFu);
    const float b2 = __builtin_amdgcn_cvt_off_f32_i4((h >> 16) & 0xFFu);
    const float b3 = __builtin_amdgcn_cvt_off_f32_i4(h >> 24);
    uint32_t p[4] = {pack_hi16(a0, a1), pack_hi16(a2, a3), pack_hi16(b0, b1), pack_hi16(b2, b3)};
    return __builtin_bit_cast(bf16x8, *reinterpret_cast<uint4*>(p));
}

// 8 Q8_0 codes (two words) -> 8 bf16 q in k order.
__device__ __forceinline__ bf16x8 cvt_q8(uint32_t w0, uint32_t w1) {
    float f[8];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        f[i] = (float)(int8_t)((w0 >> (8 * i)) & 0xFFu);
        f[4 + i] = (float)(int8_t)((w1 >> (8 * i)) & 0xFFu);
    }
    uint32_t p[4] = {pack_hi16(f[0], f[1]), pack_hi16(f[2], f[3]), pack_hi16(f[4], f[5]),
                     pack_hi16(f[6], f[7])};
    return __builtin_bit_cast(bf16x8, *reinterpret_cast<uint4*>(p));
}

// Chunk geometry the GEMM reads, by weight format (layouts in qmm_internal.hpp).
template <int kFmt>
struct GFmt {
    static constexpr bool kQ8 = kFmt == OPENMINI_QMM_Q8_0;
    static constexpr bool kQ4K = kFmt == OPENMINI_QMM_Q4_K;
    static constexpr bool kQ6K = kFmt == OPENMINI_QMM_Q6_K;
    static constexpr bool kKQ = kQ4K || kQ6K;
    static constexpr bool kNib = !kQ8 && !kQ6K;            // Q4_0 / Q4_K: 16 B of nibbles per slot
    static constexpr int kCB = kQ8 ? 32 : 16;               // bytes of a slot's (low) codes
    static constexpr int kWords = kNib ? 1 : 2;             // code words per lane and block
    static constexpr int kScaleOff = kTileEntries * (kQ6K ? 24 : kCB);
    static constexpr int kDOff = kScaleOff + (kQ6K ? 2 : 1) * kTileEntries;  // K-quant: fp16 d per row
    static constexpr int kChunk = kQ4K ? kQ4KChunk : kQ6K ? kQ6KChunk : chunk_bytes_for(!kQ8);
};

// A wave's weight operands for one group of 4 blocks, as loaded: per weight tile chunk
// slot `lane` (block lane / 16, column lane % 16) whole -- its codes in one or two 16-byte
// loads, its scale -- and for K-quants the column's d.  One wide load per tile and group
// costs the address unit what one narrow load per block would.
template <int kFmt, int kWT>
struct BRaw {
    uint4 c[kWT][GFmt<kFmt>::kQ8 ? 2 : 1];
    uint2 h[GFmt<kFmt>::kQ6K ? kWT : 1];  // Q6_K: the slot's top code bits
    uint32_t s[kWT];
    uint32_t d[GFmt<kFmt>::kKQ ? kWT : 1];
};

// The same after the transpose across the wave's four 16-lane rows: for block t the
// lane's 8 codes (elements 8 kq .. 8 kq + 7 of column li: Q4_0 / Q4_K one word of nibbles,
// Q8_0 two words of bytes, Q6_K the low-nibble word and the top-bit word) and the block
// factor (Q6_K: the column's scale pair as bits, its d in `d`).
template <int kFmt, int kWT>
struct BGroup {
    uint32_t c[kWT][4][GFmt<kFmt>::kWords];
    float f[kWT][4];
    float d[GFmt<kFmt>::kQ6K ? kWT : 1];
};

// 8 Q6_K codes of lane quarter kq -> bf16 hi / lo parts of q * sc, q * sc exact (at
// most 13 significant bits): hi keeps the top 8 bits, lo = q * sc - hi has at most 5.
// w: the slot's low-nibble word kq; hm: its top-bit word kq / 2 (qmm_internal.hpp).
__device__ __forceinline__ void split_q6(uint32_t w, uint32_t hm, int kq, float sc4, bf16x8& hi, bf16x8& lo) {
    // 4 q per int8 byte: low 4 bits at 2..5, the top 2 bits (fields 2 (kq & 1) and
    // 2 (kq & 1) + 1 of each byte of hm) at 6..7; elements 8 kq + 0..3, then + 4..7
    const int sh = (kq & 1) * 4;
    const uint32_t b0 = ((w << 2) & 0x3C3C3C3Cu) | ((hm << (6 - sh)) & 0xC0C0C0C0u);
    const uint32_t b1 = ((w >> 2) & 0x3C3C3C3Cu) | ((hm << (4 - sh)) & 0xC0C0C0C0u);
    float f[8];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        // (4 q) * (sc / 4): exact
        f[i] = (float)(int8_t)((b0 >> (8 * i)) & 0xFFu) * sc4;
        f[4 + i] = (float)(int8_t)((b1 >> (8 * i)) & 0xFFu) * sc4;
    }
    uint32_t h[4], l[4];
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        const uint32_t u0 = __float_as_uint(f[2 * p]), u1 = __float_as_uint(f[2 * p + 1]);
        const float r0 = f[2 * p] - __uint_as_float(u0 & 0xFFFF0000u);
        const float r1 = f[2 * p + 1] - __uint_as_float(u1 & 0xFFFF0000u);
        h[p] = __builtin_amdgcn_perm(u1, u0, 0x07060302u);
        l[p] = pack_hi16(r0, r1);
    }
    hi = __builtin_bit_cast(bf16x8, *reinterpret_cast<uint4*>(h));
    lo = __builtin_bit_cast(bf16x8, *reinterpret_cast<uint4*>(l));
}

// The same q * sc as fp16 hi (rounded toward zero: 11 significant bits) + lo (the
// remaining at most 2 bits), both exact.
__device__ __forceinline__ void split_q6_f16(uint32_t w, uint32_t hm, int kq, float sc4, f16x8& hi, f16x8& lo) {
    const int sh = (kq & 1) * 4;
    const uint32_t b0 = ((w << 2) & 0x3C3C3C3Cu) | ((hm << (6 - sh)) & 0xC0C0C0C0u);
    const uint32_t b1 = ((w >> 2) & 0x3C3C3C3Cu) | ((hm << (4 - sh)) & 0xC0C0C0C0u);
    float f[8];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        f[i] = (float)(int8_t)((b0 >> (8 * i)) & 0xFFu) * sc4;
        f[4 + i] = (float)(int8_t)((b1 >> (8 * i)) & 0xFFu) * sc4;
    }
    uint32_t h[4], l[4];
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        const auto hp = __builtin_amdgcn_cvt_pkrtz(f[2 * p], f[2 * p + 1]);
        h[p] = __builtin_bit_cast(uint32_t, hp);
        l[p] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(f[2 * p] - (float)hp[0], f[2 * p + 1] - (float)hp[1]));
    }
    hi = __builtin_bit_cast(f16x8, *reinterpret_cast<uint4*>(h));
    lo = __builtin_bit_cast(f16x8, *reinterpret_cast<uint4*>(l));
}

// Workgroup shape: kBM x rows, kNW column slices x kKS K parts of waves, two x stages in
// LDS.  A step is one 128-byte piece of every x row: two blocks of bf16 x, one block of
// split x (its hi and lo parts).
template <int kBM, int kNW, int kKS, int kWT_>
struct Shape {
    static constexpr int kWT = kWT_;                       // weight tiles (16 columns each) per wave
    static constexpr int kMI = kBM / 16;                   // MFMA row subtiles per wave
    static constexpr int kThreads = 64 * kNW * kKS;
    static constexpr int kBT = kNW * kWT;                 // weight tiles per workgroup
    static constexpr int kRowB = 128;                      // bytes of one x row per step
    static constexpr int kSegs = kRowB / 16;               // 16-byte segments per row
    static constexpr int kSlabB = kBM * kRowB;             // one K part's x slab per step
    static constexpr int kStageB = kKS * kSlabB;
    static constexpr int kRowsPerCopy = 1024 / kRowB;      // one 1 KB copy instruction
    static constexpr int kCopies = kSlabB / kNW / 1024;     // copies per wave per step
    static constexpr int kRedSlots = (kKS - 1) * kMI * kWT;  // K-part partials: 1 KB subtiles per column slice
    // subtiles per column slice one stage array holds, and its bytes
    static constexpr int kSlotsPerStage =
        kStageB / 1024 / kNW > (kRedSlots + 1) / 2 ? kStageB / 1024 / kNW : (kRedSlots + 1) / 2;
    static constexpr int kArrB = kSlotsPerStage * kNW * 1024;
    static_assert(kCopies * kNW * 1024 == kSlabB, "whole copies per wave");
    static_assert(kArrB >= kStageB, "a stage array holds a stage");
};

// Waves per SIMD the kernel is built for: two (one workgroup per CU, at most 256
// registers).  The 64-row tiles of two weight tiles per wave come out at 115-130, and up to
// 128 a CU runs two of them; Q8_0's 64 x 128 on bf16 x misses that by two, and held to it
// runs 11008 x 4096 at 512 rows in 80 us instead of 91 (the other Q8_0 instances would
// spill in the main loop: 64 x 64 40 -> 56 us at 100 rows of 4096 x 11008).
template <int kFmt, int kBM, int kNW, int kWT, bool kX2>
constexpr int kGemmWaves = kBM == 64 && kNW == 4 && kWT == 2 && kFmt == OPENMINI_QMM_Q8_0 && !kX2 ? 4 : 2;

// gate_in_y: y holds the gate projection on entry and each element is replaced by
// silu(gate) * (x . W^T), silu(v) = v / (1 + exp(-v)) (model.rs:713-735, :1187-1189).
// kX2: x holds split fp32 activations (split_rows_kernel), scaled by 2^e per row
// (x_exp[m] = e).  Each block runs two chained fp16 MFMAs per subtile (hi, then lo, into
// one fp32 sum) with fp16 codes, then the same rescale; outputs are scaled back by 2^-e.
template <int kFmt, int kBM, int kNW, int kKS, int kWT, bool kX2>
__global__ __launch_bounds__(64 * kNW * kKS, (kGemmWaves<kFmt, kBM, kNW, kWT, kX2>)) void gemm_kernel(
    const uint16_t* __restrict__ x, const int* __restrict__ x_exp, const uint8_t* __restrict__ chunks,
    float* __restrict__ y, int m_rows, int n_rows, int n_tiles, int groups, int k, int gate_in_y) {
    using S = Shape<kBM, kNW, kKS, kWT>;
    using F = GFmt<kFmt>;
    constexpr int kMI = S::kMI;
    constexpr int kChunk = F::kChunk;
    constexpr int kWB = kX2 ? 1 : 2;  // weight blocks per step
    constexpr int kSPG = kTileBlocks / kWB;  // steps per group
    // One array per x stage: the compiler then knows that a copy into one stage does not
    // alias the fragment reads of another.  (With a single array it waited for every
    // outstanding load before each step's first read, so nothing was in flight across
    // a step.)
    __shared__ __attribute__((aligned(16))) uint8_t lds0[S::kArrB];
    __shared__ __attribute__((aligned(16))) uint8_t lds1[S::kArrB];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int kh = wave / kNW, wn = wave % kNW;
    const int li = lane & 15;  // A row / B column inside a 16 x 16 subtile
    const int kq = lane >> 4;  // which 8-element quarter of the 32-element block
    const int bx = blockIdx.x, by = blockIdx.y;
    const int m0 = by * kBM;
    const int tile0 = bx * S::kBT + wn * kWT;

    // this K part's groups; all parts step together (barriers), a shorter one idles
    const int g0 = (int)((int64_t)groups * kh / kKS);
    const int g1 = (int)((int64_t)groups * (kh + 1) / kKS);
    const int g_last = max(g1 - 1, 0);
    const int part_groups = (groups + kKS - 1) / kKS;

    // x is < 2 GiB (the launcher splits m); the chunks < 4 GiB (checked at upload)
    const __amdgpu_buffer_rsrc_t x_rs = make_rsrc(x, (uint32_t)m_rows * (uint32_t)k * (kX2 ? 4u : 2u));
    const __amdgpu_buffer_rsrc_t w_rs = make_rsrc(chunks, (uint32_t)n_tiles * groups * kChunk);

    // ---- x slab copies: kCopies x 1 KB per wave per step.
    // bf16 x: kRowsPerCopy rows each; LDS position p of row r holds the row's 16-byte
    // segment s = p ^ (r % kSegs), so the fragment reads are bank-conflict free.
    // Split x: copy c is the hi (c even) or lo part of row subtile c / 2, which lies in
    // memory as the MFMA reads it.
    const int r_lane = wn * (kBM / kNW) + lane / S::kSegs;
    const int p_lane = lane % S::kSegs;
    const int nb = k / kQK;
    const int x_tiles = (m_rows + 15) / 16;
    auto issue_x = [&](int s, uint8_t* stage) {  // s: step of this part; past its end: zeros
        const int g = g0 + s / kSPG, sub = s % kSPG;
        const uint32_t k_lim = g < g1 ? (uint32_t)k : 0u;
        uint8_t* base = stage + kh * S::kSlabB + wn * S::kCopies * 1024;
#pragma unroll
        for (int j = 0; j < S::kCopies; ++j) {
            uint32_t voff, soff = 0;
            if constexpr (kX2) {
                // a row tile is k / 32 pieces of 128 bytes per row; the last one may have
                // fewer rows.  All offsets stay inside x: blocks past K repeat the last
                // one (their weights are zero), tiles past m and rows past the tile
                // repeat the last.
                const int c = wn * S::kCopies + j;
                const int rt = min(by * kMI + c / 2, x_tiles - 1);
                const int rows = min(16, m_rows - rt * 16);
                voff = (uint32_t)(kq * rows + min(li, rows - 1)) * 16u | (k_lim ? 0u : 0x80000000u);
                soff = (uint32_t)rt * 64u * (uint32_t)k +
                       (uint32_t)(min(min(g, g_last) * kTileBlocks + sub, nb - 1) * 2 + (c & 1)) * (uint32_t)rows * 64u;
            } else {
                const int r = r_lane + j * S::kRowsPerCopy;
                const uint32_t seg = (uint32_t)((p_lane ^ (r % S::kSegs)) * 8) + (uint32_t)(g * kTileBlocks + sub * kWB) * kQK;
                const uint32_t gm = (uint32_t)min(m0 + r, m_rows - 1);  // rows past m repeat the last one
                // segments past K read zero (an out-of-range buffer offset)
                voff = seg < k_lim ? (gm * (uint32_t)k + seg) * 2u : 0x80000000u;
            }
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                x_rs, (__attribute__((address_space(3))) void*)(base + j * 1024), 16, voff, soff, 0, 0);
        }
    };

    // ---- weight operands of one group
    uint32_t tile_off[kWT];
#pragma unroll
    for (int j = 0; j < kWT; ++j) tile_off[j] = (uint32_t)min(tile0 + j, n_tiles - 1) * groups * kChunk;
    auto load_b = [&](BRaw<kFmt, kWT>& R, int g) {
#pragma unroll
        for (int j = 0; j < kWT; ++j) {
            const uint32_t soff = tile_off[j] + (uint32_t)g * kChunk;
            R.c[j][0] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(w_rs, lane * F::kCB, soff, 0));
            if constexpr (F::kQ8)
                R.c[j][1] =
                    __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(w_rs, lane * F::kCB + 16, soff, 0));
            if constexpr (F::kQ6K)
                R.h[j] = __builtin_bit_cast(
                    uint2, __builtin_amdgcn_raw_buffer_load_b64(w_rs, kTileEntries * 16 + lane * 8, soff, 0));
            if constexpr (F::kQ4K)
                R.s[j] = __builtin_amdgcn_raw_buffer_load_b8(w_rs, F::kScaleOff + lane, soff, 0);
            else
                R.s[j] = __builtin_amdgcn_raw_buffer_load_b16(w_rs, F::kScaleOff + lane * 2, soff, 0);
            if constexpr (F::kKQ) R.d[j] = __builtin_amdgcn_raw_buffer_load_b16(w_rs, F::kDOff + li * 2, soff, 0);
        }
    };
    // bf16 x runs Q4 codes as (q - 8) / 16: the block factor carries the 16 (exact)
    constexpr float kUnit = F::kNib && !kX2 ? 16.0f : 1.0f;
    auto unpack_b = [&](BGroup<kFmt, kWT>& B, const BRaw<kFmt, kWT>& R, bool live) {  // !live: factors 0
#pragma unroll
        for (int j = 0; j < kWT; ++j) {
            uint32_t e[4], o[4];
            const uint4 c = R.c[j][0];
            if constexpr (F::kQ8) {
                const uint4 c1 = R.c[j][1];
                e[0] = c.x; o[0] = c.y; e[1] = c.z; o[1] = c.w;
                e[2] = c1.x; o[2] = c1.y; e[3] = c1.z; o[3] = c1.w;
                transpose4(e[0], e[1], e[2], e[3]);
                transpose4(o[0], o[1], o[2], o[3]);
            } else {
                e[0] = c.x; e[1] = c.y; e[2] = c.z; e[3] = c.w;
                transpose4(e[0], e[1], e[2], e[3]);
                if constexpr (F::kQ6K) {  // lane (kq, i) takes top-bit word kq / 2
                    o[0] = R.h[j].x; o[1] = R.h[j].x; o[2] = R.h[j].y; o[3] = R.h[j].y;
                    transpose4(o[0], o[1], o[2], o[3]);
                }
            }
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                B.c[j][t][0] = e[t];
                if constexpr (F::kWords == 2) B.c[j][t][1] = o[t];
            }
            if constexpr (F::kQ6K) {
                broadcast4(__uint_as_float(R.s[j]), B.f[j]);
                B.d[j] = live ? f16_bits_to_f32((uint16_t)R.d[j]) : 0.0f;
            } else if constexpr (F::kQ4K) {
                broadcast4(live ? f16_bits_to_f32((uint16_t)R.d[j]) * (float)(R.s[j] & 0xFFu) * kUnit : 0.0f, B.f[j]);
            } else {
                broadcast4(live ? f16_bits_to_f32((uint16_t)R.s[j]) * kUnit : 0.0f, B.f[j]);
            }
        }
    };
    // Q6_K: a quarter of the scale of the lane's 16-element half of block t (exact)
    auto q6_scale = [&](const BGroup<kFmt, kWT>& B, int j, int t) {
        return (float)(int8_t)((__float_as_uint(B.f[j][t]) >> ((kq >> 1) * 8)) & 0xFFu) * 0.25f;
    };

    f32x4 acc[kMI][kWT];
    // Q6_K on bf16 x: the sums of the current super-block, before its d (one per tile
    // row and super-block); the other instances leave them unused.
    constexpr bool kChain = F::kQ6K && !kX2;
    f32x4 sacc[kMI][kWT];
#pragma unroll
    for (int i = 0; i < kMI; ++i)
#pragma unroll
        for (int j = 0; j < kWT; ++j) acc[i][j] = sacc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    // A fragments of half h of the step in `stage`: rows i * 16 + li, elements 8 kq ..
    // 8 kq + 7 of bf16 block h; or of split x's row subtiles h kMI / 2 + i / 2 the fp16 hi
    // (i even) / lo (i odd) parts.
    typedef uint4 AFrags[kMI];
    auto read_a = [&](AFrags& a, const uint8_t* stage, int h) {
        const uint8_t* slab = stage + kh * S::kSlabB;
#pragma unroll
        for (int i = 0; i < kMI; ++i) {
            if constexpr (kX2) {
                a[i] = *reinterpret_cast<const uint4*>(slab + (h * kMI + i) * 1024 + lane * 16);
            } else {
                const int r = i * 16 + li;
                a[i] = *reinterpret_cast<const uint4*>(slab + r * S::kRowB + (((h * 4 + kq) ^ (r % S::kSegs)) * 16));
            }
        }
    };
    auto bf = [](const uint4& v) { return __builtin_bit_cast(bf16x8, v); };
    auto hf = [](const uint4& v) { return __builtin_bit_cast(f16x8, v); };
    // Q6_K block t: the scale changes every 16 elements, inside an MFMA's 32, so it
    // is folded into the codes: q * sc (exact integers) as bf16 hi + lo.  The d is one per
    // tile row and super-block, so the blocks of a super-block chain into one sum per
    // output (sacc; all hi MFMAs, then all lo ones, so no MFMA waits on the one before),
    // and flush_q6 applies d once per super-block: one FMA per output per 8 blocks
    // instead of one per block.
    auto compute_q6 = [&](const BGroup<kFmt, kWT>& B, const AFrags& a, int t) {
        if constexpr (kChain) {
            bf16x8 bh[kWT], bl[kWT];
#pragma unroll
            for (int j = 0; j < kWT; ++j) split_q6(B.c[j][t][0], B.c[j][t][1], kq, q6_scale(B, j, t), bh[j], bl[j]);
#pragma unroll
            for (int q = 0; q < kMI * kWT; ++q)
                sacc[q / kWT][q % kWT] =
                    __builtin_amdgcn_mfma_f32_16x16x32_bf16(bf(a[q / kWT]), bh[q % kWT], sacc[q / kWT][q % kWT], 0, 0, 0);
#pragma unroll
            for (int q = 0; q < kMI * kWT; ++q)
                sacc[q / kWT][q % kWT] =
                    __builtin_amdgcn_mfma_f32_16x16x32_bf16(bf(a[q / kWT]), bl[q % kWT], sacc[q / kWT][q % kWT], 0, 0, 0);
        }
    };
    // Q6_K: after the last group of a super-block, or of this K part, acc += sacc * d.
    auto flush_q6 = [&](const BGroup<kFmt, kWT>& B) {
        if constexpr (kChain) {
#pragma unroll
            for (int j = 0; j < kWT; ++j)
#pragma unroll
                for (int i = 0; i < kMI; ++i) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) acc[i][j][r] = fmaf(sacc[i][j][r], B.d[j], acc[i][j][r]);
                    sacc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
                }
        }
    };
    // Block t of the group on bf16 fragments `a`: kMI x kWT MFMAs and their rescales.
    auto compute = [&](const BGroup<kFmt, kWT>& B, const AFrags& a, int t) {
        if constexpr (F::kQ6K) {
            compute_q6(B, a, t);
            return;
        }
        bf16x8 b[kWT];
#pragma unroll
        for (int j = 0; j < kWT; ++j) {
            if constexpr (F::kNib)
                b[j] = cvt_q4(B.c[j][t][0]);
            else
                b[j] = cvt_q8(B.c[j][t][0], B.c[j][t][1]);
        }
        // MFMA q + 1 is issued before the FMAs of q (two result registers)
        f32x4 pp[2];
        pp[0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bf(a[0]), b[0], f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
        for (int q = 0; q < kMI * kWT; ++q) {
            if (q + 1 < kMI * kWT)
                pp[(q + 1) & 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                    bf(a[(q + 1) / kWT]), b[(q + 1) % kWT], f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
            for (int r = 0; r < 4; ++r)
                acc[q / kWT][q % kWT][r] = fmaf(pp[q & 1][r], B.f[q % kWT][t], acc[q / kWT][q % kWT][r]);
        }
    };
    // Split x, block t, half h of its row subtiles: per subtile the hi and the lo
    // fragments times the same fp16 codes, chained into one fp32 sum (exact products),
    // then the rescale.  Q6_K: q * scale as fp16 hi + lo codes, four chained MFMAs per
    // subtile.  (Chaining a super-block's blocks as on bf16 x was slower here: 194 -> 225
    // us at M = 512; these four MFMAs per block outweigh the rescale, and the chained
    // sums' registers rule out the wide tiles.)
    constexpr int kCodes = F::kQ6K ? 2 : 1;
    typedef f16x8 BX2[kWT][kCodes];
    auto convert_x2 = [&](BX2& b, const BGroup<kFmt, kWT>& B, int t) {
#pragma unroll
        for (int j = 0; j < kWT; ++j) {
            if constexpr (F::kQ6K)
                split_q6_f16(B.c[j][t][0], B.c[j][t][1], kq, q6_scale(B, j, t), b[j][0], b[j][kCodes - 1]);
            else if constexpr (F::kNib)
                b[j][0] = codes_q4_perm(B.c[j][t][0]);  // split x is stored in its order
            else
                b[j][0] = codes_q8(B.c[j][t][0], B.c[j][t][F::kWords - 1]);
        }
    };
    auto compute_x2 = [&](const BX2& b, const BGroup<kFmt, kWT>& B, const AFrags& a, int t, int h) {
        constexpr int kHalf = kMI / 2;
        auto block = [&](int q) {
            const int i = q / kWT, j = q % kWT;
            f32x4 v = __builtin_amdgcn_mfma_f32_16x16x32_f16(hf(a[2 * i]), b[j][0], f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
            v = __builtin_amdgcn_mfma_f32_16x16x32_f16(hf(a[2 * i + 1]), b[j][0], v, 0, 0, 0);
#pragma unroll
            for (int c = 1; c < kCodes; ++c) {
                v = __builtin_amdgcn_mfma_f32_16x16x32_f16(hf(a[2 * i]), b[j][c], v, 0, 0, 0);
                v = __builtin_amdgcn_mfma_f32_16x16x32_f16(hf(a[2 * i + 1]), b[j][c], v, 0, 0, 0);
            }
            return v;
        };
        // the MFMAs of subtile q + 1 are issued before the FMAs of q
        f32x4 pp[2];
        pp[0] = block(0);
#pragma unroll
        for (int q = 0; q < kHalf * kWT; ++q) {
            if (q + 1 < kHalf * kWT) pp[(q + 1) & 1] = block(q + 1);
            const int i = h * kHalf + q / kWT, j = q % kWT;
            float d;
            if constexpr (F::kQ6K) d = B.d[j]; else d = B.f[j][t];
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[i][j][r] = fmaf(pp[q & 1][r], d, acc[i][j][r]);
        }
    };

    // Step s runs as two halves, each with the fragments of the next half on their way
    // from LDS.  Between the halves the wave waits for x(s + 1) -- until at most the loads
    // issued after its copies are outstanding -- and for its own fragment reads of
    // step s; one barrier then makes every wave's copies visible and frees the stage of
    // step s, which takes x(s + 2).  A group's first step loads the next group's
    // weights, after its first half (issued right after the copies, every wave of the
    // CU would queue its vector-memory instructions at once and stall its MFMAs behind
    // them).  The loads are unconditional (steps past this part's end repeat its last
    // group, cache hits), so the count of outstanding loads is the same on every path; the
    // memory clobbers keep their order.  With one column slice every wave reads only
    // what it copied itself, and no barrier is needed.
    // A half's MFMAs and rescale run at raised wave priority, so the SIMD's other wave
    // yields issue slots to them.
    constexpr int kBLoads = kWT * ((F::kQ8 || F::kQ6K ? 3 : 2) + (F::kKQ ? 1 : 0));
    static_assert(kBLoads <= 63, "vmcnt counts up to 63");
    // Q6_K's 128-row tiles have no registers for a second set: they read each half's
    // fragments just before it (the second half's before the wait, its stage being
    // overwritten after it).
    constexpr bool kAhead = !(F::kQ6K && kBM == 128);
    AFrags f0, f1;
    // Keeps memory operations in order, and the scheduler from moving one half's work (the
    // next blocks' code conversions above all) into another, which would not fit the
    // registers.
    auto fence = [] {
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    auto step = [&](int gi, int sub, const BGroup<kFmt, kWT>& B, BRaw<kFmt, kWT>& next, uint8_t* now,
                    const uint8_t* after) {
        const int s = gi * kSPG + sub;
        BX2 bx;
        if constexpr (kAhead) read_a(f1, now, 1);
        else read_a(f0, now, 0);
        fence();
        __builtin_amdgcn_s_setprio(3);
        if constexpr (kX2) {
            convert_x2(bx, B, sub);
            compute_x2(bx, B, f0, sub, 0);
        } else {
            compute(B, f0, sub * 2);
        }
        __builtin_amdgcn_s_setprio(0);
        fence();
        if (sub == 0) load_b(next, min(g0 + gi + 1, g_last));
        if constexpr (!kAhead) read_a(f0, now, 1);
        fence();
        if (sub == 0)  // constant after unrolling
            __builtin_amdgcn_s_waitcnt(vmcnt_only(kBLoads) & ~0x0F00);
        else
            __builtin_amdgcn_s_waitcnt(vmcnt_only(0) & ~0x0F00);
        if constexpr (kNW > 1) __builtin_amdgcn_s_barrier();
        fence();
        issue_x(s + 2, now);
        fence();
        if constexpr (kAhead) read_a(f0, after, 0);
        fence();
        __builtin_amdgcn_s_setprio(3);
        if constexpr (kX2)
            compute_x2(bx, B, kAhead ? f1 : f0, sub, 1);
        else
            compute(B, kAhead ? f1 : f0, sub * 2 + 1);
        __builtin_amdgcn_s_setprio(0);
        const int g = g0 + gi;
        if (sub == kSPG - 1 && kChain && ((g & 1) == 1 || g >= g1 - 1)) flush_q6(B);
    };
    issue_x(0, lds0);
    issue_x(1, lds1);
    BRaw<kFmt, kWT> raw;
    load_b(raw, min(g0, g_last));
    __builtin_amdgcn_s_waitcnt(vmcnt_only(0));
    if constexpr (kNW > 1) __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if constexpr (kAhead) read_a(f0, lds0, 0);
    BGroup<kFmt, kWT> B;
    unpack_b(B, raw, g0 < g1);
    for (int gi = 0; gi < part_groups; ++gi) {
        step(gi, 0, B, raw, lds0, lds1);
        step(gi, 1, B, raw, lds1, lds0);
        if constexpr (kSPG == 4) {
            step(gi, 2, B, raw, lds0, lds1);
            step(gi, 3, B, raw, lds1, lds0);
        }
        unpack_b(B, raw, g0 + gi + 1 < g1);
    }
    __builtin_amdgcn_s_waitcnt(vmcnt_only(0));  // no copy may land after the stages are reused

    // ---- K parts meet in LDS (the stages are free after this barrier), then store.  A part
    // hands its sums of a subtile over as one 16-byte LDS write per lane; they are added in part
    // order (fixed, so the bits do not depend on timing).  Lane holds D[4 kq + r][li] of each
    // 16 x 16 subtile.
    // Four and eight parts: the slice's subtiles are dealt out, subtile q to part q % kKS, so that
    // the sums, the gate and the stores run on all waves and not on one in kKS (fp32 x, Q8_0
    // 5632 x 2048 gate and up at 160 rows 54.7 -> 44.9 us; bf16 x, Q8_0 3072 x 2048 at 384 rows
    // 14.3 -> 13.7; 0.4 - 0.6 us on every size of these shapes).
    // Two parts: part 0 takes all; dealt out, the 128-row tiles had to spill in the main loop
    // (split x, Q8_0 11008 x 4096 at 384 rows 94 -> 109 us) and the others gained nothing.
    __syncthreads();
    auto all = [](int, int, int) { return true; };
    if constexpr (kKS > 2) {
        // lane indexes of their own: the main loop's would have to live across it
        const int ln = (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)), lr = ln & 15, lq = ln >> 4;
        constexpr int kSub = kMI * kWT, kOwn = kSub / kKS;  // subtiles of the slice, of a part
        static_assert(kSub % kKS == 0 && (kKS == 4 || kKS == 8), "every K part takes the same number of subtiles");
        auto slot = [&](int part, int q) {
            const int owner = q % kKS, l = q * (kKS - 1) + (part < owner ? part : part - 1), arr = l / S::kSlotsPerStage;
            uint8_t* base = arr == 0 ? lds0 : lds1;
            return reinterpret_cast<f32x4*>(base) + ((l % S::kSlotsPerStage) * kNW + wn) * 64 + ln;
        };
        auto out = [&](int i, int j) { return y + (size_t)(m0 + i * 16 + lq * 4) * n_rows + (tile0 + j) * kTileRows + lr; };
        auto some = [&](int i, int j, int r) {
            return m0 + i * 16 + lq * 4 + r < m_rows && (tile0 + j) * kTileRows + lr < n_rows;
        };
        auto finish = [&](auto own, auto gated, auto inside) {
            constexpr int h = decltype(own)::value;
            // split x: the row scale 2^-e; these and the gate's loads on their way before the first sum
            int rexp[kX2 ? kMI : 1][4];
            if constexpr (kX2) {
#pragma unroll
                for (int i = 0; i < kMI; ++i)
#pragma unroll
                    for (int r = 0; r < 4; ++r) rexp[i][r] = -x_exp[min(m0 + i * 16 + lq * 4 + r, m_rows - 1)];
            }
            float gate[kOwn][4];
            if constexpr (gated) {
#pragma unroll
                for (int o = 0; o < kOwn; ++o) {
                    const int q = o * kKS + h, i = q / kWT, j = q % kWT;
#pragma unroll
                    for (int r = 0; r < 4; ++r) gate[o][r] = inside(i, j, r) ? out(i, j)[(size_t)r * n_rows] : 0.0f;
                }
            }
#pragma unroll
            for (int o = 0; o < kOwn; ++o) {
                const int q = o * kKS + h, i = q / kWT, j = q % kWT;
                f32x4 sum = h == 0 ? acc[i][j] : *slot(0, q);
#pragma unroll
                for (int part = 1; part < kKS; ++part) sum += part == h ? acc[i][j] : *slot(part, q);
                float* yp = out(i, j);
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    float v = sum[r];
                    if constexpr (kX2) v = __builtin_amdgcn_ldexpf(v, rexp[i][r]);
                    if constexpr (gated) v = gate[o][r] / (1.0f + expf(-gate[o][r])) * v;
                    if (inside(i, j, r)) yp[(size_t)r * n_rows] = v;
                }
            }
        };
#pragma unroll
        for (int h = 0; h < kKS; ++h)
            if (kh == h) {
#pragma unroll
                for (int q = 0; q < kSub; ++q)
                    if (q % kKS != h) *slot(h, q) = acc[q / kWT][q % kWT];
            }
        __syncthreads();
        auto part = [&](auto own) {
            if (kh != decltype(own)::value) return;
            if (gate_in_y)
                finish(own, std::true_type{}, some);
            else if (m0 + kBM <= m_rows && (tile0 + kWT) * kTileRows <= n_rows)  // whole tile inside y
                finish(own, std::false_type{}, all);
            else
                finish(own, std::false_type{}, some);
        };
        part(std::integral_constant<int, 0>{});
        part(std::integral_constant<int, 1>{});
        part(std::integral_constant<int, 2>{});
        part(std::integral_constant<int, 3>{});
        if constexpr (kKS == 8) {
            part(std::integral_constant<int, 4>{});
            part(std::integral_constant<int, 5>{});
            part(std::integral_constant<int, 6>{});
            part(std::integral_constant<int, 7>{});
        }
    } else {
        auto slot = [&](int i, int j) {
            const int l = i * kWT + j, arr = l / S::kSlotsPerStage;
            uint8_t* base = arr == 0 ? lds0 : lds1;
            return reinterpret_cast<f32x4*>(base) + ((l % S::kSlotsPerStage) * kNW + wn) * 64 + lane;
        };
        if (kh == 1) {
#pragma unroll
            for (int i = 0; i < kMI; ++i)
#pragma unroll
                for (int j = 0; j < kWT; ++j) *slot(i, j) = acc[i][j];
        }
        __syncthreads();
        if (kh == 0) {
            fence();
            f32x4 part[kMI][kWT];  // all reads in flight before the first add
#pragma unroll
            for (int i = 0; i < kMI; ++i)
#pragma unroll
                for (int j = 0; j < kWT; ++j) part[i][j] = *slot(i, j);
#pragma unroll
            for (int i = 0; i < kMI; ++i)
#pragma unroll
                for (int j = 0; j < kWT; ++j) acc[i][j] += part[i][j];
            // split x: the row scale 2^-e of each of the lane's output rows
            int rexp[kX2 ? kMI : 1][4];
            if constexpr (kX2) {
#pragma unroll
                for (int i = 0; i < kMI; ++i)
#pragma unroll
                    for (int r = 0; r < 4; ++r) rexp[i][r] = -x_exp[min(m0 + i * 16 + kq * 4 + r, m_rows - 1)];
            }
            // a row subtile's gate values are read together, before its first store
            auto put = [&](int j, auto gated, auto inside) {
#pragma unroll
                for (int i = 0; i < kMI; ++i) {
                    float* yp = y + (size_t)(m0 + i * 16 + kq * 4) * n_rows + (tile0 + j) * kTileRows + li;
                    float gate[4] = {0.f, 0.f, 0.f, 0.f};
                    if constexpr (gated) {
#pragma unroll
                        for (int r = 0; r < 4; ++r)
                            if (inside(i, j, r)) gate[r] = yp[(size_t)r * n_rows];
                    }
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        float v = acc[i][j][r];
                        if constexpr (kX2) v = __builtin_amdgcn_ldexpf(v, rexp[i][r]);
                        if constexpr (gated) v = gate[r] / (1.0f + expf(-gate[r])) * v;
                        if (inside(i, j, r)) yp[(size_t)r * n_rows] = v;
                    }
                }
            };
            auto some = [&](int i, int j, int r) {
                return m0 + i * 16 + kq * 4 + r < m_rows && (tile0 + j) * kTileRows + li < n_rows;
            };
            if (m0 + kBM <= m_rows && (tile0 + kWT) * kTileRows <= n_rows && !gate_in_y) {
#pragma unroll
                for (int j = 0; j < kWT; ++j) put(j, std::false_type{}, all);
            } else if (!gate_in_y) {
#pragma unroll
                for (int j = 0; j < kWT; ++j) put(j, std::false_type{}, some);
            } else {
#pragma unroll
                for (int j = 0; j < kWT; ++j) put(j, std::true_type{}, some);
            }
        }
    }
}

// x rows of k elements (bf16, or split fp32: 4 bytes per element).
template <int kFmt, int kBM, int kNW, int kKS, int kWT, bool kX2>
hipError_t launch_shape(const Weight& w, const uint16_t* x, const int* x_exp, float* y, int64_t m, bool gate_in_y,
                        hipStream_t s) {
    using S = Shape<kBM, kNW, kKS, kWT>;
    const dim3 grid((unsigned)((w.n_tiles + S::kBT - 1) / S::kBT), (unsigned)((m + kBM - 1) / kBM));
    hipLaunchKernelGGL((gemm_kernel<kFmt, kBM, kNW, kKS, kWT, kX2>), grid, dim3(S::kThreads), 0, s, x, x_exp, w.chunks,
                       y, (int)m, (int)w.n, (int)w.n_tiles, (int)w.groups, (int)w.k, (int)gate_in_y);
    return hipGetLastError();
}

// Workgroups of `kernel` (at `threads` per workgroup) one CU holds at once.
int blocks_per_cu(const void* kernel, int threads) {
    int n = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, kernel, threads, 0) != hipSuccess) return 1;
    return n;
}

// The launch shapes' rows per workgroup, column slices, K parts and weight tiles per wave, in
// the order of choose_gemm_shape.
constexpr int kForm[kShapes][4] = {{128, 4, 2, 3}, {128, 4, 2, 2}, {64, 2, 4, 3}, {64, 4, 2, 2},
                                   {64, 2, 4, 2},  {64, 1, 8, 2},  {64, 2, 2, 2}, {128, 2, 2, 3}};
// Not built for Q6_K on bf16 x: shapes 0 and 7 (the super-block sums of 128 rows x 3 weight tiles
// would not fit the registers) and 3 (two per CU do not fit, and alone it is nowhere the fastest).
template <int kFmt, bool kX2, int kShape>
constexpr bool kBuilt = kFmt != OPENMINI_QMM_Q6_K || kX2 || (kShape != 0 && kShape != 3 && kShape != 7);

// Workgroups per CU of a shape's kernel; -1: not built.
template <int kFmt, bool kX2, int kShape>
int occupancy() {
    constexpr const int* f = kForm[kShape];
    if constexpr (kBuilt<kFmt, kX2, kShape>)
        return blocks_per_cu((const void*)gemm_kernel<kFmt, f[0], f[1], f[2], f[3], kX2>, 64 * f[1] * f[2]);
    else
        return -1;
}

// Of all shapes, queried once per instantiation.
template <int kFmt, bool kX2>
const int (&shape_occupancy())[kShapes] {
    static const int per_cu[kShapes] = {occupancy<kFmt, kX2, 0>(), occupancy<kFmt, kX2, 1>(), occupancy<kFmt, kX2, 2>(),
                                        occupancy<kFmt, kX2, 3>(), occupancy<kFmt, kX2, 4>(), occupancy<kFmt, kX2, 5>(),
                                        occupancy<kFmt, kX2, 6>(), occupancy<kFmt, kX2, 7>()};
    return per_cu;
}

template <int kFmt, bool kX2>
hipError_t launch_kind(const Weight& w, const uint16_t* x, const int* x_exp, float* y, int64_t m, bool gate,
                       hipStream_t s) {
#define QMM_SHAPE_CASE(I_)                                                                                    \
    case I_:                                                                                                  \
        if constexpr (kBuilt<kFmt, kX2, I_>)                                                                  \
            return launch_shape<kFmt, kForm[I_][0], kForm[I_][1], kForm[I_][2], kForm[I_][3], kX2>(           \
                w, x, x_exp, y, m, gate, s);                                                                  \
        break;
    switch (choose_gemm_shape(w.type, w.n_tiles, w.k, m, shape_occupancy<kFmt, kX2>(), kX2)) {
        QMM_SHAPE_CASE(0)
        QMM_SHAPE_CASE(1)
        QMM_SHAPE_CASE(2)
        QMM_SHAPE_CASE(3)
        QMM_SHAPE_CASE(4)
        QMM_SHAPE_CASE(5)
        QMM_SHAPE_CASE(6)
        QMM_SHAPE_CASE(7)
    default: break;
    }
#undef QMM_SHAPE_CASE
    return hipErrorInvalidValue;
}

template <bool kX2>
hipError_t launch_type(const Weight& w, const uint16_t* x, const int* x_exp, float* y, int64_t m, bool gate,
                       hipStream_t s) {
    switch (w.type) {
    case OPENMINI_QMM_Q4_0: return launch_kind<OPENMINI_QMM_Q4_0, kX2>(w, x, x_exp, y, m, gate, s);
    case OPENMINI_QMM_Q8_0: return launch_kind<OPENMINI_QMM_Q8_0, kX2>(w, x, x_exp, y, m, gate, s);
    case OPENMINI_QMM_Q4_K: return launch_kind<OPENMINI_QMM_Q4_K, kX2>(w, x, x_exp, y, m, gate, s);
    case OPENMINI_QMM_Q6_K: return launch_kind<OPENMINI_QMM_Q6_K, kX2>(w, x, x_exp, y, m, gate, s);
    default: return hipErrorInvalidValue;
    }
}

// fp32 activations for the fp16 MFMA: row m of x [m, k] is scaled by 2^e, e chosen so
// the row's largest |x| lands in [2^14, 2^15), and each element x' = x 2^e is split
// into hi = x' rounded toward zero to fp16 (11 significant bits) and lo = x' - hi
// (exact in fp32, at most 13 bits, |lo| < 2^-10 |x'|) rounded to nearest fp16: the
// pair carries x' to within 2^-22 |x'|, and to within 2^-25 absolute (2^-39 of the
// row maximum) for elements more than 2^17 below it, where lo is an fp16 subnormal.
// e goes to x_exp[m].  A row holding inf or NaN is written as NaN (hi) and 0 (lo) with
// e = 0, so every output of that row is NaN (the decode GEMVs do the same).
//
// Written in the order the GEMM's fragments take it, so that its copies are contiguous:
// per 16-row tile (the last one of r <= 16 rows) and 32-element block, r x 4 pieces of 8
// hi values, piece kq * r + i = elements 8 kq .. 8 kq + 7 of row i, then the lo values
// the same way.  With `nib` a piece holds its elements in the order (0, 2, 1, 3, 4, 6, 5,
// 7), which makes the nibble codes three operations cheaper to build (codes_q4_perm).
// One workgroup per row, which it reads once into registers (K <= 16384; the rest twice).
// Rows go to workgroups so that a tile's 16 rows, which share cache lines of x2, run on
// one XCD (workgroups are dealt out to the 8 XCDs in turn).  x rows 16-byte aligned
// (k % 32 == 0).
constexpr int kSplitThreads = 512;
constexpr int kSplitHeld = 4;  // pieces of 8 elements a thread holds
__global__ __launch_bounds__(kSplitThreads) void split_rows_kernel(const float* __restrict__ x,
                                                                   uint16_t* __restrict__ x2,
                                                                   int* __restrict__ x_exp, int m, int k, int nib) {
    __shared__ uint32_t wave_max[kSplitThreads / 64];
    const int tile = (int)(blockIdx.x >> 7) * 8 + (int)(blockIdx.x & 7), ri = (int)(blockIdx.x >> 3) & 15;
    const int row = tile * 16 + ri;
    if (row >= m) return;  // uniform
    const float4* xr = reinterpret_cast<const float4*>(x + (size_t)row * k);
    const int pieces = k / 8;
    float4 h[kSplitHeld][2];
    auto load = [&](int p, float4* v) {
        v[0] = xr[2 * p];
        v[1] = xr[2 * p + 1];
    };
    uint32_t mx = 0;  // largest |x| as bits (inf / NaN above every finite value)
    auto fold = [&](const float4* v) {
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            mx = max(max(mx, __float_as_uint(v[q].x) & 0x7FFFFFFFu), __float_as_uint(v[q].y) & 0x7FFFFFFFu);
            mx = max(max(mx, __float_as_uint(v[q].z) & 0x7FFFFFFFu), __float_as_uint(v[q].w) & 0x7FFFFFFFu);
        }
    };
#pragma unroll
    for (int c = 0; c < kSplitHeld; ++c) {
        const int p = (int)threadIdx.x + c * kSplitThreads;
        h[c][0] = h[c][1] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (p < pieces) load(p, h[c]);
    }
#pragma unroll
    for (int c = 0; c < kSplitHeld; ++c) fold(h[c]);
    for (int p = (int)threadIdx.x + kSplitHeld * kSplitThreads; p < pieces; p += kSplitThreads) {
        float4 v[2];
        load(p, v);
        fold(v);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) mx = max(mx, (uint32_t)__shfl_xor((int)mx, o));
    if ((threadIdx.x & 63) == 0) wave_max[threadIdx.x >> 6] = mx;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < kSplitThreads / 64; ++w) mx = max(mx, wave_max[w]);
    const bool bad = mx >= 0x7F800000u;
    // max |x| in [2^(f - 1), 2^f): e = 15 - f puts it in [2^14, 2^15)
    const int e = (bad || mx == 0) ? 0 : 15 - __builtin_amdgcn_frexp_expf(__uint_as_float(mx));
    const int rows = min(16, m - tile * 16);
    uint4* out = reinterpret_cast<uint4*>(x2 + (size_t)tile * 32 * k);  // 16-byte pieces
    auto put = [&](int p, const float4* q) {
        float v[8] = {q[0].x, q[0].y, q[0].z, q[0].w, q[1].x, q[1].y, q[1].z, q[1].w};
        if (nib) {
            v[1] = q[0].z; v[2] = q[0].y;
            v[5] = q[1].z; v[6] = q[1].y;
        }
        uint32_t hi[4], lo[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float a = __builtin_amdgcn_ldexpf(v[2 * i], e), b = __builtin_amdgcn_ldexpf(v[2 * i + 1], e);
            const auto t = __builtin_amdgcn_cvt_pkrtz(a, b);
            const f16x2 l = {(_Float16)(a - (float)t[0]), (_Float16)(b - (float)t[1])};
            hi[i] = bad ? 0x7E007E00u : __builtin_bit_cast(uint32_t, t);  // fp16 NaN
            lo[i] = bad ? 0u : __builtin_bit_cast(uint32_t, l);
        }
        uint4* at = out + (size_t)(p >> 2) * 8 * rows + (p & 3) * rows + ri;
        at[0] = make_uint4(hi[0], hi[1], hi[2], hi[3]);
        at[4 * rows] = make_uint4(lo[0], lo[1], lo[2], lo[3]);
    };
#pragma unroll
    for (int c = 0; c < kSplitHeld; ++c) {
        const int p = (int)threadIdx.x + c * kSplitThreads;
        if (p < pieces) put(p, h[c]);
    }
    for (int p = (int)threadIdx.x + kSplitHeld * kSplitThreads; p < pieces; p += kSplitThreads) {
        float4 v[2];
        load(p, v);
        put(p, v);
    }
    if (threadIdx.x == 0) x_exp[row] = e;
}

// Compute-only ceiling of the prefill GEMM (Q4_0 / Q8_0): gemm_kernel's grid and
// waves, each running only its per-block register work -- kCeilWT code conversions,
// kMI x kCeilWT MFMAs and their rescale FMAs, in the same order -- for as many blocks as
// its K part holds, on operands that stay in registers.  No loads, LDS, barriers or
// stores (a sentinel store keeps the work live), so its time is what the GEMM's
// instruction mix alone costs under the same clock and power conditions.
template <int kFmt, int kMI>
__global__ __launch_bounds__(512) void gemm_ceiling_kernel(int blocks, float* __restrict__ sink) {
    constexpr bool kNib = kFmt == OPENMINI_QMM_Q4_0;
    const int lane = threadIdx.x & 63;
    bf16x8 a[kMI];
#pragma unroll
    for (int i = 0; i < kMI; ++i)
#pragma unroll
        for (int e = 0; e < 8; ++e) a[i][e] = (__bf16)((float)((lane + 7 * i + e) & 15) * 0.125f);
    uint32_t c0[kCeilWT], c1[kCeilWT], sc[kCeilWT];
#pragma unroll
    for (int j = 0; j < kCeilWT; ++j) {
        c0[j] = 0x01030507u * (uint32_t)(lane + j + 1);
        c1[j] = 0x02040608u * (uint32_t)(lane + j + 1);
        sc[j] = 0x3C00u;  // fp16 1.0
    }
    f32x4 acc[kMI][kCeilWT];
#pragma unroll
    for (int i = 0; i < kMI; ++i)
#pragma unroll
        for (int j = 0; j < kCeilWT; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int b = 0; b < blocks; ++b) {
        // new operands every block, as the A-fragment reads and weight loads give
#pragma unroll
        for (int i = 0; i < kMI; ++i) asm volatile("" : "+v"(a[i]));
#pragma unroll
        for (int j = 0; j < kCeilWT; ++j) asm volatile("" : "+v"(c0[j]), "+v"(c1[j]), "+v"(sc[j]));
        bf16x8 bq[kCeilWT];
        float d[kCeilWT];
#pragma unroll
        for (int j = 0; j < kCeilWT; ++j) {
            if constexpr (kNib) {
                bq[j] = cvt_q4(c0[j]);
                d[j] = f16_bits_to_f32((uint16_t)sc[j]) * 16.0f;
            } else {
                bq[j] = cvt_q8(c0[j], c1[j]);
                d[j] = f16_bits_to_f32((uint16_t)sc[j]);
            }
        }
        f32x4 pp[2];
        pp[0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[0], bq[0], f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
        for (int q = 0; q < kMI * kCeilWT; ++q) {
            if (q + 1 < kMI * kCeilWT)
                pp[(q + 1) & 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                    a[(q + 1) / kCeilWT], bq[(q + 1) % kCeilWT], f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
            for (int r = 0; r < 4; ++r)
                acc[q / kCeilWT][q % kCeilWT][r] = fmaf(pp[q & 1][r], d[q % kCeilWT], acc[q / kCeilWT][q % kCeilWT][r]);
        }
    }
    float t = 0.0f;
#pragma unroll
    for (int i = 0; i < kMI; ++i)
#pragma unroll
        for (int j = 0; j < kCeilWT; ++j) t += acc[i][j][0] + acc[i][j][1] + acc[i][j][2] + acc[i][j][3];
    if (t == 1234.5f) sink[0] = t;
}

template <int kFmt>
hipError_t launch_ceiling(int64_t m, int64_t n_tiles, int64_t k, float* sink, hipStream_t s) {
    // the grid, workgroup and K split of the launch shapes 128 x 192 and (few rows) 64 x 96
    const bool small = m <= kBMMax;
    const int bm = small ? 64 : 128, threads = 512, parts = small ? 4 : 2;
    const int64_t bt = (small ? 2 : 4) * kCeilWT;  // weight tiles per workgroup (column slices)
    const dim3 grid((unsigned)((n_tiles + bt - 1) / bt), (unsigned)((m + bm - 1) / bm));
    const int blocks = (int)((k / kQK + parts - 1) / parts);
    if (small)
        hipLaunchKernelGGL((gemm_ceiling_kernel<kFmt, 4>), grid, dim3(threads), 0, s, blocks, sink);
    else
        hipLaunchKernelGGL((gemm_ceiling_kernel<kFmt, 8>), grid, dim3(threads), 0, s, blocks, sink);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_gemm_ceiling(int type, int64_t m, int64_t n, int64_t k, float* sink, hipStream_t s) {
    const int64_t n_tiles = (n + kTileRows - 1) / kTileRows;
    if (m <= 0 || n <= 0 || k <= 0 || (m + 127) / 128 > 65535 || n_tiles > INT32_MAX) return hipErrorInvalidValue;
    if (type == OPENMINI_QMM_Q4_0) return launch_ceiling<OPENMINI_QMM_Q4_0>(m, n_tiles, k, sink, s);
    if (type == OPENMINI_QMM_Q8_0) return launch_ceiling<OPENMINI_QMM_Q8_0>(m, n_tiles, k, sink, s);
    return hipErrorInvalidValue;
}

// Rows of one launch: x offsets are 32-bit, so x stays below 2 GiB (row_bytes per row), and
// the grid's y dimension counts at most 65535 tiles of 64 rows.
static int64_t rows_of_launch(int64_t row_bytes) {
    const int64_t rows = (((int64_t)1 << 31) - 1) / row_bytes, grid = (int64_t)65535 * 64;
    return (rows < grid ? rows : grid) / kBMMax * kBMMax;
}

hipError_t launch_gemm_bf16(const Weight& w, const uint16_t* x, float* y, int64_t m, hipStream_t s,
                            bool gate_in_y) {
    const int64_t rows_per_launch = rows_of_launch(w.k * 2);
    if (rows_per_launch <= 0) return hipErrorInvalidValue;  // one row tile of x exceeds 2 GiB
    for (int64_t m_off = 0; m_off < m; m_off += rows_per_launch) {
        const int64_t mm = m - m_off < rows_per_launch ? m - m_off : rows_per_launch;
        const uint16_t* xs = x + m_off * w.k;
        float* ys = y + m_off * w.n;
        const hipError_t e = launch_type<false>(w, xs, nullptr, ys, mm, gate_in_y, s);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

int gemm_shape(const Weight& w, int64_t m, bool split_x) {
    auto pick = [&](auto fmt) {
        constexpr int kFmt = decltype(fmt)::value;
        return split_x ? choose_gemm_shape(kFmt, w.n_tiles, w.k, m, shape_occupancy<kFmt, true>(), true)
                       : choose_gemm_shape(kFmt, w.n_tiles, w.k, m, shape_occupancy<kFmt, false>(), false);
    };
    switch (w.type) {
    case OPENMINI_QMM_Q4_0: return pick(std::integral_constant<int, OPENMINI_QMM_Q4_0>{});
    case OPENMINI_QMM_Q8_0: return pick(std::integral_constant<int, OPENMINI_QMM_Q8_0>{});
    case OPENMINI_QMM_Q4_K: return pick(std::integral_constant<int, OPENMINI_QMM_Q4_K>{});
    case OPENMINI_QMM_Q6_K: return pick(std::integral_constant<int, OPENMINI_QMM_Q6_K>{});
    default: return -1;
    }
}

size_t gemm_f32_workspace_bytes(int64_t m, int64_t k) {
    return (((size_t)m * (size_t)k * 4 + 255) & ~(size_t)255) + (size_t)m * 4;
}

hipError_t split_rows(const Weight& w, const float* x, int64_t m, void* work, hipStream_t s) {
    const int64_t k = w.k;
    if (m <= 0 || m > INT32_MAX || k <= 0 || k % kQK != 0 || k > INT32_MAX / 2) return hipErrorInvalidValue;
    uint16_t* x2 = static_cast<uint16_t*>(work);
    int* x_exp = reinterpret_cast<int*>(static_cast<uint8_t*>(work) + (gemm_f32_workspace_bytes(m, k) - (size_t)m * 4));
    const int nib = w.type == OPENMINI_QMM_Q4_0 || w.type == OPENMINI_QMM_Q4_K;
    const int64_t tiles = (m + 15) / 16;
    hipLaunchKernelGGL(split_rows_kernel, dim3((unsigned)((tiles + 7) / 8 * 128)), dim3(kSplitThreads), 0, s, x, x2, x_exp,
                       (int)m, (int)k, nib);
    return hipGetLastError();
}

hipError_t launch_gemm_split(const Weight& w, const void* work, int64_t m, float* y, hipStream_t s, bool gate_in_y) {
    const uint16_t* x2 = static_cast<const uint16_t*>(work);
    const int* x_exp =
        reinterpret_cast<const int*>(static_cast<const uint8_t*>(work) + (gemm_f32_workspace_bytes(m, w.k) - (size_t)m * 4));
    const int64_t kx = 2 * w.k;  // fp16 elements per split row
    const int64_t rows_per_launch = rows_of_launch(kx * 2);
    if (rows_per_launch <= 0) return hipErrorInvalidValue;
    for (int64_t m_off = 0; m_off < m; m_off += rows_per_launch) {
        const int64_t mm = m - m_off < rows_per_launch ? m - m_off : rows_per_launch;
        const uint16_t* xs = x2 + m_off * kx;
        const int* es = x_exp + m_off;
        float* ys = y + m_off * w.n;
        const hipError_t e = launch_type<true>(w, xs, es, ys, mm, gate_in_y, s);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace qmm
