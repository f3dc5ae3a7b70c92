// gemm_tiles.hip -- LDS-tiled matrix-core GEMM over GGUF blocks:
// Y[m, n] = X[m, k] . W[n, k]^T for many activation rows, weights read in
// their GGUF block layout (matmul_f32_q4, quantize.rs:265-320).
//
// Numerics.  Each x row (of a row of wide range each block, see WIDE_ROW) is
// scaled by a power of two (its largest into [2^14, 2^15)) and split into x_hi =
// f16(x') and x_lo = f16(x' - x_hi), about 22 significant bits; the weight
// operand is the exact integer code in f16, one 16x16x32 MFMA K step is one
// 32-element block, and the block scale d multiplies the block's f32 dot
// afterwards: acc += d (x_hi.q + x_lo.q).
//
// Operands.  x is the A operand and W the B operand of
// v_mfma_f32_16x16x32_f16: lane l = 16 g + r holds x row r and weight column
// r, eight elements each, and the results of x rows 4 g .. 4 g + 3 with
// weight row r -- so one block scale serves a lane's four results.  The K
// order inside a block is free as long as both operands agree; lane group g
// takes elements {4g, 4g+2, 16+4g, 18+4g, 4g+1, 4g+3, 17+4g, 19+4g}, the
// order in which the low and high nibbles of bytes 4g .. 4g+3 of a Q4_0
// block fall out of two masks and one shift (v_and_or_b32 with the f16 magic
// 0x6400).  The x prep writes every block in that order.
//
// What bounds it.  Per 64 x 128 x 32 step a wave issues 64 MFMAs (1,024
// cycles of a SIMD's matrix core) and about 200 VALU instructions, 128 of
// them the scale FMAs; LDS moves 17.5 KB, a quarter of its rate.  Weights go
// through LDS as nibbles (16 bytes a block) and become f16 operands in the
// registers of the one wave column that uses them, so LDS holds three chunks
// of x and W and the loads run one and two chunks ahead of the matrix cores.
// Counters at 2048 x 14336 x 4096 / 4096 x 14336: matrix cores busy 54 / 57 %,
// VALU issue 58 / 59 %, bank conflicts 8 % of LDS cycles, clock 2.0 GHz.  2048
// rows, 14336 x 4096 / 4096 x 14336: 631 / 615 -> 480 / 455 us (501 / 528
// TFLOP/s; the matrix cores do twice that, x being two operands); 512 rows
// 14336 x 4096: 213 -> 127 us; 128 rows 4096 x 4096 / 14336 x 4096 / 4096 x
// 14336: 30.7 / 73 / 84 -> 25.6 / 44 / 49 us (split over K, below).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <type_traits>

#include "rdl_device.hpp"
#include "rdl_internal.hpp"

namespace rdl {

namespace {

// One product: tile shape cfg, the first `full` tiles whole, the others in S
// slices of kbs blocks.
struct TilePlan {
    int cfg, full, S, kbs;
};

typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));  // x and y start on any float

// ---- x preparation ---------------------------------------------------------
// |x| bits of a finite x, else 0.
__device__ __forceinline__ uint32_t finite_bits(float x) {
    const uint32_t b = abs_bits(x);
    return b < 0x7F800000u ? b : 0u;
}
// The row exponent e (amax 2^-e in [2^14, 2^15); 0 for a row of zeros) from
// each thread's maximum of its finite |x| bits; lo (if not NULL): each thread's
// smallest nonzero block maximum in, the row's out (~0: none).
template <int NT>
__device__ __forceinline__ int split_exponent(uint32_t am, uint32_t* red, uint32_t* lo = nullptr) {
    am = max8_u32(am);
    am = max(am, (uint32_t)dpp_i32<DPP_ROW_MIRROR>((int)am));
    am = max(am, (uint32_t)__shfl_xor((int)am, 16));
    am = max(am, (uint32_t)__shfl_xor((int)am, 32));
    uint32_t mn = ~0u;
    if (lo) {
        mn = min(*lo, (uint32_t)dpp_i32<DPP_ROW_MIRROR>((int)*lo));  // (alike in a block's eight threads)
        mn = min(mn, (uint32_t)__shfl_xor((int)mn, 16));
        mn = min(mn, (uint32_t)__shfl_xor((int)mn, 32));
    }
    if ((threadIdx.x & 63) == 0) {
        red[threadIdx.x >> 6] = am;
        if (lo) red[NT / 64 + (threadIdx.x >> 6)] = mn;
    }
    __syncthreads();
    am = red[0];
#pragma unroll
    for (int w = 1; w < NT / 64; w++) am = max(am, red[w]);
    if (lo) {
        mn = red[NT / 64];
#pragma unroll
        for (int w = 1; w < NT / 64; w++) mn = min(mn, red[NT / 64 + w]);
        *lo = mn;
    }
    return am != 0 ? ilogbf(__builtin_bit_cast(float, am)) - 14 : 0;
}

// The low half of a block's sum is stored times 2^12 (at most 8 before): its own
// last place, 2^-24, would be that of single elements, and 10 times their error in a
// block far below its row's largest.
constexpr float SUM_LO = 4096.0f;

// The split of elements 4 p .. 4 p + 3 of a row (p = t modulo 8).  Thread c = t %
// 8 of a block's eight holds elements 4c .. 4c+3.  Threads c and c ^ 4 trade
// halves: c < 4 ends with the block's x_hi piece g = c (elements of 4c and 16 +
// 4c in K order), c >= 4 with the x_lo piece c - 4.  Every thread of a group of
// eight takes part; p >= k4 stores nothing.
__device__ __forceinline__ void split_piece(const f32x4& v, int e, int p, int k4, _Float16* xh, _Float16* xl,
                                            uint32_t* xs) {
    const bool upper = (threadIdx.x & 4) != 0;
    _Float16 h[4], l[4];
    float bs = 0.0f;
#pragma unroll
    for (int t = 0; t < 4; t++) {
        const float s = ldexpf(v[t], -e);
        h[t] = (_Float16)s;
        l[t] = (_Float16)(fabsf(s) == INFINITY ? 0.0f : s - (float)h[t]);  // (an infinite x: no inf - inf)
        bs += s;
    }
    const uint32_t h02 = __builtin_bit_cast(uint32_t, half2_t{h[0], h[2]});
    const uint32_t h13 = __builtin_bit_cast(uint32_t, half2_t{h[1], h[3]});
    const uint32_t l02 = __builtin_bit_cast(uint32_t, half2_t{l[0], l[2]});
    const uint32_t l13 = __builtin_bit_cast(uint32_t, half2_t{l[1], l[3]});
    const uint32_t r0 = (uint32_t)__shfl_xor((int)(upper ? h02 : l02), 4);
    const uint32_t r1 = (uint32_t)__shfl_xor((int)(upper ? h13 : l13), 4);
    const u32x4 o = upper ? u32x4{r0, l02, r1, l13} : u32x4{h02, r0, h13, r1};
    if (p < k4) *reinterpret_cast<u32x4*>((upper ? xl : xh) + (size_t)(p >> 3) * 32 + (p & 3) * 8) = o;
    if (xs) {  // the block's sum of x', over 32, as an f16 hi / lo pair, lo times SUM_LO
        bs = sum8_f32(bs) * 0.03125f;
        const _Float16 sh = (_Float16)bs;
        const half2_t sp = {sh, (_Float16)((bs - (float)sh) * SUM_LO)};
        if ((threadIdx.x & 7) == 0 && p < k4) xs[p >> 3] = __builtin_bit_cast(uint32_t, sp);
    }
}

// Q4_0 rows of wide range.  x_lo's last place is 2^-24 of x', so a row with a
// block more than 2^-WB below its largest would lose bits of that block, which
// counts for all of a result where the larger blocks meet zero weights.  Where
// x is held with a scale a block otherwise (the x-tile kernel's rows, WB = 14: such
// a block keeps its 22 bits; Q8_0 values, WB = 20: they stay exact), such a row has a
// scale 2^e for every block instead: XE = WIDE_ROW and XB[block][row] = 2^e.  A
// byte a row says which are (XF, zeros up to a multiple of XF_PAD rows).
constexpr int XF_PAD = 128;
constexpr int WIDE_ROW = INT_MIN;
constexpr int WIDE_FLOAT = 14, WIDE_NATIVE = 20;

// One workgroup a row: thread t holds elements 4 (t + j NT) .. +3 (k <= 4 NV
// NT), so x is read once.  PRO 1: RMSNorm first; PRO 2: SwiGLU of rows of 2k
// interleaved (gate_j, up_j) values; PRO 3: x as its Q8_0 blocks hold it
// (quantize_row_q8_0, quantize.rs:164-193).
template <int PRO, int NT, int NV, int WB>
__global__ __launch_bounds__(NT) void gemm_split_kernel(const float* __restrict__ X, int k,
                                                        const float* __restrict__ g, float eps,
                                                        _Float16* __restrict__ XH, _Float16* __restrict__ XL,
                                                        int* __restrict__ XE, uint32_t* __restrict__ XS,
                                                        float* __restrict__ XB, int xb_rows, uint8_t* __restrict__ XF) {
    __shared__ uint32_t red[(WB ? 2 : 1) * NT / 64];
    __shared__ float red2[NT / 64];
    const int row = blockIdx.x;
    const int k4 = k >> 2;  // k % 32 == 0
    f32x4 v[NV];
    if constexpr (PRO == 2) {
        const f32x4u* x = reinterpret_cast<const f32x4u*>(X + (size_t)row * 2 * k);
        auto silu_mul = [](float gv, float uv) {
            const float sig = 1.0f / (1.0f + expf(-gv));
            return (gv * sig) * uv;
        };
#pragma unroll
        for (int j = 0; j < NV; j++) {
            const int p = threadIdx.x + j * NT;
            if (p < k4) {
                const f32x4 a = x[2 * p], b = x[2 * p + 1];
                v[j] = f32x4{silu_mul(a[0], a[1]), silu_mul(a[2], a[3]), silu_mul(b[0], b[1]), silu_mul(b[2], b[3])};
            } else {
                v[j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            }
        }
    } else {
        const f32x4u* x = reinterpret_cast<const f32x4u*>(X + (size_t)row * k);
#pragma unroll
        for (int j = 0; j < NV; j++) {
            const int p = threadIdx.x + j * NT;
            v[j] = p < k4 ? (f32x4)x[p] : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        }
    }
    if constexpr (PRO == 3) {
        // code times scale, 7 + 11 bits: exact in f32 and, by the row's or the block's
        // exponent, in the hi / lo pair; a NaN scores as 0 in the block maximum and
        // as code 0, an overflowing scale makes the block NaN
#pragma unroll
        for (int j = 0; j < NV; j++) {
            float am = 0.0f;
#pragma unroll
            for (int t = 0; t < 4; t++) am = fmaxf(am, fabsf(v[j][t]));
            am = max8_f32(am);
            const float rt = h2f(f2h_rne(am == 0.0f ? 0.0f : am / 127.0f));
            const float inv = rt == 0.0f ? 0.0f : 1.0f / rt;
#pragma unroll
            for (int t = 0; t < 4; t++) {
                const float q = roundf(v[j][t] * inv);
                v[j][t] = (q != q ? 0.0f : fminf(fmaxf(q, -128.0f), 127.0f)) * rt;
            }
        }
    }
    if constexpr (PRO == 1) {
        float ss = 0.0f;
#pragma unroll
        for (int j = 0; j < NV; j++)
            ss += (v[j][0] * v[j][0] + v[j][1] * v[j][1]) + (v[j][2] * v[j][2] + v[j][3] * v[j][3]);
        ss = sum8_f32(ss);
        ss += dpp_f32<DPP_ROW_MIRROR>(ss);
        ss += __shfl_xor(ss, 16);
        ss += __shfl_xor(ss, 32);
        if ((threadIdx.x & 63) == 0) red2[threadIdx.x >> 6] = ss;
        __syncthreads();
        ss = red2[0];
#pragma unroll
        for (int w = 1; w < NT / 64; w++) ss += red2[w];
        const float inv = 1.0f / sqrtf(ss / (float)k + eps);
        const f32x4* g4 = reinterpret_cast<const f32x4*>(g);
#pragma unroll
        for (int j = 0; j < NV; j++) {
            const int p = threadIdx.x + j * NT;
            if (p < k4) v[j] = (v[j] * inv) * g4[p];
        }
    }
    // largest finite |x| of the row as an integer maximum of |x| bits
    uint32_t am = 0, bm[WB ? NV : 1];
#pragma unroll
    for (int j = 0; j < NV; j++) {
        uint32_t a = 0;
#pragma unroll
        for (int t = 0; t < 4; t++) a = max(a, finite_bits(v[j][t]));
        if (WB) bm[j] = a = max8_u32(a);  // the block's
        am = max(am, a);
    }
    uint32_t lo = ~0u;
    if constexpr (WB != 0)
#pragma unroll
        for (int j = 0; j < NV; j++) lo = min(lo, bm[j] - 1u);  // (a block of zeros: ~0)
    const int e = split_exponent<NT>(am, red, WB ? &lo : nullptr);
    const bool wide = WB && lo != ~0u && ilogbf(__builtin_bit_cast(float, lo + 1u)) < e + 14 - WB;
    if (threadIdx.x == 0) XE[row] = wide ? WIDE_ROW : e;
    if constexpr (WB != 0) {
        if (threadIdx.x == 0) XF[row] = wide;
        const int pad = row + 1 + (int)threadIdx.x;
        if (row + 1 == (int)gridDim.x && pad < ((int)gridDim.x + XF_PAD - 1) / XF_PAD * XF_PAD) XF[pad] = 0;
    }
#pragma unroll
    for (int j = 0; j < NV; j++) {
        const int p = threadIdx.x + j * NT;
        int eb = e;
        if (WB && wide) {
            eb = bm[j] != 0 ? ilogbf(__builtin_bit_cast(float, bm[j])) - 14 : 0;
            if ((p & 7) == 0 && p < k4) XB[(size_t)(p >> 3) * xb_rows + row] = ldexpf(1.0f, eb);
        }
        split_piece(v[j], eb, p, k4, XH + (size_t)row * k, XL + (size_t)row * k,
                    XS ? XS + (size_t)row * (k >> 5) : nullptr);
    }
}

// The split of rows longer than a workgroup's registers hold: two reads of x.
__global__ __launch_bounds__(1024) void gemm_split_long_kernel(const float* __restrict__ X, int k,
                                                               _Float16* __restrict__ XH, _Float16* __restrict__ XL,
                                                               int* __restrict__ XE) {
    __shared__ uint32_t red[1024 / 64];
    const int row = blockIdx.x, k4 = k >> 2;
    const f32x4u* x = reinterpret_cast<const f32x4u*>(X + (size_t)row * k);
    uint32_t am = 0;
    for (int p = threadIdx.x; p < k4; p += 1024) {
        const f32x4 v = (f32x4)x[p];
#pragma unroll
        for (int t = 0; t < 4; t++) am = max(am, finite_bits(v[t]));
    }
    const int e = split_exponent<1024>(am, red);
    if (threadIdx.x == 0) XE[row] = e;
    for (int p = threadIdx.x; p - (int)threadIdx.x < k4; p += 1024)
        split_piece(p < k4 ? (f32x4)x[p] : f32x4{0.0f, 0.0f, 0.0f, 0.0f}, e, p, k4, XH + (size_t)row * k,
                    XL + (size_t)row * k, nullptr);
}

// ---- GEMM --------------------------------------------------------------------
// Cache policy bits of buffer loads / stores (gfx950): nt (no stale L1 line),
// sc1 (device scope).
constexpr int CPOL_NT = 2, CPOL_SC1 = 16;

// Weight formats: Q4_0 (d (q - 8)) and Q8_0 (d q, tensor.rs:535-639), whose
// blocks have f16 scales of their own; Q4_K ((d sc) q - dmin mn, parser.rs:
// 549-593) and Q6_K ((d sc) (q - 32), parser.rs:510-547), whose 256-element
// super-blocks have one f16 scale over small integer ones.  There the integer
// scale goes into the operand and the MFMAs of a super-block chain in their
// accumulators, T: acc += d T once a super-block instead of one FMA an output
// a block.
//  * Q4_K: (q - 8) sc is exact in f16.  What remains, e_j = 8 d sc_j - dmin
//    mn_j times S_j, the sum of x' over sub-block j, is one more MFMA a
//    super-block: eight sub-blocks times the four products of the f16 hi / lo
//    pairs of e_j 2^-t (t by the larger of the row's 8 d and dmin) and of S_j / 32
//    (lo times SUM_LO, against e_j / SUM_LO, which is staged too: multiplied as it
//    is read it cost the loop 7 %).  e_j keeps its 22 bits down to 2^-17 of the
//    super-block's largest, S_j always.
//    (e_j first, in f32: d q sc and dmin mn nearly cancel, and summing them
//    apart doubled the error against 64 bits.)
//  * Q6_K: (q - 32) sc has up to 13 bits: hi = f16(.) and the exact rest lo (at
//    most 1 in 4096), T += x_hi hi + x_lo hi + x_hi lo (x_lo lo < 2^-23 of a
//    product, below x's own split).
constexpr int WF_Q4_0 = 0, WF_Q8_0 = 1, WF_Q4_K = 2, WF_Q6_K = 3;

template <int WF, int FI, int WJ, int KS, bool WIDE>
struct TileCfg {
    static constexpr int FJ = 4;                 // weight rows of a wave: 64, four a lane
    static constexpr int NW = WJ * KS, NT = NW * 64;
    static constexpr int TJ = WJ * 64, TI = FI * 16;
    static constexpr int CB = KS;                // blocks a chunk: one a K group of waves
    // one block's codes: [wj][g][64 rows] dwords of nibbles, or (Q8_0) that twice,
    // bytes 4g .. 4g+3 and 16+4g .. 16+4g+3
    static constexpr bool BYTES = WF == WF_Q8_0 || WF == WF_Q6_K;
    static constexpr bool CHAIN = WF == WF_Q4_K || WF == WF_Q6_K;
    static_assert(WF != WF_Q6_K || KS == 4, "Q6_K chunks are half super-blocks");
    static constexpr int HALF = WJ * 1024;
    static constexpr int NIB_BLOCK = (BYTES ? 2 : 1) * HALF;
    static constexpr int W_BYTES = CB * NIB_BLOCK;
    // f16 d (Q4_K: sc; Q6_K: the pair of its two 16-element scales): [block][row]
    static constexpr int D_BYTES = CB * TJ * (WF == WF_Q6_K ? 4 : 2);
    static constexpr int X_PART = 1024;          // one 16-row tile of one block, hi or lo
    static constexpr int X_BYTES = CB * (TI / 16) * 2 * X_PART;
    // WIDE: the scale of each (block, x row), and as much where threads without one store
    static constexpr int F_AT = W_BYTES + D_BYTES + X_BYTES, F_BYTES = WIDE ? NT * 4 : 0;
    static_assert(!WIDE || TI * CB <= NT, "a scale a thread");
    static constexpr int STAGE = F_AT + F_BYTES;
    static constexpr int WWORDS = WF == WF_Q6_K ? 11 : WF == WF_Q4_K ? 8 : BYTES ? 9 : 5;  // dwords a unit's loads bring
    static constexpr int WU = (TJ * CB + NT - 1) / NT;      // weight blocks a thread stages
    static constexpr int XU = (TI * CB * 4 + NT - 1) / NT;  // 16-byte pieces a thread stages, hi and lo each
    static constexpr int RED = (KS - 1) * WJ * FI * FJ * 1024;
    // a super-block's own data (CHAIN): d (and Q4_K's t) of each row, Q4_K's e
    // [row][hi, hi / SUM_LO, lo, lo / SUM_LO][8] f16 and x sums [tile][hi / lo][16 rows][8] f16
    static constexpr int SU = WF == WF_Q4_K ? (TI * CB + NT - 1) / NT : 0;  // sum pairs a thread stages
    static constexpr int MN_AT = TJ * 4, SS_AT = MN_AT + TJ * 64;
    static constexpr int AUX = !CHAIN ? 0 : WF == WF_Q4_K ? SS_AT + TI * 32 : MN_AT;
    // three stages and three super-blocks' data, or the sums at the end; the x
    // rows' exponents behind them
    static constexpr int AUX_AT = 3 * STAGE, MAIN = 3 * STAGE + 3 * AUX;
    static constexpr int XE_AT = MAIN > RED ? MAIN : RED;
    static constexpr int DUMP_AT = XE_AT + TI * 4;  // where threads without a sum pair store
    static constexpr int LDS = DUMP_AT + (WF == WF_Q4_K ? 272 : 0);
    static constexpr bool W_ALL = TJ * CB % NT == 0;        // no idle threads in the last weight unit
    static_assert(TI * CB * 4 % NT == 0, "whole x pieces a thread");
    static_assert(CB % 2 == 0, "eight consecutive pieces of an x row");
};

// f16 (q - 8) of the eight nibbles of n (bytes 4g .. 4g+3 of a Q4_0 block) in
// the K order above: 0x6400 | q = 1024 + q and 0x6400 | 16 q = 1024 + 16 q.
// The masks come in scalar registers and the magic in a vector one (opaque to
// the compiler), so each pair is one v_and_or_b32.
struct Q4Consts { uint32_t lo, hi, magic; };
__device__ __forceinline__ Q4Consts q4_consts() {
    Q4Consts c = {0x000F000Fu, 0x00F000F0u, 0x64006400u};
    asm volatile("" : "+s"(c.lo), "+s"(c.hi), "+v"(c.magic));
    return c;
}
__device__ __forceinline__ half8_t q4_f16(uint32_t n, const Q4Consts& k) {
    const half2_t lo_off = {(_Float16)1032.0f, (_Float16)1032.0f};
    const half2_t hi_mul = {(_Float16)0.0625f, (_Float16)0.0625f};
    const half2_t hi_off = {(_Float16)-72.0f, (_Float16)-72.0f};
    const uint32_t n8 = n >> 8;
    const half2_t a = __builtin_bit_cast(half2_t, (n & k.lo) | k.magic) - lo_off;
    const half2_t b = __builtin_elementwise_fma(__builtin_bit_cast(half2_t, (n & k.hi) | k.magic), hi_mul, hi_off);
    const half2_t c = __builtin_bit_cast(half2_t, (n8 & k.lo) | k.magic) - lo_off;
    const half2_t d = __builtin_elementwise_fma(__builtin_bit_cast(half2_t, (n8 & k.hi) | k.magic), hi_mul, hi_off);
    return half8_t{a[0], a[1], b[0], b[1], c[0], c[1], d[0], d[1]};
}

// f16 q of the eight codes n0, n1 (staged as q + 128), in the K order above:
// 0x6400 | (q + 128) = 1152 + q.
__device__ __forceinline__ half8_t q8_f16(uint32_t n0, uint32_t n1) {
    const half2_t off = {(_Float16)1152.0f, (_Float16)1152.0f};
    constexpr uint32_t MAGIC = 0x64646464u;
    const half2_t a = __builtin_bit_cast(half2_t, perm(MAGIC, n0, 0x04020400u)) - off;
    const half2_t b = __builtin_bit_cast(half2_t, perm(MAGIC, n1, 0x04020400u)) - off;
    const half2_t c = __builtin_bit_cast(half2_t, perm(MAGIC, n0, 0x04030401u)) - off;
    const half2_t d = __builtin_bit_cast(half2_t, perm(MAGIC, n1, 0x04030401u)) - off;
    return half8_t{a[0], a[1], b[0], b[1], c[0], c[1], d[0], d[1]};
}

// f16 (q - 8) sc of eight Q4_K nibbles (bytes 4g .. in n0, 16+4g .. in n1;
// mask picks the low or the high ones, whose 0x6400 | 16 q takes mul 1 / 16, off
// -72 to q - 8 where the low ones take 1 and -1032); exact.
__device__ __forceinline__ half8_t q4k_f16(uint32_t n0, uint32_t n1, uint32_t mask, uint32_t magic, half2_t mul,
                                           half2_t off, _Float16 sc) {
    const half2_t s2 = {sc, sc};
    const half2_t a = __builtin_elementwise_fma(__builtin_bit_cast(half2_t, (n0 & mask) | magic), mul, off) * s2;
    const half2_t b = __builtin_elementwise_fma(__builtin_bit_cast(half2_t, (n1 & mask) | magic), mul, off) * s2;
    const half2_t c = __builtin_elementwise_fma(__builtin_bit_cast(half2_t, ((n0 >> 8) & mask) | magic), mul, off) * s2;
    const half2_t d = __builtin_elementwise_fma(__builtin_bit_cast(half2_t, ((n1 >> 8) & mask) | magic), mul, off) * s2;
    return half8_t{a[0], a[1], b[0], b[1], c[0], c[1], d[0], d[1]};
}
// hi and lo of (q - 32) sc for eight Q6_K codes (n0: sub-block 0, n1: 1).
__device__ __forceinline__ void q6k_f16(uint32_t n0, uint32_t n1, uint32_t scales, half8_t& hi, half8_t& lo) {
    const half2_t off = {(_Float16)1056.0f, (_Float16)1056.0f};
    const half2_t sp = __builtin_bit_cast(half2_t, scales);
    const half2_t s0 = {sp[0], sp[0]}, s1 = {sp[1], sp[1]};
    constexpr uint32_t MAGIC = 0x64646464u;
    const half2_t q0 = __builtin_bit_cast(half2_t, perm(MAGIC, n0, 0x04020400u)) - off;
    const half2_t q1 = __builtin_bit_cast(half2_t, perm(MAGIC, n1, 0x04020400u)) - off;
    const half2_t q2 = __builtin_bit_cast(half2_t, perm(MAGIC, n0, 0x04030401u)) - off;
    const half2_t q3 = __builtin_bit_cast(half2_t, perm(MAGIC, n1, 0x04030401u)) - off;
    const half2_t h0 = q0 * s0, h1 = q1 * s1, h2 = q2 * s0, h3 = q3 * s1;
    const half2_t l0 = __builtin_elementwise_fma(q0, s0, -h0), l1 = __builtin_elementwise_fma(q1, s1, -h1);
    const half2_t l2 = __builtin_elementwise_fma(q2, s0, -h2), l3 = __builtin_elementwise_fma(q3, s1, -h3);
    hi = half8_t{h0[0], h0[1], h1[0], h1[1], h2[0], h2[1], h3[0], h3[1]};
    lo = half8_t{l0[0], l0[1], l1[0], l1[1], l2[0], l2[1], l3[0], l3[1]};
}

// The launch computes rows r0 .. r1 - 1 of the product's m (r0 a multiple of
// the tile's rows): the split holds those, the tiles and their K slices are
// the whole product's, so the results do not depend on the rows of a launch.
// WIDE: x may have rows of wide range (WIDE_ROW).  A tile with one takes the
// loop with a scale a block and row, one multiplication a result more; the
// others take the plain loop (a byte a row tells, read through scalar registers:
// no barrier; 0.4 to 0.8 us a call).  us without such rows, with them, and on the
// x-tile or int8 kernel, which always scale so: 64 x 14336 x 4096 32 / 37 / 58, 16 x
// 32000 x 4096 43 / 52 / 57, native 512 x 14336 x 4096 135 / 199 / 190.
template <int WF, int FI, int WJ, int KS, bool LOCAL, bool WIDE>
__global__ __launch_bounds__(WJ * KS * 64, 2) void gemm_tile_kernel(
    const uint8_t* __restrict__ W, int n, int nb, const void* __restrict__ XH, const void* __restrict__ XL,
    const int* __restrict__ XE, int m, int r0, int r1, const uint32_t* __restrict__ XS, const float* __restrict__ XB,
    int xb_rows, const uint32_t* __restrict__ XF, float* __restrict__ Y, int accy, int full, int SR, int kbs,
    float* __restrict__ part, int* __restrict__ cnt) {
    using C = TileCfg<WF, FI, WJ, KS, WIDE>;
    constexpr int CB = C::CB, FJ = 4;
    constexpr bool BYTES = C::BYTES, Q4K = WF == WF_Q4_K, Q6K = WF == WF_Q6_K, CHAIN = C::CHAIN;
    constexpr uint32_t BB = BYTES ? 34u : 18u;  // bytes a block (not CHAIN)
    static_assert(FI == 4 || FI == 8, "x tiles of a wave");
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    const int tid = threadIdx.x, lane = tid & 63, wave = C::CHAIN ? __builtin_amdgcn_readfirstlane(tid >> 6) : tid >> 6;
    const int ks = wave % KS, wj = wave / KS;
    const int g = lane >> 4, r = lane & 15;
    // The first `full` tiles (whole rounds of workgroups, or all) are unsplit,
    // the others take SR slices of kbs blocks.  Workgroups go round-robin to the
    // 8 XCDs: each XCD takes a contiguous run of the unsplit tiles (one L2),
    // four x tiles deep before the next weight tile; a split tile's slices have
    // one b % 8 (LOCAL: one XCD, whose L2 holds their partials; full % 8 == 0).
    const int nj = (n + C::TJ - 1) / C::TJ, ni = (m + C::TI - 1) / C::TI, total = nj * ni;
    int t = blockIdx.x, slice = 0, S = 1;
    if (t < full) {
        if (full % 8 == 0) t = (t % 8) * (full / 8) + t / 8;
    } else {
        const int b = t - full;
        S = SR;
        if constexpr (LOCAL) {
            slice = (b / 8) % S;
            t = full + b / (8 * S) * 8 + b % 8;
        } else {
            slice = b % S;
            t = full + b / S;
        }
        if (t >= total) return;  // grid rounded up to whole XCD rounds (whole workgroup)
    }
    constexpr int GI = 4;
    const int band = t / (GI * nj), rem = t % (GI * nj);
    const int bh = min(GI, ni - band * GI);
    const int j0 = (rem / bh) * C::TJ, i0 = (band * GI + rem % bh) * C::TI;
    if (i0 < r0 || i0 >= r1) return;  // (whole workgroup)
    const int kb0 = slice * kbs, kb1 = S > 1 ? min(nb, kb0 + kbs) : nb;  // this slice's blocks (kb0 a multiple of CB)

    const uint32_t k = (uint32_t)nb * 32u, row_bytes = Q4K   ? (uint32_t)(nb / 8) * 144u
                                                             : Q6K ? (uint32_t)(nb / 8) * 210u
                                                                   : (uint32_t)nb * BB,
                   wbytes = (uint32_t)n * row_bytes;
    const __amdgpu_buffer_rsrc_t wrs = make_rsrc(W, wbytes);
    const __amdgpu_buffer_rsrc_t hrs = make_rsrc(XH, (uint32_t)(r1 - r0) * k * 2u);
    const __amdgpu_buffer_rsrc_t lrs = make_rsrc(XL, (uint32_t)(r1 - r0) * k * 2u);
    const int nchunks = (kb1 - kb0 + CB - 1) / CB;

    struct WRegs { uint32_t w[C::WU][C::WWORDS]; };
    struct XRegs {
        u32x4 h[C::XU], l[C::XU];
        uint32_t s[Q4K ? C::SU : 1];
        uint32_t f;
    };
    // unit u of a thread: block b0 + c CB of row j; CB is even, so a Q4_0 or Q8_0
    // block's place within its dword (2 bytes past it when j nb + b is odd) is
    // the same in every chunk.  Rows past n start out of range.
    uint32_t wbase[C::WU], wsel[C::WU];
    int wblk[C::WU];
#pragma unroll
    for (int u = 0; u < C::WU; u++) {
        const int idx = tid + u * C::NT, j = j0 + idx / CB;
        wblk[u] = idx % CB;
        const bool ok = (C::W_ALL || idx < C::TJ * CB) && j < n;
        if constexpr (CHAIN)  // the row's first super-block of the slice (kb0 % 8 == 0)
            wbase[u] = ok ? (uint32_t)j * row_bytes + (uint32_t)(kb0 / 8) * (Q4K ? 144u : 210u) : RSRC_OOB;
        else
            wbase[u] = ok ? ((uint32_t)j * row_bytes + (uint32_t)(kb0 + wblk[u]) * BB) & ~3u : RSRC_OOB;
        wsel[u] = (((uint32_t)j * (uint32_t)nb + (uint32_t)wblk[u]) & 1u) ? 0x07060504u : 0x05040302u;
    }
    // the matrix may end 2 bytes into a window's last dword: that dword is read
    // 2 bytes early and shifted when stored
    const uint32_t wlast = wbytes - 4u;
    auto load_w = [&](int c, WRegs& R) {
#pragma unroll
        for (int u = 0; u < C::WU; u++) {
            if constexpr (Q4K) {
                // sub-block b: the super-block's 16-byte header and the 16 bytes 16 (b %
                // 8) of its nibbles (half b % 2 of the run that sub-blocks b & ~1, b | 1 share)
                const uint32_t b = (uint32_t)(c * CB + wblk[u]), sb = (b >> 3) * 144u;
                const bool ok = kb0 + (int)b < kb1;
                const u32x4 h = buf_load_b128(wrs, ok ? wbase[u] + sb : RSRC_OOB);
                const u32x4 q = buf_load_b128(wrs, ok ? wbase[u] + sb + 16u + 16u * (b & 7u) : RSRC_OOB);
                R.w[u][0] = h.x, R.w[u][1] = h.y, R.w[u][2] = h.z, R.w[u][3] = h.w;
                R.w[u][4] = q.x, R.w[u][5] = q.y, R.w[u][6] = q.z, R.w[u][7] = q.w;
                continue;
            }
            if constexpr (Q6K) {
                // chunk c is half hh of a super-block; unit e takes elements 8 e .. 8 e +
                // 7 of its four groups: 8 bytes of each ql run and of qh (12-byte windows
                // from the dword below: super-blocks start on even bytes), group e's two
                // scales and d
                const uint32_t b = (uint32_t)(c * CB), hh = (b >> 2) & 1u, e = (uint32_t)wblk[u];
                const uint32_t base = wbase[u] + (b >> 3) * 210u;
                const bool ok = kb0 + (int)b < kb1 && wbase[u] != RSRC_OOB;
                const uint32_t q0 = ok ? (base + 64u * hh + 8u * e) & ~3u : RSRC_OOB;
                const uint32_t qh = ok ? (base + 128u + 32u * hh + 8u * e) & ~3u : RSRC_OOB;
                const auto v0 = __builtin_amdgcn_raw_buffer_load_b96(wrs, (int)q0, 0, 0);
                const auto v1 = __builtin_amdgcn_raw_buffer_load_b96(wrs, (int)(ok ? q0 + 32u : RSRC_OOB), 0, 0);
                const auto v2 = __builtin_amdgcn_raw_buffer_load_b96(wrs, (int)qh, 0, 0);
                R.w[u][0] = v0[0], R.w[u][1] = v0[1], R.w[u][2] = v0[2];
                R.w[u][3] = v1[0], R.w[u][4] = v1[1], R.w[u][5] = v1[2];
                R.w[u][6] = v2[0], R.w[u][7] = v2[1], R.w[u][8] = v2[2];
                R.w[u][9] = buf_load_b16(wrs, ok ? base + 192u + 8u * hh + 2u * e : RSRC_OOB);
                R.w[u][10] = buf_load_b16(wrs, ok ? base + 208u : RSRC_OOB);
                continue;
            }
            const uint32_t base = kb0 + wblk[u] + c * CB < kb1 ? wbase[u] + (uint32_t)c * (CB * BB) : RSRC_OOB;
            const u32x4 v = buf_load_b128(wrs, base);
            R.w[u][0] = v.x, R.w[u][1] = v.y, R.w[u][2] = v.z, R.w[u][3] = v.w;
            if constexpr (BYTES) {
                const u32x4 v1 = buf_load_b128(wrs, base == RSRC_OOB ? RSRC_OOB : base + 16u);
                R.w[u][4] = v1.x, R.w[u][5] = v1.y, R.w[u][6] = v1.z, R.w[u][7] = v1.w;
                R.w[u][8] = buf_load_b32(wrs, min(base + 32u, wlast));
            } else {
                R.w[u][4] = buf_load_b32(wrs, min(base + 16u, wlast));
            }
        }
    };
    int* const xe = reinterpret_cast<int*>(lds + C::XE_AT);
    if (tid < C::TI) xe[tid] = i0 + tid < r1 ? XE[i0 + tid - r0] : 0;

    uint32_t xbase[C::XU];
#pragma unroll
    for (int u = 0; u < C::XU; u++) {
        const int idx = tid + u * C::NT, i = i0 + idx / (CB * 4), q = idx % (CB * 4);
        xbase[u] = i < r1 ? ((uint32_t)(i - r0) * k + (uint32_t)kb0 * 32u + (uint32_t)q * 8u) * 2u : RSRC_OOB;
    }
    // part q of a chunk's x loads: unit q / 2, hi or lo
    auto load_x_part = [&](int c, XRegs& R, int q) {
        const int u = q >> 1, blk = ((tid + u * C::NT) % (CB * 4)) >> 2;
        const uint32_t off = kb0 + blk + c * CB < kb1 ? xbase[u] + (uint32_t)c * (CB * 64u) : RSRC_OOB;
        if (q & 1) R.l[u] = buf_load_b128(lrs, off);
        else R.h[u] = buf_load_b128(hrs, off);
    };
    const __amdgpu_buffer_rsrc_t srs = make_rsrc(Q4K ? (const void*)XS : XH, Q4K ? (uint32_t)(r1 - r0) * (uint32_t)nb * 4u : 0u);
    auto load_sums = [&](int c, XRegs& R) {
        if constexpr (Q4K) {
#pragma unroll
            for (int u = 0; u < C::SU; u++) {
                const int idx = tid + u * C::NT, i = i0 + idx / CB, b = kb0 + c * CB + idx % CB;
                R.s[u] = buf_load_b32(srs, idx < C::TI * CB && i < r1 && b < kb1
                                               ? ((uint32_t)(i - r0) * (uint32_t)nb + (uint32_t)b) * 4u
                                               : RSRC_OOB);
            }
        }
    };
    // WIDE: thread t's scale is that of block t / TI of a chunk and row t % TI
    const __amdgpu_buffer_rsrc_t brs =
        make_rsrc(WIDE ? (const void*)XB : XH, WIDE ? (uint32_t)xb_rows * (uint32_t)nb * 4u : 0u);
    uint32_t fbase = RSRC_OOB;  // (a row without scales, and until the loop that uses them)
    auto load_scale = [&](int c, XRegs& R) {  // (past the last block: out of range)
        R.f = buf_load_b32(brs, fbase + (uint32_t)c * (uint32_t)(CB * 4) * (uint32_t)xb_rows);
    };
    auto load_x = [&](int c, XRegs& R, auto w_tag) {
#pragma unroll
        for (int q = 0; q < 2 * C::XU; q++) load_x_part(c, R, q);
        load_sums(c, R);
        if constexpr (decltype(w_tag)::value) load_scale(c, R);
    };
    // aux: the super-block's own data (CHAIN)
    auto store_w = [&](int c, uint8_t* st, uint8_t* aux, const WRegs& R) {
#pragma unroll
        for (int u = 0; u < C::WU; u++) {
            const int idx = tid + u * C::NT, jl = idx / CB, bl = idx % CB;
            if (!C::W_ALL && idx >= C::TJ * CB) continue;
            if constexpr (Q4K) {
                uint32_t* dst = reinterpret_cast<uint32_t*>(st + bl * C::NIB_BLOCK + (jl >> 6) * 1024) + (jl & 63);
#pragma unroll
                for (int q = 0; q < 4; q++) dst[q * 64] = R.w[u][4 + q];
                // every dword of the header stays live to here: a load whose last one
                // is known dead (sub-blocks 0-3 do not use s[8..11]) has its register
                // reused at once, behind a wait for the load
                asm volatile("" ::"v"(R.w[u][0]), "v"(R.w[u][1]), "v"(R.w[u][2]), "v"(R.w[u][3]));
                // sub-block j's 6-bit scale and min (parser.rs:562-569)
                const uint32_t j = (uint32_t)(c * CB + bl) & 7u, sh = 8u * (j & 3u);
                const uint32_t si = R.w[u][1] >> sh, ti = R.w[u][2] >> sh, ui = R.w[u][3] >> sh;
                const uint32_t sc = j < 4 ? si & 63u : ((si >> 6) & 3u) | ((ui & 15u) << 2);
                const uint32_t mn = j < 4 ? ti & 63u : ((ti >> 6) & 3u) | ((ui >> 2) & 60u);
                reinterpret_cast<_Float16*>(st + C::W_BYTES)[bl * C::TJ + jl] = (_Float16)(float)sc;
                const float d8 = 8.0f * h2f(R.w[u][0] & 0xFFFFu), dm = h2f(R.w[u][0] >> 16);
                // t by the exponent bits of the larger that any sub-block uses: |e 2^-t| < 2^15
                const uint32_t bd = (R.w[u][1] | (R.w[u][3] & 0x0F0F0F0Fu)) != 0 ? abs_bits(d8) : 0u;
                const uint32_t bm = (R.w[u][2] | (R.w[u][3] & 0xF0F0F0F0u)) != 0 ? abs_bits(dm) : 0u;
                const int t = (int)(max(bd, bm) >> 23) - 134;
                const float e = ldexpf(d8 * (float)sc - dm * (float)mn, -t);
                const _Float16 eh = (_Float16)e;
                const _Float16 el = (_Float16)(e - (float)eh), inv = (_Float16)(1.0f / SUM_LO);
                _Float16* em = reinterpret_cast<_Float16*>(aux + C::MN_AT) + jl * 32 + j;
                em[0] = eh;
                em[8] = eh * inv;
                em[16] = el;
                em[24] = el * inv;
                reinterpret_cast<uint32_t*>(aux)[jl] = (R.w[u][0] & 0xFFFFu) | ((uint32_t)t << 16);  // d, t
                continue;
            }
            if constexpr (Q6K) {
                const uint32_t b = (uint32_t)(c * CB);
                const uint32_t sel = ((wbase[u] + (b >> 3) * 210u) & 2u) ? 0x05040302u : 0x03020100u;
                uint8_t* dst0 = st + (jl >> 6) * 1024 + (jl & 63) * 4;
#pragma unroll
                for (int i = 0; i < 2; i++) {
                    const uint32_t A = perm(R.w[u][i + 1], R.w[u][i], sel), B = perm(R.w[u][i + 4], R.w[u][i + 3], sel);
                    const uint32_t H = perm(R.w[u][i + 7], R.w[u][i + 6], sel);
                    const int dq = 2 * bl + i;  // dword of the group's 32 codes
                    uint8_t* dst = dst0 + (dq >> 2) * C::HALF + (dq & 3) * 256;
                    constexpr uint32_t LO = 0x0F0F0F0Fu, TWO = 0x30303030u;
                    *reinterpret_cast<uint32_t*>(dst) = (A & LO) | ((H << 4) & TWO);
                    *reinterpret_cast<uint32_t*>(dst + C::NIB_BLOCK) = (B & LO) | ((H << 2) & TWO);
                    *reinterpret_cast<uint32_t*>(dst + 2 * C::NIB_BLOCK) = ((A >> 4) & LO) | (H & TWO);
                    *reinterpret_cast<uint32_t*>(dst + 3 * C::NIB_BLOCK) = ((B >> 4) & LO) | ((H >> 2) & TWO);
                }
                const half2_t sp = {(_Float16)(float)(int8_t)(R.w[u][9] & 0xFFu), (_Float16)(float)(int8_t)(R.w[u][9] >> 8)};
                reinterpret_cast<uint32_t*>(st + C::W_BYTES)[bl * C::TJ + jl] = __builtin_bit_cast(uint32_t, sp);
                reinterpret_cast<uint32_t*>(aux)[jl] = R.w[u][10];
                continue;
            }
            const uint32_t end = wbase[u] + (uint32_t)c * (CB * BB) + (BYTES ? 32u : 16u);
            const uint32_t tail = R.w[u][C::WWORDS - 1];
            const uint32_t wt = end > wlast ? tail >> 16 : tail;
            uint32_t* dst = reinterpret_cast<uint32_t*>(st + bl * C::NIB_BLOCK + (jl >> 6) * 1024) + (jl & 63);
            if constexpr (BYTES) {
#pragma unroll
                for (int q = 0; q < 8; q++)
                    dst[(q & 3) * 64 + (q >> 2) * (C::HALF / 4)] =
                        perm(q == 7 ? wt : R.w[u][q + 1], R.w[u][q], wsel[u]) ^ 0x80808080u;
            } else {
#pragma unroll
                for (int q = 0; q < 4; q++) dst[q * 64] = perm(q == 3 ? wt : R.w[u][q + 1], R.w[u][q], wsel[u]);
            }
            uint16_t* wd = reinterpret_cast<uint16_t*>(st + C::W_BYTES);
            wd[bl * C::TJ + jl] = (uint16_t)(R.w[u][0] >> ((wsel[u] & 2u) << 3 ^ 16u));
        }
    };
    // x piece (row il, block bl, group gq) at slot 16 gq + (row ^ (4 (bl % 2) + gq)) of its tile's
    // part: eight consecutive threads (one row's pieces) and eight consecutive
    // lanes of a fragment read (one group's rows) each touch all LDS banks once
    auto store_x = [&](int c, uint8_t* st, uint8_t* aux, const XRegs& R, auto w_tag) {
        if constexpr (decltype(w_tag)::value)
            reinterpret_cast<float*>(st + C::F_AT)[tid] = fbase != RSRC_OOB ? __builtin_bit_cast(float, R.f) : 1.0f;
        uint8_t* xs = st + C::W_BYTES + C::D_BYTES;
#pragma unroll
        for (int u = 0; u < C::XU; u++) {
            const int idx = tid + u * C::NT, il = idx / (CB * 4), q = idx % (CB * 4);
            const int slot = (q & 3) * 16 + ((il & 15) ^ (q & 7));
            uint8_t* p = xs + (((q >> 2) * (C::TI / 16) + (il >> 4)) * 2) * C::X_PART + slot * 16;
            *reinterpret_cast<u32x4*>(p) = R.h[u];
            *reinterpret_cast<u32x4*>(p + C::X_PART) = R.l[u];
        }
        if constexpr (Q4K) {
#pragma unroll
            for (int u = 0; u < C::SU; u++) {
                const int idx = tid + u * C::NT, il = idx / CB, j = (c * CB + idx % CB) & 7;
                // (no branch in the loop body: what follows it would sink past it)
                uint16_t* ss = reinterpret_cast<uint16_t*>(
                    idx < C::TI * CB ? aux + C::SS_AT + (il >> 4) * 512 + (il & 15) * 16 + j * 2 : lds + C::DUMP_AT);
                ss[0] = (uint16_t)R.s[u];
                ss[128] = (uint16_t)(R.s[u] >> 16);
            }
        }
    };

    f32x4 acc[FI][FJ];
#pragma unroll
    for (int b = 0; b < FI; b++)
#pragma unroll
        for (int a = 0; a < FJ; a++) acc[b][a] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    // The main loop runs in steps: one block of one 16-row x tile, 2 FJ MFMAs
    // each.  A step reads the next step's x and adds the previous step's scaled
    // results between its MFMAs.  LDS holds three chunks: while chunk c is
    // multiplied, chunk c + 1 is stored in the first half of its steps, one
    // barrier follows, and the second half reads and converts chunk c + 1's
    // first weights, so the matrix cores are fed across the chunk boundary.
    // Past the end every load reads zeros (x 0, d 0).
    constexpr int RB = FI / 2;
    const Q4Consts qc = q4_consts();
    constexpr bool ONE = Q6K;  // no registers for two sets of operands: converted between the chunks
    u32x4 nv, nv2;  // codes of the next block (nv2: bytes 16+4g .., Q8_0 and the super-block formats)
    uint32_t dd[Q6K ? 4 : 2];
    half8_t wq[ONE ? 1 : 2][4], wl[Q6K ? 4 : 1];
    float dv[2][4];
    f32x4 fv[2];  // WIDE: the scales of a step's rows
    half8_t xh[2], xl[2];
    f32x4 p[CHAIN ? 1 : 2][FJ], T[CHAIN ? FI : 1][FJ];
    // Q4_K: even sub-blocks are low nibbles, odd ones high; this wave's are all alike
    const uint32_t kmask = ks & 1 ? qc.hi : qc.lo;
    const uint32_t kmul = ks & 1 ? 0x2C002C00u : 0x3C003C00u;  // f16 1 / 16, 1
    const uint32_t koff = ks & 1 ? 0xD480D480u : 0xE408E408u;  // f16 -72, -1032
    auto read_w = [&](const uint8_t* st) {
        const int lo = wj * 1024 + g * 256 + r * 16;
        if constexpr (Q4K) {  // both halves of the run of sub-blocks ks & ~1, ks | 1
            nv = *reinterpret_cast<const u32x4*>(st + (ks & ~1) * C::NIB_BLOCK + lo);
            nv2 = *reinterpret_cast<const u32x4*>(st + (ks | 1) * C::NIB_BLOCK + lo);
        } else {
            nv = *reinterpret_cast<const u32x4*>(st + ks * C::NIB_BLOCK + lo);
            if constexpr (BYTES) nv2 = *reinterpret_cast<const u32x4*>(st + ks * C::NIB_BLOCK + C::HALF + lo);
        }
        const uint8_t* dp = st + C::W_BYTES + (ks * C::TJ + wj * 64 + r * 4) * (Q6K ? 4 : 2);
        if constexpr (Q6K) {
            const u32x4 v = *reinterpret_cast<const u32x4*>(dp);
            dd[0] = v.x, dd[1] = v.y, dd[2] = v.z, dd[3] = v.w;
        } else {
            const uint2 v = *reinterpret_cast<const uint2*>(dp);
            dd[0] = v.x, dd[1] = v.y;
        }
    };
    auto read_x = [&](const uint8_t* st, int s) {
        const uint8_t* xb = st + C::W_BYTES + C::D_BYTES + (ks * FI + s) * 2 * C::X_PART +
                            (g * 16 + (r ^ ((ks & 1) * 4 + g))) * 16;
        xh[s & 1] = *reinterpret_cast<const half8_t*>(xb);
        xl[s & 1] = *reinterpret_cast<const half8_t*>(xb + C::X_PART);
    };
    auto conv = [&](int o, int a) {
        const uint32_t n0 = a == 0 ? nv.x : a == 1 ? nv.y : a == 2 ? nv.z : nv.w;
        const uint32_t n1 = a == 0 ? nv2.x : a == 1 ? nv2.y : a == 2 ? nv2.z : nv2.w;
        if constexpr (Q6K) {
            q6k_f16(n0, n1, dd[a], wq[0][a], wl[a]);
            return;
        }
        const uint32_t d16 = a & 1 ? dd[a >> 1] >> 16 : dd[a >> 1] & 0xFFFFu;
        if constexpr (Q4K) {
            const _Float16 sc = __builtin_bit_cast(_Float16, (uint16_t)d16);
            wq[o][a] = q4k_f16(n0, n1, kmask, qc.magic, __builtin_bit_cast(half2_t, kmul),
                               __builtin_bit_cast(half2_t, koff), sc);
            return;
        }
        if constexpr (BYTES) wq[o][a] = q8_f16(n0, n1);
        else wq[o][a] = q4_f16(n0, qc);
        dv[o][a] = h2f(d16);
        // f32 here once a block: left to itself the compiler folds the conversion
        // into every scale FMA (v_fma_mix_f32: 1,240 against 546 us, 2048 x 14336 x 4096)
        asm volatile("" : "+v"(dv[o][a]));
    };
    auto add = [&](int b, int o, int ps, auto w_tag) {
#pragma unroll
        for (int a = 0; a < FJ; a++)
#pragma unroll
            for (int u = 0; u < 4; u++)
                acc[b][a][u] = fmaf(decltype(w_tag)::value ? dv[o][a] * fv[ps][u] : dv[o][a], p[ps][a][u], acc[b][a][u]);
    };
    // CHAIN: a finished super-block (its own data at aux) goes into the sums in
    // the FI steps of the next chunk: step b adds x tile b, and Q4_K's remainder
    // of weight column b for the FO tiles ks FO .. that this K group ends with
    // (um, so that the KS groups share them).  K elements 8 g .. of that MFMA:
    // S hi, lo, hi, lo times e hi, hi, lo, lo (against S lo: over SUM_LO).
    constexpr int FO = FI / KS;
    static_assert(!CHAIN || FI == FJ, "a weight column a step");
    f32x4 um[Q4K ? FO : 1][FJ];
    u32x4 fd;                       // d (and t) of the lane's four columns
    half8_t fs[Q4K ? FO : 1], fe;   // S of the tiles, e of the step's column
    auto flush_e = [&](int a, const uint8_t* aux) {
        if constexpr (Q4K)
            fe = *reinterpret_cast<const half8_t*>(aux + C::MN_AT + (wj * 64 + r * 4 + a) * 64 + g * 16);
    };
    auto flush_begin = [&](const uint8_t* aux) {
        fd = *reinterpret_cast<const u32x4*>(aux + (wj * 64 + r * 4) * 4);
        if constexpr (Q4K) {
#pragma unroll
            for (int b = 0; b < FO; b++)
                fs[b] = *reinterpret_cast<const half8_t*>(aux + C::SS_AT + (ks * FO + b) * 512 + (g & 1) * 256 + r * 16);
        }
        flush_e(0, aux);
    };
    auto flush = [&](int b, const uint8_t* aux) {
        const uint32_t db[4] = {fd.x, fd.y, fd.z, fd.w};
        f32x4 u4[Q4K ? FO : 1];
        if constexpr (Q4K) {
            const f32x4 z = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int o = 0; o < FO; o++) u4[o] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fs[o], fe, z, 0, 0, 0);
            if (b + 1 < FJ) flush_e(b + 1, aux);
        }
#pragma unroll
        for (int a = 0; a < FJ; a++) {
            const float d = h2f(db[a] & 0xFFFFu);
#pragma unroll
            for (int u = 0; u < 4; u++) acc[b][a][u] = fmaf(d, T[b][a][u], acc[b][a][u]);
        }
        if constexpr (Q4K) {
            const float dm = ldexpf(32.0f, (int)db[b] >> 16);
#pragma unroll
            for (int o = 0; o < FO; o++)
#pragma unroll
                for (int u = 0; u < 4; u++) um[o][b][u] = fmaf(dm, u4[o][u], um[o][b][u]);
        }
    };
    // chunks the loads run ahead (no registers for more)
    constexpr int DX = FI == 8 || CHAIN ? 1 : 2, DW = (FI == 8 && BYTES) || CHAIN ? 1 : 2;
    constexpr int UN = 2;  // chunks a turn of the loop (CHAIN: a super-block)
    static_assert(!CHAIN || UN * CB == 8, "a super-block a turn");
    WRegs w[DW];
    XRegs x1[DX];
    uint8_t *bc = lds, *bn = lds + C::STAGE, *bf = lds + 2 * C::STAGE;  // chunk c, c + 1, free
    // super-block being multiplied, the next one, the previous one
    uint8_t *ac = lds + C::AUX_AT, *an = ac + C::AUX, *ap = an + C::AUX;
    // chunk c = U modulo UN (register sets by parity)
    auto chunk = [&](int c, auto u_tag, auto w_tag) {
        constexpr int U = decltype(u_tag)::value, H = U & 1, WS = (U + 1) % DW, XS1 = (U + 1) % DX;
        uint8_t* const as = CHAIN && U == UN - 1 ? an : ac;  // chunk c + 1's super-block
#pragma unroll
        for (int s = 0; s < FI; s++) {
            if (s + 1 < FI) read_x(bc, s + 1);
            else read_x(bn, 0);
            if (s == RB && !ONE) read_w(bn);
            const f32x4 z = {0.0f, 0.0f, 0.0f, 0.0f};
            if constexpr (CHAIN) {
                if (U == 0) {
                    flush(s, ap);
                    __builtin_amdgcn_sched_barrier(0);
                }
                // Q6_K: one operand at a time, four independent MFMAs between
                // dependent ones (2 % faster); Q4_K: a column at a time (3 %)
                auto mul = [&](int a, const half8_t& xv, const half8_t& wv, bool first) {
                    T[s][a] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xv, wv, U == 0 && first ? z : T[s][a], 0, 0, 0);
                };
                if constexpr (Q6K) {
#pragma unroll
                    for (int a = 0; a < FJ; a++) mul(a, xh[s & 1], wq[0][a], true);
#pragma unroll
                    for (int a = 0; a < FJ; a++) mul(a, xl[s & 1], wq[0][a], false);
#pragma unroll
                    for (int a = 0; a < FJ; a++) mul(a, xh[s & 1], wl[a], false);
                } else {
#pragma unroll
                    for (int a = 0; a < FJ; a++) {
                        mul(a, xh[s & 1], wq[H][a], true);
                        mul(a, xl[s & 1], wq[H][a], false);
                    }
                }
            } else {
#pragma unroll
                for (int a = 0; a < FJ; a++) {
                    p[s & 1][a] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xh[s & 1], wq[H][a], z, 0, 0, 0);
                    p[s & 1][a] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xl[s & 1], wq[H][a], p[s & 1][a], 0, 0, 0);
                }
                add(s == 0 ? FI - 1 : s - 1, s == 0 ? H ^ 1 : H, (s & 1) ^ 1, w_tag);
                if constexpr (decltype(w_tag)::value)
                    fv[s & 1] = *reinterpret_cast<const f32x4*>(bc + C::F_AT + (ks * C::TI + s * 16 + g * 4) * 4);
            }
            if (s > RB && !ONE) {
#pragma unroll
                for (int a = 0; a < FJ; a++)
                    if (a * (FI - 1 - RB) / FJ == s - 1 - RB) conv(H ^ 1, a);
            }
            if (s == 0) {
                store_w(c + 1, bn, as, w[WS]);
                if (DW == 1) load_w(c + 2, w[0]);
            }
            if (s == 1) store_x(c + 1, bn, as, x1[XS1], w_tag);
            // the loads into the freed registers, spread over the later steps (a
            // burst of them stalls the waves at issue)
            if (DW == 2 && s == FI - 1) load_w(c + 3, w[WS]);
            if (s >= 2) {
#pragma unroll
                for (int q = 0; q < 2 * C::XU; q++)
                    if (2 + q * (FI - 2) / (2 * C::XU) == s) load_x_part(c + 1 + DX, x1[XS1], q);
                if (s == FI - 1) load_sums(c + 1 + DX, x1[XS1]);
                if constexpr (decltype(w_tag)::value)
                    if (s == FI - 1) load_scale(c + 1 + DX, x1[XS1]);
            }
            if constexpr (!Q6K) {
#pragma unroll
                for (int a = 0; a < FJ; a++) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
                    __builtin_amdgcn_sched_group_barrier(0x002, 6, 0);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
            if (s == RB - 1) __syncthreads();
        }
        if (CHAIN && U == UN - 1) flush_begin(ac);
        if constexpr (ONE) {
            read_w(bn);
#pragma unroll
            for (int a = 0; a < FJ; a++) conv(0, a);
        }
        uint8_t* t3 = bc;
        bc = bn;
        bn = bf;
        bf = t3;
        if (CHAIN && U == UN - 1) {
            uint8_t* t4 = ap;
            ap = ac;
            ac = an;
            an = t4;
        }
    };
    constexpr std::false_type plain{};
    if constexpr (!WIDE) {
        // chunks 0 .. DW - 1 of W and 0 .. DX - 1 of x first, then on to DW / DX
        // once chunk 0 is stored
#pragma unroll
        for (int q = 0; q < DW; q++) load_w(q, w[q]);
#pragma unroll
        for (int q = 0; q < DX; q++) load_x(q, x1[q], plain);
        if constexpr (CHAIN)  // nothing to flush before the first super-block: zeros
            for (int q = tid; q < C::AUX / 4; q += C::NT) reinterpret_cast<uint32_t*>(ap)[q] = 0;
        store_w(0, bc, ac, w[0]);
        store_x(0, bc, ac, x1[0], plain);
        load_w(DW, w[0]);
        load_x(DX, x1[0], plain);
        __syncthreads();
        read_w(bc);
        read_x(bc, 0);
        if constexpr (CHAIN) flush_begin(ap);
#pragma unroll
        for (int a = 0; a < FJ; a++) {
            conv(0, a);
            if constexpr (!CHAIN) {
                dv[1][a] = 0.0f;
                p[1][a] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            } else {
#pragma unroll
                for (int b = 0; b < FI; b++) T[b][a] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
                if constexpr (Q4K)
#pragma unroll
                    for (int b = 0; b < FO; b++) um[b][a] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            }
        }
        // (chunks past the slice's end: zeros; no branch, so that the waits stay exact)
        for (int c = 0; c < nchunks; c += UN) {
            chunk(c, std::integral_constant<int, 0>{}, plain);
            chunk(c + 1, std::integral_constant<int, 1>{}, plain);
        }
        if constexpr (CHAIN) {
#pragma unroll
            for (int b = 0; b < FI; b++) flush(b, ap);  // (begun at the end of the last chunk)
        } else {
            add(FI - 1, 1, 1, plain);
        }
    } else {
        // The same steps.  The loads before the loop stay in the loop's order, for
        // its first wait covers both (reordered it waits for all loads but two: 64 x
        // 14336 x 4096 27.6 -> 29.4 us).
        auto first_w = [&]() {
#pragma unroll
            for (int q = 0; q < DW; q++) {
                load_w(q, w[q]);
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        // weights, and chunk 0 of x, on their way before the flags are waited for
        // (0.2 to 1 us a call) where there are registers for them across the branch
        constexpr int EX = FI == 4 && C::NT == 512 ? 1 : 0;
        if constexpr (FI == 4) first_w();
#pragma unroll
        for (int q = 0; q < EX; q++) {
            load_x(q, x1[q], plain);
            __builtin_amdgcn_sched_barrier(0);
        }
        uint32_t any = 0;
#pragma unroll
        for (int q = 0; q < C::TI / 4; q++) any |= XF[(i0 - r0) / 4 + q];
        const bool wide = __builtin_amdgcn_readfirstlane(any) != 0;
        auto multiply = [&](auto w_tag) {
            if constexpr (FI != 4) first_w();
#pragma unroll
            for (int q = 0; q < DX; q++) {
                if (q >= EX) load_x(q, x1[q], w_tag);
                else if constexpr (decltype(w_tag)::value) load_scale(q, x1[q]);
                __builtin_amdgcn_sched_barrier(0);
            }
            store_w(0, bc, ac, w[0]);
            store_x(0, bc, ac, x1[0], w_tag);
            load_w(DW, w[0]);
            __builtin_amdgcn_sched_barrier(0);
            load_x(DX, x1[0], w_tag);
            __builtin_amdgcn_sched_barrier(0);
            __syncthreads();
            read_w(bc);
            read_x(bc, 0);
            fv[1] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int a = 0; a < FJ; a++) {
                conv(0, a);
                dv[1][a] = 0.0f;
                p[1][a] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            }
            for (int c = 0; c < nchunks; c += UN) {
                chunk(c, std::integral_constant<int, 0>{}, w_tag);
                chunk(c + 1, std::integral_constant<int, 1>{}, w_tag);
            }
            add(FI - 1, 1, 1, w_tag);
        };
        if (wide) {
            __syncthreads();  // (the rows' exponents are in LDS)
            if (tid < C::TI * CB && xe[tid % C::TI] == WIDE_ROW)
                fbase = ((uint32_t)(kb0 + tid / C::TI) * (uint32_t)xb_rows + (uint32_t)(i0 - r0 + tid % C::TI)) * 4u;
            multiply(std::true_type{});
        } else {
            multiply(plain);
        }
    }

    // lane (g, r) holds y[i = 4 g + u][j = 4 r .. 4 r + 3] of 16-row tile b
    auto store_rows = [&](int b, const f32x4 (&v4)[FJ]) {
        const int j = j0 + wj * 64 + r * 4;
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int i = i0 + b * 16 + g * 4 + u;
            if (i >= r1) continue;
            const int e = WIDE && xe[i - i0] == WIDE_ROW ? 0 : xe[i - i0];
            f32x4 v = {ldexpf(v4[0][u], e), ldexpf(v4[1][u], e), ldexpf(v4[2][u], e), ldexpf(v4[3][u], e)};
            float* yp = Y + (size_t)i * n + j;
            // accy: y += the product (the residual add, one rounding as x + y)
            if (j + 3 < n && (n & 3) == 0) {
                if (accy) v = (f32x4)*reinterpret_cast<const f32x4u*>(yp) + v;
                *reinterpret_cast<f32x4u*>(yp) = v;
            } else {
#pragma unroll
                for (int q = 0; q < 4; q++)
                    if (j + q < n) yp[q] = accy ? yp[q] + v[q] : v[q];
            }
        }
    };
    // The KS waves of a column group share its 16-row tiles: wave ks ends with
    // the sums of tiles ks FO .. ks FO + FO - 1.  Each wave hands the tiles of
    // the others through LDS (the stages are free once every wave is here).
    __syncthreads();
    if constexpr (KS > 1) {
        f32x4* red = reinterpret_cast<f32x4*>(lds) + wj * (KS * (KS - 1) * FO * FJ * 64) + lane;
#pragma unroll
        for (int o = 0; o < KS; o++) {
            if (o == ks) continue;  // (slot of sender ks among the owner's KS - 1)
            const int slot = o * (KS - 1) + (ks < o ? ks : ks - 1);
#pragma unroll
            for (int b = 0; b < FO; b++)
#pragma unroll
                for (int a = 0; a < FJ; a++) red[((slot * FO + b) * FJ + a) * 64] = acc[o * FO + b][a];
        }
        __syncthreads();
    }
    f32x4 own[FO][FJ];
#pragma unroll
    for (int o = 0; o < KS; o++)
        if (o == ks) {
#pragma unroll
            for (int b = 0; b < FO; b++)
#pragma unroll
                for (int a = 0; a < FJ; a++) own[b][a] = acc[o * FO + b][a];
        }
    if constexpr (KS > 1) {
        const f32x4* red = reinterpret_cast<const f32x4*>(lds) + wj * (KS * (KS - 1) * FO * FJ * 64) + lane;
#pragma unroll
        for (int q = 0; q < KS - 1; q++)
#pragma unroll
            for (int b = 0; b < FO; b++)
#pragma unroll
                for (int a = 0; a < FJ; a++) own[b][a] += red[(((ks * (KS - 1) + q) * FO + b) * FJ + a) * 64];
    }

    if constexpr (Q4K)
#pragma unroll
        for (int b = 0; b < FO; b++)
#pragma unroll
            for (int a = 0; a < FJ; a++) own[b][a] += um[b][a];

    // ---- slices of the tile: partials, counter, the last one adds them in slice order
    if (S > 1) {
        constexpr int UNITS = C::NW * FO * FJ * 64;  // f32x4 results of a tile
        const __amdgpu_buffer_rsrc_t prs = make_rsrc(part + (size_t)(t - full) * S * UNITS * 4, (uint32_t)S * UNITS * 16u);
        const uint32_t u0 = (uint32_t)wave * (FO * FJ * 64) + lane;
#pragma unroll
        for (int b = 0; b < FO; b++)
#pragma unroll
            for (int a = 0; a < FJ; a++)
                __builtin_amdgcn_raw_buffer_store_b128(
                    __builtin_bit_cast(u32x4, own[b][a]), prs,
                    (int)(((uint32_t)slice * UNITS + u0 + (b * FJ + a) * 64) * 16u), 0, LOCAL ? 0 : CPOL_SC1);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this thread's partial has completed
        __syncthreads();  // (and every wave is done with the LDS sums)
        int* last_sh = reinterpret_cast<int*>(lds);
        if (tid == 0) {
            constexpr int SCOPE = LOCAL ? __HIP_MEMORY_SCOPE_WORKGROUP : __HIP_MEMORY_SCOPE_AGENT;
            const int old = __hip_atomic_fetch_add(cnt + t - full, 1, __ATOMIC_RELAXED, SCOPE);
            *last_sh = old == S - 1;
            if (old == S - 1) __hip_atomic_store(cnt + t - full, 0, __ATOMIC_RELAXED, SCOPE);
        }
        __syncthreads();
        if (!*last_sh) return;
        // four slices' loads in flight (slots past S read zeros, which add nothing)
#pragma unroll
        for (int b = 0; b < FO; b++)
#pragma unroll
            for (int a = 0; a < FJ; a++) own[b][a] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        for (int s0 = 0; s0 < S; s0 += 4) {
            f32x4 v[4][FO][FJ];
#pragma unroll
            for (int q = 0; q < 4; q++)
#pragma unroll
                for (int b = 0; b < FO; b++)
#pragma unroll
                    for (int a = 0; a < FJ; a++) {
                        const uint32_t off = ((uint32_t)(s0 + q) * UNITS + u0 + (b * FJ + a) * 64) * 16u;
                        v[q][b][a] = __builtin_bit_cast(
                            f32x4, __builtin_amdgcn_raw_buffer_load_b128(prs, (int)(s0 + q < S ? off : RSRC_OOB), 0,
                                                                         LOCAL ? CPOL_NT : CPOL_SC1));
                    }
#pragma unroll
            for (int q = 0; q < 4; q++)
#pragma unroll
                for (int b = 0; b < FO; b++)
#pragma unroll
                    for (int a = 0; a < FJ; a++) own[b][a] += v[q][b][a];
        }
    }
#pragma unroll
    for (int b = 0; b < FO; b++) store_rows(ks * FO + b, own[b]);
}

// x split of m rows in the scratch (gemm_tiles_scratch_bytes(m, k), or
// gemm_wide_scratch_bytes(m, k) where rows may be wide); lo: where x_lo goes
// instead (m k 2 bytes), or NULL.
struct XSplit {
    _Float16 *h, *l;
    int* e;
    uint32_t* s;  // x' sums of each block (hi / lo pairs), or NULL
    float* b;     // [block][b_rows] scales of wide rows, or NULL
    int b_rows;
    uint8_t* f;   // whether a row is wide
};
XSplit x_split_at(void* scratch, void* lo, size_t m, size_t k, bool sums, bool wide) {
    const size_t xb = (m * k * 2 + 255) & ~(size_t)255, eb = (m * 4 + 255) & ~(size_t)255;
    uint8_t* p = reinterpret_cast<uint8_t*>(scratch);
    uint8_t* e = p + (lo ? xb : 2 * xb);
    uint8_t* f = e + eb;  // (first: a multiple of XF_PAD bytes)
    const size_t fb = (m + 255) & ~(size_t)255;
    return {reinterpret_cast<_Float16*>(p), reinterpret_cast<_Float16*>(lo ? lo : p + xb), reinterpret_cast<int*>(e),
            sums ? reinterpret_cast<uint32_t*>(e + eb) : nullptr, wide ? reinterpret_cast<float*>(f + fb) : nullptr,
            (int)m, f};
}

// One tile shape: 64 WJ weight rows x 16 FI x rows, KS wave groups sharing
// each chunk's blocks.
template <int WF, int FI, int WJ, int KS, bool WIDE>
hipError_t launch_tile_cfg(const uint8_t* w, int n, int nb, const XSplit& x, int m, int r0, int r1, float* y, int accy,
                           const TilePlan& p, float* part, int* cnt, hipStream_t s) {
    using C = TileCfg<WF, FI, WJ, KS, WIDE>;
    static_assert(C::LDS <= 160 * 1024, "LDS per workgroup");
    const bool local = p.S > 1 && xcd_round_robin(s);
    auto kern = local ? gemm_tile_kernel<WF, FI, WJ, KS, true, WIDE> : gemm_tile_kernel<WF, FI, WJ, KS, false, WIDE>;
    if (C::LDS > 65536) {
        static const hipError_t e[2] = {
            hipFuncSetAttribute((const void*)gemm_tile_kernel<WF, FI, WJ, KS, false, WIDE>,
                                hipFuncAttributeMaxDynamicSharedMemorySize, C::LDS),
            hipFuncSetAttribute((const void*)gemm_tile_kernel<WF, FI, WJ, KS, true, WIDE>,
                                hipFuncAttributeMaxDynamicSharedMemorySize, C::LDS)};  // once a process
        if (e[local] != hipSuccess) return e[local];
    }
    unsigned rest = (unsigned)((n + C::TJ - 1) / C::TJ) * (unsigned)((m + C::TI - 1) / C::TI) - (unsigned)p.full;
    if (local) rest = (rest + 7) / 8 * 8;
    launch_kernel(kern, dim3((unsigned)p.full + rest * (unsigned)p.S), dim3(C::NT), (size_t)C::LDS, s, w, n, nb, x.h,
                  x.l, x.e, m, r0, r1, x.s, x.b, x.b_rows,
                  reinterpret_cast<const uint32_t*>(x.f), y, accy, p.full, p.S, p.kbs, part, cnt);
    return hipGetLastError();
}

// The tile shapes, largest first: weight rows, x rows, K groups, and the time
// one workgroup takes a 32-element block (one workgroup a CU; measured at n =
// 4096, 128 rows: 117 / 66 / 39 / 35 us for 128 blocks).
struct TileShape {
    int tj, ti, ks;
    double us_block;
};
constexpr TileShape TILE_SHAPES[4] = {{256, 128, 2, 0.90}, {256, 64, 2, 0.50}, {128, 64, 4, 0.29}, {64, 64, 4, 0.26}};
// The super-block formats run on one shape: their sums take the registers of
// the larger ones (Q4_K in 256 x 64 tiles spills: 211 x 14336 x 4096 115 us there, 114 here),
// and 64 x 64 tiles spill too (72 us against 58 at 128 x 4096 x 4096).
constexpr int SUPER_SHAPE = 2;
constexpr double SUPER_US_BLOCK = 0.43;

// Tile shape and K slices of a product by estimated time.  Whole rounds of
// one workgroup a CU run unsplit; the tiles past them are split over K, where
// that is estimated to pay, into up to as many slices as fill a round.  Time:
// a round's blocks, plus, split, the last slice's reading of the others'
// partials (about 40 KB a us; 2 us for the stores and the counter).  Against
// sweeps over shapes and slices at 80-2048 rows, n = 1024 .. 28672, k = 4096
// and 14336 the choice was the best or within 5 % of it: at 128 rows 4096 x
// 4096 64 tiles of 128 x 64 in 4 slices (25.6 us; unsplit 40.4, 2 slices 28.7,
// 8 slices 36.2), 14336 x 4096 the same tiles unsplit (44 us; 256 x 128 117,
// 64 x 64 67), 512 rows 14336 x 4096 256 x 128 (127 us; 256 x 64 162).
TilePlan tile_plan(WType t, size_t m, size_t n, size_t nb, bool can_split) {
    const bool super = t == WType::Q4_K || t == WType::Q6_K;
    const size_t round = std::max(8, device_cu_count() / 8 * 8);
    TilePlan best{};
    double best_us = 1e30;
    for (int c = 0; c < 4; c++) {
        if (super && c != SUPER_SHAPE) continue;
        const TileShape& sh = TILE_SHAPES[c];
        const double us_block = super ? SUPER_US_BLOCK : sh.us_block;
        const size_t tiles = ((n + sh.tj - 1) / sh.tj) * ((m + sh.ti - 1) / sh.ti);
        const size_t unit = super ? 8 : 2 * (size_t)sh.ks;  // a turn of the main loop: two chunks, or a super-block
        const size_t full = tiles / round * round, rest = tiles - full;
        const double whole = nb * us_block + 6.0;  // us a round of unsplit tiles
        for (size_t S = 1; S <= 16; S++) {
            const size_t kbs = ((nb + S - 1) / S + unit - 1) / unit * unit;
            double us = (double)(full / round) * whole;
            if (S == 1) {
                us += rest ? whole : 0.0;
            } else {
                if (!can_split || rest * S > round) break;
                if ((S - 1) * kbs >= nb) continue;  // (an empty slice)
                const size_t bytes = S * sh.tj * sh.ti * sizeof(float);
                if (rest == 0 || rest * bytes > GEMM_PART_BYTES) break;
                us += kbs * us_block + 6.0 + 2.0 + (double)bytes / 40e3;
            }
            if (us < best_us) best_us = us, best = {c, (int)(S == 1 ? tiles : full), (int)S, (int)kbs};
        }
    }
    return best;
}

template <int PRO, int WB>
hipError_t launch_split(const float* x, size_t m, size_t k, const float* g, float eps, const XSplit& o, hipStream_t s) {
    // 256 threads hold 4096 elements of a row, 1024 threads GEMM_SPLIT_MAX_K
    if (k > GEMM_SPLIT_MAX_K) {
        if (PRO != 0 || WB != 0 || o.s) return hipErrorInvalidValue;
        launch_kernel(gemm_split_long_kernel, dim3((unsigned)m), dim3(1024), 0, s, x, (int)k, o.h, o.l, o.e);
        return hipGetLastError();
    }
    if (k <= 4096)
        launch_kernel(gemm_split_kernel<PRO, 256, 4, WB>, dim3((unsigned)m), dim3(256), 0, s, x, (int)k, g, eps, o.h,
                      o.l, o.e, o.s, o.b, o.b_rows, o.f);
    else
        launch_kernel(gemm_split_kernel<PRO, 1024, 4, WB>, dim3((unsigned)m), dim3(1024), 0, s, x, (int)k, g, eps, o.h,
                      o.l, o.e, o.s, o.b, o.b_rows, o.f);
    return hipGetLastError();
}

}  // namespace

// Native mode (x as Q8_0 blocks hold it, the same codes and scales times the
// same blocks): the int8 kernel of gemm.hip forms sx d and scales every int32
// dot, three VALU instructions a result where one FMA does here, and its tiles
// are not split over K (us, int8 kernel / here: 512 x 14336 x 4096 184 / 114,
// 512 x 4096 x 14336 171 / 134, 2048 x 14336 x 4096 601 / 448, 65 x 4096 x 4096 25.3 /
// 22.4, 128 x 14336 x 4096 88 / 42, 256 x 1024 x 4096 50 / 21.5, 1024 x 64 x 4096 46 /
// 25).  It keeps short products over small matrices (128 x 2048 x 2048 10.6 / 15.4,
// 200 x 1024 x 4096 17.4 / 19.3, 1024 x 512 x 992 15.4 / 17) and rows past one
// workgroup's registers.
bool gemm_native_tile_takes(size_t m, size_t n, size_t k) {
    if (m <= GEMM_XTILE_M || k > GEMM_SPLIT_MAX_K) return false;
    if (m < 256) return n * k >= (size_t)1 << 24;
    return m < 1024 || n >= 2048 || k >= 2048;
}

// The small-tile kernel of gemm.hip keeps short products over small matrices:
// its 16 x 32 tiles reach all CUs without a split over K, and its code is
// smaller (us, here against there: Q4_0 100 x 512 x 992 10.7 / 9.1, 200 x 2048 x
// 992 13.6 / 12.7, 100 x 4096 x 1024 12.9 / 11.8, 200 x 4096 x 1024 16.2 / 15.4, 200 x
// 2048 x 2048 18.8 / 16.6 (100 rows: 14.1 / 15.0), 100 x 64 x 4096 13.4 / 17.3;
// Q8_0 100 x 512 x 992 11.0 / 8.9, 1000 x 512 x 992 17.5 / 16.4, 333 x 4096 x 992
// 19.5 / 25.7, 17 x 4096 x 4096 17.9 / 17.2, 33 x 4096 x 4096 18.6 / 24.4; Q4_K 64 x
// 2048 x 2048 16.5 / 14.7, 128 x 2048 x 2048 18.5 / 19.1, 32 x 512 x 4096 17.3 / 22.3, 16 x
// 4096 x 4096 19.5 / 17.3, 16 x 14336 x 1024 17.6 / 24.1, 500 x 4096 x 1024 23.4 / 26.8,
// 211 x 4096 x 1024 19.7 / 17.4; Q6_K alike).
// Q4_0 calls of 5 to 64 rows have the x-tile kernel, one launch that splits x in
// every strip of 128 weight rows.  The tiles compute 64 rows whatever m is, but
// split x once: they take matrices of many strips or long rows, and short wide
// ones whose few strips leave CUs idle there (us, here / x-tile kernel: 16 x 32000
// x 4096 38 / 44, 16 x 14336 x 4096 27 / 23, 16 x 512 x 4096 12.8 / 14.8; 32 x 32000 x
// 4096 39 / 53, 32 x 4096 x 14336 29.6 / 33.1, 32 x 9000 x 7168 31.6 / 30.4, 32 x 11008
// x 4096 26.6 / 23.9, 32 x 64 x 4096 12.6 / 16.3; 33 x 6144 x 4096 19.8 / 24.2, 64 x
// 14336 x 4096 28.6 / 54, 64 x 4096 x 14336 31 / 65, 33 x 4096 x 4096 17.1 / 14.9, 33 x
// 1024 x 4096 14.2 / 16.5, 33 x 4096 x 2048 13.4 / 10.3).
bool gemm_tile_takes(WType t, size_t m, size_t n, size_t k) {
    if (t == WType::Q4_0 && m <= GEMM_XTILE_M) {
        if (k > GEMM_SPLIT_MAX_K) return false;
        const size_t nk = n * k;
        if (m <= 16) return nk >= (size_t)3 << 25 || (n <= 512 && nk >= (size_t)1 << 21);
        if (m <= 32) return nk >= (size_t)3 << 25 || (nk >= (size_t)3 << 24 && k >= 2 * n) || (n <= 512 && nk >= (size_t)1 << 18);
        return nk > (size_t)1 << 24 || (nk >= (size_t)1 << 18 && (n <= 512 || (n <= 1024 && nk <= (size_t)1 << 22)));
    }
    if (t == WType::Q4_0) return m > GEMM_XTILE_M && !(m < 256 && n <= 4096 && k <= 2048 && n * k <= (size_t)1 << 22);
    if (k > GEMM_SPLIT_MAX_K) return false;
    if (t == WType::Q4_K || t == WType::Q6_K) {
        if (n >= 8192) return m >= KQ_GEMM_MIN_M;
        return m >= 32 && (k >= 4096 || (m >= 128 && k >= 2048 && n >= 2048) || m * n >= (size_t)3 << 19);
    }
    if (t != WType::Q8_0 || m < KQ_GEMM_MIN_M) return false;
    if (k <= 2048 && (m * n <= (size_t)1 << 19 || (m <= 256 && n * k <= (size_t)1 << 23))) return false;
    return m > 24 || n * k > (size_t)1 << 24;
}

size_t gemm_part_bytes(WType t, size_t m, size_t n, size_t k) {
    const TilePlan p = tile_plan(t, m, n, k / QK, true);
    const TileShape& sh = TILE_SHAPES[p.cfg];
    const size_t rest = ((n + sh.tj - 1) / sh.tj) * ((m + sh.ti - 1) / sh.ti) - (size_t)p.full;
    return rest * p.S * sh.tj * sh.ti * sizeof(float);
}

template <int WF, bool WIDE = false>
static hipError_t launch_tile_wf(const uint8_t* w, int n, int nb, const XSplit& x, int m, int r0, int r1, float* y,
                                 int accy, const TilePlan& p, float* part, int* cnt, hipStream_t s) {
    auto go = [&](auto fi, auto wj, auto ks) {
        return launch_tile_cfg<WF, decltype(fi)::value, decltype(wj)::value, decltype(ks)::value, WIDE>(
            w, n, nb, x, m, r0, r1, y, accy, p, part, cnt, s);
    };
    using I1 = std::integral_constant<int, 1>;
    using I2 = std::integral_constant<int, 2>;
    using I4 = std::integral_constant<int, 4>;
    using I8 = std::integral_constant<int, 8>;
    if constexpr (WF == WF_Q4_0 || WF == WF_Q8_0) {
        if (p.cfg == 0) return go(I8{}, I4{}, I2{});
        if (p.cfg == 1) return go(I4{}, I4{}, I2{});
        if (p.cfg == 3) return go(I4{}, I1{}, I4{});
    }
    return go(I4{}, I2{}, I4{});
}

hipError_t launch_gemm_tile(WType t, const uint8_t* w, size_t n, size_t k, const float* x, size_t m, float* y,
                            void* scratch, float* part, int* cnt, int pro, const float* g, float eps, bool accumulate,
                            hipStream_t s, void* lo, size_t chunk) {
    if (pro == 3 ? t != WType::Q4_0 || k == 0 || !gemm_native_tile_takes(m, n, k)
                 : k == 0 || !gemm_tile_takes(t, m, n, k) || (pro != 0 && k > GEMM_SPLIT_MAX_K))
        return hipErrorInvalidValue;
    if (chunk == 0 && lo) return hipErrorInvalidValue;  // (not one row fits)
    if (chunk == 0) chunk = m;
    if (chunk < m && chunk % TILE_SHAPES[0].ti != 0) return hipErrorInvalidValue;
    const TilePlan p = tile_plan(t, m, n, k / QK, part != nullptr && cnt != nullptr);
    const int ni = (int)n, nb = (int)(k / QK), mi = (int)m, acc = accumulate ? 1 : 0;
    const bool few = t == WType::Q4_0 && pro == 0 && m <= GEMM_XTILE_M;  // (the x-tile kernel's rows)
    for (size_t r0 = 0; r0 < m; r0 += chunk) {
        const size_t rows = std::min(chunk, m - r0);
        const int a = (int)r0, b = (int)(r0 + rows);
        const XSplit xo = x_split_at(scratch, lo, rows, k, t == WType::Q4_K, few || pro == 3);
        const float* xr = x + r0 * k * (pro == 2 ? 2 : 1);
        hipError_t e = pro == 1   ? launch_split<1, 0>(xr, rows, k, g, eps, xo, s)
                       : pro == 2 ? launch_split<2, 0>(xr, rows, k, g, eps, xo, s)
                       : pro == 3 ? launch_split<3, WIDE_NATIVE>(xr, rows, k, g, eps, xo, s)
                       : few      ? launch_split<0, WIDE_FLOAT>(xr, rows, k, g, eps, xo, s)
                                  : launch_split<0, 0>(xr, rows, k, g, eps, xo, s);
        if (e != hipSuccess) return e;
        switch (t) {
            case WType::Q4_0:
                e = xo.b ? launch_tile_wf<WF_Q4_0, true>(w, ni, nb, xo, mi, a, b, y, acc, p, part, cnt, s)
                         : launch_tile_wf<WF_Q4_0>(w, ni, nb, xo, mi, a, b, y, acc, p, part, cnt, s);
                break;
            case WType::Q8_0: e = launch_tile_wf<WF_Q8_0>(w, ni, nb, xo, mi, a, b, y, acc, p, part, cnt, s); break;
            case WType::Q4_K: e = launch_tile_wf<WF_Q4_K>(w, ni, nb, xo, mi, a, b, y, acc, p, part, cnt, s); break;
            default: e = launch_tile_wf<WF_Q6_K>(w, ni, nb, xo, mi, a, b, y, acc, p, part, cnt, s);
        }
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

size_t gemm_wide_scratch_bytes(size_t m, size_t k) {
    const size_t xb = (m * k * 2 + 255) & ~(size_t)255;
    return 2 * xb + ((m * 4 + 255) & ~(size_t)255) + ((m + 255) & ~(size_t)255) + ((m * (k / QK) * 4 + 255) & ~(size_t)255);
}

size_t gemm_tile_chunk_rows(size_t k, size_t bytes, size_t lo_bytes) {
    const size_t ti = TILE_SHAPES[0].ti;  // (the other shapes' rows divide it)
    size_t rows = lo_bytes / (k * 2) / ti * ti;
    // x_hi, the exponents and the blocks' scales
    while (rows > 0 && gemm_wide_scratch_bytes(rows, k) - ((rows * k * 2 + 255) & ~(size_t)255) > bytes) rows -= ti;
    return rows;
}

}  // namespace rdl
