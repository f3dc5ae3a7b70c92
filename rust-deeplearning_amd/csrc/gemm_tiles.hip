// gemm_tiles.hip -- LDS-tiled matrix-core GEMM over GGUF blocks:
// Y[m, n] = X[m, k] . W[n, k]^T for many activation rows, weights read in
// their GGUF block layout (matmul_f32_q4, quantize.rs:265-320).
//
// Numerics.  Each x row is scaled by a power of two (row max into [2^14,
// 2^15)) and split into x_hi = f16(x') and x_lo = f16(x' - x_hi), about 22
// significant bits; the weight operand is the exact integer code in f16, one
// 16x16x32 MFMA K step is one 32-element block, and the block scale d
// multiplies the block's f32 dot afterwards: acc += d (x_hi.q + x_lo.q).
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
// Counters at 2048 x 4096 x 14336: matrix cores busy 53 %, VALU issue 55 %,
// bank conflicts 8 % of LDS cycles; the clock settles near 1.95 GHz.  2048
// rows, 14336 x 4096 / 4096 x 14336: 631 / 615 -> 480 / 455 us (501 / 528
// TFLOP/s; the matrix cores do twice that, x being two operands); 512 rows
// 14336 x 4096: 213 -> 127 us; 128 rows 4096 x 4096 / 14336 x 4096 / 4096 x
// 14336: 30.7 / 73 / 84 -> 25.6 / 44 / 49 us (split over K, below).
#include <hip/hip_runtime.h>

#include <algorithm>
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

// ---- x preparation ---------------------------------------------------------
// One workgroup a row: thread t holds elements 4 (t + j NT) .. +3 (k <= 4 NV
// NT), so x is read once.  PRO 1: RMSNorm first; PRO 2: SwiGLU of rows of 2k
// interleaved (gate_j, up_j) values.
template <int PRO, int NT, int NV>
__global__ __launch_bounds__(NT) void gemm_split_kernel(const float* __restrict__ X, int k,
                                                        const float* __restrict__ g, float eps,
                                                        _Float16* __restrict__ XH, _Float16* __restrict__ XL,
                                                        int* __restrict__ XE, float* __restrict__ XS) {
    __shared__ float red[NT / 64], red2[NT / 64];
    const int row = blockIdx.x;
    const int k4 = k >> 2;  // k % 32 == 0
    f32x4 v[NV];
    if constexpr (PRO == 2) {
        const f32x4* x = reinterpret_cast<const f32x4*>(X + (size_t)row * 2 * k);
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
        const f32x4* x = reinterpret_cast<const f32x4*>(X + (size_t)row * k);
#pragma unroll
        for (int j = 0; j < NV; j++) {
            const int p = threadIdx.x + j * NT;
            v[j] = p < k4 ? x[p] : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
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
    // largest |x| of the row as an integer maximum of |x| bits (non-finite on top)
    uint32_t am = 0;
#pragma unroll
    for (int j = 0; j < NV; j++)
#pragma unroll
        for (int t = 0; t < 4; t++) am = max(am, abs_bits(v[j][t]));
    am = max8_u32(am);
    am = max(am, (uint32_t)dpp_i32<DPP_ROW_MIRROR>((int)am));
    am = max(am, (uint32_t)__shfl_xor((int)am, 16));
    am = max(am, (uint32_t)__shfl_xor((int)am, 32));
    uint32_t* redu = reinterpret_cast<uint32_t*>(red);
    if ((threadIdx.x & 63) == 0) redu[threadIdx.x >> 6] = am;
    __syncthreads();
    am = redu[0];
#pragma unroll
    for (int w = 1; w < NT / 64; w++) am = max(am, redu[w]);
    // e: amax * 2^-e in [2^14, 2^15); non-finite or zero rows keep e = 0
    int e = 0;
    if (am != 0 && am < 0x7F800000u) e = ilogbf(__builtin_bit_cast(float, am)) - 14;
    if (threadIdx.x == 0) XE[row] = e;
    // Thread c = t % 8 of a block's eight holds elements 4c .. 4c+3.  Threads c
    // and c ^ 4 trade halves: c < 4 ends with the block's x_hi piece g = c
    // (elements of 4c and 16 + 4c in K order), c >= 4 with the x_lo piece c - 4.
    const bool upper = (threadIdx.x & 4) != 0;
#pragma unroll
    for (int j = 0; j < NV; j++) {
        const int p = threadIdx.x + j * NT;
        _Float16 h[4], l[4];
        float bs = 0.0f;
#pragma unroll
        for (int t = 0; t < 4; t++) {
            const float s = ldexpf(v[j][t], -e);
            h[t] = (_Float16)s;
            l[t] = (_Float16)(s - (float)h[t]);
            bs += s;
        }
        const uint32_t h02 = __builtin_bit_cast(uint32_t, half2_t{h[0], h[2]});
        const uint32_t h13 = __builtin_bit_cast(uint32_t, half2_t{h[1], h[3]});
        const uint32_t l02 = __builtin_bit_cast(uint32_t, half2_t{l[0], l[2]});
        const uint32_t l13 = __builtin_bit_cast(uint32_t, half2_t{l[1], l[3]});
        const uint32_t r0 = (uint32_t)__shfl_xor((int)(upper ? h02 : l02), 4);
        const uint32_t r1 = (uint32_t)__shfl_xor((int)(upper ? h13 : l13), 4);
        const u32x4 o = upper ? u32x4{r0, l02, r1, l13} : u32x4{h02, r0, h13, r1};
        if (p < k4) {
            _Float16* dst = (upper ? XL : XH) + (size_t)row * k + (size_t)(p >> 3) * 32 + (p & 3) * 8;
            *reinterpret_cast<u32x4*>(dst) = o;
        }
        if (XS) {  // the block's f32 sum of x'
            bs = sum8_f32(bs);
            if ((threadIdx.x & 7) == 0 && p < k4) XS[(size_t)row * (k >> 5) + (p >> 3)] = bs;
        }
    }
}

// ---- GEMM --------------------------------------------------------------------
// Cache policy bits of buffer loads / stores (gfx950): nt (no stale L1 line),
// sc1 (device scope).
constexpr int CPOL_NT = 2, CPOL_SC1 = 16;

// Weight formats: Q4_0 (d (q - 8)) and Q8_0 (d q, tensor.rs:535-639).
constexpr int WF_Q4_0 = 0, WF_Q8_0 = 1;

template <int WF, int FI, int WJ, int KS>
struct TileCfg {
    static constexpr int FJ = 4;                 // weight rows of a wave: 64, four a lane
    static constexpr int NW = WJ * KS, NT = NW * 64;
    static constexpr int TJ = WJ * 64, TI = FI * 16;
    static constexpr int CB = KS;                // blocks a chunk: one a K group of waves
    // one block's codes: [wj][g][64 rows] dwords of nibbles, or (Q8_0) that twice,
    // bytes 4g .. 4g+3 and 16+4g .. 16+4g+3
    static constexpr bool BYTES = WF == WF_Q8_0;
    static constexpr int HALF = WJ * 1024;
    static constexpr int NIB_BLOCK = (BYTES ? 2 : 1) * HALF;
    static constexpr int W_BYTES = CB * NIB_BLOCK;
    static constexpr int D_BYTES = CB * TJ * 2;    // f16 d: [block][row]
    static constexpr int X_PART = 1024;          // one 16-row tile of one block, hi or lo
    static constexpr int X_BYTES = CB * (TI / 16) * 2 * X_PART;
    static constexpr int STAGE = W_BYTES + D_BYTES + X_BYTES;
    static constexpr int WWORDS = BYTES ? 9 : 5;            // dwords a weight block's loads bring
    static constexpr int WU = (TJ * CB + NT - 1) / NT;      // weight blocks a thread stages
    static constexpr int XU = (TI * CB * 4 + NT - 1) / NT;  // 16-byte pieces a thread stages, hi and lo each
    static constexpr int RED = (KS - 1) * WJ * FI * FJ * 1024;
    // three stages, or the sums at the end; the x rows' exponents behind them
    static constexpr int XE_AT = 3 * STAGE > RED ? 3 * STAGE : RED;
    static constexpr int LDS = XE_AT + TI * 4;
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

template <int WF, int FI, int WJ, int KS, bool LOCAL>
__global__ __launch_bounds__(WJ * KS * 64, 2) void gemm_tile_kernel(
    const uint8_t* __restrict__ W, int n, int nb, const void* __restrict__ XH, const void* __restrict__ XL,
    const int* __restrict__ XE, int m, float* __restrict__ Y, int accy, int full, int SR, int kbs, float* __restrict__ part,
    int* __restrict__ cnt) {
    using C = TileCfg<WF, FI, WJ, KS>;
    constexpr int CB = C::CB, FJ = 4;
    constexpr bool BYTES = C::BYTES;
    constexpr uint32_t BB = BYTES ? 34u : 18u;  // bytes a block
    static_assert(FI == 4 || FI == 8, "x tiles of a wave");
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
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
    const int kb0 = slice * kbs, kb1 = S > 1 ? min(nb, kb0 + kbs) : nb;  // this slice's blocks (kb0 a multiple of CB)

    const uint32_t k = (uint32_t)nb * 32u, row_bytes = (uint32_t)nb * BB, wbytes = (uint32_t)n * row_bytes;
    const __amdgpu_buffer_rsrc_t wrs = make_rsrc(W, wbytes);
    const __amdgpu_buffer_rsrc_t hrs = make_rsrc(XH, (uint32_t)m * k * 2u);
    const __amdgpu_buffer_rsrc_t lrs = make_rsrc(XL, (uint32_t)m * k * 2u);
    const int nchunks = (kb1 - kb0 + CB - 1) / CB;

    struct WRegs { uint32_t w[C::WU][C::WWORDS]; };
    struct XRegs { u32x4 h[C::XU], l[C::XU]; };
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
        wbase[u] = ok ? ((uint32_t)j * row_bytes + (uint32_t)(kb0 + wblk[u]) * BB) & ~3u : RSRC_OOB;
        wsel[u] = (((uint32_t)j * (uint32_t)nb + (uint32_t)wblk[u]) & 1u) ? 0x07060504u : 0x05040302u;
    }
    // the matrix may end 2 bytes into a window's last dword: that dword is read
    // 2 bytes early and shifted when stored
    const uint32_t wlast = wbytes - 4u;
    auto load_w = [&](int c, WRegs& R) {
#pragma unroll
        for (int u = 0; u < C::WU; u++) {
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
    if (tid < C::TI) xe[tid] = i0 + tid < m ? XE[i0 + tid] : 0;

    uint32_t xbase[C::XU];
#pragma unroll
    for (int u = 0; u < C::XU; u++) {
        const int idx = tid + u * C::NT, i = i0 + idx / (CB * 4), q = idx % (CB * 4);
        xbase[u] = i < m ? ((uint32_t)i * k + (uint32_t)kb0 * 32u + (uint32_t)q * 8u) * 2u : RSRC_OOB;
    }
    // part q of a chunk's x loads: unit q / 2, hi or lo
    auto load_x_part = [&](int c, XRegs& R, int q) {
        const int u = q >> 1, blk = ((tid + u * C::NT) % (CB * 4)) >> 2;
        const uint32_t off = kb0 + blk + c * CB < kb1 ? xbase[u] + (uint32_t)c * (CB * 64u) : RSRC_OOB;
        if (q & 1) R.l[u] = buf_load_b128(lrs, off);
        else R.h[u] = buf_load_b128(hrs, off);
    };
    auto load_x = [&](int c, XRegs& R) {
#pragma unroll
        for (int q = 0; q < 2 * C::XU; q++) load_x_part(c, R, q);
    };
    auto store_w = [&](int c, uint8_t* st, const WRegs& R) {
#pragma unroll
        for (int u = 0; u < C::WU; u++) {
            const int idx = tid + u * C::NT, jl = idx / CB, bl = idx % CB;
            if (!C::W_ALL && idx >= C::TJ * CB) continue;
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
    auto store_x = [&](uint8_t* st, const XRegs& R) {
        uint8_t* xs = st + C::W_BYTES + C::D_BYTES;
#pragma unroll
        for (int u = 0; u < C::XU; u++) {
            const int idx = tid + u * C::NT, il = idx / (CB * 4), q = idx % (CB * 4);
            const int slot = (q & 3) * 16 + ((il & 15) ^ (q & 7));
            uint8_t* p = xs + (((q >> 2) * (C::TI / 16) + (il >> 4)) * 2) * C::X_PART + slot * 16;
            *reinterpret_cast<u32x4*>(p) = R.h[u];
            *reinterpret_cast<u32x4*>(p + C::X_PART) = R.l[u];
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
    u32x4 nv, nv2;    // codes of the next block (nv2: Q8_0's second half)
    uint2 dd;
    half8_t wq[2][4];
    float dv[2][4];
    half8_t xh[2], xl[2];
    f32x4 p[2][FJ];
    auto read_w = [&](const uint8_t* st) {
        nv = *reinterpret_cast<const u32x4*>(st + ks * C::NIB_BLOCK + wj * 1024 + g * 256 + r * 16);
        if constexpr (BYTES)
            nv2 = *reinterpret_cast<const u32x4*>(st + ks * C::NIB_BLOCK + C::HALF + wj * 1024 + g * 256 + r * 16);
        dd = *reinterpret_cast<const uint2*>(st + C::W_BYTES + (ks * C::TJ + wj * 64 + r * 4) * 2);
    };
    auto read_x = [&](const uint8_t* st, int s) {
        const uint8_t* xb = st + C::W_BYTES + C::D_BYTES + (ks * FI + s) * 2 * C::X_PART +
                            (g * 16 + (r ^ ((ks & 1) * 4 + g))) * 16;
        xh[s & 1] = *reinterpret_cast<const half8_t*>(xb);
        xl[s & 1] = *reinterpret_cast<const half8_t*>(xb + C::X_PART);
    };
    auto conv = [&](int o, int a) {
        const uint32_t n0 = a == 0 ? nv.x : a == 1 ? nv.y : a == 2 ? nv.z : nv.w;
        if constexpr (BYTES) {
            const uint32_t n1 = a == 0 ? nv2.x : a == 1 ? nv2.y : a == 2 ? nv2.z : nv2.w;
            wq[o][a] = q8_f16(n0, n1);
        } else {
            wq[o][a] = q4_f16(n0, qc);
        }
        dv[o][a] = h2f(a == 0 ? dd.x & 0xFFFFu : a == 1 ? dd.x >> 16 : a == 2 ? dd.y & 0xFFFFu : dd.y >> 16);
        // f32 here once a block: left to itself the compiler folds the conversion
        // into every scale FMA (v_fma_mix_f32: 1,240 against 546 us, 2048 x 14336 x 4096)
        asm volatile("" : "+v"(dv[o][a]));
    };
    auto add = [&](int b, int o, int ps) {
#pragma unroll
        for (int a = 0; a < FJ; a++)
#pragma unroll
            for (int u = 0; u < 4; u++) acc[b][a][u] = fmaf(dv[o][a], p[ps][a][u], acc[b][a][u]);
    };
    // chunks the loads run ahead (FI 8: no registers for more)
    constexpr int DX = FI == 8 ? 1 : 2, DW = FI == 8 && BYTES ? 1 : 2;
    WRegs w[DW];
    XRegs x1[DX];
    uint8_t *bc = lds, *bn = lds + C::STAGE, *bf = lds + 2 * C::STAGE;  // chunk c, c + 1, free
    // chunk c; H = c % 2 (register sets by parity)
    auto chunk = [&](int c, auto u_tag) {
        constexpr int U = decltype(u_tag)::value, H = U & 1, WS = (U + 1) % DW, XS = (U + 1) % DX;
#pragma unroll
        for (int s = 0; s < FI; s++) {
            if (s + 1 < FI) read_x(bc, s + 1);
            else read_x(bn, 0);
            if (s == RB) read_w(bn);
            const f32x4 z = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int a = 0; a < FJ; a++) {
                p[s & 1][a] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xh[s & 1], wq[H][a], z, 0, 0, 0);
                p[s & 1][a] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xl[s & 1], wq[H][a], p[s & 1][a], 0, 0, 0);
            }
            add(s == 0 ? FI - 1 : s - 1, s == 0 ? H ^ 1 : H, (s & 1) ^ 1);
            if (s > RB) {
#pragma unroll
                for (int a = 0; a < FJ; a++)
                    if (a * (FI - 1 - RB) / FJ == s - 1 - RB) conv(H ^ 1, a);
            }
            if (s == 0) store_w(c + 1, bn, w[WS]);
            if (s == 1) store_x(bn, x1[XS]);
            // the loads into the freed registers, spread over the later steps (a
            // burst of them stalls the waves at issue)
            if (s == FI - 1) load_w(c + 1 + DW, w[WS]);
            if (s >= 2) {
#pragma unroll
                for (int q = 0; q < 2 * C::XU; q++)
                    if (2 + q * (FI - 2) / (2 * C::XU) == s) load_x_part(c + 1 + DX, x1[XS], q);
            }
#pragma unroll
            for (int a = 0; a < FJ; a++) {
                __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, 6, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
            if (s == RB - 1) __syncthreads();
        }
        uint8_t* t3 = bc;
        bc = bn;
        bn = bf;
        bf = t3;
    };
    // chunks 0 .. DW - 1 of W and 0 .. DX - 1 of x first, then on to DW / DX
    // once chunk 0 is stored
#pragma unroll
    for (int q = 0; q < DW; q++) {
        load_w(q, w[q]);
    }
#pragma unroll
    for (int q = 0; q < DX; q++) load_x(q, x1[q]);
    store_w(0, bc, w[0]);
    store_x(bc, x1[0]);
    load_w(DW, w[0]);
    load_x(DX, x1[0]);
    __syncthreads();
    read_w(bc);
    read_x(bc, 0);
#pragma unroll
    for (int a = 0; a < FJ; a++) {
        conv(0, a);
        dv[1][a] = 0.0f;
        p[1][a] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    }
    // (chunks past the slice's end: zeros; no branch, so that the waits stay exact)
    for (int c = 0; c < nchunks; c += 2) {
        chunk(c, std::integral_constant<int, 0>{});
        chunk(c + 1, std::integral_constant<int, 1>{});
    }
    add(FI - 1, 1, 1);

    // lane (g, r) holds y[i = 4 g + u][j = 4 r .. 4 r + 3] of 16-row tile b
    auto store_rows = [&](int b, const f32x4 (&v4)[FJ]) {
        const int j = j0 + wj * 64 + r * 4;
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int i = i0 + b * 16 + g * 4 + u;
            if (i >= m) continue;
            const int e = xe[i - i0];
            f32x4 v = {ldexpf(v4[0][u], e), ldexpf(v4[1][u], e), ldexpf(v4[2][u], e), ldexpf(v4[3][u], e)};
            float* yp = Y + (size_t)i * n + j;
            // accy: y += the product (the residual add, one rounding as x + y)
            if (j + 3 < n && (n & 3) == 0) {
                if (accy) v = *reinterpret_cast<const f32x4*>(yp) + v;
                *reinterpret_cast<f32x4*>(yp) = v;
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
    constexpr int FO = FI / KS;
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

// x split of one product in the scratch (gemm_tiles_scratch_bytes(m, k)).
struct XSplit {
    _Float16 *h, *l;
    int* e;
    float* s;  // x' sums of each block, or NULL
};
XSplit x_split_at(void* scratch, size_t m, size_t k, bool sums) {
    const size_t xb = (m * k * 2 + 255) & ~(size_t)255, eb = (m * 4 + 255) & ~(size_t)255;
    uint8_t* p = reinterpret_cast<uint8_t*>(scratch);
    return {reinterpret_cast<_Float16*>(p), reinterpret_cast<_Float16*>(p + xb), reinterpret_cast<int*>(p + 2 * xb),
            sums ? reinterpret_cast<float*>(p + 2 * xb + eb) : nullptr};
}

// One tile shape: 64 WJ weight rows x 16 FI x rows, KS wave groups sharing
// each chunk's blocks.
template <int WF, int FI, int WJ, int KS>
hipError_t launch_tile_cfg(const uint8_t* w, int n, int nb, const XSplit& x, int m, float* y, int accy,
                           const TilePlan& p, float* part, int* cnt, hipStream_t s) {
    using C = TileCfg<WF, FI, WJ, KS>;
    static_assert(C::LDS <= 160 * 1024, "LDS per workgroup");
    const bool local = p.S > 1 && xcd_round_robin(s);
    auto kern = local ? gemm_tile_kernel<WF, FI, WJ, KS, true> : gemm_tile_kernel<WF, FI, WJ, KS, false>;
    if (C::LDS > 65536) {
        static const hipError_t e[2] = {
            hipFuncSetAttribute((const void*)gemm_tile_kernel<WF, FI, WJ, KS, false>,
                                hipFuncAttributeMaxDynamicSharedMemorySize, C::LDS),
            hipFuncSetAttribute((const void*)gemm_tile_kernel<WF, FI, WJ, KS, true>,
                                hipFuncAttributeMaxDynamicSharedMemorySize, C::LDS)};  // once a process
        if (e[local] != hipSuccess) return e[local];
    }
    unsigned rest = (unsigned)((n + C::TJ - 1) / C::TJ) * (unsigned)((m + C::TI - 1) / C::TI) - (unsigned)p.full;
    if (local) rest = (rest + 7) / 8 * 8;
    launch_kernel(kern, dim3((unsigned)p.full + rest * (unsigned)p.S), dim3(C::NT), (size_t)C::LDS, s, w, n, nb, x.h, x.l, x.e, m, y,
                  accy, p.full, p.S, p.kbs, part, cnt);
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
TilePlan tile_plan(size_t m, size_t n, size_t nb, bool can_split) {
    const size_t round = std::max(8, device_cu_count() / 8 * 8);
    TilePlan best{};
    double best_us = 1e30;
    for (int c = 0; c < 4; c++) {
        const TileShape& t = TILE_SHAPES[c];
        const size_t tiles = ((n + t.tj - 1) / t.tj) * ((m + t.ti - 1) / t.ti);
        const size_t unit = 2 * (size_t)t.ks;  // the main loop's step: two chunks
        const size_t full = tiles / round * round, rest = tiles - full;
        const double whole = nb * t.us_block + 6.0;  // us a round of unsplit tiles
        for (size_t S = 1; S <= 16; S++) {
            const size_t kbs = ((nb + S - 1) / S + unit - 1) / unit * unit;
            double us = (double)(full / round) * whole;
            if (S == 1) {
                us += rest ? whole : 0.0;
            } else {
                if (!can_split || rest * S > round) break;
                if ((S - 1) * kbs >= nb) continue;  // (an empty slice)
                const size_t bytes = S * t.tj * t.ti * sizeof(float);
                if (rest == 0 || rest * bytes > GEMM_PART_BYTES) break;
                us += kbs * t.us_block + 6.0 + 2.0 + (double)bytes / 40e3;
            }
            if (us < best_us) best_us = us, best = {c, (int)(S == 1 ? tiles : full), (int)S, (int)kbs};
        }
    }
    return best;
}

template <int PRO>
hipError_t launch_split(const float* x, size_t m, size_t k, const float* g, float eps, const XSplit& o, hipStream_t s) {
    // 256 threads hold 4096 elements of a row, 1024 threads 16384
    if (k <= 4096)
        launch_kernel(gemm_split_kernel<PRO, 256, 4>, dim3((unsigned)m), dim3(256), 0, s, x, (int)k, g, eps, o.h, o.l,
                      o.e, o.s);
    else
        launch_kernel(gemm_split_kernel<PRO, 1024, 4>, dim3((unsigned)m), dim3(1024), 0, s, x, (int)k, g, eps, o.h,
                      o.l, o.e, o.s);
    return hipGetLastError();
}

}  // namespace

// The small-tile kernel of gemm.hip keeps short products over small matrices:
// its 16 x 32 tiles reach all CUs without a split over K, and its code is
// smaller (us, here against there: Q4_0 100 x 512 x 992 10.7 / 9.1, 200 x 2048 x
// 992 13.6 / 12.7, 100 x 2048 x 2048 14.2 / 15.8, 100 x 64 x 4096 13.4 / 17.3;
// Q8_0 100 x 512 x 992 11.0 / 8.9, 1000 x 512 x 992 17.5 / 16.4, 333 x 4096 x 992
// 19.5 / 25.7, 17 x 4096 x 4096 17.9 / 17.2, 33 x 4096 x 4096 18.6 / 24.4).
bool gemm_tile_takes(WType t, size_t m, size_t n, size_t k) {
    if (k > GEMM_TILE_MAX_K) return false;
    if (t == WType::Q4_0) return m > GEMM_XTILE_M && !(m <= 256 && k <= 2048 && n * k <= (size_t)1 << 22);
    if (t != WType::Q8_0 || m < KQ_GEMM_MIN_M) return false;
    if (k <= 2048 && (m * n <= (size_t)1 << 19 || (m <= 256 && n * k <= (size_t)1 << 23))) return false;
    return m > 24 || n * k > (size_t)1 << 24;
}

size_t gemm_part_bytes(size_t m, size_t n, size_t k) {
    const TilePlan p = tile_plan(m, n, k / QK, true);
    const TileShape& t = TILE_SHAPES[p.cfg];
    const size_t rest = ((n + t.tj - 1) / t.tj) * ((m + t.ti - 1) / t.ti) - (size_t)p.full;
    return rest * p.S * t.tj * t.ti * sizeof(float);
}

template <int WF>
static hipError_t launch_tile_wf(const uint8_t* w, int n, int nb, const XSplit& x, int m, float* y, int accy,
                                 float* part, int* cnt, hipStream_t s) {
    const TilePlan p = tile_plan(m, n, nb, part != nullptr && cnt != nullptr);
    switch (p.cfg) {
        case 0: return launch_tile_cfg<WF, 8, 4, 2>(w, n, nb, x, m, y, accy, p, part, cnt, s);
        case 1: return launch_tile_cfg<WF, 4, 4, 2>(w, n, nb, x, m, y, accy, p, part, cnt, s);
        case 2: return launch_tile_cfg<WF, 4, 2, 4>(w, n, nb, x, m, y, accy, p, part, cnt, s);
        default: return launch_tile_cfg<WF, 4, 1, 4>(w, n, nb, x, m, y, accy, p, part, cnt, s);
    }
}

hipError_t launch_gemm_tile(WType t, const uint8_t* w, size_t n, size_t k, const float* x, size_t m, float* y,
                            void* scratch, float* part, int* cnt, int pro, const float* g, float eps, bool accumulate,
                            hipStream_t s) {
    if (k == 0 || !gemm_tile_takes(t, m, n, k)) return hipErrorInvalidValue;
    const XSplit xo = x_split_at(scratch, m, k, false);
    const hipError_t e = pro == 1   ? launch_split<1>(x, m, k, g, eps, xo, s)
                         : pro == 2 ? launch_split<2>(x, m, k, g, eps, xo, s)
                                    : launch_split<0>(x, m, k, g, eps, xo, s);
    if (e != hipSuccess) return e;
    const int ni = (int)n, nb = (int)(k / QK), mi = (int)m, acc = accumulate ? 1 : 0;
    return t == WType::Q4_0 ? launch_tile_wf<WF_Q4_0>(w, ni, nb, xo, mi, y, acc, part, cnt, s)
                            : launch_tile_wf<WF_Q8_0>(w, ni, nb, xo, mi, y, acc, part, cnt, s);
}

}  // namespace rdl
