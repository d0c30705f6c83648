// gemm_split.hip -- fp32 GEMM on the bf16 matrix cores: every operand split into
// three bf16 parts (common.h), six MFMAs per product step, fp32 accumulators.
//
// Row-major C = alpha * op(A) op(B) + beta * C (+ bias per row).  One workgroup
// = 8 waves = a 256 x 128 tile of C, each wave 64 x 64 of it (2 x 2 MFMA blocks: a
// block's operand is read from LDS once for two of them), K in steps of 32.  A
// step's operands are loaded two steps ahead into registers, split, and stored to
// double-buffered LDS as 16-byte units of 8 consecutive k of one row of A or
// column of B, which is what an MFMA lane takes: one barrier per step.
//   K-contiguous operand (A, or B transposed): a thread loads 8 k of a row (two
//     16-byte loads; 4 threads cover the row's step).
//   K-strided operand (A transposed, or B): a thread loads 8 k of one column
//     (eight 4-byte loads, each a run over the lanes), so the transposition costs
//     no store.
// The operands are taken times 2^24 and the results times 2^-48, which moves the
// range that three bf16 parts hold exactly to all of fp32's small numbers; a sum that
// this takes past the largest float is formed again in plain fp32 (below).
// The matrix cores' sums round a little towards -infinity (2e-8 of a result's rms
// on average, which a sum over thousands of rows of C would show): half of the rows
// and columns, by the parity of their index's bits, are negated, so that half of
// the results are formed as their negatives and what is left cancels in sums over
// rows or columns of C.  The small part products have accumulators of their own.
// A non-finite element makes its row's or column's results NaN; the wave that has one
// forms its 64 x 64 again on the fp32 matrix cores, so infinities come out as before.
//
// Few tiles and a long K: the K range is split over workgroups, their partial
// tiles go to the workspace and a second kernel sums them in order.
//
// Bound by the MFMAs and the splitting VALU work beside them, at a shader clock that
// falls with the load: 4096^3 at 1.18 PFLOP/s of MFMAs, where a large library product
// in bf16 reaches 1.25.  Against the vendor library's fp32 kernels (us): 8192 x 3072 x
// 768 342 -> 253, 8192 x 768 x 3072 308 -> 249, 768 x 3072 x 8192 300 -> 220, 4096^3
// 917 -> 701, 2905 x 2240 x 560 115 -> 55, 3309 x 664 x 2656 114 -> 85; the distance of
// the MLP's outputs to 64 bits 1.7e-6 -> 4e-7.  Two fp16 parts with a scale per row
// and column and three MFMAs took 185, 177, 159, 466, 52 and 73, but lost the bits
// of what lies far below its row's largest (2e-3 of the result where features and
// their weights are scaled against each other by 2^13).
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "common.h"
#include "gemm_split_rule.h"
#include "kernels.h"

namespace inf {

namespace {

constexpr int kBM = kSplitBM, kBN = kSplitBN, kBK = kSplitBK, kNT = 512;
constexpr int kKG = kBK / 8;  // 8-k units per row and step
constexpr float kUp = 0x1p24f, kDown = 0x1p-48f;  // the operands' factor, and what takes it from a result

// v, negated where i has an odd number of bits
__device__ __forceinline__ float with_parity(float v, uint32_t i) {
    return __uint_as_float(__float_as_uint(v) ^ (uint32_t)__popc(i) << 31);
}

struct GemmSplitParams {
    const float* A;
    const float* B;
    float* C;
    const float* bias;
    float* part;              // split K: [ksplit, M, N] partial products
    int M, N, K;
    int64_t lda, ldb, ldc, sa, sb, sc;
    float alpha, beta;
    int tiles_m, tiles_n;
    int ksplit, kchunk;       // K range per split, a multiple of kBK
    int items;                // tiles x K ranges x batch
};

// One operand's staging: rows row0 .. row0 + ROWS - 1, U units of 8 k per thread
// (NT = ROWS * 4 / U threads).
template <bool KC, int ROWS, int U>
struct Stage {
    static constexpr int US = ROWS + 4;  // units per 8-k group in LDS (64 bytes of padding)
    using Raw = f32x4[U][2];
    Raw raw[2];          // two steps' loads
    float sgn[U];        // 2^kUp or -2^kUp, the unit's row's factor
    const float* base;   // KC: row row0, k 0; else: k 0, column row0
    int64_t ld;
    int rows, row_a;     // rows of the operand in this tile; this thread's first row
    int kg;              // this thread's first 8-k group
    uint32_t voff;

    __device__ __forceinline__ void init(const float* op, int64_t ld_, int row0, int rows_total, int tid) {
        const int lane = tid & 63, wave = tid >> 6;
        ld = ld_;
        rows = min(rows_total - row0, ROWS);
        if constexpr (KC) {  // 16 rows a wave, 4 neighbouring lanes a row (128 bytes)
            base = op + (int64_t)row0 * ld;
            row_a = 16 * wave + (lane >> 2);
            kg = lane & 3;
            voff = (uint32_t)(((int64_t)row_a * ld + 8 * kg) * 4);
        } else {
            base = op + row0;
            row_a = U == 2 ? 32 * wave + (lane & 31) : 16 * wave + (lane & 15);
            kg = U == 2 ? lane >> 5 : lane >> 4;
            voff = (uint32_t)(((int64_t)(8 * kg) * ld + row_a) * 4);
        }
#pragma unroll
        for (int i = 0; i < U; ++i) sgn[i] = with_parity(kUp, KC ? row_a + ROWS / 2 * i : row_a);
    }
    // k0 .. k0 + 31 below kend; elements outside read as zeros.
    __device__ __forceinline__ void load(Raw& r, int k0, int kend) const {
        const int ks = min(kend - k0, kBK);
        if constexpr (KC) {
            const uint32_t bytes = ks > 0 ? (uint32_t)(((int64_t)(rows - 1) * ld + ks) * 4) : 0u;
            const auto rs = buffer_rsrc(base + k0, bytes);
            const uint32_t end = 0x40000000u;  // past the end of every resource
            const uint32_t v = 8 * kg < ks ? voff : end, v2 = 8 * kg + 4 < ks ? voff + 16 : end;
#pragma unroll
            for (int i = 0; i < U; ++i) {
                const uint32_t so = (uint32_t)((int64_t)(ROWS / 2 * i) * ld * 4);
                r[i][0] = buffer_ld4(rs, v, so);
                r[i][1] = buffer_ld4(rs, v2, so);
            }
        } else {
            const uint32_t bytes = ks > 0 ? (uint32_t)(((int64_t)(ks - 1) * ld + rows) * 4) : 0u;
            const auto rs = buffer_rsrc(base + (int64_t)k0 * ld, bytes);
#pragma unroll
            for (int i = 0; i < U; ++i)
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    r[i][e >> 2][e & 3] = buffer_ld1(rs, voff, (uint32_t)((int64_t)(16 * i + e) * ld * 4));
        }
    }
    // Split the loaded step into LDS (no branch, so that it can be scheduled between
    // the MFMAs of the step before: 3-5% of the time).
    __device__ __forceinline__ void store(const Raw& r, bf16x8 (&L)[3][kKG][US]) const {
#pragma unroll
        for (int i = 0; i < U; ++i) {
            const Bf3x8 h = split3(r[i][0] * sgn[i], r[i][1] * sgn[i]);
            const int g = KC ? kg : kg + 2 * i, row = KC ? row_a + ROWS / 2 * i : row_a;
            L[0][g][row] = h.h;
            L[1][g][row] = h.m;
            L[2][g][row] = h.l;
        }
    }
};

}  // namespace

template <bool AKC, bool BKC>
__global__ __launch_bounds__(kNT, 2) void gemm_split_kernel(GemmSplitParams p) {
    using StageA = Stage<AKC, kBM, 2>;
    using StageB = Stage<BKC, kBN, 1>;
    __shared__ bf16x8 Ua[2][3][kKG][StageA::US];  // [buffer][part][8-k group][row]
    __shared__ bf16x8 Ub[2][3][kKG][StageB::US];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31;
    const int g = lane >> 5;
    const int wm = wave >> 1, wn = wave & 1;

    // Consecutive workgroups go to the 8 XCDs in turn: each XCD takes an even share
    // of the work as one run of tiles (of one K range, then the next), so that it
    // finds their operand panels in its own L2.
    const int n_tiles = p.tiles_m * p.tiles_n, xcd = blockIdx.x % 8;
    const int item = (int)((int64_t)p.items * xcd / 8) + (int)(blockIdx.x / 8);
    if (item >= (int)((int64_t)p.items * (xcd + 1) / 8)) return;
    const int tile = item % n_tiles, split = item / n_tiles % p.ksplit, batch = item / n_tiles / p.ksplit;
    const int m0 = tile / p.tiles_n * kBM, n0 = tile % p.tiles_n * kBN;
    const int kb = split * p.kchunk, ke = min(p.K, kb + p.kchunk);
    const int nt = (ke - kb + kBK - 1) / kBK;
    const float* A = p.A + batch * p.sa;
    const float* B = p.B + batch * p.sb;
    float* C = p.C + batch * p.sc;

    StageA sa;
    StageB sb;
    sa.init(A, p.lda, m0, p.M, tid);
    sb.init(B, p.ldb, n0, p.N, tid);

    f32x16 acc[2][2], lo[2][2];  // the main part products, and the small ones apart: their roundings stay off the result's last bits
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = lo[i][j] = f32x16{};

    sa.load(sa.raw[0], kb, ke);
    sb.load(sb.raw[0], kb, ke);
    sa.load(sa.raw[1], kb + kBK, ke);
    sb.load(sb.raw[1], kb + kBK, ke);
    sa.store(sa.raw[0], Ua[0]);
    sb.store(sb.raw[0], Ub[0]);
    __syncthreads();

    // Step t computes on buffer BUF = t % 2; step t + 1, loaded in the previous
    // step, is split into the other buffer, and step t + 2's loads go out.
    auto step = [&](int t, auto buf_c) {
        constexpr int BUF = decltype(buf_c)::value;
        sa.load(sa.raw[BUF], kb + (t + 2) * kBK, ke);
        sb.load(sb.raw[BUF], kb + (t + 2) * kBK, ke);
#pragma unroll
        for (int kk = 0; kk < kBK / 16; ++kk) {
            Bf3x8 a[2], b[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int ra = 64 * wm + 32 * i + l32, rb = 64 * wn + 32 * i + l32;
                a[i] = Bf3x8{Ua[BUF][0][2 * kk + g][ra], Ua[BUF][1][2 * kk + g][ra], Ua[BUF][2][2 * kk + g][ra]};
                b[i] = Bf3x8{Ub[BUF][0][2 * kk + g][rb], Ub[BUF][1][2 * kk + g][rb], Ub[BUF][2][2 * kk + g][rb]};
            }
            // four independent accumulators in turn
            auto product = [&](f32x16 (&c)[2][2], auto pa, auto pb) {
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int j = 0; j < 2; ++j) c[i][j] = mfma32x32x16bf16(a[i].*pa, b[j].*pb, c[i][j]);
            };
            product(lo, &Bf3x8::l, &Bf3x8::h);
            product(lo, &Bf3x8::h, &Bf3x8::l);
            product(lo, &Bf3x8::m, &Bf3x8::m);
            product(lo, &Bf3x8::m, &Bf3x8::h);
            product(lo, &Bf3x8::h, &Bf3x8::m);
            product(acc, &Bf3x8::h, &Bf3x8::h);
        }
        sa.store(sa.raw[BUF ^ 1], Ua[BUF ^ 1]);
        sb.store(sb.raw[BUF ^ 1], Ub[BUF ^ 1]);
        __syncthreads();
    };
    using B0 = std::integral_constant<int, 0>;
    using B1 = std::integral_constant<int, 1>;
    for (int t = 0; t < nt; t += 2) {
        step(t, B0{});
        if (t + 1 < nt) step(t + 1, B1{});
    }

    // ---- epilogue ------------------------------------------------------------------
    float chk = 0.f;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            acc[i][j] += lo[i][j];
#pragma unroll
            for (int r = 0; r < 16; ++r) chk = fmaf(acc[i][j][r], 0.f, chk);
        }
    // A result that is not finite: an infinity or NaN in its operands, or a sum that only
    // their factors took past the largest float.  The wave's 64 x 64 results are formed
    // again in plain fp32, straight from memory.
    const bool plain = __any(chk != 0.f);
    if (plain) {
        const float* ap[2];
        const float* bp[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {  // null: zeros
            const int m = m0 + 64 * wm + 32 * i + l32, n = n0 + 64 * wn + 32 * i + l32;
            ap[i] = m < p.M ? A + (AKC ? (int64_t)m * p.lda : m) : nullptr;
            bp[i] = n < p.N ? B + (BKC ? (int64_t)n * p.ldb : n) : nullptr;
#pragma unroll
            for (int j = 0; j < 2; ++j) acc[i][j] = f32x16{};
        }
        auto load4 = [&](const float* q, int64_t ld, bool kc, int k) {  // k .. k + 3 below ke
            f32x4 v = {0.f, 0.f, 0.f, 0.f};
            if (q && k < ke) {
                if (kc) {  // (ke is a multiple of 4 then)
                    v = *reinterpret_cast<const f32x4*>(q + k);
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[e] = k + e < ke ? q[(int64_t)(k + e) * ld] : 0.f;
                }
            }
            return v;
        };
#pragma unroll 1
        for (int k = kb + 4 * g; k - 4 * g < ke; k += 8) {
            f32x4 a[2], b[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                a[i] = load4(ap[i], p.lda, AKC, k);
                b[i] = load4(bp[i], p.ldb, BKC, k);
            }
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int j = 0; j < 2; ++j) acc[i][j] = mfma32x32x2(a[i][e], b[j][e], acc[i][j]);
        }
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int nl = 64 * wn + 32 * j + l32, n = n0 + nl;
        const float bias = p.bias && n < p.N && p.ksplit == 1 ? p.bias[n] : 0.f;
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int ml = 64 * wm + 32 * i + 8 * (r >> 2) + 4 * g + (r & 3), m = m0 + ml;
                float v = acc[i][j][r] * (plain ? 1.f : with_parity(kDown, ml ^ nl));
                if (m < p.M && n < p.N) {
                    if (p.ksplit > 1) {
                        p.part[((int64_t)split * p.M + m) * p.N + n] = v;
                    } else {
                        float* c = C + (int64_t)m * p.ldc + n;
                        v = fmaf(v, p.alpha, bias);
                        *c = p.beta != 0.f ? fmaf(p.beta, *c, v) : v;
                    }
                }
            }
    }
}

// C from the partial products of a split K, summed in order.
__global__ __launch_bounds__(256) void gemm_split_reduce_kernel(GemmSplitParams p) {
    const int64_t mn = (int64_t)p.M * p.N;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < mn; i += (int64_t)gridDim.x * 256) {
        float v = 0.f;
        for (int s = 0; s < p.ksplit; ++s) v += p.part[s * mn + i];
        const uint32_t m = (uint32_t)(i / (uint32_t)p.N), n = (uint32_t)(i - (int64_t)m * p.N);
        float* c = p.C + (int64_t)m * p.ldc + n;
        v = fmaf(v, p.alpha, p.bias ? p.bias[n] : 0.f);
        *c = p.beta != 0.f ? fmaf(p.beta, *c, v) : v;
    }
}

// Whether the kernel can read the operands: a K-contiguous one 8 elements at a time in
// halves (16-byte rows).  (alpha = 0 must not read operands that may hold infinities.)
static bool split_reads(const GemmArgs& g) {
    if (g.bf16 || g.alpha == 0.f) return false;
    auto rows16 = [](const void* p, int64_t ld, int64_t stride) {
        return reinterpret_cast<uintptr_t>(p) % 16 == 0 && ld % 4 == 0 && stride % 4 == 0;
    };
    if (!g.ta && !rows16(g.A, g.lda, g.batch > 1 ? g.sa : 0)) return false;
    if (g.tb && !rows16(g.B, g.ldb, g.batch > 1 ? g.sb : 0)) return false;
    return true;
}

int launch_gemm_split(const GemmArgs& g, hipStream_t s, bool* taken) {
    *taken = false;
    if (!split_reads(g)) return 0;
    const bool ws_ok = reinterpret_cast<uintptr_t>(g.ws) % 16 == 0;
    const int ks = gemm_split_ranges(g.ta, g.tb, g.M, g.N, g.K, g.batch, g.lda, g.ldb, ws_ok ? g.ws_bytes : 0);
    if (!ks) return 0;
    GemmSplitParams p{};
    p.A = (const float*)g.A;
    p.B = (const float*)g.B;
    p.C = (float*)g.C;
    p.bias = (const float*)g.bias;
    p.M = (int)g.M;
    p.N = (int)g.N;
    p.K = (int)g.K;
    p.lda = g.lda;
    p.ldb = g.ldb;
    p.ldc = g.ldc;
    p.sa = g.batch > 1 ? g.sa : 0;
    p.sb = g.batch > 1 ? g.sb : 0;
    p.sc = g.batch > 1 ? g.sc : 0;
    p.alpha = g.alpha;
    p.beta = g.beta;
    p.tiles_m = (int)((g.M + kBM - 1) / kBM);
    p.tiles_n = (int)((g.N + kBN - 1) / kBN);
    const int64_t tiles = (int64_t)p.tiles_m * p.tiles_n * g.batch;
    const int nk = (p.K + kBK - 1) / kBK;
    p.kchunk = (nk + ks - 1) / ks * kBK;
    p.ksplit = (p.K + p.kchunk - 1) / p.kchunk;
    p.part = (float*)g.ws;
    p.items = (int)(tiles * p.ksplit);
    const dim3 grid((unsigned)((p.items + 7) / 8 * 8)), block(kNT);
    if (!g.ta && !g.tb) hipLaunchKernelGGL((gemm_split_kernel<true, false>), grid, block, 0, s, p);
    else if (!g.ta) hipLaunchKernelGGL((gemm_split_kernel<true, true>), grid, block, 0, s, p);
    else if (!g.tb) hipLaunchKernelGGL((gemm_split_kernel<false, false>), grid, block, 0, s, p);
    else hipLaunchKernelGGL((gemm_split_kernel<false, true>), grid, block, 0, s, p);
    if (p.ksplit > 1)
        hipLaunchKernelGGL(gemm_split_reduce_kernel, dim3((unsigned)std::min<int64_t>((g.M * g.N + 255) / 256, 2048)),
                           dim3(256), 0, s, p);
    *taken = true;
    return (int)hipGetLastError();
}

}  // namespace inf
