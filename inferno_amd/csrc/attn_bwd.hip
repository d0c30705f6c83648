// attn_bwd.hip -- fused causal attention backward for gfx950 (recompute).
//
// Kernel 1 (bwd_pre): delta[i] = sum_d dO[i,d] * O[i,d] per query row (the
// row dot that SoftmaxBackward computes as sum_j dP_ij P_ij), zeroes the
// fp32 dQ accumulator and, for fp32, leaves the largest |q| and |dO| of its
// rows.  (The bf16 main kernel at D <= 64 forms delta itself, and then this
// pass only zeroes.)
//
// Kernel 2 (bwd_main, fp32): its products run on the fp16 matrix cores, every
// operand split into two fp16 parts (common.h), three MFMAs per product step.
// One workgroup = 8 waves = 4 pairs, each pair with 64 keys (or 32) of one
// (b, h).  In a pair, wave 0 (role 0) holds the keys' K operand and dV^T
// accumulators in VGPRs, wave 1 (role 1) their V operand and dK^T accumulators,
// 64 + 64 registers each at D = 64 and 128, so two waves fit a SIMD, one of each
// role.  dK and dV are written exactly once, with no atomics.  The workgroup
// walks query tiles of 32 rows, split into LDS once for all waves; per tile,
// in three phases with a barrier after each:
//
//   A  role 0: S = Q K^T, P = exp2(S c - lse log2e) (masked entries exactly 0),
//      P handed to role 1 through LDS;   role 1: dP = dO V^T
//   B  role 0: dV^T += dO^T P;   role 1: dS = P (dP - delta), split, to LDS
//   C  role 0: dQ tile += dS K over the workgroup's keys, fp32 atomics into the
//      global accumulator;   role 1: dK^T += Q^T dS;   both: the next tile
//
// Keys lie on the lane axis in S, dP, dV^T and dK^T, so P and dS are operands
// straight from the accumulators; the transposed operands (dO^T, Q^T, dS) are
// transposed LDS reads, and K^T for dQ is staged transposed once.  S is formed
// in the forward's order, to the same bits, so P is consistent with the LSE.
// Bound by the phases' latency: a tile's MFMAs take 3840 of its 8100 (D = 128)
// or 9100 (D = 64) cycles per SIMD, and at config 4 the fp16 MFMAs run at a
// 2.0 GHz shader clock.  The backward call against the fp32-MFMA kernel that this
// one replaced (us): config 2 308 -> 163, config 4 5980 -> 2170, B8 H12 T1024 D32
// 178 -> 128, B1 H12 T333 D64 34 -> 27.
//
// bf16 inputs use the bf16-MFMA main kernel (attn_bwd_bf16.hip) between the
// same pre kernel and a final bwd_cvt that turns the fp32 dQ accumulator into
// bf16 dq.
#include <type_traits>

#include <algorithm>
#include <array>
#include <cmath>
#include <map>
#include <mutex>
#include <vector>

#include "bwd_split.h"
#include "common.h"
#include "kernels.h"

namespace inf {

// Batch, head and position of row `row` of the [B, H, Tq] rows: 32-bit
// divisions when the row count fits (every practical shape), as 64-bit ones
// cost tens of instructions per thread in these memory-bound passes.
__device__ __forceinline__ void bwd_row_split(const BwdParams& p, int64_t rows, int64_t row, int64_t& b, int64_t& h,
                                              int64_t& i) {
    if (rows <= 0xffffffffLL) {
        const uint32_t r = (uint32_t)row, bh = r / (uint32_t)p.Tq;
        i = r - bh * (uint32_t)p.Tq;
        b = bh / (uint32_t)p.H;
        h = bh - (uint32_t)b * (uint32_t)p.H;
    } else {
        const int64_t bh = row / p.Tq;
        i = row % p.Tq;
        b = bh / p.H;
        h = bh % p.H;
    }
}

// delta = rowsum(dO * O) per query row, and the zeroing of the fp32 dQ
// accumulator and the split plan's arrival counters.  Each thread takes one
// 16-byte chunk of O and dO (4 fp32 or 8 bf16 elements; TPR threads per row)
// and the row's threads sum their products with DPP moves.
template <int D, typename E>
constexpr int bwd_pre_tpr() { return D / (16 / (int)sizeof(E)); }
template <int D, typename E>
constexpr int bwd_pre_rows_per_block() { return 256 / bwd_pre_tpr<D, E>(); }

template <int D, typename E>
__global__ __launch_bounds__(256) void bwd_pre_kernel(BwdParams p) {
    constexpr int VEC = 16 / (int)sizeof(E);   // elements per 16-byte chunk
    constexpr int TPR = bwd_pre_tpr<D, E>();    // threads per row
    constexpr int RPB = bwd_pre_rows_per_block<D, E>();
    const int tid = threadIdx.x;
    const int c = tid % TPR;
    const int64_t rows = (int64_t)p.B * p.H * p.Tq;
    // fp32: p.n_amax workgroups per head; bf16: flat over the rows
    int64_t row, b, h, i;
    bool in;
    if constexpr (sizeof(E) == 4) {
        const unsigned bh = blockIdx.x / (unsigned)p.n_amax;
        i = (int64_t)(blockIdx.x % (unsigned)p.n_amax) * RPB + tid / TPR;
        b = bh / (unsigned)p.H;
        h = bh % (unsigned)p.H;
        in = i < p.Tq;
        row = (int64_t)bh * p.Tq + i;
    } else {
        row = (int64_t)blockIdx.x * RPB + tid / TPR;
        in = row < rows;
        if (in) bwd_row_split(p, rows, row, b, h, i);
    }
    float s = 0.f, aq = 0.f, ad = 0.f;
    if (in) {
        if (p.pre_delta) {
            const E* po = (const E*)p.o + b * p.so.b + h * p.so.h + i * p.so.t + VEC * c;
            const E* pd = (const E*)p.dout + b * p.sdo.b + h * p.sdo.h + i * p.sdo.t + VEC * c;
            if constexpr (sizeof(E) == 4) {
                const f32x4 o4 = ld4(po), d4 = ld4(pd);
                s = o4[0] * d4[0] + o4[1] * d4[1] + o4[2] * d4[2] + o4[3] * d4[3];
                const f32x4 q4 = ld4((const E*)p.q + b * p.sq.b + h * p.sq.h + i * p.sq.t + VEC * c);
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    aq = fmaxf(aq, finite_abs(q4[k]));
                    ad = fmaxf(ad, finite_abs(d4[k]));
                }
            } else {
                const u16x8 o8 = *reinterpret_cast<const u16x8*>(po);
                const u16x8 d8 = *reinterpret_cast<const u16x8*>(pd);
#pragma unroll
                for (int k = 0; k < 8; ++k) s = fmaf(bf16_to_f32(o8[k]), bf16_to_f32(d8[k]), s);
            }
        }
        if (!p.dq_direct) {
            f32x4* acc = reinterpret_cast<f32x4*>(p.dq_acc + b * p.sacc.b + h * p.sacc.h + i * p.sacc.t + VEC * c);
#pragma unroll
            for (int k = 0; k < VEC / 4; ++k) acc[k] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
    }
    // (p.pre_delta is uniform: the whole grid takes or skips the exchange)
    if (p.pre_delta) {
        s = group_sum<TPR>(s);
        if (in && c == 0) p.delta[row] = s;
    }
    if constexpr (sizeof(E) == 4) {
        __shared__ float red[2][4];
        aq = wave_max(aq);
        ad = wave_max(ad);
        if ((tid & 63) == 0) {
            red[0][tid >> 6] = aq;
            red[1][tid >> 6] = ad;
        }
        __syncthreads();
        if (tid < 2)
            p.amax[(int64_t)blockIdx.x * 2 + tid] =
                fmaxf(fmaxf(red[tid][0], red[tid][1]), fmaxf(red[tid][2], red[tid][3]));
    }
    if (blockIdx.x == 0)
        for (int i = tid; i < p.n_split * p.B * p.H; i += 256) p.counters[i] = 0u;
}

// bwd_pre without delta (the bf16 main kernel at D <= 64 forms it): the fp32
// dQ accumulator is one dense [B, H, Tq, D] block, so it is cleared as a flat
// array (16-byte stores over a grid-stride loop), with the split plan's
// arrival counters.
__global__ __launch_bounds__(256) void bwd_zero_kernel(BwdParams p) {
    const int64_t n4 = (int64_t)p.B * p.H * p.Tq * p.D / 4;
    f32x4* acc = reinterpret_cast<f32x4*>(p.dq_acc);
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n4; i += (int64_t)gridDim.x * 256)
        acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (blockIdx.x == 0)
        for (int i = threadIdx.x; i < p.n_split * p.B * p.H; i += 256) p.counters[i] = 0u;
}

// KP: keys per pair of waves (32 at D = 128, else 32 or 64)
template <int D, int KP>
struct BwdTile {
    static constexpr int BK = 4 * KP;              // keys per workgroup
    // Q / dO row stride in LDS (fp16 elements): row reads want an odd number of
    // 16-byte units, transposed reads the 32-byte windows of 4 rows in disjoint banks
    static constexpr int QS = D == 128 ? 152 : D == 64 ? 72 : 56;
    static constexpr int SS = 36;                  // dS row stride (queries of one key, fp16 elements)
};
constexpr float kBwdPBits = 14.f, kBwdPInv = 1.f / 16384.f;  // P enters its products as 2^14 P

// A operand (32 rows of 16 values) read transposed from `t`, rows = the
// reduction index r0 + {0..3} and + 8 + {0..3} per lane half (r0 includes 4 g),
// columns c0 + lane % 32.
template <typename Addr>
__device__ __forceinline__ f16x8 tr_frag(Addr addr) {
    const f16x4 lo = ds_read_tr16_f16(addr(0));
    const f16x4 hi = ds_read_tr16_f16(addr(8));
    return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
}

// SHORT: the launch has short rows (p.n_short > 0); without them the kernel
// carries neither the prologue nor the low part of delta.
// DQD: dQ comes from the query-major pass (bwd_dq_kernel), not from here.
template <int D, int KP, bool SHORT, bool DQD>
__global__ __launch_bounds__(512, 2) void bwd_main_kernel(BwdParams p) {
    using T = BwdTile<D, KP>;
    constexpr int NT = 512;
    constexpr int BQ = kBwdBQ;
    constexpr int BK = T::BK, QS = T::QS, SS = T::SS;
    constexpr int NKB = KP / 32;           // 32-key blocks per pair
    constexpr int NKK = D / 16;            // MFMA steps along the head dim
    constexpr int NDB = D / 32;            // 32-wide head-dim blocks
    constexpr int C8 = D / 8;              // 8-element chunks per row
    constexpr int NCH = BQ * C8;           // chunks of a Q or dO tile, staged by 256 threads
    constexpr int CPT = (NCH + 255) / 256;
    constexpr int XB = 32 * SS * 2;        // bytes of one dS part of a 32-key block
    constexpr int DQP = NDB;               // dQ: pairs of keys per wave (4 / NDB waves share a head-dim block)
    constexpr int KU = BK / 8 * D / NT;    // K^T units per thread

    __shared__ __attribute__((aligned(16))) _Float16 Qs[2][2][BQ][QS];  // [buffer][part]
    __shared__ __attribute__((aligned(16))) _Float16 dOs[2][BQ][QS];    // [part]
    __shared__ f16x8 Kt[2][BK / 8][D];  // [part][8 keys][head dim]: K^T in the dQ product's operand order
    __shared__ __attribute__((aligned(16))) char Xs[4][NKB * 2 * XB];   // P, then dS, of each pair
    __shared__ __attribute__((aligned(16))) float lse_s[BQ];
    __shared__ __attribute__((aligned(16))) float dl_s[BQ];
    __shared__ __attribute__((aligned(16))) float dlo_s[BQ];
    __shared__ float dinv_s[SHORT ? BQ : 1];  // units of the dO rows
    __shared__ int dqcls_s[4];     // sum of the classes of a pair's dS, V and K
    __shared__ int kcls_s[4];
    __shared__ float red_s[2][8];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int role = wave >> 2;  // 0: K, S, P, dV; 1: V, dP, dS, dK
    const int pr = wave & 3;     // pair
    const int l32 = lane & 31;
    const int g = lane >> 5;

    const BwdWork wk = bwd_work<BK>(p);
    if (wk.bh >= p.B * p.H) return;  // padding workgroup of a split plan's grid
    const int kblk = wk.kblk;
    const int bh = wk.bh;
    const int b = bh / p.H;
    const int h = bh % p.H;

    const float* Q = (const float*)p.q + b * p.sq.b + h * p.sq.h;
    const float* dO = (const float*)p.dout + b * p.sdo.b + h * p.sdo.h;
    float* dQa = p.dq_acc + b * p.sacc.b + h * p.sacc.h;
    const float* LSE = p.lse + (int64_t)bh * p.Tq;
    const float* DL = p.delta + (int64_t)bh * p.Tq;
    const float* DLO = p.delta_lo + (int64_t)bh * p.Tq;
    const int k0 = kblk * BK;
    const int k0p = k0 + pr * KP;  // the pair's first key

    const int q_begin = wk.q_begin;
    const int q_end = wk.q_end;

    // Role 1's threads stage the Q tiles, role 0's the dO tiles, with the rows'
    // LSE and delta.  Rows at or past `lim` read as zeros.
    const int ts = tid & 255;
    const float* Y = role ? Q : dO;
    const int64_t yt = role ? p.sq.t : p.sdo.t;
    const uint32_t y_voff = (uint32_t)(((int64_t)(ts / C8) * yt + 8 * (ts % C8)) * 4);
    f32x4 yr[CPT][2];
    float r_lse[CPT], r_dl[CPT], r_dlo[CPT];
    auto gload = [&](int q0, int lim) {
        const int rows = min(lim - q0, BQ);
        const auto ry = row_rsrc(Y, yt, q0, rows, D);
#pragma unroll
        for (int i = 0; i < CPT; ++i) {
            const uint32_t so = (uint32_t)((int64_t)(256 * i / C8) * yt * 4);
            yr[i][0] = buffer_ld4(ry, y_voff, so);
            yr[i][1] = buffer_ld4(ry, y_voff + 16, so);
        }
        if (role == 0) {
            const int n_sh = SHORT && kblk == 0 ? max(0, min(p.n_short - q0, rows)) : 0;
            const auto rl = row_rsrc(LSE, 1, q0, rows, 1), rd = row_rsrc(DL, 1, q0, rows, 1), ro = row_rsrc(DLO, 1, q0, n_sh, 1);
#pragma unroll
            for (int i = 0; i < CPT; ++i) {
                const uint32_t off = (uint32_t)((ts + 256 * i) / C8) * 4;
                r_lse[i] = buffer_ld1(rl, off, 0);
                r_dl[i] = buffer_ld1(rd, off, 0);
                r_dlo[i] = SHORT ? buffer_ld1(ro, off, 0) : 0.f;
            }
        }
    };
    // Everything that the workgroup starts from is loaded at once: its operand
    // rows, K^T, the first Q / dO tile and the maxima of the head's Q and dO rows.
    // The wave's operand, K or V rows of its pair's keys: MFMA step kk takes
    // row key, columns 16 kk + 8 g .. + 7.
    Half2x8 xf[NKB][NKK];
    int xcls;  // its scale class
    // K^T for the dQ product: unit f holds column f % D of the 8 keys that an
    // operand takes together (16 m + 4 g' + {0..3} and + 8 for key group f / D =
    // 2 m + g'), scaled as its pair's K rows are.
    f32x4 kt[DQD ? 1 : KU][2];
    auto kt_key = [](int f) { return 16 * (f / D >> 1) + 4 * (f / D & 1); };
    {
        const float* X = role ? (const float*)p.v + b * p.sv.b + h * p.sv.h : (const float*)p.k + b * p.sk.b + h * p.sk.h;
        const int64_t xt = role ? p.sv.t : p.sk.t;
        f32x4 raw[NKB][NKK][2];
#pragma unroll
        for (int kb = 0; kb < NKB; ++kb) {
            const int key = k0p + kb * 32 + l32;
#pragma unroll
            for (int kk = 0; kk < NKK; ++kk) {
                raw[kb][kk][0] = raw[kb][kk][1] = f32x4{0.f, 0.f, 0.f, 0.f};
                if (key < p.Tk) {
                    raw[kb][kk][0] = ld4(X + (int64_t)key * xt + 16 * kk + 8 * g);
                    raw[kb][kk][1] = ld4(X + (int64_t)key * xt + 16 * kk + 8 * g + 4);
                }
            }
        }
        if constexpr (!DQD) {
            const float* K = (const float*)p.k + b * p.sk.b + h * p.sk.h;
            const auto rk = row_rsrc(K, p.sk.t, k0, min(p.Tk - k0, BK), D);
#pragma unroll
            for (int i = 0; i < KU; ++i) {
                const int f = tid + NT * i;
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    kt[i][e >> 2][e & 3] = buffer_ld1(rk, (uint32_t)(((int64_t)kt_key(f) * p.sk.t + f % D) * 4),
                                                      (uint32_t)((int64_t)((e & 3) + 8 * (e >> 2)) * p.sk.t * 4));
            }
        }
        gload(q_begin, p.Tq);
        const float* am = p.amax + (int64_t)bh * p.n_amax * 2;
        float aq = 0.f, ad = 0.f;
        for (int i = tid; i < p.n_amax; i += NT) {
            aq = fmaxf(aq, am[2 * i]);
            ad = fmaxf(ad, am[2 * i + 1]);
        }
        aq = wave_max(aq);
        ad = wave_max(ad);
        if (lane == 0) {
            red_s[0][wave] = aq;
            red_s[1][wave] = ad;
        }
        float amax = 0.f;
#pragma unroll
        for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
            for (int kk = 0; kk < NKK; ++kk) amax = absmax8_finite(amax, raw[kb][kk][0], raw[kb][kk][1]);
        xcls = __builtin_amdgcn_readfirstlane(scale_class(wave_max(amax)));
        const float xs = class_scale(xcls);
#pragma unroll
        for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
            for (int kk = 0; kk < NKK; ++kk) xf[kb][kk] = split2(raw[kb][kk][0], raw[kb][kk][1], xs);
        if (role == 0 && lane == 0) kcls_s[pr] = xcls;
    }
    int qcls, docls;  // scale classes of the head's Q and dO rows, from bwd_pre's maxima
    __syncthreads();
    {
        float aq = 0.f, ad = 0.f;
#pragma unroll
        for (int w = 0; w < 8; ++w) {
            aq = fmaxf(aq, red_s[0][w]);
            ad = fmaxf(ad, red_s[1][w]);
        }
        qcls = __builtin_amdgcn_readfirstlane(scale_class(aq));
        docls = __builtin_amdgcn_readfirstlane(scale_class(ad));
    }
    if constexpr (!DQD) {
#pragma unroll
        for (int i = 0; i < KU; ++i) {
            const int f = tid + NT * i;
            const Half2x8 k = split2(kt[i][0], kt[i][1], class_scale(kcls_s[kt_key(f) / KP]));
            Kt[0][f / D][f % D] = k.h;
            Kt[1][f / D][f % D] = k.l;
        }
    }
    const float qinv = class_inv(qcls), doinv = class_inv(docls);
    const float xinv = class_inv(xcls);
    const float ytile = class_scale(role ? qcls : docls);  // scale of the rows this wave stages
    const float cs = p.c * xinv * qinv;                     // role 0: scores in exp2 units are S cs
    const float dsu = kBwdPInv * xinv * doinv;              // role 1: dS = ds dsu, ds = (2^14 P) (dP' - delta')
    const float xscale = class_scale(xcls);                 // role 1

    auto sstore = [&](int buf) {
        int ts = tid & 255;
        if constexpr (D == 64 && KP == 64) asm volatile("" : "+v"(ts));
        _Float16* dst = role ? &Qs[buf][0][0][0] : &dOs[0][0][0];
#pragma unroll
        for (int i = 0; i < CPT; ++i) {
            const int f = ts + 256 * i;
            float ys = ytile;
            int rc = docls;
            if (role == 0) {  // a dO row by its own class: rows may differ by many binades
                rc = scale_class(group_max<C8>(absmax8_finite(0.f, yr[i][0], yr[i][1])));
                ys = class_scale(rc);
            }
            const Half2x8 y = split2(yr[i][0], yr[i][1], ys);
            if (NCH % 256 == 0 || f < NCH) {
                *reinterpret_cast<f16x8*>(dst + (f / C8) * QS + 8 * (f % C8)) = y.h;
                *reinterpret_cast<f16x8*>(dst + (BQ + f / C8) * QS + 8 * (f % C8)) = y.l;
                if (role == 0 && f % C8 == 0) {
                    // P carries the row's unit over the head's, so that dV and dS sum
                    // rows in one unit: 2^14 P 2^(8 (rc - docls)) = exp2(S c - lse_s)
                    const int r = f / C8;
                    lse_s[r] = fmaf(r_lse[i], kLog2e, (float)(8 * (docls - rc)) - kBwdPBits);
                    dl_s[r] = r_dl[i] * ys;
                    if constexpr (SHORT) {
                        dlo_s[r] = r_dlo[i] * ys;
                        dinv_s[r] = class_inv(rc);
                    }
                }
            }
        }
    };

    // Short rows (bwd_split.h): before the main loop, their delta from this
    // block's own S and dP.  Per short tile the pair's waves form S^T and dP^T
    // (the main loop's products with the operands swapped, in the same order, so
    // lane (l32, g) holds query q0 + l32 and keys 32 kb + 8 (r / 4) + 4 g + r % 4
    // of the pair), role 0 hands over the weights e = exp2(S c - lse log2 e) (1 for
    // a one-key row's key), and role 1 sums e and e dP in fp64 (exact products)
    // over its registers and the lane pair; the first BQ threads add the pairs'
    // sums in order and store delta = sum(e dP) / sum(e) as hi + lo.
    const int qs_end = SHORT && kblk == 0 ? min(q_end, p.n_short) : q_begin;  // short tiles: [q_begin, qs_end)
    if (SHORT && q_begin < qs_end) {
        double* part = reinterpret_cast<double*>(&Qs[1][0][0][0]);  // [4][BQ] pairs (sum e, sum e dP)
        static_assert(2 * 4 * BQ * sizeof(double) <= sizeof(Qs[1]), "the sums fit the second Q buffer");
        for (int q0 = q_begin; q0 < qs_end; q0 += BQ) {
            sstore(0);
            __syncthreads();
            gload(q0 + BQ, q0 + BQ < qs_end ? p.Tq : 0);
            const bool active = (!p.causal || (q0 + BQ - 1 + p.off >= k0p)) && k0p < p.Tk;
            f32x16 st[NKB];
            f32x4* X = reinterpret_cast<f32x4*>(&Xs[pr][0]);
            if (active) {
                const _Float16* rows = role ? &dOs[0][0][0] : &Qs[0][0][0][0];
#pragma unroll
                for (int kk = 0; kk < NKK; ++kk) {
                    Half2x8 y;
                    y.h = *reinterpret_cast<const f16x8*>(rows + l32 * QS + 16 * kk + 8 * g);
                    y.l = *reinterpret_cast<const f16x8*>(rows + (BQ + l32) * QS + 16 * kk + 8 * g);
#pragma unroll
                    for (int kb = 0; kb < NKB; ++kb) st[kb] = mfma_split<true>(xf[kb][kk], y, kk == 0 ? f32x16{} : st[kb]);
                }
                if (role == 0) {
                    const int qi = q0 + l32;
                    const float L = lse_s[l32];
#pragma unroll
                    for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
                        for (int j = 0; j < 4; ++j) {
                            f32x4 e;
#pragma unroll
                            for (int cc = 0; cc < 4; ++cc) {
                                const int kj = k0p + 32 * kb + 8 * j + 4 * g + cc;
                                const bool vis = (qi < p.Tq) && (kj < p.Tk) && (!p.causal || kj <= qi + p.off);
                                e[cc] = bwd_short_weight(p, qi, vis, fast_exp2(fmaf(st[kb][4 * j + cc], cs, -L)) * kBwdPInv);
                            }
                            X[(4 * kb + j) * 64 + lane] = e;
                        }
                }
            }
            __syncthreads();
            if (role == 1) {
                double l = 0.0, w = 0.0;
                if (active) {
#pragma unroll
                    for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
                        for (int j = 0; j < 4; ++j) {
                            const f32x4 e = X[(4 * kb + j) * 64 + lane];
#pragma unroll
                            for (int cc = 0; cc < 4; ++cc) {
                                l += (double)e[cc];
                                w += (double)e[cc] * (double)st[kb][4 * j + cc];
                            }
                        }
                }
                l += __shfl_xor(l, 32);
                w += __shfl_xor(w, 32);
                if (g == 0) {
                    part[2 * (pr * BQ + l32)] = l;
                    part[2 * (pr * BQ + l32) + 1] = w * ((double)xinv * (double)dinv_s[l32]);
                }
            }
            __syncthreads();
            if (tid < BQ) bwd_short_delta_store<4, BQ>(p, bh, q0 + tid, part + 2 * tid);
        }
        __syncthreads();  // the deltas are stored: the first tile's are read again
        gload(q_begin, p.Tq);
    }

    f32x16 acc[NDB][NKB];  // dV^T (role 0) or dK^T (role 1): row d, column key
#pragma unroll
    for (int db = 0; db < NDB; ++db)
#pragma unroll
        for (int kb = 0; kb < NKB; ++kb) acc[db][kb] = f32x16{};
    int dscls = 2;  // role 1: class of the largest |ds| so far

    sstore(0);
    __syncthreads();

    int buf = 0;
    for (int q0 = q_begin; q0 < q_end; q0 += BQ, buf ^= 1) {
        // At D = 64 the lane number passes an empty asm, so that LDS addresses are
        // formed in each tile instead of being held (and spilled) across the loop.
        int ln = lane;
        if constexpr (D == 64 && KP == 64) asm volatile("" : "+v"(ln));
        const int lane = ln, l32 = ln & 31, g = ln >> 5;
        // ---- A: S and P (role 0), dP (role 1) -----------------------------------
        gload(q0 + BQ, q0 + BQ < q_end ? p.Tq : 0);
        // Does any query of this tile see any key of this pair?
        const bool active = (!p.causal || (q0 + BQ - 1 + p.off >= k0p)) && k0p < p.Tk;
        f32x4* X = reinterpret_cast<f32x4*>(&Xs[pr][0]);
        f32x16 s[NKB];
        if (active) {
            const _Float16* rows = role ? &dOs[0][0][0] : &Qs[buf][0][0][0];
#pragma unroll
            for (int kk = 0; kk < NKK; ++kk) {
                Half2x8 y;
                y.h = *reinterpret_cast<const f16x8*>(rows + l32 * QS + 16 * kk + 8 * g);
                y.l = *reinterpret_cast<const f16x8*>(rows + (BQ + l32) * QS + 16 * kk + 8 * g);
#pragma unroll
                for (int kb = 0; kb < NKB; ++kb) s[kb] = mfma_split<false>(y, xf[kb][kk], kk == 0 ? f32x16{} : s[kb]);
            }
            // reg 4j + cc of s[kb]: query row 8 j + 4 g + cc of the tile, key 32 kb + l32 of the pair
            if (role == 0) {
                // Only tiles that cross the causal diagonal or the end of the
                // queries / keys evaluate the visibility test.
                auto prob = [&](auto masked) {
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const f32x4 L = *reinterpret_cast<const f32x4*>(&lse_s[8 * j + 4 * g]);
#pragma unroll
                        for (int kb = 0; kb < NKB; ++kb) {
                            f32x4 e;
#pragma unroll
                            for (int cc = 0; cc < 4; ++cc) {
                                float pv = fast_exp2(fmaf(s[kb][4 * j + cc], cs, -L[cc]));
                                if constexpr (decltype(masked)::value) {
                                    const int qi = q0 + 8 * j + 4 * g + cc, key = k0p + 32 * kb + l32;
                                    const bool vis = (qi < p.Tq) && (key < p.Tk) && (!p.causal || key <= qi + p.off);
                                    pv = vis ? pv : 0.f;
                                }
                                s[kb][4 * j + cc] = e[cc] = pv;
                            }
                            X[(4 * kb + j) * 64 + lane] = e;
                        }
                    }
                };
                if (q0 + BQ > p.Tq || k0p + KP > p.Tk || (p.causal && k0p + KP - 1 > q0 + p.off))
                    prob(std::true_type{});
                else
                    prob(std::false_type{});
            }
        }
        __syncthreads();

        // ---- B: dV (role 0), dS (role 1) -----------------------------------------
        Half2x8 pb[NKB][2];  // P or dS: queries 16 mm + 4 g + {0..3} and + 8 of key block kb
        if (active) {
            if (role == 1) {
                float mx = 0.f;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const f32x4 Dl = *reinterpret_cast<const f32x4*>(&dl_s[8 * j + 4 * g]);
                    const f32x4 Dlo = SHORT ? *reinterpret_cast<const f32x4*>(&dlo_s[8 * j + 4 * g])
                                            : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int kb = 0; kb < NKB; ++kb) {
                        const f32x4 pv = X[(4 * kb + j) * 64 + lane];
#pragma unroll
                        for (int cc = 0; cc < 4; ++cc) {
                            float t = fmaf(-Dl[cc], xscale, s[kb][4 * j + cc]);
                            if constexpr (SHORT) t = fmaf(-Dlo[cc], xscale, t);
                            s[kb][4 * j + cc] = pv[cc] * t;
                        }
                    }
                }
                // A row with one visible key: dS = P (dP - dP) = 0.
                if (bwd_one_key_tile(p, q0, k0p)) {
#pragma unroll
                    for (int r = 0; r < 16; ++r)
                        if (bwd_one_key_row(p, q0 + 8 * (r >> 2) + 4 * g + (r & 3))) s[0][r] = 0.f;
                }
#pragma unroll
                for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
                    for (int r = 0; r < 16; r += 8)
                        mx = absmax8(mx, f32x4{s[kb][r], s[kb][r + 1], s[kb][r + 2], s[kb][r + 3]},
                                     f32x4{s[kb][r + 4], s[kb][r + 5], s[kb][r + 6], s[kb][r + 7]});
                if (__any(mx >= class_limit(dscls))) {  // dK^T is kept in units of ds's scale
                    mx = 0.f;
#pragma unroll
                    for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
                        for (int r = 0; r < 16; ++r) mx = fmaxf(mx, finite_abs(s[kb][r]));
                    const int nc = max(dscls, min(31, __builtin_amdgcn_readfirstlane(scale_class(wave_max(mx)))));
                    const float f = class_scale(nc) * class_inv(dscls);
#pragma unroll
                    for (int db = 0; db < NDB; ++db)
#pragma unroll
                        for (int kb = 0; kb < NKB; ++kb) acc[db][kb] *= f;
                    dscls = nc;
                }
                if (lane == 0) dqcls_s[pr] = dscls + xcls + kcls_s[pr];
            }
            const float psc = role ? class_scale(dscls) : 1.f;
#pragma unroll
            for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
                for (int mm = 0; mm < 2; ++mm) {
                    const f32x16& e = s[kb];
                    pb[kb][mm] = split2(f32x4{e[8 * mm], e[8 * mm + 1], e[8 * mm + 2], e[8 * mm + 3]},
                                        f32x4{e[8 * mm + 4], e[8 * mm + 5], e[8 * mm + 6], e[8 * mm + 7]}, psc);
                }
        } else if (role == 1 && !DQD) {
#pragma unroll
            for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
                for (int mm = 0; mm < 2; ++mm) pb[kb][mm] = Half2x8{};
            if (lane == 0) dqcls_s[pr] = -1;
        }
        if (role == 1 && !DQD) {
            {
                // dS over P (read above by this wave): row key l32, queries along it
                asm volatile("" ::: "memory");
#pragma unroll
                for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
                    for (int mm = 0; mm < 2; ++mm)
#pragma unroll
                        for (int hl = 0; hl < 2; ++hl) {
                            const f16x8 v = hl ? pb[kb][mm].l : pb[kb][mm].h;
                            _Float16* row = reinterpret_cast<_Float16*>(&Xs[pr][(2 * kb + hl) * XB]) + l32 * SS + 16 * mm + 4 * g;
                            *reinterpret_cast<f16x4*>(row) = __builtin_shufflevector(v, v, 0, 1, 2, 3);
                            *reinterpret_cast<f16x4*>(row + 8) = __builtin_shufflevector(v, v, 4, 5, 6, 7);
                        }
            }
        }
        // acc += rows^T pb (dO^T P or Q^T dS), rows read transposed
        auto accumulate = [&](const _Float16* rows) {
            const int a_off = (4 * (ln >> 5) + ((ln & 15) >> 2)) * QS + 16 * ((ln >> 4) & 1) + 4 * (ln & 3);
#pragma unroll
            for (int mm = 0; mm < 2; ++mm)
#pragma unroll
                for (int db = 0; db < NDB; ++db) {
                    const _Float16* at = rows + a_off + 16 * mm * QS + db * 32;
                    Half2x8 a;
                    a.h = tr_frag([&](int r) { return at + r * QS; });
                    a.l = tr_frag([&](int r) { return at + (BQ + r) * QS; });
#pragma unroll
                    for (int kb = 0; kb < NKB; ++kb) acc[db][kb] = mfma_split(a, pb[kb][mm], acc[db][kb]);
                }
        };
        if (active && role == 0) accumulate(&dOs[0][0][0]);
        __syncthreads();

        // ---- C: dQ (both), dK (role 1), the next dO tile (role 0) ------------------
        sstore(buf ^ 1);
        if (active && role == 1) accumulate(&Qs[buf][0][0][0]);
        if constexpr (!DQD) {
            if (role == 0) {
                // dQ tile (32 x D) = dS K: a wave takes a 32-wide head-dim block, over all
                // of the workgroup's keys at D = 128 and a half (a quarter) of them at
                // D = 64 (32), and adds it to the global accumulator with fp32 atomics.
                // (One 16x16 block per wave of both roles over all keys made this phase
                // LDS-bound: twice the operand bytes.  Adding the waves' shares in LDS
                // took 160 cycles per ds_add_f32.)
                const int db = pr % NDB;
                f32x16 dq = f32x16{};
                int unit = -1;  // dq is in units of 2^(8 unit)
#pragma unroll
                for (int pi = 0; pi < DQP; ++pi) {
                    const int pp = pr / NDB * DQP + pi;
                    const int u = __builtin_amdgcn_readfirstlane(dqcls_s[pp]);  // < 0: the pair's dS is zero
                    const int d = u >= 0 && unit >= 0 ? min(max(unit - u, -15), 15) : 0;
                    unit = u >= 0 ? u : unit;
                    if (pi > 0) dq *= __uint_as_float((uint32_t)(127 + 8 * d) << 23);
#pragma unroll
                    for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
                        for (int m = 0; m < 2; ++m) {
                            const _Float16* ds = reinterpret_cast<const _Float16*>(&Xs[pp][2 * kb * XB]) +
                                                 (16 * m + 4 * g + ((lane & 15) >> 2)) * SS + 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
                            Half2x8 a, kf;
                            a.h = tr_frag([&](int r) { return ds + r * SS; });
                            a.l = tr_frag([&](int r) { return ds + XB / 2 + r * SS; });
                            kf.h = Kt[0][(pp * KP + 32 * kb + 16 * m) / 8 + g][db * 32 + l32];
                            kf.l = Kt[1][(pp * KP + 32 * kb + 16 * m) / 8 + g][db * 32 + l32];
                            dq = mfma_split(a, kf, dq);
                        }
                }
                const float f = ldexpf(kBwdPInv * doinv * p.scale, 8 * unit - 414);
                const auto rdq = row_rsrc(dQa, p.sacc.t, q0, min(p.Tq - q0, BQ), D);  // rows past Tq are dropped
                const uint32_t voff = (uint32_t)(((int64_t)(4 * g) * p.sacc.t + db * 32 + l32) * 4);
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    buffer_atomic_add(rdq, dq[r] * f, voff, (uint32_t)((int64_t)(8 * (r >> 2) + (r & 3)) * p.sacc.t * 4));
            }
        }
        __syncthreads();
    }

    // ---- dK = scale * dK^T^T, dV = dV^T^T ------------------------------------------
    const float unit = role ? class_inv(dscls) * dsu * qinv * p.scale : kBwdPInv * doinv;
    f32x16 out[NDB * NKB];
#pragma unroll
    for (int db = 0; db < NDB; ++db)
#pragma unroll
        for (int kb = 0; kb < NKB; ++kb) out[db * NKB + kb] = acc[db][kb] * unit;
    if (!bwd_fixup<NT>(p, wk, out)) return;
#pragma unroll
    for (int kb = 0; kb < NKB; ++kb) {
        const int key = k0p + 32 * kb + l32;
        if (key >= p.Tk) continue;
        float* dst = role ? (float*)p.dk + b * p.sdk.b + h * p.sdk.h + (int64_t)key * p.sdk.t
                          : (float*)p.dv + b * p.sdv.b + h * p.sdv.h + (int64_t)key * p.sdv.t;
#pragma unroll
        for (int db = 0; db < NDB; ++db)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const f32x16& v = out[db * NKB + kb];
                st4(dst + db * 32 + 8 * j + 4 * g, f32x4{v[4 * j], v[4 * j + 1], v[4 * j + 2], v[4 * j + 3]});
            }
    }
}

// dQ accumulator (fp32) -> bf16 dq, when dq has the accumulator's dense
// [B, H, Tq, D] layout and 16-byte aligned rows: a flat pass, 8 elements
// (two 16-byte loads, one 16-byte store) per thread.
__global__ __launch_bounds__(256) void bwd_cvt_flat_kernel(BwdParams p) {
    const int64_t n8 = (int64_t)p.B * p.H * p.Tq * p.D / 8;
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n8) return;
    const f32x4* a = reinterpret_cast<const f32x4*>(p.dq_acc) + 2 * i;
    const f32x4 x = a[0], y = a[1];
    u16x8 h;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        h[k] = f32_to_bf16(x[k]);
        h[4 + k] = f32_to_bf16(y[k]);
    }
    reinterpret_cast<u16x8*>(p.dq)[i] = h;
}

// dQ accumulator (fp32) -> bf16 dq on dq's own strides.
template <int D>
__global__ __launch_bounds__(256) void bwd_cvt_kernel(BwdParams p) {
    constexpr int TPR = D / 4;
    constexpr int RPB = 256 / TPR;
    const int tid = threadIdx.x;
    const int64_t row = (int64_t)blockIdx.x * RPB + tid / TPR;
    const int c4 = tid % TPR;
    const int64_t rows = (int64_t)p.B * p.H * p.Tq;
    if (row >= rows) return;
    int64_t b, h, i;
    bwd_row_split(p, rows, row, b, h, i);
    const f32x4 a = *reinterpret_cast<const f32x4*>(p.dq_acc + b * p.sacc.b + h * p.sacc.h +
                                                     i * p.sacc.t + 4 * c4);
    st4((uint16_t*)p.dq + b * p.sdq.b + h * p.sdq.h + i * p.sdq.t + 4 * c4, a);
}

// Query-major dQ pass, fp32 (the deterministic mode: the main kernel then
// skips its dQ product).  One workgroup = 4 waves x 32 query rows of one
// (b, h), laid out as the forward: each lane keeps its query row of Q and dO
// as split B operands (Q^T, dO^T) in VGPRs, with that row's log-sum-exp and
// delta; tiles of 32 keys of K and V, split, are double-buffered in LDS (loaded
// two tiles ahead, scaled by the class of the largest magnitude so far).  Per
// wave and tile:
//   S^T = K Q^T, dP^T = V dO^T        in the forward's and the main kernel's
//                                     order, to the same bits
//   P^T = exp2(S^T c - lse log2 e), dS^T = P^T (dP^T - delta)
//   dQ^T += K^T dS^T                  A = K^T read transposed from the K rows,
//                                     B = dS^T straight from the accumulators
// dQ stays in VGPRs and is stored once, times the scale: every element is the
// sum of its key tiles in key order, with no accumulator, zeroing or atomics,
// so the result is the same on every run.  It recomputes S and dP (two more
// products per score than the atomic dQ of the main kernel).
template <int D>
__global__ __launch_bounds__(256, D >= 128 ? 1 : 2) void bwd_dq_kernel(BwdParams p) {
    constexpr int BM = kBwdDqBM;
    constexpr int BN = 32;               // keys per tile
    constexpr int NKK = D / 16;          // MFMA steps along the head dim
    constexpr int NDB = D / 32;          // 32-wide d blocks of dQ^T
    constexpr int C8 = D / 8;            // 8-element chunks per row
    constexpr int NCH = BN * C8;         // chunks of a tile
    constexpr int CPT = (NCH + 255) / 256;
    constexpr int QS = BwdTile<D, 32>::QS;
    static_assert(BM == 128 && 256 % C8 == 0, "4 waves x 32 rows, whole staging passes");

    __shared__ __attribute__((aligned(16))) _Float16 Ks[2][2][BN][QS];  // [buffer][part]
    __shared__ __attribute__((aligned(16))) _Float16 Vs[2][2][BN][QS];
    __shared__ int cls_s[2][2][4];  // scale class that each wave's loads need: [K, V][tile parity]

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31;
    const int g = lane >> 5;
    const int tr_row = (lane & 15) >> 2, tr_col = 16 * ((lane >> 4) & 1) + 4 * (lane & 3);

    const int BH = p.B * p.H;
    const int w = blockIdx.x;
    const int qtile = p.n_qtiles - 1 - w / BH;  // the longest causal rows first
    const int bh = w % BH;
    const int b = bh / p.H;
    const int h = bh % p.H;

    const float* Q = (const float*)p.q + b * p.sq.b + h * p.sq.h;
    const float* K = (const float*)p.k + b * p.sk.b + h * p.sk.h;
    const float* V = (const float*)p.v + b * p.sv.b + h * p.sv.h;
    const float* dO = (const float*)p.dout + b * p.sdo.b + h * p.sdo.h;

    const int q0w = qtile * BM + wave * 32;
    const int qrow = q0w + l32;
    // B operands: MFMA step kk takes row qrow, columns 16 kk + 8 g .. + 7, scaled by the row's class.
    Half2x8 qf[NKK], df[NKK];
    float qinv, doscale, doinv;
    auto load_row = [&](const float* src, int64_t st, Half2x8 (&f)[NKK]) {
        f32x4 raw[NKK][2];
        float amax = 0.f;
#pragma unroll
        for (int kk = 0; kk < NKK; ++kk) {
            raw[kk][0] = raw[kk][1] = f32x4{0.f, 0.f, 0.f, 0.f};
            if (qrow < p.Tq) {
                raw[kk][0] = ld4(src + (int64_t)qrow * st + 16 * kk + 8 * g);
                raw[kk][1] = ld4(src + (int64_t)qrow * st + 16 * kk + 8 * g + 4);
            }
            amax = absmax8_finite(amax, raw[kk][0], raw[kk][1]);
        }
        const int k = scale_class(max_xor32(amax));
#pragma unroll
        for (int kk = 0; kk < NKK; ++kk) f[kk] = split2(raw[kk][0], raw[kk][1], class_scale(k));
        return k;
    };
    qinv = class_inv(load_row(Q, p.sq.t, qf));
    {
        const int k = load_row(dO, p.sdo.t, df);
        doscale = class_scale(k);
        doinv = class_inv(k);
    }
    const float Lq = qrow < p.Tq ? fmaf(p.lse[(int64_t)bh * p.Tq + qrow], kLog2e, -kBwdPBits) : 0.f;
    const float Dq = qrow < p.Tq ? p.delta[(int64_t)bh * p.Tq + qrow] * doscale : 0.f;
    const float Dqlo = bwd_short_row(p, qrow) ? p.delta_lo[(int64_t)bh * p.Tq + qrow] * doscale : 0.f;
    const bool one_key = qrow < p.Tq && bwd_one_key_row(p, qrow);
    const bool one_key_wave = p.causal ? (-p.off >= q0w && -p.off < q0w + 32) : p.Tk == 1;  // wave-uniform

    int kv_end = p.Tk;
    if (p.causal) kv_end = min(p.Tk, qtile * BM + BM + p.off);
    const int nt = (kv_end + BN - 1) / BN;
    const int wave_kend = p.causal ? min(kv_end, q0w + 32 + p.off) : kv_end;

    // Chunk tid + 256 i of a tile: row f / C8, 8 columns from 8 (f % C8).  Rows at
    // or past the resource's end (<= Tk) read as zeros.
    struct Raw {
        f32x4 k[CPT][2], v[CPT][2];
    };
    const uint32_t k_voff = (uint32_t)(((int64_t)(tid / C8) * p.sk.t + 8 * (tid % C8)) * 4);
    const uint32_t v_voff = (uint32_t)(((int64_t)(tid / C8) * p.sv.t + 8 * (tid % C8)) * 4);
    auto gload = [&](Raw& r, int u) {
        const int rows = u < nt ? min(p.Tk - u * BN, BN) : 0;
        const auto rk = row_rsrc(K, p.sk.t, u * BN, rows, D);
        const auto rv = row_rsrc(V, p.sv.t, u * BN, rows, D);
#pragma unroll
        for (int i = 0; i < CPT; ++i) {
            const uint32_t ko = (uint32_t)((int64_t)(256 * i / C8) * p.sk.t * 4);
            const uint32_t vo = (uint32_t)((int64_t)(256 * i / C8) * p.sv.t * 4);
            r.k[i][0] = buffer_ld4(rk, k_voff, ko);
            r.k[i][1] = buffer_ld4(rk, k_voff + 16, ko);
            r.v[i][0] = buffer_ld4(rv, v_voff, vo);
            r.v[i][1] = buffer_ld4(rv, v_voff + 16, vo);
        }
    };
    int kcls = 2, vcls = 2;  // classes of the tile in LDS (as in the forward)
    auto need_classes = [&](const Raw& r, int par) {
        float mk = 0.f, mv = 0.f;
#pragma unroll
        for (int i = 0; i < CPT; ++i) {
            mk = absmax8(mk, r.k[i][0], r.k[i][1]);
            mv = absmax8(mv, r.v[i][0], r.v[i][1]);
        }
        int nk = 0, nv = 0;
        if (__any(mk >= class_limit(kcls) || mv >= class_limit(vcls))) {
            mk = mv = 0.f;
#pragma unroll
            for (int i = 0; i < CPT; ++i) {
                mk = absmax8_finite(mk, r.k[i][0], r.k[i][1]);
                mv = absmax8_finite(mv, r.v[i][0], r.v[i][1]);
            }
            nk = scale_class(wave_max(mk));
            nv = scale_class(wave_max(mv));
        }
        if (lane == 0) {
            cls_s[0][par][wave] = nk;
            cls_s[1][par][wave] = nv;
        }
    };
    auto class_of = [&](int which, int par, int cur) {  // after the barrier
        int m = cur;
#pragma unroll
        for (int i = 0; i < 4; ++i) m = max(m, cls_s[which][par][i]);
        return __builtin_amdgcn_readfirstlane(m);
    };
    auto sstore = [&](const Raw& r, int buf, int kc, int vc) {
#pragma unroll
        for (int i = 0; i < CPT; ++i) {
            const int f = tid + 256 * i, row = f / C8, col = 8 * (f % C8);
            if (NCH % 256 == 0 || f < NCH) {
                const Half2x8 k = split2(r.k[i][0], r.k[i][1], class_scale(kc));
                const Half2x8 v = split2(r.v[i][0], r.v[i][1], class_scale(vc));
                *reinterpret_cast<f16x8*>(&Ks[buf][0][row][col]) = k.h;
                *reinterpret_cast<f16x8*>(&Ks[buf][1][row][col]) = k.l;
                *reinterpret_cast<f16x8*>(&Vs[buf][0][row][col]) = v.h;
                *reinterpret_cast<f16x8*>(&Vs[buf][1][row][col]) = v.l;
            }
        }
    };

    f32x16 dq[NDB];
#pragma unroll
    for (int i = 0; i < NDB; ++i) dq[i] = f32x16{};
    int dscls = 2;  // class of the row's largest |ds| so far, per lane

    Raw ra, rb;
    gload(ra, 0);
    need_classes(ra, 0);
    gload(rb, 1);
    __syncthreads();
    kcls = class_of(0, 0, kcls);
    vcls = class_of(1, 0, vcls);
    sstore(ra, 0, kcls, vcls);
    need_classes(rb, 1);
    __syncthreads();
    auto step = [&](int u, Raw& nxt, Raw& far) {
        const int buf = u & 1;
        const int k0 = u * BN;
        gload(far, u + 2);
        const int nk = class_of(0, (u + 1) & 1, kcls), nv = class_of(1, (u + 1) & 1, vcls);
        if (k0 < wave_kend) {
            f32x16 s, dp;
#pragma unroll
            for (int kk = 0; kk < NKK; ++kk) {
                Half2x8 k, v;
                k.h = *reinterpret_cast<const f16x8*>(&Ks[buf][0][l32][16 * kk + 8 * g]);
                k.l = *reinterpret_cast<const f16x8*>(&Ks[buf][1][l32][16 * kk + 8 * g]);
                v.h = *reinterpret_cast<const f16x8*>(&Vs[buf][0][l32][16 * kk + 8 * g]);
                v.l = *reinterpret_cast<const f16x8*>(&Vs[buf][1][l32][16 * kk + 8 * g]);
                s = mfma_split(k, qf[kk], kk == 0 ? f32x16{} : s);
                dp = mfma_split(v, df[kk], kk == 0 ? f32x16{} : dp);
            }
            // reg r: key k0 + 8 (r / 4) + 4 g + r % 4 of query qrow
            const bool need_mask = (k0 + BN > p.Tk) || (qtile * BM + BM > p.Tq) || (p.causal && (k0 + BN - 1 > q0w + p.off));
            const int lim = p.causal ? min(p.Tk - 1, qrow + p.off) : p.Tk - 1;
            const float cs = p.c * qinv * class_inv(kcls), vscale = class_scale(vcls);
            // the visibility test only on tiles that cross the diagonal or the ends
            float mx = 0.f;
            auto p_ds = [&](auto masked) {
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    float pr = fast_exp2(fmaf(s[r], cs, -Lq));
                    if constexpr (decltype(masked)::value) {
                        const int key = k0 + 8 * (r >> 2) + 4 * g + (r & 3);
                        pr = (key <= lim && qrow < p.Tq) ? pr : 0.f;
                    }
                    s[r] = pr * fmaf(-Dqlo, vscale, fmaf(-Dq, vscale, dp[r]));  // dS^T
                }
            };
            if (need_mask)
                p_ds(std::true_type{});
            else
                p_ds(std::false_type{});
            if (one_key_wave && k0 == 0 && one_key) s = f32x16{};  // one visible key: dS = P (dP - dP) = 0
#pragma unroll
            for (int r = 0; r < 16; ++r) mx = fmaxf(mx, fabsf(s[r]));
            if (__any(mx >= class_limit(dscls))) {  // a row's dQ is kept in units of its ds scale
                mx = 0.f;
#pragma unroll
                for (int r = 0; r < 16; ++r) mx = fmaxf(mx, finite_abs(s[r]));
                const int nc = max(dscls, min(31, scale_class(max_xor32(mx))));
                const float f = class_scale(nc) * class_inv(dscls);
#pragma unroll
                for (int db = 0; db < NDB; ++db) dq[db] *= f;
                dscls = nc;
            }
            const float sc = class_scale(dscls);
            // dQ^T[d][q] += K^T[d][keys] dS^T[keys][q]: step m takes keys 16 m + 4 g + {0..3} and + 8
#pragma unroll
            for (int m = 0; m < 2; ++m) {
                const Half2x8 ds = split2(f32x4{s[8 * m], s[8 * m + 1], s[8 * m + 2], s[8 * m + 3]},
                                          f32x4{s[8 * m + 4], s[8 * m + 5], s[8 * m + 6], s[8 * m + 7]}, sc);
                const int r0 = 16 * m + 4 * g + tr_row;
#pragma unroll
                for (int db = 0; db < NDB; ++db) {
                    Half2x8 kt;
                    kt.h = tr_frag([&](int r) { return &Ks[buf][0][r0 + r][db * 32 + tr_col]; });
                    kt.l = tr_frag([&](int r) { return &Ks[buf][1][r0 + r][db * 32 + tr_col]; });
                    dq[db] = mfma_split(kt, ds, dq[db]);
                }
            }
        }
        if (nk != kcls || nv != vcls) {  // ... and of K's and V's scales
            const float f = (class_scale(nk) * class_inv(kcls)) * (class_scale(nv) * class_inv(vcls));
#pragma unroll
            for (int db = 0; db < NDB; ++db) dq[db] *= f;
        }
        kcls = nk;
        vcls = nv;
        sstore(nxt, buf ^ 1, nk, nv);
        need_classes(far, u & 1);
        __syncthreads();
    };
    for (int u = 0; u < nt; u += 2) {
        step(u, rb, ra);
        if (u + 1 < nt) step(u + 1, ra, rb);
    }
    if (qrow < p.Tq) {
        const float unit = class_inv(dscls) * kBwdPInv * class_inv(vcls) * doinv * class_inv(kcls) * p.scale;
        float* dst = (float*)p.dq + b * p.sdq.b + h * p.sdq.h + (int64_t)qrow * p.sdq.t;
#pragma unroll
        for (int db = 0; db < NDB; ++db)
#pragma unroll
            for (int j = 0; j < 4; ++j)
                st4(dst + db * 32 + 8 * j + 4 * g,
                    f32x4{dq[db][4 * j], dq[db][4 * j + 1], dq[db][4 * j + 2], dq[db][4 * j + 3]} * unit);
    }
}

// ---- split plan (host) ------------------------------------------------------------
//
// Under a causal mask key block j has ~(Tq - 128 j) / 32 query tiles, so at
// config-2 sizes the first key blocks carry up to 8x the work of the last.
// Measured on MI355X: a workgroup alone on a CU runs ~1.85x faster than each
// of two sharing it (two resident workgroups give ~8% more throughput than
// one), so the heaviest workgroups, which always share their CU with lighter
// ones, set the kernel's length.  bwd_plan simulates the dispatch (workgroup w
// to XCD w % 8, each XCD's workgroups placed in order on its least-loaded CU
// with a free slot) for splits of the heaviest key blocks' tile ranges into
// chunks, and keeps the best if it beats the unsplit order by 3%.

static constexpr double kBwdPairGain = 0.08;  // throughput gained per extra resident workgroup
// Per-workgroup fixed cost (K/V loads, K^T staging) and the partial store /
// reduction of a split chunk, in query tiles of that dtype's kernel.  A bf16
// tile costs a fraction of an fp32 one while the fixed costs take about the
// same time; the bf16 figures are set from measurement (splits lost 5-8% at
// B4 H12 and config 2 with smaller ones), so bf16 splits only grids far below
// the device's size.
static constexpr double kBwdOverhead[2] = {1.0, 5.0};
static constexpr double kBwdFixup[2] = {1.0, 8.0};
// The short-row prologue of key block 0 (the S and dP chains of each short
// query tile, run once more to form delta) per short tile, in the same units.
static constexpr double kBwdShortTile[2] = {0.55, 0.5};

static double share_rate(size_t k) { return k <= 1 ? 1.0 : (1.0 + kBwdPairGain * (double)(k - 1)) / (double)k; }

// Makespan, in query tiles of a workgroup alone on a CU, of workgroups of the
// given costs in dispatch order.
static double cu_makespan(const std::vector<double>& cost, int cus_per_xcd, int slots) {
    double worst = 0.0;
    std::vector<std::vector<double>> res((size_t)cus_per_xcd);
    for (int x = 0; x < 8; ++x) {
        for (auto& r : res) r.clear();
        size_t next = (size_t)x;
        auto fill = [&]() {
            while (next < cost.size()) {
                int best = -1;
                for (int c = 0; c < cus_per_xcd; ++c)
                    if ((int)res[(size_t)c].size() < slots &&
                        (best < 0 || res[(size_t)c].size() < res[(size_t)best].size()))
                        best = c;
                if (best < 0) break;
                res[(size_t)best].push_back(cost[next]);
                next += 8;
            }
        };
        fill();
        double t = 0.0;
        for (;;) {
            double dt = INFINITY;
            for (const auto& r : res)
                for (double v : r) dt = std::min(dt, v / share_rate(r.size()));
            if (!(dt < INFINITY)) break;
            t += dt;
            for (auto& r : res) {
                const double rate = share_rate(r.size());
                for (double& v : r) v -= dt * rate;
                r.erase(std::remove_if(r.begin(), r.end(), [](double v) { return v <= 1e-9; }), r.end());
            }
            fill();
        }
        worst = std::max(worst, t);
    }
    return worst;
}

// Resident backward workgroups per CU, and CUs per XCD, on the current device.
// An error left pending by an earlier HIP call on this thread is returned
// (named in the detail text) instead of being cleared by the queries here.
static int bwd_slots(int D, int bf16, int* per_cu, int* cus_per_xcd) {
    static std::mutex mu;
    static std::map<std::array<int, 3>, std::pair<int, int>> cache;
    const hipError_t pending = hipGetLastError();
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess) {
        (void)hipGetLastError();  // no device (a CPU-only host sizing workspaces): MI355X defaults
        dev = -1;
    } else if (pending != hipSuccess) {
        return report_pending_error(pending, "attention backward planner");
    }
    std::lock_guard<std::mutex> lk(mu);
    const std::array<int, 3> key{dev, D, bf16};
    auto it = cache.find(key);
    if (it == cache.end()) {
        int cus = 256, occ = (!bf16 || D >= 64) ? 1 : 2;  // MI355X defaults
        if (dev >= 0) {
            int n = 0, o = 0;
            if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && n > 0) cus = n;
            hipError_t e = hipErrorInvalidValue;
            if (!bf16) o = 1, e = hipSuccess;  // fp32: 512 threads of 208-256 VGPRs, one workgroup per CU
            if (bf16) e = (hipError_t)bwd_main_bf16_occupancy(D, &o);
            if (e == hipSuccess && o > 0) occ = o;
            (void)hipGetLastError();  // a failed query of ours: the defaults stand
        }
        it = cache.emplace(key, std::make_pair(occ, std::max(1, cus / 8))).first;
    }
    *per_cu = it->second.first;
    *cus_per_xcd = it->second.second;
    return 0;
}

static void bwd_plan_compute(int B, int H, int Tq, int Tk, int D, int bf16, int per_cu, int cus_per_xcd,
                             BwdPlan* out) {
    const int BH = B * H;
    const int bk = bwd_keys_per_wg(bf16, D, BH, Tq, Tk);
    const int nkb = (Tk + bk - 1) / bk;
    const int off = Tk - Tq;
    if ((int64_t)nkb * BH > 8LL * 8 * cus_per_xcd * per_cu) return;  // the tail is a small share
    std::vector<int> t0((size_t)nkb), nt((size_t)nkb);
    int max_nt = 0;
    for (int j = 0; j < nkb; ++j) {
        t0[(size_t)j] = std::max(0, j * bk - off) / kBwdBQ;
        nt[(size_t)j] = (Tq + kBwdBQ - 1) / kBwdBQ - t0[(size_t)j];
        max_nt = std::max(max_nt, nt[(size_t)j]);
    }
    // query tiles [0, s_tiles) of key block 0 hold its short rows and run the prologue
    const int s_tiles = (bwd_short_rows(B, H, Tq, Tk, 1, bwd_short_keys(bf16, bk)) + kBwdBQ - 1) / kBwdBQ;
    struct G { double cost; int kb, a, b, chunk, n; };
    // A key block of more than ch tiles is split into ceil(n / ch) chunks of
    // near-equal cost, block 0's short tiles counted with the prologue's share
    // pro.  The chunk size is chosen with pro = 0: counting the prologue there
    // moved the choice to plans measured slower (config 2 fp32: ch 27-31, which
    // leave key block 1 whole, +6-10%), while cutting block 0 at the weighted
    // midpoint recovered half of the prologue's cost at the chosen size.
    auto build = [&](int ch, double pro, std::vector<G>& g) {
        g.clear();
        for (int j = 0; j < nkb; ++j) {
            const int n = nt[(size_t)j], s = j == 0 ? s_tiles : 0;
            const int k = n > ch ? (n + ch - 1) / ch : 1;
            auto work = [&](int t) { return (double)t + pro * std::min(t, s); };  // tiles [0, t)
            int a = 0;
            for (int c = 0; c < k; ++c) {
                int e = n;
                if (c + 1 < k) {  // the cut nearest cost share c + 1, leaving a tile for each later chunk
                    const double target = work(n) * (c + 1) / k;
                    e = a + 1;
                    while (e < n - (k - c - 1) && work(e) < target) ++e;
                    if (e > a + 1 && target - work(e - 1) < work(e) - target) --e;
                }
                const double cost = work(e) - work(a) + kBwdOverhead[bf16] + (k > 1 ? kBwdFixup[bf16] : 0.0);
                g.push_back({cost, j, t0[(size_t)j] + a, t0[(size_t)j] + e, c, k});
                a = e;
            }
        }
        std::stable_sort(g.begin(), g.end(), [](const G& x, const G& y) { return x.cost > y.cost; });
    };
    // dispatch order of a plan's grid: group-major, BHp heads per group (padding
    // heads cost nothing); the unsplit grid has B*H heads per key block
    auto makespan = [&](const std::vector<G>& g, int heads) {
        std::vector<double> cost;
        cost.reserve(g.size() * (size_t)heads);
        for (const G& x : g)
            for (int i = 0; i < heads; ++i) cost.push_back(i < BH ? x.cost : 0.0);
        return cu_makespan(cost, cus_per_xcd, per_cu);
    };
    std::vector<G> g;
    build(max_nt, 0.0, g);
    const double base = makespan(g, BH);
    double best = base * 0.97;
    int best_ch = 0;
    for (int ch = max_nt - 1; ch >= std::max(2, max_nt / 8); --ch) {
        build(ch, 0.0, g);
        int n_split = 0;
        for (const G& x : g) n_split += x.chunk == 0 && x.n > 1;
        if ((int)g.size() > kMaxBwdGroups || n_split == 0) continue;
        const double ms = makespan(g, bwd_padded_heads(BH));
        if (ms < best) {
            best = ms;
            best_ch = ch;
        }
    }
    if (!best_ch) return;
    build(best_ch, kBwdShortTile[bf16], g);
    std::vector<int> chunks((size_t)nkb, 1), split_of((size_t)nkb, -1), slot0((size_t)nkb, 0);
    for (const G& x : g) chunks[(size_t)x.kb] = x.n;
    int n_split = 0, n_slots = 0;
    for (int j = 0; j < nkb; ++j) {
        if (chunks[(size_t)j] > 1) {
            split_of[(size_t)j] = n_split++;
            slot0[(size_t)j] = n_slots;
            n_slots += chunks[(size_t)j];
        }
    }
    for (const G& x : g) {
        BwdGroup& o = out->groups[out->n_groups++];
        o.kb = x.kb;
        o.t0 = x.a;
        o.t1 = x.b;
        o.split = split_of[(size_t)x.kb];
        o.chunk = x.chunk;
        o.n_chunks = x.n;
        o.slot0 = slot0[(size_t)x.kb];
    }
    out->n_split = n_split;
    out->n_slots = n_slots;
}

int bwd_plan(int B, int H, int Tq, int Tk, int D, int causal, int bf16, BwdPlan* out) {
    *out = BwdPlan{};
    out->bk = bwd_keys_per_wg(bf16, D, (int64_t)B * H, Tq, Tk);
    if (!causal) return 0;
    int per_cu = 0, cus_per_xcd = 0;
    if (const int e = bwd_slots(D, bf16, &per_cu, &cus_per_xcd)) return e;
    static std::mutex mu;
    static std::map<std::array<int, 7>, BwdPlan> cache;
    const std::array<int, 7> key{B * H, Tq, Tk, D, bf16, per_cu, cus_per_xcd};
    {
        std::lock_guard<std::mutex> lk(mu);
        auto it = cache.find(key);
        if (it != cache.end()) {
            *out = it->second;
            return 0;
        }
    }
    bwd_plan_compute(B, H, Tq, Tk, D, bf16 ? 1 : 0, per_cu, cus_per_xcd, out);
    std::lock_guard<std::mutex> lk(mu);
    if (cache.size() > 256) cache.clear();
    cache[key] = *out;
    return 0;
}

size_t bwd_split_workspace_bytes(const BwdPlan& plan, int B, int H, int D) {
    if (!plan.n_split) return 0;
    const size_t bh = (size_t)B * H;
    const size_t part = (size_t)plan.n_slots * bh * 2 * (size_t)D * plan.bk * sizeof(float);
    return part + (size_t)plan.n_split * bh * sizeof(unsigned);
}

template <int D, int KP>
static void launch_bwd_main_f32(const BwdParams& p, dim3 grid, hipStream_t s) {
    if (p.dq_direct)
        hipLaunchKernelGGL((bwd_main_kernel<D, KP, true, true>), grid, dim3(512), 0, s, p);
    else if (p.n_short > 0)
        hipLaunchKernelGGL((bwd_main_kernel<D, KP, true, false>), grid, dim3(512), 0, s, p);
    else
        hipLaunchKernelGGL((bwd_main_kernel<D, KP, false, false>), grid, dim3(512), 0, s, p);
}

template <int D, typename E>
static int launch_bwd_t(const BwdParams& p_in, hipStream_t s) {
    BwdParams p = p_in;
    // The bf16 main kernel at D <= 64 forms delta itself while staging each
    // query tile; bwd_pre then only zeroes, unless the query-major dQ pass
    // (which reads delta) follows.
    p.pre_delta = (sizeof(E) == 2 && D <= 64) ? p.dq_direct : 1;
    constexpr int RPB = 256 / (D / 4);
    const int64_t rows = (int64_t)p.B * p.H * p.Tq;
    const dim3 pre_grid((unsigned)((rows + RPB - 1) / RPB));  // bwd_cvt: 4 elements per thread
    constexpr int PRE_RPB = bwd_pre_rows_per_block<D, E>();
    const dim3 delta_grid((unsigned)(sizeof(E) == 4 ? (int64_t)p.B * p.H * p.n_amax : (rows + PRE_RPB - 1) / PRE_RPB));
    if (!p.pre_delta && !p.dq_direct) {
        // zeroing only: a few grid-stride workgroups per CU
        const int64_t n4 = rows * D / 4;
        const unsigned zb = (unsigned)std::min<int64_t>((n4 + 255) / 256, 2048);
        hipLaunchKernelGGL(bwd_zero_kernel, dim3(zb), dim3(256), 0, s, p);
    } else {
        hipLaunchKernelGGL((bwd_pre_kernel<D, E>), delta_grid, dim3(256), 0, s, p);
    }
    if constexpr (sizeof(E) == 2) {
        const int e = launch_bwd_main_bf16(p, s);
        if (e) return e;
        if (p.dq_direct) {
            const int e2 = launch_bwd_dq_bf16(p, s);
            if (e2) return e2;
        } else {
            const bool dense = p.sdq.t == D && p.sdq.h == (int64_t)p.Tq * D && p.sdq.b == (int64_t)p.H * p.Tq * D &&
                               reinterpret_cast<uintptr_t>(p.dq) % 16 == 0;
            if (dense)
                hipLaunchKernelGGL(bwd_cvt_flat_kernel, dim3((unsigned)((rows * D / 8 + 255) / 256)), dim3(256), 0, s, p);
            else
                hipLaunchKernelGGL((bwd_cvt_kernel<D>), pre_grid, dim3(256), 0, s, p);
        }
    } else {
        const dim3 grid((unsigned)(p.n_groups ? p.n_groups * bwd_padded_heads(p.B * p.H) : p.n_kblocks * p.B * p.H));
        if (p.keys_per_wg == 128)
            launch_bwd_main_f32<D, 32>(p, grid, s);
        else
            launch_bwd_main_f32<D, D >= 128 ? 32 : 64>(p, grid, s);
        if (p.dq_direct)
            hipLaunchKernelGGL((bwd_dq_kernel<D>), dim3((unsigned)(p.n_qtiles * p.B * p.H)), dim3(256), 0, s, p);
    }
    return (int)hipGetLastError();
}

int launch_attn_bwd(const BwdParams& p, int bf16, hipStream_t s) {
    switch (p.D) {
        case 32: return bf16 ? launch_bwd_t<32, uint16_t>(p, s) : launch_bwd_t<32, float>(p, s);
        case 64: return bf16 ? launch_bwd_t<64, uint16_t>(p, s) : launch_bwd_t<64, float>(p, s);
        case 128: return bf16 ? launch_bwd_t<128, uint16_t>(p, s) : launch_bwd_t<128, float>(p, s);
        default: return (int)hipErrorInvalidValue;
    }
}

}  // namespace inf
