// attn_bwd.hip -- fused causal attention backward for gfx950 (recompute).
//
// Kernel 1 (bwd_pre): delta[i] = sum_d dO[i,d] * O[i,d] per query row (the
// row dot that SoftmaxBackward computes as sum_j dP_ij P_ij), and zeroes the
// fp32 dQ accumulator.  (The bf16 main kernel at D <= 64 forms delta itself, and
// then this pass only zeroes.)
//
// Kernel 2 (bwd_main, fp32): its products run on the bf16 matrix cores, every
// operand split into three bf16 parts (common.h), six MFMAs per product step.
// One workgroup = 8 waves = 4 pairs, each pair with 64 keys (or 32) of one
// (b, h).  In a pair, wave 0 (role 0) has the keys' K operand and dV^T
// accumulators, wave 1 (role 1) their V operand and dK^T accumulators, so two
// waves fit a SIMD, one of each role.  dK and dV are written exactly once, with no
// atomics.  The workgroup walks query tiles of 32 rows, split into LDS once for all
// waves; per tile, in three phases with a barrier after each:
//
//   A  role 0: S = Q K^T, P = exp2(S c - lse log2e) (masked entries exactly 0),
//      P handed to role 1 through LDS;   role 1: dP = dO V^T
//   B  role 0: dV^T += dO^T P;   role 1: dS = P (dP - delta), its parts to LDS,
//      dK^T += Q^T dS
//   C  role 0: dQ tile += dS K over the workgroup's keys, fp32 atomics into the
//      global accumulator;   both: the next tile into LDS
//
// Keys lie on the lane axis in S, dP, dV^T and dK^T, so P and dS are operands
// straight from the accumulators; dO^T, Q^T, dS and K^T are transposed LDS reads.
// The K rows' h and m parts lie in LDS, their l parts in registers, V in registers
// as fp32 (its parts don't fit; split again for each tile).  S is formed in the
// forward's order, to the same bits, so P is consistent with the LSE.
// Bound by the MFMAs: 51% busy at D = 128 (7680 of 15000 cycles per tile and SIMD) at a
// clock that the load holds at 2.0 GHz, which is 1.07 PFLOP/s of them where a large
// library product reaches 1.25; at D = 64 (39% busy) also by the phases' latency.
// Against the fp32 MFMAs, the backward call (us): config 2 308 -> 248, config 4 5980 ->
// 3870.  Two scaled fp16 parts and three MFMAs took 163 and 2170, but blocks shared
// a scale: a block of zero keys gave infinities, small rows lost bits.
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
    const int64_t row = (int64_t)blockIdx.x * RPB + tid / TPR;
    const bool in = row < rows;
    float s = 0.f;
    if (in) {
        int64_t b, h, i;
        bwd_row_split(p, rows, row, b, h, i);
        if (p.pre_delta) {
            const E* po = (const E*)p.o + b * p.so.b + h * p.so.h + i * p.so.t + VEC * c;
            const E* pd = (const E*)p.dout + b * p.sdo.b + h * p.sdo.h + i * p.sdo.t + VEC * c;
            if constexpr (sizeof(E) == 4) {
                const f32x4 o4 = ld4(po), d4 = ld4(pd);
                s = o4[0] * d4[0] + o4[1] * d4[1] + o4[2] * d4[2] + o4[3] * d4[3];
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
    // Rows in LDS (bf16 elements), without padding: the 16-byte units of a row are
    // permuted by its number, so that row reads (one unit of 8 rows at a time) and
    // transposed reads (64 bytes of 4 rows) both touch every bank once.
    static constexpr int QS = D;
    static constexpr int SS = 36;                  // dS row stride (queries of one key, bf16 elements)
    static __device__ __forceinline__ int swz(int row) {
        return D == 128 ? 4 * (row & 3) ^ ((row >> 2) & 3) : D == 64 ? 4 * ((row >> 1) & 1) ^ ((row >> 2) & 3) : (row >> 2) & 3;
    }
    // Byte offset of the 8 columns from 8 * unit of a row.
    static __device__ __forceinline__ uint32_t at(int row, int unit) { return (uint32_t)(row * QS * 2 + 16 * (unit ^ swz(row))); }
    // A lane's offset for the row operands of 32 rows (row lane % 32, columns 8 (lane /
    // 32) ..) and for the transposed ones (rows 4 (lane / 32) + {0..3}).
    static __device__ __forceinline__ uint32_t row_lane(int lane) { return at(lane & 31, lane >> 5); }
    static __device__ __forceinline__ uint32_t tr_lane(int lane) {
        return at(4 * (lane >> 5) + ((lane & 15) >> 2), 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1)) + 8 * (lane & 1);
    }
    // From a lane's offset (in LDS at `lds`, the tile's start a multiple of 256) one
    // part of the operand: the row operand of MFMA step kk (columns 16 kk ..), and the
    // transposed one with columns 32 db + lane % 32 as its rows and rows row0 + 4 (lane
    // / 32) + {0..3} and + 8 (row0 a multiple of 16) as reduction index.  The unit's
    // permutation makes a step of columns (and of 8 rows) an exclusive or.
    static __device__ __forceinline__ bf16x8 row_part(const char* lds, uint32_t off, int kk, int bytes) {
        return *reinterpret_cast<const bf16x8*>(lds + (off ^ (uint32_t)(32 * kk)) + bytes);
    }
    static __device__ __forceinline__ bf16x8 tr_part(const char* lds, uint32_t off, int row0, int db, int bytes) {
        const char* lo = lds + (off ^ (uint32_t)(64 * db)) + row0 * QS * 2 + bytes;
        const char* hi = lds + (off ^ (uint32_t)(64 * db ^ 32)) + (row0 + 8) * QS * 2 + bytes;
        return __builtin_shufflevector(ds_read_tr16(reinterpret_cast<const __bf16*>(lo)),
                                       ds_read_tr16(reinterpret_cast<const __bf16*>(hi)), 0, 1, 2, 3, 4, 5, 6, 7);
    }
    // All three parts, `part` bytes apart.
    static __device__ __forceinline__ Bf3x8 row_frag(const char* lds, uint32_t off, int kk, int part) {
        return Bf3x8{row_part(lds, off, kk, 0), row_part(lds, off, kk, part), row_part(lds, off, kk, 2 * part)};
    }
    static __device__ __forceinline__ Bf3x8 tr_frag(const char* lds, uint32_t off, int row0, int db, int part) {
        return Bf3x8{tr_part(lds, off, row0, db, 0), tr_part(lds, off, row0, db, part), tr_part(lds, off, row0, db, 2 * part)};
    }
    static __device__ __forceinline__ void put(char* at, const Bf3x8& y, int part) {
        *reinterpret_cast<bf16x8*>(at) = y.h;
        *reinterpret_cast<bf16x8*>(at + part) = y.m;
        *reinterpret_cast<bf16x8*>(at + 2 * part) = y.l;
    }
};

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
    constexpr int PART = BQ * QS * 2;      // bytes of one part of a Q or dO tile
    constexpr int KPART = BK * QS * 2;     // ... and of the K rows
    constexpr int XB = 32 * SS * 2;        // bytes of one dS part of a 32-key block
    constexpr int XPAIR = NKB * 3 * XB;
    constexpr int DQP = NDB;               // dQ: pairs of keys per wave (4 / NDB waves share a head-dim block)
    static_assert(DQP * 2 == NKK, "as many dQ steps as S steps");

    // LDS: the h and m parts of the workgroup's K rows, the Q tile and the dO tile
    // (three parts each), and for each pair P (fp32), then dS (three parts).
    constexpr int Q_OFF = 2 * KPART, DO_OFF = Q_OFF + 3 * PART, X_OFF = DO_OFF + 3 * PART;
    __shared__ __attribute__((aligned(256))) char lds[X_OFF + 4 * XPAIR];
    __shared__ __attribute__((aligned(16))) float lse_s[BQ];
    __shared__ __attribute__((aligned(16))) float dl_s[BQ];
    __shared__ __attribute__((aligned(16))) float dlo_s[SHORT ? BQ : 4];

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

    // Role 1's threads stage the Q tiles, role 0's the dO tiles, wave 0 the rows'
    // LSE and delta.  Rows at or past `lim` read as zeros.
    const int ts = tid & 255;
    const float* Y = role ? Q : dO;
    const int64_t yt = role ? p.sq.t : p.sdo.t;
    const uint32_t y_voff = (uint32_t)(((int64_t)(ts / C8) * yt + 8 * (ts % C8)) * 4);
    f32x4 yr[CPT][2];
    float r_row = 0.f, r_dlo = 0.f;  // thread ts < 32: row ts's LSE (and delta's low part), 32 + r: row r's delta
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
            const auto rl = row_rsrc(LSE, 1, q0, rows, 1), rd = row_rsrc(DL, 1, q0, rows, 1);
            if (wave == 0) {
                const uint32_t off = (uint32_t)l32 * 4;
                r_row = g == 0 ? buffer_ld1(rl, off, 0) : buffer_ld1(rd, off, 0);
                if constexpr (SHORT) {
                    const int n_sh = kblk == 0 ? max(0, min(p.n_short - q0, rows)) : 0;
                    r_dlo = buffer_ld1(row_rsrc(DLO, 1, q0, n_sh, 1), off, 0);
                }
            }
        }
    };
    // Everything that the workgroup starts from is loaded at once: its operand rows
    // (K or V rows of the pair's keys: MFMA step kk takes row key, columns 16 kk + 8
    // g .. + 7), the K^T operand of dQ and the first Q / dO tile.
    //   role 1: xr is the V rows in fp32, two thirds of the registers of their parts,
    //     split again for each tile;
    //   role 0: K's h and m parts go to LDS, where row reads serve S and transposed
    //     reads dQ; xr[..][0] is the l part in S's layout and xr[..][1], in entry
    //     step, the one in dQ's.
    f32x4 xr[NKB][NKK][2];
    bool k_past = false;
    const float* X = role ? (const float*)p.v + b * p.sv.b + h * p.sv.h : (const float*)p.k + b * p.sk.b + h * p.sk.h;
    const int64_t xt = role ? p.sv.t : p.sk.t;
    {
#pragma unroll
        for (int kb = 0; kb < NKB; ++kb) {
            const int key = k0p + kb * 32 + l32;
#pragma unroll
            for (int kk = 0; kk < NKK; ++kk) {
                xr[kb][kk][0] = xr[kb][kk][1] = f32x4{0.f, 0.f, 0.f, 0.f};
                if (key < p.Tk) {
                    xr[kb][kk][0] = ld4(X + (int64_t)key * xt + 16 * kk + 8 * g);
                    xr[kb][kk][1] = ld4(X + (int64_t)key * xt + 16 * kk + 8 * g + 4);
                }
            }
        }
        gload(q_begin, p.Tq);
        if (role == 0) {
#pragma unroll
            for (int kb = 0; kb < NKB; ++kb) k_past |= any_past_bf16(xr[kb]);
#pragma unroll
            for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
                for (int kk = 0; kk < NKK; ++kk) {
                    const Bf3x8 k = split3<true>(xr[kb][kk][0], xr[kb][kk][1]);
                    char* at = lds + T::at(pr * KP + 32 * kb + l32, 2 * kk + g);
                    *reinterpret_cast<bf16x8*>(at) = k.h;
                    *reinterpret_cast<bf16x8*>(at + KPART) = k.m;
                    xr[kb][kk][0] = __builtin_bit_cast(f32x4, k.l);
                }
            if constexpr (!DQD) {
#pragma unroll
                for (int st = 0; st < NKB * NKK; ++st) {  // step st: pair pr / NDB * DQP + st / (2 NKB), ...
                    const int pp = pr / NDB * DQP + st / (2 * NKB);
                    const int row0 = k0 + pp * KP;
                    const auto rk = row_rsrc(X, xt, row0, min(p.Tk - row0, KP), D);
                    f32x4 kt[2];
#pragma unroll
                    for (int e = 0; e < 8; ++e)  // ... keys 16 (st % (2 NKB)) + 4 g + {0..3} and + 8, column 32 (pr % NDB) + l32
                        kt[e >> 2][e & 3] =
                            buffer_ld1(rk, (uint32_t)(((int64_t)(16 * (st % (2 * NKB)) + 4 * g) * xt + 32 * (pr % NDB) + l32) * 4),
                                       (uint32_t)((int64_t)((e & 3) + 8 * (e >> 2)) * xt * 4));
                    xr[st / NKK][st % NKK][1] = __builtin_bit_cast(f32x4, split3<true>(kt[0], kt[1]).l);
                }
            }
        }
    }
    // This lane's LDS offsets: row operands of the tile whose scores the wave forms
    // and of its pair's keys, transposed operands of the tile that it sums into dV or
    // dK and of K, dS as the dQ product reads it.  Each passes an empty asm per tile:
    // what is derived from them is formed again instead of being held (and spilled).
    uint32_t row_off = (role ? DO_OFF : Q_OFF) + T::row_lane(lane), krow_off = pr * KP * QS * 2 + T::row_lane(lane);
    uint32_t tr_off = (role ? Q_OFF : DO_OFF) + T::tr_lane(lane), ktr_off = pr / NDB * DQP * KP * QS * 2 + T::tr_lane(lane);
    uint32_t ds_off = X_OFF + pr / NDB * DQP * XPAIR + (4 * g + ((lane & 15) >> 2)) * SS * 2 + 32 * ((lane >> 4) & 1) + 8 * (lane & 3);
    auto fresh_off = [&]() { asm volatile("" : "+v"(row_off), "+v"(krow_off), "+v"(tr_off), "+v"(ktr_off), "+v"(ds_off)); };
    const uint32_t st_off = (role ? Q_OFF : DO_OFF) + T::at(ts / C8, ts % C8);
    // The split parts of role 1's rows don't change from tile to tile: an empty asm
    // per tile keeps them from being formed once and held (or spilled).
    auto fresh_xr = [&]() {
#pragma unroll
        for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
            for (int kk = 0; kk < NKK; ++kk) asm volatile("" : "+v"(xr[kb][kk][0]), "+v"(xr[kb][kk][1]));
    };
    // The S (role 0) or dP (role 1) chains of the staged tile and the pair's keys;
    // SWAP: queries as the MFMA's rows (the main loop), else keys (the short rows),
    // in the same order, to the same bits.  Scores of keys with an infinity are formed
    // from memory in plain fp32: a key that scores -inf has probability 0, and
    // dK and dV of 0.  (Infinities in q, v and dO leave nothing finite that they meet.)
    auto scores = [&](f32x16 (&s)[NKB], int q0, auto swap_c) {
        constexpr bool SWAP = decltype(swap_c)::value;
        fresh_xr();
        fresh_off();
        Split3Sum sum;
        auto add = [&](const Bf3x8& y, const Bf3x8& x) {
            if constexpr (SWAP)
                mfma_split3<true>(y, x, sum);
            else
                mfma_split3<false>(x, y, sum);
        };
        // a step's LDS operands are read while the step before runs
        constexpr int N = NKB * NKK;
        if (k_past) {  // (role 0)
            const float* yp = q0 + l32 < p.Tq ? Q + (int64_t)(q0 + l32) * p.sq.t : nullptr;
#pragma unroll
            for (int kb = 0; kb < NKB; ++kb) {
                const int key = k0p + 32 * kb + l32;
                const float* xp = key < p.Tk ? X + (int64_t)key * xt : nullptr;
                s[kb] = SWAP ? dot_rows_f32<D>(yp, xp, g) : dot_rows_f32<D>(xp, yp, g);
            }
        } else if (role == 0) {
            Bf3x8 y[2];
            y[0] = T::row_frag(lds, row_off, 0, PART);
            bf16x8 k[2][2];
            auto k_read = [&](int st) {
                k[st & 1][0] = T::row_part(lds, krow_off, st % NKK, 32 * (st / NKK) * QS * 2);
                k[st & 1][1] = T::row_part(lds, krow_off, st % NKK, 32 * (st / NKK) * QS * 2 + KPART);
            };
            if constexpr (NKB == 1) k_read(0);
#pragma unroll
            for (int st = 0; st < N; ++st) {
                if constexpr (NKB > 1) k_read(st);  // (the registers of another step's K don't fit)
                if (st + 1 < N) {
                    y[(st + 1) & 1] = T::row_frag(lds, row_off, (st + 1) % NKK, PART);
                    if constexpr (NKB == 1) k_read(st + 1);
                }
                if (st % NKK == 0) sum.hi = sum.lo = f32x16{};
                __builtin_amdgcn_sched_barrier(0);
                add(y[st & 1], Bf3x8{k[st & 1][0], k[st & 1][1], __builtin_bit_cast(bf16x8, xr[st / NKK][st % NKK][0])});
                __builtin_amdgcn_sched_barrier(0);
                if (st % NKK == NKK - 1) s[st / NKK] = sum.sum();
            }
        } else {
#pragma unroll
            for (int st = 0; st < N; ++st) {
                const Bf3x8 y = T::row_frag(lds, row_off, st % NKK, PART);  // (while the rows are split)
                if (st % NKK == 0) sum.hi = sum.lo = f32x16{};
                __builtin_amdgcn_sched_barrier(0);
                add(y, split3(xr[st / NKK][st % NKK][0], xr[st / NKK][st % NKK][1]));
                __builtin_amdgcn_sched_barrier(0);
                if (st % NKK == NKK - 1) s[st / NKK] = sum.sum();
            }
        }
    };

    auto sstore = [&]() {
#pragma unroll
        for (int i = 0; i < CPT; ++i) {
            const int f = ts + 256 * i;
            const Bf3x8 y = split3<true>(yr[i][0], yr[i][1]);
            if (NCH % 256 == 0 || f < NCH) {
                T::put(lds + st_off + 256 / C8 * i * QS * 2, y, PART);  // (rows 16 or more apart: the same units)
            }
        }
        if (wave == 0) {
            if (g == 0) {
                lse_s[l32] = r_row * kLog2e;
                if constexpr (SHORT) dlo_s[l32] = r_dlo;
            } else {
                dl_s[l32] = r_row;
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
        // pairs (sum e, sum e dP) of each pair of waves, behind its P
        constexpr int PSTRIDE = XPAIR / 16;
        double* part = reinterpret_cast<double*>(lds + X_OFF + NKB * 4096);
        static_assert(2 * BQ * sizeof(double) + NKB * 4096 <= XPAIR && XPAIR % 16 == 0, "the sums fit behind P");
        for (int q0 = q_begin; q0 < qs_end; q0 += BQ) {
            sstore();
            __syncthreads();
            gload(q0 + BQ, q0 + BQ < qs_end ? p.Tq : 0);
            const bool active = (!p.causal || (q0 + BQ - 1 + p.off >= k0p)) && k0p < p.Tk;
            f32x16 st[NKB];
            f32x4* X = reinterpret_cast<f32x4*>(lds + X_OFF + pr * XPAIR);
            if (active) {
                scores(st, q0, std::false_type{});
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
                                e[cc] = bwd_short_weight(p, qi, vis, fast_exp2(fmaf(st[kb][4 * j + cc], p.c, -L)));
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
                    part[2 * (pr * PSTRIDE + l32)] = l;
                    part[2 * (pr * PSTRIDE + l32) + 1] = w;
                }
            }
            __syncthreads();
            if (tid < BQ) bwd_short_delta_store<4, PSTRIDE>(p, bh, q0 + tid, part + 2 * tid);
        }
        __syncthreads();  // the deltas are stored: the first tile's are read again
        gload(q_begin, p.Tq);
    }

    f32x16 acc[NDB][NKB];  // dV^T (role 0) or dK^T (role 1): row d, column key
#pragma unroll
    for (int db = 0; db < NDB; ++db)
#pragma unroll
        for (int kb = 0; kb < NKB; ++kb) acc[db][kb] = f32x16{};

    sstore();
    __syncthreads();

    for (int q0 = q_begin; q0 < q_end; q0 += BQ) {
        // ---- A: S and P (role 0), dP (role 1) -----------------------------------
        gload(q0 + BQ, q0 + BQ < q_end ? p.Tq : 0);
        // Does any query of this tile see any key of a pair (of this one)?
        auto sees = [&](int key0) { return (!p.causal || (q0 + BQ - 1 + p.off >= key0)) && key0 < p.Tk; };
        const bool active = sees(k0p);
        f32x4* X = reinterpret_cast<f32x4*>(lds + X_OFF + pr * XPAIR);
        f32x16 s[NKB];
        if (active) {
            scores(s, q0, std::true_type{});
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
                                float pv = fast_exp2(fmaf(s[kb][4 * j + cc], p.c, -L[cc]));
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

        // ---- B: dV (role 0), dS and dK (role 1) ------------------------------------
        if (active) {
            if (role == 1) {
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
                            float t = s[kb][4 * j + cc] - Dl[cc];
                            if constexpr (SHORT) t -= Dlo[cc];
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
                // (dS goes over P below, which this wave has read)
                asm volatile("" ::: "memory");
            }
            // dV^T += dO^T P or dK^T += Q^T dS, rows read transposed; step mm takes
            // queries 16 mm + 4 g + {0..3} and + 8
            // (a step's rows are read while the step before runs where their registers fit)
            constexpr bool AHEAD = NKB == 1;
            Bf3x8 pb[NKB], a[2];
            if constexpr (AHEAD) a[0] = T::tr_frag(lds, tr_off, 0, 0, PART);
#pragma unroll
            for (int st = 0; st < 2 * NDB; ++st) {
                const int mm = st / NDB, db = st % NDB;
                if (db == 0) {
#pragma unroll
                    for (int kb = 0; kb < NKB; ++kb) {
                        const f32x16& e = s[kb];
                        pb[kb] = split3<true>(f32x4{e[8 * mm], e[8 * mm + 1], e[8 * mm + 2], e[8 * mm + 3]},
                                              f32x4{e[8 * mm + 4], e[8 * mm + 5], e[8 * mm + 6], e[8 * mm + 7]});
                        if (role == 1 && !DQD) {  // row key l32, queries along it
                            auto put = [&](int part, const bf16x8& v) {
                                char* row = lds + X_OFF + pr * XPAIR + (3 * kb + part) * XB + (l32 * SS + 16 * mm + 4 * g) * 2;
                                *reinterpret_cast<bf16x4*>(row) = __builtin_shufflevector(v, v, 0, 1, 2, 3);
                                *reinterpret_cast<bf16x4*>(row + 16) = __builtin_shufflevector(v, v, 4, 5, 6, 7);
                            };
                            put(0, pb[kb].h);
                            put(1, pb[kb].m);
                            put(2, pb[kb].l);
                        }
                    }
                }
                const int rd = AHEAD ? st + 1 : st;
                if (rd < 2 * NDB) a[rd & 1] = T::tr_frag(lds, tr_off, 16 * (rd / NDB), rd % NDB, PART);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int kb = 0; kb < NKB; ++kb) {
                    acc[db][kb] = mfma_split3_once(a[st & 1], pb[kb], acc[db][kb]);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        }
        __syncthreads();

        // ---- C: dQ (role 0), the next tile (both) -----------------------------------
        sstore();
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
                struct Ops {
                    Bf3x8 ds;
                    bf16x8 kh, km;
                };
                // step st: pair pr / NDB * DQP + st / (2 NKB), keys 16 (st % (2 NKB)) .. + 15 of it
                auto ops = [&](int st) {
                    const int pi = st / (2 * NKB), kb = st % (2 * NKB) / 2, m = st % 2;
                    auto ds_part = [&](int part) {
                        const char* at = lds + ds_off + pi * XPAIR + (3 * kb + part) * XB + 16 * m * SS * 2;
                        return __builtin_shufflevector(ds_read_tr16(reinterpret_cast<const __bf16*>(at)),
                                                       ds_read_tr16(reinterpret_cast<const __bf16*>(at + 8 * SS * 2)), 0, 1, 2, 3, 4, 5, 6, 7);
                    };
                    const int row0 = pi * KP + 32 * kb + 16 * m;
                    Ops o;
                    o.ds.h = ds_part(0);
                    o.ds.m = ds_part(1);
                    o.ds.l = ds_part(2);
                    o.kh = T::tr_part(lds, ktr_off, row0, db, 0);
                    o.km = T::tr_part(lds, ktr_off, row0, db, KPART);
                    return o;
                };
                auto mul = [&](const Ops& o, int st) {
                    dq = mfma_split3(o.ds, Bf3x8{o.kh, o.km, __builtin_bit_cast(bf16x8, xr[st / NKK][st % NKK][1])}, dq);
                };
                const int pp0 = pr / NDB * DQP;
                if (sees(k0 + (pp0 + DQP - 1) * KP)) {
                    Ops o[2];
                    o[0] = ops(0);
#pragma unroll
                    for (int st = 0; st < NKB * NKK; ++st) {
                        if (st + 1 < NKB * NKK) o[(st + 1) & 1] = ops(st + 1);
                        __builtin_amdgcn_sched_barrier(0);
                        mul(o[st & 1], st);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                } else {
                    // (a pair that no row sees wrote no dS, and its keys must not reach these rows)
#pragma unroll
                    for (int pi = 0; pi < DQP; ++pi)
                        if (sees(k0 + (pp0 + pi) * KP)) {
#pragma unroll
                            for (int i = 0; i < 2 * NKB; ++i) mul(ops(pi * 2 * NKB + i), pi * 2 * NKB + i);
                        }
                }
                const auto rdq = row_rsrc(dQa, p.sacc.t, q0, min(p.Tq - q0, BQ), D);  // rows past Tq are dropped
                const uint32_t voff = (uint32_t)(((int64_t)(4 * g) * p.sacc.t + db * 32 + l32) * 4);
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    buffer_atomic_add(rdq, dq[r] * p.scale, voff, (uint32_t)((int64_t)(8 * (r >> 2) + (r & 3)) * p.sacc.t * 4));
            }
        }
        __syncthreads();
    }

    // ---- dK = scale * dK^T^T, dV = dV^T^T ------------------------------------------
    const float unit = role ? p.scale : 1.f;
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
// (the B operands Q^T, dO^T, split for each tile) in VGPRs, with that row's
// log-sum-exp and delta; tiles of 32 keys of K and V, split, are double-buffered in
// LDS (loaded two tiles ahead).  Per wave and tile:
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
    using T = BwdTile<D, 32>;
    constexpr int PART = BN * T::QS * 2, K_OFF = 0, V_OFF = 6 * PART;
    static_assert(BM == 128 && 256 % C8 == 0, "4 waves x 32 rows, whole staging passes");

    __shared__ __attribute__((aligned(256))) char lds[12 * PART];  // K, then V: [buffer][part]

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31;
    const int g = lane >> 5;

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
    // B operands: MFMA step kk takes row qrow, columns 16 kk + 8 g .. + 7, split for each tile.
    f32x4 qr[NKK][2], dr[NKK][2];
    auto load_row = [&](const float* src, int64_t st, f32x4 (&f)[NKK][2]) {
#pragma unroll
        for (int kk = 0; kk < NKK; ++kk) {
            f[kk][0] = f[kk][1] = f32x4{0.f, 0.f, 0.f, 0.f};
            if (qrow < p.Tq) {
                f[kk][0] = ld4(src + (int64_t)qrow * st + 16 * kk + 8 * g);
                f[kk][1] = ld4(src + (int64_t)qrow * st + 16 * kk + 8 * g + 4);
            }
        }
    };
    load_row(Q, p.sq.t, qr);
    load_row(dO, p.sdo.t, dr);
    const float Lq = qrow < p.Tq ? p.lse[(int64_t)bh * p.Tq + qrow] * kLog2e : 0.f;
    const float Dq = qrow < p.Tq ? p.delta[(int64_t)bh * p.Tq + qrow] : 0.f;
    const float Dqlo = bwd_short_row(p, qrow) ? p.delta_lo[(int64_t)bh * p.Tq + qrow] : 0.f;
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
    auto sstore = [&](const Raw& r, int buf) {
#pragma unroll
        for (int i = 0; i < CPT; ++i) {
            const int f = tid + 256 * i;
            if (NCH % 256 == 0 || f < NCH) {
                char* at = lds + 3 * buf * PART + T::at(f / C8, f % C8);
                T::put(at + K_OFF, split3<true>(r.k[i][0], r.k[i][1]), PART);
                T::put(at + V_OFF, split3(r.v[i][0], r.v[i][1]), PART);
            }
        }
    };

    f32x16 dq[NDB];
#pragma unroll
    for (int i = 0; i < NDB; ++i) dq[i] = f32x16{};

    Raw ra, rb;
    gload(ra, 0);
    gload(rb, 1);
    sstore(ra, 0);
    __syncthreads();
    auto step = [&](int u, Raw& nxt, Raw& far) {
        const int buf = u & 1;
        const int k0 = u * BN;
        gload(far, u + 2);
#pragma unroll
        for (int kk = 0; kk < NKK; ++kk)  // split again for each tile, not held (as in the main kernel)
            asm volatile("" : "+v"(qr[kk][0]), "+v"(qr[kk][1]), "+v"(dr[kk][0]), "+v"(dr[kk][1]));
        if (k0 < wave_kend) {
            Split3Sum ss, dps;
            ss.hi = ss.lo = dps.hi = dps.lo = f32x16{};
#pragma unroll
            for (int kk = 0; kk < NKK; ++kk) {
                mfma_split3(T::row_frag(lds + K_OFF + 3 * buf * PART, T::row_lane(lane), kk, PART), split3(qr[kk][0], qr[kk][1]), ss);
                mfma_split3(T::row_frag(lds + V_OFF + 3 * buf * PART, T::row_lane(lane), kk, PART), split3(dr[kk][0], dr[kk][1]), dps);
            }
            f32x16 s = ss.sum(), dp = dps.sum();
            if (any_nonfinite(s))  // (as in the main kernel)
                s = dot_rows_f32<D>(k0 + l32 < p.Tk ? K + (int64_t)(k0 + l32) * p.sk.t : nullptr,
                                    qrow < p.Tq ? Q + (int64_t)qrow * p.sq.t : nullptr, g);
            // reg r: key k0 + 8 (r / 4) + 4 g + r % 4 of query qrow
            const bool need_mask = (k0 + BN > p.Tk) || (qtile * BM + BM > p.Tq) || (p.causal && (k0 + BN - 1 > q0w + p.off));
            const int lim = p.causal ? min(p.Tk - 1, qrow + p.off) : p.Tk - 1;
            // the visibility test only on tiles that cross the diagonal or the ends
            auto p_ds = [&](auto masked) {
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    float pr = fast_exp2(fmaf(s[r], p.c, -Lq));
                    if constexpr (decltype(masked)::value) {
                        const int key = k0 + 8 * (r >> 2) + 4 * g + (r & 3);
                        pr = (key <= lim && qrow < p.Tq) ? pr : 0.f;
                    }
                    s[r] = pr * ((dp[r] - Dq) - Dqlo);  // dS^T
                }
            };
            if (need_mask)
                p_ds(std::true_type{});
            else
                p_ds(std::false_type{});
            if (one_key_wave && k0 == 0 && one_key) s = f32x16{};  // one visible key: dS = P (dP - dP) = 0
            // dQ^T[d][q] += K^T[d][keys] dS^T[keys][q]: step m takes keys 16 m + 4 g + {0..3} and + 8
#pragma unroll
            for (int m = 0; m < 2; ++m) {
                const Bf3x8 ds = split3(f32x4{s[8 * m], s[8 * m + 1], s[8 * m + 2], s[8 * m + 3]},
                                        f32x4{s[8 * m + 4], s[8 * m + 5], s[8 * m + 6], s[8 * m + 7]});
#pragma unroll
                for (int db = 0; db < NDB; ++db)
                    dq[db] = mfma_split3(T::tr_frag(lds + K_OFF + 3 * buf * PART, T::tr_lane(lane), 16 * m, db, PART), ds, dq[db]);
            }
        }
        sstore(nxt, buf ^ 1);
        __syncthreads();
    };
    for (int u = 0; u < nt; u += 2) {
        step(u, rb, ra);
        if (u + 1 < nt) step(u + 1, ra, rb);
    }
    if (qrow < p.Tq) {
        float* dst = (float*)p.dq + b * p.sdq.b + h * p.sdq.h + (int64_t)qrow * p.sdq.t;
#pragma unroll
        for (int db = 0; db < NDB; ++db)
#pragma unroll
            for (int j = 0; j < 4; ++j)
                st4(dst + db * 32 + 8 * j + 4 * g,
                    f32x4{dq[db][4 * j], dq[db][4 * j + 1], dq[db][4 * j + 2], dq[db][4 * j + 3]} * p.scale);
    }
}

// ---- split plan (host) ------------------------------------------------------------
//
// Under a causal mask key block j has ~(Tq - bk j) / 32 query tiles, so the first key
// blocks carry many times the work of the last, and the heaviest workgroups set the
// kernel's length.  bwd_plan simulates the dispatch (workgroup w to XCD w % 8, each
// XCD's workgroups placed in order on its least-loaded CU with a free slot) for
// splits of the heaviest key blocks' tile ranges into chunks, and keeps the best if it
// beats the unsplit order by 3%.
//
// fp32 (one workgroup per CU): against splits forced into halves to eighths, at 77
// shapes of 1 to 192 heads, T 100 to 8192, D 32 to 128, the plan's choice is within 5%
// of the fastest but for B H 4, T 512, D 128 (48 and 45 us); without a split 2 to 5
// times as slow at few heads (1 x 1024 x 64 136 us, split 41).

static constexpr double kBwdPairGain = 0.08;  // throughput gained per extra resident workgroup (bf16 at D = 32: two per CU)
// Per-workgroup fixed cost (K/V loads, K staging) and the partial store /
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
    const int bk = bwd_keys_per_wg(bf16, D, BH, Tq, Tk, 1);
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
    // pro.  The chunk size is chosen with pro = 0 (block 0's short tiles alone must
    // not move it); the cuts of block 0 are then made with the prologue's share.
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
    out->bk = bwd_keys_per_wg(bf16, D, (int64_t)B * H, Tq, Tk, 1);
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
    const dim3 delta_grid((unsigned)((rows + PRE_RPB - 1) / PRE_RPB));
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
