// attn_fwd.hip -- fused causal attention forward for gfx950, fp32.
//
// One workgroup = 8 waves = 256 query rows of one (b, h); each wave owns 32
// rows for the whole kernel.  Both products run on the bf16 matrix cores, every
// operand split into three bf16 parts (common.h), six MFMAs per product step: no
// scales, so a row depends on what it sees alone, at any magnitude.
// K and V tiles of BN keys are loaded two tiles ahead into registers, split
// once for all eight waves into double-buffered LDS, one barrier per tile.  Per
// wave and tile:
//
//   S^T (keys x queries) = K Q^T      v_mfma_f32_32x32x16_bf16, A = K from LDS,
//                                     B = Q^T resident in VGPRs, split
//   online softmax on S^T             query = lane%32, so the row max needs one
//                                     xor-32 exchange; the row sum stays
//                                     per-lane until the end; fp32
//   O^T (d x queries) += V^T P^T      A = V^T from LDS, B = P^T split from
//                                     the S^T accumulators (reduction index
//                                     permuted to match their layout)
//
// V lies transposed in LDS in the operand's order, one 16-byte read per operand
// part: a thread loads one column of the 8 keys that an operand takes together,
// so the transposition costs no store.
//
// At D = 128 the kernel keeps the matrix cores 67% busy at a shader clock that the
// load holds at 1.9 GHz (VALU work, 30% of the issue slots, overlaps in part): 1.65
// PFLOP of MFMAs in 1.27 ms, the rate of a large library product in bf16.  At D = 64 a
// workgroup's serial chain of tiles sets causal grids of a round or two (51% busy).
// Against the fp32 MFMAs (us): config 2 128.8 -> 82.6, config 4 2281 -> 1270.  Two
// fp16 parts per operand, scaled by the largest value of a tile, and three MFMAs took
// 58.4 and 726, but a value 2^10 below its tile's largest lost bits, also to a key
// that the row can't see.  128-row workgroups of four waves split each tile twice as
// often.
//
// Keeping queries on the lane axis in both products is what lets P stay in
// registers.  The scale is folded into exp2: p = exp2(s*c - m) with
// c = scale*log2(e).  Masked scores (key > query + Tk - Tq, or key >= Tk)
// become -inf, so their probabilities are exactly 0, as the reference's
// -1e9f fill followed by exp((double)(-1e9 - max)) is.  The row
// log-sum-exp (natural log) is stored for the backward pass.
//
// Scheduling: dispatch group g = w / (B*H) of head w % (B*H).  Without a
// split plan, group g is query tile n_qtiles - 1 - g, so the longest causal
// rows start first; when B*H is a multiple of 8, all tiles of a head land on
// the same XCD (dispatch is round-robin over the 8 XCDs), so a head's K/V is
// fetched into one L2.  With a split plan (fwd_plan, causal shapes whose
// heaviest query tiles would otherwise set the makespan), the heaviest query
// tiles' key ranges are cut into chunks run by separate groups, the groups are
// ordered heaviest first, and each chunk leaves (unnormalised O, row max, row
// sum) in a workspace slot that attn_fwd_merge_kernel combines with the same
// log-sum-exp weighting as the decode combine.
#include <algorithm>
#include <array>
#include <functional>
#include <map>
#include <mutex>
#include <type_traits>
#include <vector>

#include "common.h"
#include "kernels.h"

namespace inf {

template <int D>
struct FwdTile {
    static constexpr int NW = 8;  // waves per workgroup, 32 query rows each
    static constexpr int BM = 32 * NW;
    static constexpr int BN = D == 32 ? 128 : D == 64 ? 64 : 32;  // keys per LDS tile: one 8-element unit per thread
    static constexpr int KS = D + 8;                              // K row stride in LDS (bf16 elements)
};

// Headroom of the forward's lazy rescaling, in exp2 units: P <= 2^8.
constexpr float kLazyLog2 = 8.f;

template <int D>
__global__ __launch_bounds__(64 * FwdTile<D>::NW, 2) void attn_fwd_kernel(FwdParams p) {
    constexpr int NT = 64 * FwdTile<D>::NW;
    constexpr int BM = FwdTile<D>::BM;
    constexpr int BN = FwdTile<D>::BN;
    constexpr int KS = FwdTile<D>::KS;
    constexpr int NKK = D / 16;          // MFMA steps along the head dim for S^T
    constexpr int NKB = BN / 32;         // 32-key blocks per tile
    constexpr int NDB = D / 32;          // 32-wide head-dim blocks of O^T
    constexpr int C8 = D / 8;            // 8-element chunks per K row
    constexpr int UPT = BN * C8 / NT;    // 8-element units per thread per tensor per tile
    static_assert(BN * C8 % NT == 0 && NT % D == 0 && NT % C8 == 0, "whole staging passes");

    __shared__ __attribute__((aligned(16))) __bf16 Ks0[3][BN][KS];
    __shared__ __attribute__((aligned(16))) __bf16 Ks1[3][BN][KS];
    __shared__ bf16x8 Vt0[3][BN / 8][D];
    __shared__ bf16x8 Vt1[3][BN / 8][D];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int l32 = lane & 31;
    const int g = lane >> 5;

    const int BH = p.B * p.H;
    const int w = blockIdx.x;
    int qtile, t_begin = 0, t_end = 0x7fffffff, slot = -1;
    if (p.n_groups) {
        const FwdGroup grp = p.groups[w / BH];
        qtile = grp.qt;
        t_begin = grp.t0;
        t_end = grp.t1;
        slot = grp.slot;
    } else {
        qtile = p.n_qtiles - 1 - w / BH;
    }
    const int bh = w % BH;
    const int b = bh / p.H;
    const int h = bh % p.H;

    const float* Q = (const float*)p.q + b * p.sq.b + h * p.sq.h;
    const float* K = (const float*)p.k + b * p.sk.b + h * p.sk.h;
    const float* V = (const float*)p.v + b * p.sv.b + h * p.sv.h;
    float* O = (float*)p.o + b * p.so.b + h * p.so.h;

    const int q0w = qtile * BM + wave * 32;  // first query row of this wave
    const int qrow = q0w + l32;              // this lane's query row

    // Q^T operand: MFMA step kk takes Q[qrow][16 kk + 8 g .. + 7].
    Bf3x8 qf[NKK];
#pragma unroll
    for (int kk = 0; kk < NKK; ++kk) {
        f32x4 a = f32x4{0.f, 0.f, 0.f, 0.f}, b2 = a;
        if (qrow < p.Tq) {
            a = ld4(Q + (int64_t)qrow * p.sq.t + 16 * kk + 8 * g);
            b2 = ld4(Q + (int64_t)qrow * p.sq.t + 16 * kk + 8 * g + 4);
        }
        qf[kk] = split3(a, b2);
    }

    // Keys this workgroup needs, and this wave's visible limit (exclusive).
    int kv_end = p.Tk;
    if (p.causal) kv_end = min(p.Tk, qtile * BM + BM + p.off);
    const int n_tiles = min((kv_end + BN - 1) / BN, t_end);
    const int wave_kend = p.causal ? min(kv_end, q0w + 32 + p.off) : kv_end;

    // K unit tid + NT i: row f / C8, 8 columns from 8 (f % C8): two 16-byte
    // loads.  V unit: column f % D of the 8 keys that the P V operand takes
    // together (keys 16 m + 4 g' + {0..3} and + 8 for key group f / D = 2 m + g'):
    // eight 4-byte loads, each a run of a row over the wave's lanes, so V lands
    // transposed without a transposing store.  Loads go through a buffer
    // resource per tile: rows at or past `lim` read as zeros.
    struct Raw {
        f32x4 k[UPT][2];
        float v[UPT][8];
    };
    const uint32_t k_voff = (uint32_t)(((int64_t)(tid / C8) * p.sk.t + 8 * (tid % C8)) * 4);
    auto vrow0 = [](int kg) { return 16 * (kg >> 1) + 4 * (kg & 1); };
    const uint32_t vd = (uint32_t)(tid % D) * 4;
    auto gload = [&](Raw& r, int t) {
        const int rows = t < n_tiles ? min(p.Tk - t * BN, BN) : 0;
        const auto rk = row_rsrc(K, p.sk.t, t * BN, rows, D);
        const auto rv = row_rsrc(V, p.sv.t, t * BN, rows, D);
#pragma unroll
        for (int i = 0; i < UPT; ++i) {
            const uint32_t so = (uint32_t)((int64_t)(NT * i / C8) * p.sk.t * 4);
            r.k[i][0] = buffer_ld4(rk, k_voff, so);
            r.k[i][1] = buffer_ld4(rk, k_voff + 16, so);
            const int r0 = __builtin_amdgcn_readfirstlane(vrow0((tid + NT * i) / D));  // D >= 64: wave-uniform
            const uint32_t v_voff = D >= 64 ? vd : (uint32_t)((int64_t)vrow0((tid + NT * i) / D) * p.sv.t * 4) + vd;
#pragma unroll
            for (int e = 0; e < 8; ++e)
                r.v[i][e] = buffer_ld1(rv, v_voff,
                                       (uint32_t)((int64_t)((D >= 64 ? r0 : 0) + (e & 3) + 8 * (e >> 2)) * p.sv.t * 4));
        }
    };
    auto v4 = [](const float (&v)[8], int j) { return f32x4{v[j], v[j + 1], v[j + 2], v[j + 3]}; };
    auto sstore = [&](const Raw& r, __bf16 (&Kd)[3][BN][KS], bf16x8 (&Vd)[3][BN / 8][D]) {
#pragma unroll
        for (int i = 0; i < UPT; ++i) {
            const int f = tid + NT * i;
            const Bf3x8 k = split3(r.k[i][0], r.k[i][1]);
            *reinterpret_cast<bf16x8*>(&Kd[0][f / C8][8 * (f % C8)]) = k.h;
            *reinterpret_cast<bf16x8*>(&Kd[1][f / C8][8 * (f % C8)]) = k.m;
            *reinterpret_cast<bf16x8*>(&Kd[2][f / C8][8 * (f % C8)]) = k.l;
            const Bf3x8 v = split3(v4(r.v[i], 0), v4(r.v[i], 4));
            Vd[0][f / D][f % D] = v.h;
            Vd[1][f / D][f % D] = v.m;
            Vd[2][f / D][f % D] = v.l;
        }
    };

    f32x16 o[NDB];
#pragma unroll
    for (int i = 0; i < NDB; ++i) o[i] = f32x16{};
    float m_run = -INFINITY;  // reference max of row qrow's scores, in exp2 units
    float l_run = 0.f;        // this lane's partial sum of p (its half of the keys)

    Raw ra, rb;
    gload(ra, t_begin);
    gload(rb, t_begin + 1);
    sstore(ra, Ks0, Vt0);
    __syncthreads();

    // Step t reads tile t from buffer BUF = (t - t_begin) % 2 while tile t + 2
    // loads into registers; tile t + 1, loaded in the previous step, is split
    // into the other buffer, which every wave finished reading before the
    // previous step's barrier.
    auto step = [&](int t, auto buf_c, Raw& nxt, Raw& far) {
        constexpr int BUF = decltype(buf_c)::value;
        __bf16(&Kc)[3][BN][KS] = BUF ? Ks1 : Ks0;
        bf16x8(&Vc)[3][BN / 8][D] = BUF ? Vt1 : Vt0;
        const int k0 = t * BN;
        gload(far, t + 2);
        if (k0 < wave_kend) {
            f32x16 s[NKB];
            {
                Split3Sum st[NKB];
#pragma unroll
                for (int kb = 0; kb < NKB; ++kb) st[kb].hi = st[kb].lo = f32x16{};
#pragma unroll
                for (int kk = 0; kk < NKK; ++kk)
#pragma unroll
                    for (int kb = 0; kb < NKB; ++kb) {
                        Bf3x8 a;
                        a.h = *reinterpret_cast<const bf16x8*>(&Kc[0][kb * 32 + l32][16 * kk + 8 * g]);
                        a.m = *reinterpret_cast<const bf16x8*>(&Kc[1][kb * 32 + l32][16 * kk + 8 * g]);
                        a.l = *reinterpret_cast<const bf16x8*>(&Kc[2][kb * 32 + l32][16 * kk + 8 * g]);
                        mfma_split3(a, qf[kk], st[kb]);
                    }
#pragma unroll
                for (int kb = 0; kb < NKB; ++kb) s[kb] = st[kb].sum();
            }
            // reg 4j+cc of s[kb] holds key kb*32 + 8j + 4g + cc
            const bool need_mask = (k0 + BN > p.Tk) || (p.causal && (k0 + BN - 1 > q0w + p.off));
            if (need_mask) {
                const int lim = p.causal ? min(p.Tk - 1, qrow + p.off) : p.Tk - 1;
#pragma unroll
                for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        const int key = k0 + kb * 32 + 8 * (r >> 2) + 4 * g + (r & 3);
                        if (key > lim) s[kb][r] = -INFINITY;
                    }
            }
            float mp[4] = {-INFINITY, -INFINITY, -INFINITY, -INFINITY};
#pragma unroll
            for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
                for (int r = 0; r < 16; ++r) mp[r & 3] = fmaxf(mp[r & 3], s[kb][r]);
            const float mloc = max_xor32(fmaxf(fmaxf(mp[0], mp[1]), fmaxf(mp[2], mp[3]))) * p.c;
            // Lazy rescaling: a row's reference max m_run moves only when the row
            // sees a score more than kLazyLog2 above it, so P stays
            // <= 2^kLazyLog2; the O / l rescale and its exp2 run only on tiles where
            // some row of the wave moved, and for the other rows it multiplies by
            // exactly 1, so every row depends on its own scores only.  O / l and the
            // LSE do not depend on the reference.  m_run = -inf with a visible key
            // always moves it.
            const bool grow = mloc > m_run + kLazyLog2;
            if (__any(grow)) {
                // A row can see no key of a chunk that does not start at key 0:
                // keep m = -inf, l = 0, O = 0 for it instead of exp2(NaN).
                const float alpha = grow ? fast_exp2(m_run - mloc) : 1.f;  // m_run = -inf -> 0
                l_run *= alpha;
#pragma unroll
                for (int db = 0; db < NDB; ++db) o[db] *= alpha;
                m_run = grow ? mloc : m_run;
            }
            const float mc = m_run == -INFINITY ? 0.f : -m_run;
            // row sum as four independent partial chains
            float ls[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const float e = fast_exp2(fmaf(s[kb][r], p.c, mc));
                    s[kb][r] = e;
                    ls[r & 3] += e;
                }
            l_run += (ls[0] + ls[1]) + (ls[2] + ls[3]);
#pragma unroll
            for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
                for (int mm = 0; mm < 2; ++mm) {
                    const f32x16& e = s[kb];
                    const Bf3x8 pb = split3(f32x4{e[8 * mm], e[8 * mm + 1], e[8 * mm + 2], e[8 * mm + 3]},
                                            f32x4{e[8 * mm + 4], e[8 * mm + 5], e[8 * mm + 6], e[8 * mm + 7]});
#pragma unroll
                    for (int db = 0; db < NDB; ++db) {
                        Bf3x8 a;
                        a.h = Vc[0][4 * kb + 2 * mm + g][db * 32 + l32];
                        a.m = Vc[1][4 * kb + 2 * mm + g][db * 32 + l32];
                        a.l = Vc[2][4 * kb + 2 * mm + g][db * 32 + l32];
                        o[db] = mfma_split3(a, pb, o[db]);
                    }
                }
        }
        if constexpr (BUF)
            sstore(nxt, Ks0, Vt0);
        else
            sstore(nxt, Ks1, Vt1);
        __syncthreads();
    };
    using B0 = std::integral_constant<int, 0>;
    using B1 = std::integral_constant<int, 1>;
    for (int t = t_begin; t < n_tiles; t += 2) {
        step(t, B0{}, rb, ra);
        if (t + 1 < n_tiles) step(t + 1, B1{}, ra, rb);
    }

    // ---- non-finite inputs ------------------------------------------------------
    // An infinity in q, k or v, or a value past the largest bf16, is NaN in its
    // split parts, where the fp32 formula may still be finite or infinite (a
    // score of -inf is a probability of 0).  A wave whose sums are not finite forms
    // its rows again from memory in plain fp32: by MFMAs where every row sees all 32
    // keys of a block (keys past Tk are zeros there), else one key at a time, as a
    // hidden key's value must not meet a probability of 0.  (One such key in
    // 8192 of B1 H16 D128: 1.3 ms -> 5.6; one key at a time everywhere 246.)
    float chk = l_run * 0.f;
#pragma unroll
    for (int db = 0; db < NDB; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) chk = fmaf(o[db][r], 0.f, chk);
    if (__any(chk != 0.f)) {
        m_run = -INFINITY;
        l_run = 0.f;
#pragma unroll
        for (int db = 0; db < NDB; ++db) o[db] = f32x16{};
        const float* qp = qrow < p.Tq ? Q + (int64_t)qrow * p.sq.t : nullptr;
        const int b_end = min(n_tiles * BN, wave_kend);
        // the row's reference moves to mn: the factor of its sums, and mn as a finite reference
        auto move = [&](float mn) {
            const float ref = mn == -INFINITY ? 0.f : mn, alpha = m_run == -INFINITY ? 0.f : fast_exp2(m_run - ref);
            m_run = mn;
            l_run *= alpha;
#pragma unroll
            for (int db = 0; db < NDB; ++db) o[db] *= alpha;
            return ref;
        };
#pragma unroll 1
        for (int j0 = t_begin * BN; j0 < b_end; j0 += 32) {
            if (!p.causal || j0 + 31 <= q0w + p.off) {
                const float* kp = j0 + l32 < p.Tk ? K + (int64_t)(j0 + l32) * p.sk.t : nullptr;
                f32x16 s = dot_rows_f32<D, 4>(kp, qp, g);
                float mx = -INFINITY;
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    if (j0 + 8 * (r >> 2) + 4 * g + (r & 3) >= p.Tk) s[r] = -INFINITY;
                    mx = fmaxf(mx, s[r]);
                }
                const float ref = move(fmaxf(m_run, max_xor32(mx) * p.c));
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    s[r] = fast_exp2(fmaf(s[r], p.c, -ref));
                    l_run += s[r];
                }
#pragma unroll 1
                for (int db = 0; db < NDB; ++db) {  // 16 loads in flight
                    float v[16];
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        const int key = j0 + 8 * (r >> 2) + 4 * g + (r & 3);
                        v[r] = key < p.Tk ? V[(int64_t)key * p.sv.t + db * 32 + l32] : 0.f;
                    }
                    f32x16 t = f32x16{};
#pragma unroll
                    for (int r = 0; r < 16; ++r) t = mfma32x32x2(v[r], s[r], t);
#pragma unroll
                    for (int i = 0; i < NDB; ++i)  // (a loop variable can't index registers)
                        if (i == db) o[i] += t;
                }
                continue;
            }
            const int j_end = qp ? min(min(b_end, j0 + 32), qrow + p.off + 1) : 0;
#pragma unroll 1
            for (int j = j0; j < j_end; ++j) {
                const float* kp = K + (int64_t)j * p.sk.t;
                float s = 0.f;
#pragma unroll 4
                for (int d = 0; d < D; ++d) s = fmaf(qp[d], kp[d], s);
                s *= p.c;
                const float e = fast_exp2(s - move(fmaxf(m_run, s)));
                l_run += g == 0 ? e : 0.f;
                const float* vp = V + (int64_t)j * p.sv.t + 4 * g;
#pragma unroll
                for (int db = 0; db < NDB; ++db)
#pragma unroll
                    for (int r = 0; r < 16; ++r) o[db][r] = fmaf(e, vp[db * 32 + 8 * (r >> 2) + (r & 3)], o[db][r]);
            }
        }
    }

    // ---- epilogue ---------------------------------------------------------------
    const float l_tot = l_run + shfl_xor(l_run, 32);
    if (slot >= 0) {
        // partial of a split query tile: unnormalised O, row max, row sum
        if (qrow < p.Tq) {
            const int r = wave * 32 + l32;
            float* po = p.part + ((int64_t)slot * BH + bh) * (BM * D) + (int64_t)r * D;
#pragma unroll
            for (int db = 0; db < NDB; ++db)
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    st4(po + db * 32 + 8 * j + 4 * g,
                        f32x4{o[db][4 * j + 0], o[db][4 * j + 1], o[db][4 * j + 2], o[db][4 * j + 3]});
            if (g == 0) {
                float* pml = p.part + (int64_t)p.n_slots * BH * BM * D + (((int64_t)slot * BH + bh) * BM + r) * 2;
                pml[0] = m_run;
                pml[1] = l_tot;
            }
        }
        return;
    }
    const float inv = 1.f / l_tot;
    if (qrow < p.Tq) {
        float* dst = O + (int64_t)qrow * p.so.t;
#pragma unroll
        for (int db = 0; db < NDB; ++db)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                f32x4 val;
                val[0] = o[db][4 * j + 0] * inv;
                val[1] = o[db][4 * j + 1] * inv;
                val[2] = o[db][4 * j + 2] * inv;
                val[3] = o[db][4 * j + 3] * inv;
                st4(dst + db * 32 + 8 * j + 4 * g, val);
            }
        if (g == 0 && p.lse) p.lse[(int64_t)bh * p.Tq + qrow] = fmaf(m_run, kLn2, logf(l_tot));
    }
}

// Combines the partial slots of each split query tile: per row M = max_s m_s,
// w_s = 2^(m_s - M), O = sum_s w_s O_s / sum_s w_s l_s, LSE = M ln 2 + ln(sum_s w_s l_s),
// where m is in exp2 units (fp32; bf16: in units of the scores, so times c, and
// the scale).  One thread per (row, 4 columns).
template <int D, typename E>
__global__ __launch_bounds__(256) void attn_fwd_merge_kernel(FwdParams p) {
    constexpr int BM = fwd_bm(sizeof(E) == 2);
    constexpr int C4 = D / 4;
    constexpr int TPT = BM * C4;  // threads per (split tile, head)
    const int BH = p.B * p.H;
    const int64_t gid = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int64_t unit = gid / TPT;  // (split tile, head)
    if (unit >= (int64_t)p.n_split * BH) return;
    const int si = (int)(unit / BH);
    const int bh = (int)(unit % BH);
    const int rem = (int)(gid % TPT);
    const int r = rem / C4;
    const int c4 = rem % C4;
    const int qrow = p.split_qt[si] * BM + r;
    if (qrow >= p.Tq) return;
    const int s0 = p.split_slot0[si], ns = p.split_count[si];
    const float* ml = p.part + (int64_t)p.n_slots * BH * BM * D;
    float M = -INFINITY;
    for (int s = 0; s < ns; ++s) M = fmaxf(M, ml[(((int64_t)(s0 + s) * BH + bh) * BM + r) * 2]);
    float L = 0.f;
    f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int s = 0; s < ns; ++s) {
        const int64_t base = ((int64_t)(s0 + s) * BH + bh) * BM + r;
        const float m = ml[base * 2];
        if (m == -INFINITY) continue;
        const float wgt = fast_exp2(sizeof(E) == 4 ? m - M : (m - M) * p.c);
        L = fmaf(ml[base * 2 + 1], wgt, L);
        const f32x4 v = *reinterpret_cast<const f32x4*>(p.part + base * D + 4 * c4);
        acc[0] = fmaf(v[0], wgt, acc[0]);
        acc[1] = fmaf(v[1], wgt, acc[1]);
        acc[2] = fmaf(v[2], wgt, acc[2]);
        acc[3] = fmaf(v[3], wgt, acc[3]);
    }
    const float inv = 1.f / L;
    const int b = bh / p.H, h = bh % p.H;
    E* dst = (E*)p.o + b * p.so.b + h * p.so.h + (int64_t)qrow * p.so.t + 4 * c4;
    st4(dst, f32x4{acc[0] * inv, acc[1] * inv, acc[2] * inv, acc[3] * inv});
    if (c4 == 0 && p.lse) p.lse[(int64_t)bh * p.Tq + qrow] =
            sizeof(E) == 4 ? fmaf(M, kLn2, logf(L)) : M * p.scale + logf(L);
}

template <int D, typename E>
static void launch_merge_t(const FwdParams& p, hipStream_t s) {
    const int64_t threads = (int64_t)p.n_split * p.B * p.H * fwd_bm(sizeof(E) == 2) * (D / 4);
    hipLaunchKernelGGL((attn_fwd_merge_kernel<D, E>), dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, s, p);
}

template <int D>
static int launch_fwd_t(const FwdParams& p, hipStream_t s) {
    const int BH = p.B * p.H;
    const dim3 grid((unsigned)((p.n_groups ? p.n_groups : p.n_qtiles) * BH));
    hipLaunchKernelGGL((attn_fwd_kernel<D>), grid, dim3(64 * FwdTile<D>::NW), 0, s, p);
    if (p.n_split) launch_merge_t<D, float>(p, s);
    return (int)hipGetLastError();
}

// ---- split plan ----------------------------------------------------------------
// Makespan of a dispatch order on the device: workgroup w goes to XCD w % 8,
// and inside an XCD each workgroup starts on the slot that frees first (slots =
// resident workgroups).  Costs are in key tiles plus a fixed per-workgroup
// overhead (Q load, first K/V tile not hidden behind compute, epilogue).
static double fwd_makespan(const int* cost, int n_groups, int BH, int slots_per_xcd, double overhead) {
    double worst = 0.0;
    std::vector<double> heap((size_t)slots_per_xcd);
    for (int x = 0; x < 8; ++x) {
        std::fill(heap.begin(), heap.end(), 0.0);  // min-heap of slot free times
        int64_t w = 0;
        for (int gi = 0; gi < n_groups; ++gi)
            for (int i = 0; i < BH; ++i, ++w) {
                if (w % 8 != x) continue;
                std::pop_heap(heap.begin(), heap.end(), std::greater<double>());
                heap.back() += cost[gi] + overhead;
                std::push_heap(heap.begin(), heap.end(), std::greater<double>());
            }
        worst = std::max(worst, *std::max_element(heap.begin(), heap.end()));
    }
    return worst;
}

// Resident forward workgroups per XCD on the current device (8 XCDs), and
// the device's CU count.
struct FwdSlots {
    int per_xcd, cus;
};
// An error left pending by an earlier HIP call on this thread is returned
// (named in the detail text) instead of being cleared by the queries here.
static int fwd_slots(int D, int bf16, FwdSlots* out) {
    static std::mutex mu;
    static std::map<std::array<int, 3>, FwdSlots> cache;
    const hipError_t pending = hipGetLastError();
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess) {
        (void)hipGetLastError();  // no device (a CPU-only host sizing workspaces): MI355X defaults
        dev = -1;
    } else if (pending != hipSuccess) {
        return report_pending_error(pending, "attention forward planner");
    }
    std::lock_guard<std::mutex> lk(mu);
    const std::array<int, 3> key{dev, D, bf16};
    auto it = cache.find(key);
    if (it != cache.end()) {
        *out = it->second;
        return 0;
    }
    // MI355X: 256 CUs; fp32: one workgroup per CU.
    int cus = 256, per_cu = bf16 ? (D >= 128 ? 2 : 4) : 1;
    if (dev >= 0) {
        int n = 0, occ = 0;
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && n > 0) cus = n;
        hipError_t e = hipErrorInvalidValue;
        if (bf16) e = (hipError_t)fwd_bf16_occupancy(D, &occ);
        else if (D == 32) e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, attn_fwd_kernel<32>, 64 * FwdTile<32>::NW, 0);
        else if (D == 64) e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, attn_fwd_kernel<64>, 64 * FwdTile<64>::NW, 0);
        else if (D == 128) e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, attn_fwd_kernel<128>, 64 * FwdTile<128>::NW, 0);
        if (e == hipSuccess && occ > 0) per_cu = occ;
        (void)hipGetLastError();  // a failed query of ours: the defaults stand
    }
    const FwdSlots slots{std::max(1, cus * per_cu / 8), cus};
    cache[key] = slots;
    *out = slots;
    return 0;
}

// Causal forward split plan.  Without a split the query tiles run heaviest
// first, one workgroup per (tile, head).  When the whole grid fits in the
// resident slots at once, the heaviest tile alone sets the kernel time (fp32, us,
// unsplit and split: B H 1, T 8192, D 64 490 and 126; 4, 2048, 128 240 and 58), so its
// key range is cut.  With more workgroups than slots the tail balances itself: such
// grids never split (96 x 1024 x 64 93 us, cut 90 to 128; 192 x 512 x 64 61 and 79 to 98;
// 96 x 1024 x 128 152 and 160 to 217).  Each candidate chunk length CH cuts every tile
// with more than CH key tiles into ceil(n / CH) near-equal chunks; the candidate with
// the smallest simulated makespan (plus the merge pass) wins if it beats the unsplit
// order by more than 2%.
//
// fp32: a key tile (128, 64, 32 keys at D = 32, 64, 128) takes about 4 us; the merge costs
// two of them and the time that the partials take to memory and back (4 TB/s).  Over
// 77 shapes the plan's time is 1.4% above the fastest of six forced splits (3.4% with
// half a tile and nothing for the partials: 96 x 333 x 64 split 40 us, unsplit 30; one
// workgroup of 200 rows 24 and 20).
//
// bf16 (constants fitted to measurements at T = 1024..8192, D = 32..128): a
// bf16 key tile costs about a fifth of an fp32-MFMA one, so the workgroup's fixed
// cost and the merge weigh more in its units; up to four workgroups share a CU,
// whose resident workgroups together run about 1.1 tiles in the time one runs
// alone, so the makespan is also bounded below by the total work over the
// CUs; and tiles under 32 key tiles (2048 keys) never split (B1 H12 T1024 D64
// measured 19.9 us unsplit, 24.1 us split).
static constexpr double kFwdOverhead[2] = {0.35, 2.0};   // per-workgroup fixed cost, in key tiles (fp32, bf16)
static constexpr double kFwdMergeCost[2] = {2.0, 12.0};  // merge kernel, in key tiles
// ... and per float of the partials (written and read: 8 bytes at 4 TB/s over 4 us)
static constexpr double kFwdMergeFloat[2] = {8.0 / 16e6, 0.0};
static constexpr double kFwdCuRate[2] = {0.0, 1.1};      // tiles per CU per tile time (0: no bound)
static constexpr int kFwdMinSplitTiles[2] = {0, 32};

static void fwd_plan_compute(int B, int H, int Tq, int Tk, int D, int bf16, FwdSlots slots, FwdPlan* out) {
    const int BM = fwd_bm(bf16), BN = bf16 ? kFwdBf16BN : D >= 128 ? FwdTile<128>::BN : D >= 64 ? FwdTile<64>::BN : FwdTile<32>::BN;
    const int ix = bf16 ? 1 : 0;
    const double overhead = kFwdOverhead[ix], merge_cost = kFwdMergeCost[ix], cap = kFwdCuRate[ix] * slots.cus;
    const int slots_per_xcd = slots.per_xcd;
    const int nq = (Tq + BM - 1) / BM;
    const int BH = B * H;
    const int off = Tk - Tq;
    if ((int64_t)nq * BH > 8LL * slots_per_xcd) return;
    std::vector<int> nt((size_t)nq);
    int max_nt = 0;
    for (int q = 0; q < nq; ++q) {
        const int kend = std::min(Tk, (q + 1) * BM + off);
        nt[(size_t)q] = std::max(0, (kend + BN - 1) / BN);
        max_nt = std::max(max_nt, nt[(size_t)q]);
    }
    if (max_nt < kFwdMinSplitTiles[ix]) return;
    auto span = [&](const std::vector<int>& c) {
        double m = fwd_makespan(c.data(), (int)c.size(), BH, slots_per_xcd, overhead);
        if (cap > 0) {
            double work = 0.0;
            for (int x : c) work += x + overhead;
            m = std::max(m, work * BH / cap);
        }
        return m;
    };
    std::vector<int> cost;
    for (int q = nq - 1; q >= 0; --q) cost.push_back(nt[(size_t)q]);
    const double base = span(cost);
    double best = base * 0.98;
    int best_ch = 0;
    struct G { int n, qt, t0, t1; };
    auto build = [&](int ch, std::vector<G>& g, int& n_split) {
        g.clear();
        n_split = 0;
        for (int q = 0; q < nq; ++q) {
            const int n = nt[(size_t)q];
            if (n > ch) {
                const int k = (n + ch - 1) / ch;
                ++n_split;
                for (int j = 0; j < k; ++j) {
                    const int a = (int)((int64_t)n * j / k), b = (int)((int64_t)n * (j + 1) / k);
                    g.push_back({b - a, q, a, b});
                }
            } else {
                g.push_back({n, q, 0, n});
            }
        }
        std::stable_sort(g.begin(), g.end(), [](const G& x, const G& y) {
            return x.n != y.n ? x.n > y.n : x.qt > y.qt;
        });
    };
    std::vector<G> g;
    for (int ch = max_nt - 1; ch >= std::max(2, max_nt / 8); --ch) {
        int n_split = 0;
        build(ch, g, n_split);
        if ((int)g.size() > kMaxFwdGroups || n_split > kMaxFwdGroups / 2) continue;
        cost.resize(g.size());
        for (size_t i = 0; i < g.size(); ++i) cost[i] = g[i].n;
        int64_t parts = 0;
        for (const G& x : g) parts += x.t1 - x.t0 < nt[(size_t)x.qt];
        const double ms = span(cost) + merge_cost + kFwdMergeFloat[ix] * (double)(parts * BH * BM * (D + 2));
        if (ms < best) {
            best = ms;
            best_ch = ch;
        }
    }
    if (!best_ch) return;
    int n_split = 0;
    build(best_ch, g, n_split);
    // slots: consecutive per split tile, in query-tile order
    std::vector<int> slot0((size_t)nq, -1), count((size_t)nq, 0);
    for (const G& x : g)
        if (x.t1 - x.t0 < nt[(size_t)x.qt]) ++count[(size_t)x.qt];
    int ns = 0;
    for (int q = 0; q < nq; ++q)
        if (count[(size_t)q]) {
            slot0[(size_t)q] = ns;
            out->split_qt[out->n_split] = q;
            out->split_slot0[out->n_split] = ns;
            out->split_count[out->n_split] = count[(size_t)q];
            ++out->n_split;
            ns += count[(size_t)q];
        }
    std::vector<int> next((size_t)nq, 0);
    for (const G& x : g) {
        FwdGroup& o = out->groups[out->n_groups++];
        o.qt = x.qt;
        o.t0 = x.t0;
        o.t1 = x.t1;
        o.slot = count[(size_t)x.qt] ? slot0[(size_t)x.qt] + next[(size_t)x.qt]++ : -1;
    }
    out->n_slots = ns;
}

int fwd_plan(int B, int H, int Tq, int Tk, int D, int causal, int bf16, FwdPlan* out) {
    *out = FwdPlan{};
    bf16 = bf16 ? 1 : 0;
    if (!causal || (D != 32 && D != 64 && D != 128)) return 0;
    FwdSlots slots{};
    if (const int e = fwd_slots(D, bf16, &slots)) return e;
    static std::mutex mu;
    static std::map<std::array<int, 7>, FwdPlan> cache;
    const std::array<int, 7> key{B * H, Tq, Tk, D, bf16, slots.per_xcd, slots.cus};
    {
        std::lock_guard<std::mutex> lk(mu);
        auto it = cache.find(key);
        if (it != cache.end()) {
            *out = it->second;
            return 0;
        }
    }
    fwd_plan_compute(B, H, Tq, Tk, D, bf16, slots, out);
    // The bf16 D = 128 forward raises the P.V MFMAs' wave priority (a wave that
    // reaches them issues them ahead of the other wave's softmax VALU work on
    // its SIMD); on grids that fit one round of workgroup slots that measured
    // 5-7% slower (B2 H8 T4096, B1 H16 T4096, B4 H8 T2048, B1 H8 T8192: 512
    // workgroups on 512 slots) and on larger ones 1-10% faster (config 4, B4
    // H16 T2048, B8 H16 T1024, B8 H12 T1024).
    out->pv_prio = (int64_t)((Tq + fwd_bm(bf16) - 1) / fwd_bm(bf16)) * B * H > 8LL * slots.per_xcd;
    std::lock_guard<std::mutex> lk(mu);
    if (cache.size() > 256) cache.clear();
    cache[key] = *out;
    return 0;
}

size_t fwd_workspace_bytes(const FwdPlan& plan, int B, int H, int D, int bf16) {
    return (size_t)plan.n_slots * B * H * fwd_bm(bf16) * (size_t)(D + 2) * sizeof(float);
}

int launch_attn_fwd(const FwdParams& p, int bf16, hipStream_t s) {
    if (bf16) {
        const int e = launch_attn_fwd_bf16(p, s);
        if (e || !p.n_split) return e;
        switch (p.D) {  // the merge reads fp32 partials and writes bf16 O
            case 32: launch_merge_t<32, uint16_t>(p, s); break;
            case 64: launch_merge_t<64, uint16_t>(p, s); break;
            case 128: launch_merge_t<128, uint16_t>(p, s); break;
            default: return (int)hipErrorInvalidValue;
        }
        return (int)hipGetLastError();
    }
    switch (p.D) {
        case 32: return launch_fwd_t<32>(p, s);
        case 64: return launch_fwd_t<64>(p, s);
        case 128: return launch_fwd_t<128>(p, s);
        default: return (int)hipErrorInvalidValue;
    }
}

}  // namespace inf
