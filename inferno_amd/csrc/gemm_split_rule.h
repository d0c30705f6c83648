// gemm_split_rule.h -- which fp32 products the split-operand GEMM takes, and in how
// many K ranges.  Plain host C++ without HIP, so that it can be checked anywhere.
#pragma once

#include <algorithm>
#include <cmath>
#include <cstddef>
#include <cstdint>

namespace inf {

constexpr int kSplitBM = 256, kSplitBN = 128, kSplitBK = 32;  // a workgroup's tile of C, a step of K

// The number of K ranges, or 0 where the vendor library runs the product: sizes that the
// kernel can't address (32-bit row, column and step counts and offsets inside a
// tile's panel; a K-contiguous operand is read 4 elements at a time), and
// those where the library is no slower.
inline int gemm_split_ranges(int ta, int tb, int64_t M, int64_t N, int64_t K, int64_t batch, int64_t lda, int64_t ldb,
                             size_t ws_bytes) {
    constexpr int64_t kMax = int64_t(1) << 30;
    if (M < 1 || N < 1 || K < 1 || batch < 1 || M > kMax || N > kMax || K > kMax) return 0;
    if ((K % 4 != 0 && !(ta && !tb)) || lda > (1 << 20) || ldb > (1 << 20)) return 0;
    const int64_t tm = (M + kSplitBM - 1) / kSplitBM, tn = (N + kSplitBN - 1) / kSplitBN;
    if (tm * tn > (1 << 24) || tm * tn * batch > (1 << 24)) return 0;
    const int64_t tiles = tm * tn * batch, nk = (K + kSplitBK - 1) / kSplitBK;
    // The cheapest under a model (microseconds, within 8% rms of 31 measured shapes): the
    // longest chain of K steps on a CU (2.2 a step, 5 steps for a workgroup's start
    // and end) or, where the device is full and its clock falls with the load, the
    // steps over the rate that large products reach; partials pass through memory
    // once more.
    double best = 1e30;
    int ks = 1;
    for (int c = 1; c <= 8; ++c) {
        if (c > 1 && (batch > 1 || nk / c < 8 || (double)c * M * N * sizeof(float) > (double)ws_bytes)) break;
        const double wgs = (double)(tiles * c), steps = (double)((nk + c - 1) / c + 5);
        double cost = std::max(steps * 2.2 * std::ceil(wgs / 256), wgs * steps / 100.0);
        if (c > 1) cost += 4.0 + (double)(c + 1) * M * N * 4 / 4e6;
        if (cost < best) {
            best = cost;
            ks = c;
        }
    }
    // The vendor library's fp32 kernels (about 142 TFLOP/s, 118 at ragged sizes, and
    // better split for small problems) where the model says that they are no
    // slower, us there and here: 1024^3 20 and 37, 1200 x 512 x 2048 28 and 39, 1024 x 768
    // x 3072 40 and 48, 8192 x 256 x 1024 38 and 41; but 8192 x 1024 x 256 40 and 34,
    // 2048^3 122 and 102.
    const bool whole = M % 128 == 0 && N % 128 == 0 && K % 32 == 0;
    return best > 2.0 * M * N * K * batch / (whole ? 142e6 : 118e6) + 8.0 ? 0 : ks;
}

}  // namespace inf
