// gemm_routes.h -- whether a matrix product runs on operands packed to fp16
// (gemm_packed.hip) or on the tiles that read fp32 operands (igemm.h; below
// "direct"). Host code without HIP, so that the rules are checked on the CPU
// against the times they were taken from (tests/golden/gemm_routes.csv).
#pragma once

#include <algorithm>
#include <cmath>
#include <cstdint>

namespace seera {

// The share of the chip's 256 CUs that have work over the rounds of 256x256
// tiles of an M x N result.
inline double tile_fill(int M, int N) {
    const double t = (double)((M + 255) / 256) * ((N + 255) / 256);
    return t / (256.0 * std::ceil(t / 256.0));
}

// Whether an M x N product over K with float4-aligned rows that reads its
// operands `reuse` times over is better off packed: the 256x256 tiles of the
// streaming kernel leave CUs idle in their last round, and the contraction is
// long enough for that to weigh more than packing.
inline bool tiles_leave_idle(int M, int N, int K, double reuse, double most_fill) {
    if (K < 400) return false;
    const double fill = tile_fill(M, N);
    return (int64_t)((M + 255) / 256) * ((N + 255) / 256) > 256 ? fill < most_fill && reuse >= 600
                                                                : fill < 0.6 && reuse >= 1250;
}

// Whether a call runs on operands packed to fp16 (gemm_packed.hip). Reuse: the
// multiply-adds per value packed. Measured direct -> packed (us, M x N x K; dA and
// dB in brackets):
//  - rows that are not whole float4s, from kPackMin* multiply-adds on: below,
//    the packing launch costs what it saves (332 x 539 x 103: 7.2 -> 8.8; 65 x
//    4000 x 65 [15.4 -> 16.5]), and from a reuse of 12 [80] on (3 x 100001 x 101:
//    18 -> 22; 16 x 4001 x 4001: 36 -> 29; 33 x 9001 x 2001: 54 -> 34 [reuse 65,
//    76 -> 81]; 85 x 3687 x 2236 [reuse 160, 171 -> 34]); 511^3: 15.6 -> 9.7 [23.9 ->
//    15.0], 3001 x 2047 x 1501: 60 -> 38 [141 -> 79], 4095^3: 190 -> 175 [378 -> 350].
//    Ragged in N alone, A streams as it is and only B's loads are scalar: short sums
//    (60160 x 57 x 156 19 -> 25, 1523 x 278 x 100 5.4 -> 6.3; 24608 x 1633 x 20 68 -> 59),
//    fewer than 32 columns (62592 x 26 x 1312 76 -> 120) and split sums on narrow results
//    (1064 x 57 x 3856 12 -> 17) stay direct below 4e9 multiply-adds; 65568 x 57 x 2616
//    442 -> 268.
//  - a contraction that is not whole 32-deep slices, where the kernel cannot
//    stream: with a reuse of 600 and a K of 480 on (1000^3, reuse 500: 13.2 -> 14.8
//    [reuse 667, 26.8 -> 25.1]; 1200^3: 22 -> 18 [46 -> 29]; 16384 x 512 x 500: 27 -> 32;
//    100000 x 256 x 252: 63 -> 80 [reuse 253, 133 -> 191]; 7168 x 6128 x 80 41 -> 63, 6112 x
//    1188 x 396 22 -> 24, 4476 x 1820 x 528 58 -> 37).
//  - tiles_leave_idle: 2560^3: 61 -> 52 [128 -> 96], 4608^3: 338 -> 240, 6144^3:
//    759 -> 515 [1884 -> 995]; not 5120^3 forward (fill 0.78, 283 -> 329; [627 -> 653, but
//    7424 x 3328 x 3520, 0.79 and 0.71, 555 -> 453]), 4096^3
//    (144 -> 167), 3584^3 (125 -> 131) or 4096 x 11008 x 4096 (412 -> 438), whose tiles fill
//    their rounds, nor 9984 x 4896 x 32 (34 -> 56), 2752 x 2752 x 256 (14 -> 19).
constexpr double kPackMinFwd = 3e7, kPackMinBwd = 2e7;

// a16, b16, c16: the operands' first elements lie on 16 bytes.
inline bool packed_gemm_fwd_pays(bool a16, bool b16, int M, int N, int K) {
    const double macs = (double)M * N * K;
    if (macs < kPackMinFwd) return false;
    const double reuse = 1.0 / (1.0 / M + 1.0 / N);
    if (K % 4 != 0 || !a16) return reuse >= 12;
    if (N % 4 != 0 || !b16) {
        if (reuse < 12) return false;
        if (macs >= 4e9) return true;
        if (N < 32 || (K > 3000 && std::min(M, N) <= 64)) return false;
        return K >= (N <= 64 ? 512 : 120) || (N >= 400 && macs >= 1.5e8);
    }
    if (K % 32 != 0) return reuse >= 600 && K >= 480;
    return tiles_leave_idle(M, N, K, reuse, 0.77);
}

inline bool packed_gemm_bwd_pays(bool a16, bool b16, bool c16, int M, int N, int K) {
    const double macs = (double)M * N * K;
    if (macs < kPackMinBwd) return false;
    const double reuse = 2.0 / (1.0 / M + 1.0 / N + 1.0 / K);
    if (K % 4 != 0 || N % 4 != 0 || !a16 || !b16 || !c16) return reuse >= 80;
    if (M % 32 != 0 || N % 32 != 0) return reuse >= 600;
    return tiles_leave_idle(M, K, N, reuse, 0.8) || tiles_leave_idle(K, N, M, reuse, 0.8);
}

}  // namespace seera
