// gemm_packed.hip -- matrix products over operands packed to fp16: shapes whose
// rows are not whole float4s or whose contraction is not whole 32-deep slices,
// and large ones that 256x256 tiles cut badly.
//
// The tiles of igemm.h load fp32 operands 16 bytes at a time and round them on
// the way to LDS; a row length that is not a multiple of 4 leaves them scalar
// loads (511^3: 15.6 us, here 9.7; 4095^3 over zero-padded fp32 copies of both
// operands, 8 bytes moved per value each: 190 us, here 175). Here one launch
// writes every operand of the call once as fp16 [cols / 64][rows][64], rows and
// columns rounded up to 64 with zeros (6 bytes moved per value); a 64-deep slice
// of a tile is then one run of memory whichever way the operand is contracted,
// and goes to LDS by DMA (half_tile.h): along its columns as a K-contiguous tile,
// along its rows as an MN-contiguous one. The forward packs A and B; the backward
// A, B and dC once for both of its products (3001 x 2047 x 1501: 141 -> 79 us).
// Reference: engine_cuda/src/GEMM.cu:13-103, 164-225.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "half_tile.h"
#include "kernels.h"
#include "plan.h"

namespace seera {
namespace {

struct PackMat {
    const float* in;  // [rows, cols]
    half_t* out;      // [colsP / 64][rowsP][64]
    float* sums;      // [rowsP / 32][colsP] column sums of 32 rows, or nullptr
    int64_t total;
    int rows, cols, rowsP, colsP;
    FastDiv by_blocks;  // 64-column blocks
    int block0;
};
struct PackMats {
    PackMat m[3];
    int n;
};

// A wave takes 32 rows of 64 columns: lane (8 rows) x (8 columns), four times.
// Columns past the end of a row load what follows in memory (never past the
// tensor: make_rsrc_in) and are replaced by zeros.
__global__ __launch_bounds__(256) void pack_matrices(const PackMats a) {
    int z = 0;
    while (z + 1 < a.n && (int)blockIdx.x >= a.m[z + 1].block0) ++z;
    const PackMat& p = a.m[z];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int unit = ((int)blockIdx.x - p.block0) * 4 + wave;
    const int rg = p.by_blocks.div(unit), cb = unit - rg * (p.colsP >> 6);
    if (rg * 32 >= p.rowsP) return;
    const int r0 = rg * 32, c = cb * 64 + (lane & 7) * 8;
    const rsrc_t rs = make_rsrc_in(p.in, p.total, (int64_t)r0 * p.cols);
    floatx4 v[4][2];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int r = 8 * i + (lane >> 3);
#pragma unroll
        for (int h = 0; h < 2; ++h)
            v[i][h] = buf_load4(rs, r0 + r < p.rows && c + 4 * h < p.cols
                                        ? (uint32_t)(r * p.cols + c + 4 * h) * 4u : kBufOOB);
    }
    float s[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) s[j] = 0.f;
    half_t* out = p.out + ((int64_t)cb * p.rowsP + r0) * 64 + lane * 8;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        float x[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            x[j] = c + j < p.cols ? v[i][j >> 2][j & 3] : 0.f;
            s[j] += x[j];
        }
        *reinterpret_cast<half8*>(out + i * 512) = pack8(x);
    }
    if (p.sums) {
#pragma unroll
        for (int m = 8; m < 64; m <<= 1)
#pragma unroll
            for (int j = 0; j < 8; ++j) s[j] += __shfl_xor(s[j], m);
        if (lane < 8) {
#pragma unroll
            for (int j = 0; j < 8; ++j) p.sums[(int64_t)rg * p.colsP + c + j] = s[j];
        }
    }
}

// One operand as packed; KC: contracted along its columns.
struct HalfMat {
    const half_t* p;
    int rowsP, colsP;
};
struct PackedGemmArgs {
    HalfMat a, b;
    float* C;
    int M, N;
    int64_t ldc, split_stride;
    int slices, sps;      // 64-deep slices in all and per split
    int tiles, tiles_n;
    const float* bias;    // EPI
    float* mask;
    int act;
};

template <int R, int NT, bool KC>
struct HalfOperand {
    using Tile = std::conditional_t<KC, KcTile<R, 64, NT>, McTile<R, 64, NT>>;
    // Where slice s of the tile at r0 begins, the bytes to the next slice, and
    // the bytes from there to piece i. Rows (columns) past the matrix repeat
    // its last row (first column of the tile): their results are never stored.
    static __device__ __forceinline__ const char* base(const HalfMat& m, int r0, int s) {
        const int64_t at = KC ? (int64_t)r0 * 64 : (int64_t)(r0 >> 6) * m.rowsP * 64;
        return reinterpret_cast<const char*>(m.p + at) + s * step(m);
    }
    static __device__ __forceinline__ int64_t step(const HalfMat& m) {
        return KC ? (int64_t)m.rowsP * 128 : 64 * 128;
    }
    static __device__ __forceinline__ uint32_t offset(const HalfMat& m, int r0, int i) {
        int row, chunk;
        Tile::item(i, row, chunk);
        if constexpr (KC)
            return (uint32_t)(min(row, m.rowsP - 1 - r0) * 64 + chunk * 8) * 2u;
        else
            return r0 + chunk * 8 < m.colsP ? (uint32_t)((chunk >> 3) * m.rowsP + row) * 128u + (chunk & 7) * 16u : 0u;
    }
};

// BM x BN tile, WM x WN waves in KG groups that share each slice's K and add up
// at the end, three LDS stages (half_pipeline); blockIdx.y is the split over K.
// Up to 64x64 per wave the sums run in parts of 8 (one group) or 16 steps, as registers allow
// (error against 64 bits at 2000^3 1.1e-7 of the result); at 128x64 over the
// whole length of a group's K (2.0e-7; the single chain of igemm.h 2.8e-7).
template <int BM, int BN, int WM, int WN, int KG, bool AKC, bool BKC, bool EPI>
__global__ __launch_bounds__(64 * WM * WN * KG, 1) void packed_gemm_kernel(const PackedGemmArgs g) {
    constexpr int NT = 64 * WM * WN * KG, NS = 3, KK = 4 / KG;
    using A = HalfOperand<BM, NT, AKC>;
    using B = HalfOperand<BN, NT, BKC>;
    using TA = typename A::Tile;
    using TB = typename B::Tile;
    constexpr int STAGE = TA::HALVES + TB::HALVES, LOADS = TA::PASSES + TB::PASSES;
    constexpr int TM = BM / WM / 32, TN = BN / WN / 32;
    extern __shared__ __align__(16) half_t smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // The blocks of one XCD walk groups of 4 tile rows column by column.
    const int id = xcd_order(blockIdx.x, g.tiles), tiles_m = g.tiles / g.tiles_n;
    const int group = id / (4 * g.tiles_n), in_group = id - group * 4 * g.tiles_n;
    const int rows = min(tiles_m - group * 4, 4);
    const int tm = group * 4 + in_group % rows, tn = in_group / rows;
    const int m0 = tm * BM, n0 = tn * BN, z = blockIdx.y;
    uint32_t ao[TA::PASSES], bo[TB::PASSES];
#pragma unroll
    for (int p = 0; p < TA::PASSES; ++p) ao[p] = A::offset(g.a, m0, p * NT + tid);
#pragma unroll
    for (int p = 0; p < TB::PASSES; ++p) bo[p] = B::offset(g.b, n0, p * NT + tid);
    const int64_t da = A::step(g.a), db = B::step(g.b);
    const int s0 = z * g.sps, n = min(g.sps, g.slices - s0);
    const char *pa = A::base(g.a, m0, s0), *pb = B::base(g.b, n0, s0);
    auto load = [&](int l, half_t* stage) {
        half_t* d = stage + wave * 512 + l * NT * 8;
        if (l < TA::PASSES)
            dma16(make_dma_rsrc(pa, kMaxTileSpanBytes), d, ao[l < TA::PASSES ? l : 0], 0u);
        else
            dma16(make_dma_rsrc(pb, kMaxTileSpanBytes), d, bo[l < TA::PASSES ? 0 : l - TA::PASSES], 0u);
        if (l == LOADS - 1) {
            pa += da;
            pb += db;
        }
    };
    constexpr bool PARTS = TM * TN <= 4;
    floatx16 part[TM][TN], acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) part[i][j][r] = acc[i][j][r] = 0.f;
    constexpr int GW = WM * WN;
    const int grp = wave / GW, gw = wave % GW;
    const int wm = (gw % WM) * (BM / WM), wn = (gw / WM) * (BN / WN);
    half_pipeline<TA, TB, KK, NS, LOADS, TM, TN>(smem, STAGE, TA::HALVES, wm, wn, grp * KK, lane, n, part,
                                                 load, [&](int s) {
                                                     if constexpr (PARTS) add_part<KG == 1 ? 2 : 8>(s, part, acc);
                                                 });
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] += part[i][j][r];
    sum_groups<KG, GW, TM, TN>(reinterpret_cast<float*>(smem), wave, lane, acc);
    if (grp > 0) return;

    float* const out = g.C + z * g.split_stride;
    const int mb = m0 + wm + 4 * (lane >> 5);
    const rsrc_t ro = make_rsrc(out + (int64_t)m0 * g.ldc);
    rsrc_t rm = ro;
    if (EPI && g.mask) rm = make_rsrc(g.mask + (int64_t)m0 * g.ldc);
    const uint32_t step = (uint32_t)g.ldc * 4u;
#pragma unroll
    for (int j = 0; j < TN; ++j) {
        const int col = n0 + wn + 32 * j + (lane & 31);
        const float bias = EPI && g.bias && col < g.N ? g.bias[col] : 0.f;
        const uint32_t o = (uint32_t)(mb - m0) * step + (uint32_t)col * 4u;
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            auto row = [&](int e) { return 32 * i + 8 * (e >> 2) + (e & 3); };
            auto at = [&](int e) { return col < g.N && mb + row(e) < g.M ? o : kBufOOB; };
            floatx16 v = acc[i][j];
            if constexpr (EPI) {  // (as epilogue() of mfma_core.h; a column's masks before its first store)
                if (g.act == kActReluGrad) {
                    float m[16];
#pragma unroll
                    for (int e = 0; e < 16; ++e) m[e] = buf_load1s(rm, at(e), row(e) * step);
#pragma unroll
                    for (int e = 0; e < 16; ++e) v[e] *= m[e];
                } else {
#pragma unroll
                    for (int e = 0; e < 16; ++e) v[e] += bias;
                    if (g.act == kActRelu) {
                        if (g.mask) {
#pragma unroll
                            for (int e = 0; e < 16; ++e)
                                buf_store1s(rm, at(e), row(e) * step, v[e] > 0.f ? 1.f : 0.f);
                        }
#pragma unroll
                        for (int e = 0; e < 16; ++e) v[e] = v[e] > 0.f ? v[e] : 0.f;
                    }
                }
            }
#pragma unroll
            for (int e = 0; e < 16; ++e) buf_store1s(ro, at(e), row(e) * step, v[e]);
        }
    }
}

constexpr int64_t kMost = 0x7F000000ll;
int64_t up64(int64_t n) { return (n + 63) & ~(int64_t)63; }

template <int BM, int BN, int WM, int WN, int KG, bool AKC, bool BKC, bool EPI>
hipError_t launch_packed_gemm(PackedGemmArgs g, int splits, hipStream_t st) {
    constexpr int lds = std::max(3 * (BM + BN) * 64 * 2, KG > 1 ? BM * BN * 4 : 0);
    auto kern = packed_gemm_kernel<BM, BN, WM, WN, KG, AKC, BKC, EPI>;
    if (lds > 65536) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, lds);
        if (e != hipSuccess) return e;
    }
    g.tiles_n = (g.N + BN - 1) / BN;
    g.tiles = g.tiles_n * ((g.M + BM - 1) / BM);
    hipLaunchKernelGGL(kern, dim3((unsigned)g.tiles, (unsigned)splits), dim3(64 * WM * WN * KG), lds, st, g);
    return hipGetLastError();
}

// Tile and splits of an M x N product of `slices` 64-deep slices, from times over
// 73 shapes of 64 to 16385 rows with every tile and 1 to 16 splits (us, a fit within
// 10 % on average). A block takes a start-up (first loads, stores) and its slices:
//   256x128  8.7 + 0.71 a slice, one per CU, bound by the matrix cores
//   128x128  4.9 + 0.47 a slice, one per CU, bound by LDS (1.5 cycles of it per
//            matrix-core cycle, against 1.1)
//   64x64    2.1 + 0.35, 0.44 or 0.54 a slice with one, two or three on a CU
// and a split adds 2.8 (a launch) and a pass over the partials at 3.1 TB/s. The chosen tile,
// us with the packing: 4097^3 256x128 214 (128x128 223, 64x64 266), 3001x2047x1501 256x128
// 39 (64x64 43), 2047^3 128x128 35 (256x128 41), 1301^3 64x64 20 (128x128 24); of 73 shapes
// two lose more than 8 %: 795x1046x4432 35 (31), 1597x4059x379 25 (23).
enum { kTile64, kTile128, kTile256 };
struct PackedPlan {
    int tile, splits, sps;
    PackedPlan(int M, int N, int slices) : tile(kTile128), splits(1) {
        auto tiles = [&](int bm, int bn) { return (int64_t)((M + bm - 1) / bm) * ((N + bn - 1) / bn); };
        auto per_cu = [](int64_t blocks) { return (double)((blocks + 255) / 256); };
        double best = 1e30;
        for (int s = 1; s <= 32; s *= 2) {
            if (s > 1 && slices / s < 4) break;
            const double n = (slices + s - 1) / s;
            auto consider = [&](int t, double us) {
                if (s > 1) us += 2.8 + (double)s * M * N * 4 / 3.1e6;
                if (us < best) {
                    best = us;
                    tile = t;
                    splits = s;
                }
            };
            consider(kTile256, per_cu(tiles(256, 128) * s) * (8.7 + 0.71 * n));
            consider(kTile128, per_cu(tiles(128, 128) * s) * (4.9 + 0.47 * n));
            const double b = per_cu(tiles(64, 64) * s), full = std::floor(b / 3), rest = b - 3 * full;
            consider(kTile64, (full + (rest > 0 ? 1 : 0)) * 2.1 +
                                  n * (full * 0.54 + (rest == 1 ? 0.35 : rest == 2 ? 0.44 : 0.0)));
        }
        sps = (slices + splits - 1) / splits;
        splits = (slices + sps - 1) / sps;
    }
};

template <bool AKC, bool BKC, bool EPI>
hipError_t launch_tile(const PackedGemmArgs& g, const PackedPlan& pl, hipStream_t st) {
    if (pl.tile == kTile256) return launch_packed_gemm<256, 128, 2, 2, 2, AKC, BKC, EPI>(g, pl.splits, st);
    if (pl.tile == kTile128) return launch_packed_gemm<128, 128, 2, 2, 2, AKC, BKC, EPI>(g, pl.splits, st);
    return launch_packed_gemm<64, 64, 2, 2, 1, AKC, BKC, EPI>(g, pl.splits, st);
}

// C = A . B over packed operands; partials (splits) go to `part`.
template <bool AKC, bool BKC, bool EPI>
int run_packed(const HalfMat& a, const HalfMat& b, float* C, int M, int N, int64_t ldc, int slices,
               const PackedPlan& pl, float* part, const float* bias, float* mask, int act, hipStream_t st) {
    PackedGemmArgs g{};
    g.a = a; g.b = b;
    g.C = C; g.ldc = ldc;
    g.M = M; g.N = N;
    g.slices = slices; g.sps = pl.sps;
    g.bias = bias; g.mask = mask; g.act = act;
    hipError_t e;
    if (pl.splits > 1) {
        g.C = part;
        g.ldc = N;
        g.split_stride = (int64_t)M * N;
        e = launch_tile<AKC, BKC, false>(g, pl, st);
    } else {
        e = launch_tile<AKC, BKC, EPI>(g, pl, st);
    }
    if (e != hipSuccess) return fail_hip(e, "packed GEMM launch");
    if (pl.splits > 1) {
        const int64_t n = (int64_t)M * N;
        const unsigned nb = (unsigned)((n + 255) / 256);
        if constexpr (EPI)
            hipLaunchKernelGGL(splitk_reduce_epi, dim3(nb), dim3(256), 0, st, part, C, M, N, ldc, pl.splits, n,
                               bias, mask, act);
        else
            hipLaunchKernelGGL(splitk_reduce, dim3(nb), dim3(256), 0, st, part, C, M, N, ldc, pl.splits, n, (int)nb,
                               (const float*)nullptr, (float*)nullptr);
        SEERA_HIP_TRY(hipGetLastError());
    }
    return SEERA_OK;
}

struct Operand2D {
    const float* in;
    int rows, cols;
    int64_t halves() const { return up64(rows) * up64(cols); }
    // 32 rows as read, a tile's 256 columns as packed, and the packing units
    // within 32 bits
    bool ok() const {
        return (int64_t)cols * 4 * 32 < kMost && up64(rows) * 512 < kMost && halves() / 2048 < 0x7f000000;
    }
};

HalfMat add_matrix(PackMats& pk, int& block, const Operand2D& m, half_t* out, float* sums) {
    PackMat& p = pk.m[pk.n++];
    p.in = m.in; p.out = out; p.sums = sums;
    p.total = (int64_t)m.rows * m.cols;
    p.rows = m.rows; p.cols = m.cols;
    p.rowsP = (int)up64(m.rows); p.colsP = (int)up64(m.cols);
    p.by_blocks = FastDiv(p.colsP / 64);
    p.block0 = block;
    block += (int)(((int64_t)(p.rowsP / 32) * (p.colsP / 64) + 3) / 4);
    return HalfMat{out, p.rowsP, p.colsP};
}

size_t align256(size_t n) { return (n + 255) & ~(size_t)255; }

// The rows of one tile of the result within 32-bit offsets.
bool result_ok(int64_t ld) { return ld * 4 * 256 < kMost; }

}  // namespace

int packed_gemm_fwd(const float* A, const float* B, const float* bias, float* C, float* mask, int M, int N, int K,
                    int act, bool epi, hipStream_t st, bool* used) {
    *used = false;
    const Operand2D a{A, M, K}, b{B, K, N};
    if (!a.ok() || !b.ok() || !result_ok(N)) return SEERA_OK;
    const int slices = (int)(up64(K) / 64);
    const PackedPlan pl(M, N, slices);
    const size_t na = align256(a.halves() * 2), nb = align256(b.halves() * 2);
    const size_t np = pl.splits > 1 ? (size_t)pl.splits * M * N * 4 : 0;
    void* ws = nullptr;
    bool got = false;
    // (operands and partials in one piece: what fits the fixed array of the
    // no-allocation entry point runs there in the same order of sums)
    SEERA_TRY(staging_workspace_try(na + nb + np, &ws, st, &got, true));
    if (!got) return SEERA_OK;
    char* p = static_cast<char*>(ws);
    PackMats pk{};
    int block = 0;
    const HalfMat ha = add_matrix(pk, block, a, reinterpret_cast<half_t*>(p), nullptr);
    const HalfMat hb = add_matrix(pk, block, b, reinterpret_cast<half_t*>(p + na), nullptr);
    hipLaunchKernelGGL(pack_matrices, dim3((unsigned)block), dim3(256), 0, st, pk);
    SEERA_HIP_TRY(hipGetLastError());
    float* part = reinterpret_cast<float*>(p + na + nb);
    if (epi)
        SEERA_TRY((run_packed<true, false, true>(ha, hb, C, M, N, N, slices, pl, part, bias, mask, act, st)));
    else
        SEERA_TRY((run_packed<true, false, false>(ha, hb, C, M, N, N, slices, pl, part, nullptr, nullptr, 0, st)));
    *used = true;
    return SEERA_OK;
}

int packed_gemm_bwd(const float* A, const float* B, const float* dC, const float* mask, float* dA, float* dB,
                    float* db, int M, int N, int K, hipStream_t st, bool* used) {
    *used = false;
    const Operand2D a{A, M, K}, b{B, K, N}, c{dC, M, N};
    if (!a.ok() || !b.ok() || !c.ok() || !result_ok(K) || !result_ok(N)) return SEERA_OK;
    const int sa = (int)(up64(N) / 64), sb = (int)(up64(M) / 64);
    const PackedPlan pa(M, K, sa), pb(K, N, sb);
    const size_t na = align256(a.halves() * 2), nb = align256(b.halves() * 2), nc = align256(c.halves() * 2);
    const size_t np = align256(std::max(pa.splits > 1 ? (size_t)pa.splits * M * K * 4 : 0,
                                        pb.splits > 1 ? (size_t)pb.splits * K * N * 4 : 0));
    const size_t ns = db ? (size_t)(up64(M) / 32) * up64(N) * 4 : 0;
    void* ws = nullptr;
    bool got = false;
    SEERA_TRY(staging_workspace_try(na + nb + nc + np + ns, &ws, st, &got));
    if (!got) return SEERA_OK;
    char* p = static_cast<char*>(ws);
    float* part = reinterpret_cast<float*>(p + na + nb + nc);
    float* sums = db ? reinterpret_cast<float*>(p + na + nb + nc + np) : nullptr;
    PackMats pk{};
    int block = 0;
    const HalfMat ha = add_matrix(pk, block, a, reinterpret_cast<half_t*>(p), nullptr);
    const HalfMat hb = add_matrix(pk, block, b, reinterpret_cast<half_t*>(p + na), nullptr);
    const HalfMat hc = add_matrix(pk, block, c, reinterpret_cast<half_t*>(p + na + nb), sums);
    hipLaunchKernelGGL(pack_matrices, dim3((unsigned)block), dim3(256), 0, st, pk);
    SEERA_HIP_TRY(hipGetLastError());
    // dA [M, K] = dC . B^T: both contracted along their columns. dB [K, N] =
    // A^T . dC: both along their rows.
    if (mask)
        SEERA_TRY((run_packed<true, true, true>(hc, hb, dA, M, K, K, sa, pa, part, nullptr,
                                                const_cast<float*>(mask), kActReluGrad, st)));
    else
        SEERA_TRY((run_packed<true, true, false>(hc, hb, dA, M, K, K, sa, pa, part, nullptr, nullptr, 0, st)));
    SEERA_TRY((run_packed<false, false, false>(ha, hc, dB, K, N, N, sb, pb, part, nullptr, nullptr, 0, st)));
    if (db) SEERA_TRY(column_sums(sums, db, (int)(up64(M) / 32), up64(N), N, st));
    *used = true;
    return SEERA_OK;
}

}  // namespace seera
