// conv_pointwise.hip -- 1x1 stride-1 convolutions as one pass over fp32 memory.
//
// With few filters a 1x1 layer is bound by reading its input and writing its
// outputs once: the products are a tenth of that time, so the operands need no
// packing and the only matter is bytes in flight. One block per CU runs over
// tiles of 128 pixels; [64 channels][128 pixels] pieces of fp32 go to LDS by DMA
// (no registers, no conversion on the way) into a ring of three, so 64 KB per CU
// are under way at any time, across the tiles' ends. Fragments are read from LDS
// as fp32 and rounded there. The weights stay in LDS as fp16, rounded by
// each block, for the whole kernel.
//   forward   Y [F, px] = W . X over 64-channel slices
//   backward  one pass over dY and X: a tile's dY becomes fragments in registers
//             once, and per 64 channels dX [c, px] = W^T . dY is stored and
//             dW [f, c] += dY . X^T kept in registers until the block ends (then a
//             reduce over the blocks, with db)
// 64x256x56x56 -> 64, with the kernels that stream image rows before: forward 80
// -> 62 us (257 MB, 4.1 TB/s), backward 168 -> 126 us (460 MB, 3.7 TB/s), of which
// the reduce is 5. The rows' blocks, 64 of them in the backward, had few bytes
// in flight; dX and dW each read dY.
// Reference: engine_cuda/src/conv2D.cu (the same layer through im2col + GEMM).
#include <algorithm>

#include "conv_pointwise.h"
#include "half_tile.h"
#include "kernels.h"

namespace seera {
namespace {

constexpr int kPix = 128, kSlice = 64, kStage = kPix * kSlice, kStages = 3;

struct PointArgs {
    const float *x, *dy, *w;  // [B, C, HW], [B, F, HW], [F, C]
    float *y, *dx, *part;     // part: [blocks][64 * Cp + 64]
    int B, C, F, HW, Cp;
    int tiles;
    FastDiv per_image;  // tiles of an image
    int image_tiles;
    ConvEpi epi;
};

// Piece p of a stage: thread t moves 16 bytes of row 8 p + t / 32, chunk (4
// pixels) (t % 32) ^ (row % 16): both kinds of fragment then read without bank
// conflicts (32 consecutive pixels of the rows k and k + 8; 16 bytes of 16 rows).
__device__ __forceinline__ void load_stage(const float* src, int rows, int HW, int pixels, float* stage, int tid) {
    const dma_rsrc_t r = make_dma_rsrc(src, kMaxTileSpanBytes);
    const int row = tid >> 5, chunk = (tid & 31) ^ row;
    const uint32_t base = (uint32_t)row * HW * 4u;
    const uint32_t even = chunk * 4 < pixels ? base + chunk * 16 : kBufOOB;
    const uint32_t odd = (chunk ^ 8) * 4 < pixels ? base + (chunk ^ 8) * 16 : kBufOOB;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
#pragma unroll
    for (int p = 0; p < 8; ++p) {
        const uint32_t off = p & 1 ? odd : even;
        dma16(r, reinterpret_cast<half_t*>(stage + (p * 256 + wave * 64) * 4), 8 * p + row < rows ? off : kBufOOB,
              (uint32_t)p * 32u * HW);
    }
}

// Channels 16 kk + 8 (lane / 32) .. + 7 of pixel px, rounded.
__device__ __forceinline__ half8 channel_frag(const float* stage, int px, int kk, int lane) {
    const int h = lane >> 5;
    float v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j)
        v[j] = stage[(kk * 16 + 8 * h + j) * kPix + (((px >> 2) ^ (8 * h + j)) << 2) + (px & 3)];
    return pack8(v);
}

// Pixels 16 ks + 8 (lane / 32) .. + 7 of row r0 + lane % 32.
__device__ __forceinline__ void pixel_values(const float* stage, int r0, int ks, int lane, float (&v)[8]) {
    const float* row = stage + (r0 + (lane & 31)) * kPix;
    const int c = ks * 4 + 2 * (lane >> 5), x = lane & 15;
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        const floatx4 f = *reinterpret_cast<const floatx4*>(row + (((c + q) ^ x) << 2));
#pragma unroll
        for (int j = 0; j < 4; ++j) v[4 * q + j] = f[j];
    }
}

// ---- forward: TF 32-filter tiles ----
template <int TF>
__global__ __launch_bounds__(256, 1) void pointwise_fwd_kernel(const PointArgs g) {
    extern __shared__ __align__(16) float lds[];
    half_t* const wl = reinterpret_cast<half_t*>(lds + kStages * kStage);  // [Cp / 64][32 TF][64]
    float* const bias = reinterpret_cast<float*>(wl + 32 * TF * g.Cp);     // [32 TF]
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int slices = g.Cp >> 6;
    int lt = blockIdx.x, ls = 0, ring = 0;
    auto load = [&] {
        if (lt >= g.tiles) return;
        const int b = g.per_image.div(lt), p0 = (lt - b * g.image_tiles) * kPix;
        load_stage(g.x + ((int64_t)b * g.C + ls * 64) * g.HW + p0, g.C - ls * 64, g.HW, g.HW - p0, lds + ring * kStage,
                   tid);
        ring = ring == kStages - 1 ? 0 : ring + 1;
        if (++ls == slices) {
            ls = 0;
            lt += gridDim.x;
        }
    };
    load();
    load();
    const int chunks = g.Cp >> 3;
    for (int i = tid; i < 32 * TF * chunks; i += 256) {
        const int f = i / chunks, c = (i - f * chunks) * 8;
        float v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = f < g.F && c + j < g.C ? g.w[(int64_t)f * g.C + c + j] : 0.f;
        lds_write8<64>(wl + (c >> 6) * 32 * TF * 64, f, (c & 63) >> 3, pack8(v));
    }
    if (tid < 32 * TF) bias[tid] = g.epi.bias && tid < g.F ? g.epi.bias[tid] : 0.f;

    const int px = 32 * wave + (lane & 31);
    int cur = 0;
    for (int t = blockIdx.x; t < g.tiles; t += gridDim.x) {
        floatx16 acc[TF];
#pragma unroll
        for (int i = 0; i < TF; ++i)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][r] = 0.f;
        for (int s = 0; s < slices; ++s) {
            // This piece has landed: behind it are at most the next one and the
            // stores of the last two iterations.
            if (t + (int)gridDim.x >= g.tiles && s == slices - 1)
                wait_vm<0>();
            else if (t != (int)blockIdx.x && s <= 1)
                wait_vm<8 + (TF > 3 ? 48 : 16 * TF)>();
            else
                wait_vm<8>();
            lds_barrier();
            load();
            const float* stage = lds + cur * kStage;
            cur = cur == kStages - 1 ? 0 : cur + 1;
            const half_t* ws = wl + s * 32 * TF * 64;
#pragma unroll
            for (int kk = 0; kk < 4; ++kk) {
                const half8 x = channel_frag(stage, px, kk, lane);
#pragma unroll
                for (int i = 0; i < TF; ++i)
                    acc[i] = mfma32x32x16(lds_read8<64>(ws, 32 * i + (lane & 31), kk * 2 + (lane >> 5)), x, acc[i]);
            }
        }
        const int b = g.per_image.div(t), p0 = (t - b * g.image_tiles) * kPix;
        const int64_t at = (int64_t)b * g.F * g.HW + p0;
        const rsrc_t ry = make_rsrc(g.y + at);
        rsrc_t rm = ry;
        if (g.epi.mask) rm = make_rsrc(g.epi.mask + at);
        const int f0 = 4 * (lane >> 5);
        const uint32_t o = p0 + px < g.HW ? ((uint32_t)f0 * g.HW + px) * 4u : kBufOOB;
#pragma unroll
        for (int i = 0; i < TF; ++i)
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int row = 32 * i + 8 * (e >> 2) + (e & 3);
                const uint32_t v = f0 + row < g.F ? o : kBufOOB;
                float r = acc[i][e] + bias[f0 + row];
                if (g.epi.act == kActRelu) {
                    if (g.epi.mask) buf_store1s(rm, v, (uint32_t)row * g.HW * 4u, r > 0.f ? 1.f : 0.f);
                    r = r > 0.f ? r : 0.f;
                }
                buf_store1s(ry, v, (uint32_t)row * g.HW * 4u, r);
            }
    }
}

// ---- backward: up to 64 filters, NCH 64-channel slices ----
template <int NCH>
__global__ __launch_bounds__(256, 1) void pointwise_bwd_kernel(const PointArgs g) {
    extern __shared__ __align__(16) float lds[];
    half_t* const wl = reinterpret_cast<half_t*>(lds + kStages * kStage);  // [64 NCH channels][64 filters]
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int lt = blockIdx.x, part = 0, ring = 0;  // part 0: dY, 1 + q: channels 64 q ..
    auto load = [&] {
        if (lt >= g.tiles) return;
        const int b = g.per_image.div(lt), p0 = (lt - b * g.image_tiles) * kPix;
        const int q = part - 1;
        const float* src = part == 0 ? g.dy + (int64_t)b * g.F * g.HW : g.x + ((int64_t)b * g.C + 64 * q) * g.HW;
        load_stage(src + p0, part == 0 ? g.F : g.C - 64 * q, g.HW, g.HW - p0, lds + ring * kStage, tid);
        ring = ring == kStages - 1 ? 0 : ring + 1;
        if (++part > NCH) {
            part = 0;
            lt += gridDim.x;
        }
    };
    load();
    load();
    for (int i = tid; i < 64 * NCH * 8; i += 256) {
        const int c = i % (64 * NCH), f = (i / (64 * NCH)) * 8;
        float v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = c < g.C && f + j < g.F ? g.w[(int64_t)(f + j) * g.C + c] : 0.f;
        lds_write8<64>(wl, c, f >> 3, pack8(v));
    }

    const int px = 32 * wave + (lane & 31), wf = (wave & 1) * 32, wc = (wave >> 1) * 32;
    floatx16 dw[NCH];
#pragma unroll
    for (int q = 0; q < NCH; ++q)
#pragma unroll
        for (int r = 0; r < 16; ++r) dw[q][r] = 0.f;
    float db = 0.f;
    int cur = 0;
    auto next_stage = [&] {
        const float* s = lds + cur * kStage;
        cur = cur == kStages - 1 ? 0 : cur + 1;
        return s;
    };
    for (int t = blockIdx.x; t < g.tiles; t += gridDim.x) {
        const bool first = t == (int)blockIdx.x, last = t + (int)gridDim.x >= g.tiles;
        const int b = g.per_image.div(t), p0 = (t - b * g.image_tiles) * kPix;
        // (waits: the next piece and 32 stores of dX may still be under way)
        if (first)
            wait_vm<8>();
        else
            wait_vm<40>();
        lds_barrier();
        load();
        const float* stage = next_stage();
        half8 yc[4], yp[8];  // dY by channel (for dX) and by pixel (for dW)
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) yc[kk] = channel_frag(stage, px, kk, lane);
        float s = 0.f;
#pragma unroll
        for (int ks = 0; ks < 8; ++ks) {
            float v[8];
            pixel_values(stage, wf, ks, lane, v);
            yp[ks] = pack8(v);
            s += ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
        }
        db += s;
        const uint32_t o = p0 + px < g.HW ? ((uint32_t)(4 * (lane >> 5)) * g.HW + px) * 4u : kBufOOB;
#pragma unroll
        for (int q = 0; q < NCH; ++q) {
            if (last && q == NCH - 1)
                wait_vm<0>();
            else if (first && q == 0)
                wait_vm<8>();
            else
                wait_vm<40>();
            lds_barrier();
            load();
            stage = next_stage();
            floatx16 acc[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[i][r] = 0.f;
#pragma unroll
                for (int kk = 0; kk < 4; ++kk)
                    acc[i] = mfma32x32x16(lds_read8<64>(wl, 64 * q + 32 * i + (lane & 31), kk * 2 + (lane >> 5)),
                                          yc[kk], acc[i]);
            }
            floatx16 sum;  // (of one tile: a chain over all of the block's would round more)
#pragma unroll
            for (int r = 0; r < 16; ++r) sum[r] = 0.f;
#pragma unroll
            for (int ks = 0; ks < 8; ++ks) {
                float v[8];
                pixel_values(stage, wc, ks, lane, v);
                sum = mfma32x32x16(yp[ks], pack8(v), sum);
            }
#pragma unroll
            for (int r = 0; r < 16; ++r) dw[q][r] += sum[r];
            const rsrc_t rx = make_rsrc(g.dx + ((int64_t)b * g.C + 64 * q) * g.HW + p0);
            const int left = g.C - 64 * q - 4 * (lane >> 5);
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    const int row = 32 * i + 8 * (e >> 2) + (e & 3);
                    buf_store1s(rx, row < left ? o : kBufOOB, (uint32_t)row * g.HW * 4u, acc[i][e]);
                }
        }
    }
    float* const out = g.part + (int64_t)blockIdx.x * (64 * g.Cp + 64);
#pragma unroll
    for (int q = 0; q < NCH; ++q)
#pragma unroll
        for (int e = 0; e < 16; ++e)
            out[(wf + 4 * (lane >> 5) + 8 * (e >> 2) + (e & 3)) * g.Cp + 64 * q + wc + (lane & 31)] = dw[q][e];
    db += __shfl_xor(db, 32);
    if (wc == 0 && lane < 32) out[64 * g.Cp + wf + lane] = db;
}

// dW and db: the blocks' sums, four classes of blocks each in order.
__global__ __launch_bounds__(256) void pointwise_reduce(const float* __restrict__ part, int blocks, int n, int F, int C,
                                                        int Cp, float* __restrict__ dW, float* __restrict__ db) {
    __shared__ float red[256];
    const int tid = threadIdx.x, k = tid >> 6, i = blockIdx.x * 64 + (tid & 63);
    float s = 0.f;
    for (int z = k; z < blocks; z += 4 * 8) {
        float v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = z + 4 * j < blocks ? part[(int64_t)(z + 4 * j) * n + i] : 0.f;
        s += ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
    }
    red[tid] = s;
    __syncthreads();
    if (k > 0) return;
    s = ((red[tid] + red[tid + 64]) + red[tid + 128]) + red[tid + 192];
    const int f = i / Cp, c = i - f * Cp;
    if (i < 64 * Cp) {
        if (f < F && c < C) dW[(int64_t)f * C + c] = s;
    } else if (db && i - 64 * Cp < F) {
        db[i - 64 * Cp] = s;
    }
}

constexpr int kBlocks = 256;

template <class K>
int launch_point(K kern, const PointArgs& g, int blocks, int64_t lds, hipStream_t st) {
    SEERA_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                                      (int)lds));
    hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(256), (unsigned)lds, st, g);
    SEERA_HIP_TRY(hipGetLastError());
    return SEERA_OK;
}

bool aligned(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

// Sizes that the pieces and 32-bit offsets allow.
bool point_args(PointArgs& g, int B, int C, int64_t HW, int F) {
    const int64_t per = (HW + kPix - 1) / kPix;
    if (HW < 1 || B < 1 || HW % 4 != 0 || HW * 4 * 128 >= kMaxTileSpanBytes || B * per > 0x7f000000) return false;
    g.B = B; g.C = C; g.F = F; g.HW = (int)HW;
    g.Cp = (C + 63) & ~63;
    g.image_tiles = (int)per;
    g.per_image = FastDiv((uint32_t)per);
    g.tiles = (int)(B * per);
    return true;
}

}  // namespace

int pointwise_conv_fwd(const float* X, const float* Wt, float* Y, int B, int C, int64_t HW, int F, const ConvEpi& epi,
                       hipStream_t st, bool* used) {
    *used = false;
    PointArgs g{};
    const int TF = F <= 32 ? 1 : F <= 64 ? 2 : 4;
    if (C < 1 || F < 1 || F > 128 || !aligned(X) || !point_args(g, B, C, HW, F) || 32 * TF * g.Cp > 32 * 1024) return SEERA_OK;
    g.x = X; g.w = Wt; g.y = Y;
    g.epi = epi;
    const int64_t lds = kStages * kStage * 4 + 32 * TF * g.Cp * 2 + 32 * TF * 4;
    if (lds > 160 * 1024) return SEERA_OK;
    const int blocks = std::min(g.tiles, kBlocks);
    if (TF == 1) SEERA_TRY(launch_point(pointwise_fwd_kernel<1>, g, blocks, lds, st));
    else if (TF == 2) SEERA_TRY(launch_point(pointwise_fwd_kernel<2>, g, blocks, lds, st));
    else SEERA_TRY(launch_point(pointwise_fwd_kernel<4>, g, blocks, lds, st));
    *used = true;
    return SEERA_OK;
}

int pointwise_conv_bwd(const float* dY, const float* Wt, const float* X, float* dX, float* dW, float* db, int B, int C,
                       int64_t HW, int F, hipStream_t st, bool* used) {
    *used = false;
    PointArgs g{};
    if (C < 1 || F < 1 || F > 64 || C > 512 || !aligned(X) || !aligned(dY) || !point_args(g, B, C, HW, F)) return SEERA_OK;
    const int blocks = std::min(g.tiles, kBlocks), n = 64 * g.Cp + 64;
    void* ws = nullptr;
    bool got = false;
    SEERA_TRY(workspace_try(sizeof(float) * (size_t)blocks * n, &ws, st, &got));
    if (!got) return SEERA_OK;
    g.x = X; g.dy = dY; g.w = Wt; g.dx = dX;
    g.part = static_cast<float*>(ws);
    const int64_t lds = kStages * kStage * 4 + 64 * g.Cp * 2;
    typedef void (*Kernel)(const PointArgs);
    static constexpr Kernel kernels[] = {pointwise_bwd_kernel<1>, pointwise_bwd_kernel<2>, pointwise_bwd_kernel<3>,
                                         pointwise_bwd_kernel<4>, pointwise_bwd_kernel<5>, pointwise_bwd_kernel<6>,
                                         pointwise_bwd_kernel<7>, pointwise_bwd_kernel<8>};
    SEERA_TRY(launch_point(kernels[g.Cp / 64 - 1], g, blocks, lds, st));
    hipLaunchKernelGGL(pointwise_reduce, dim3((unsigned)(n / 64)), dim3(256), 0, st, g.part, blocks, n, F, C, g.Cp, dW,
                       db);
    SEERA_HIP_TRY(hipGetLastError());
    *used = true;
    return SEERA_OK;
}

}  // namespace seera
