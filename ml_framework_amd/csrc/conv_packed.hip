// conv_packed.hip -- convolutions as matrix products over operands packed to
// fp16, channels innermost.
//
// The band and row-streaming kernels (conv_band.hip, conv_stream.hip,
// conv_wgrad.hip) read NCHW fp32 and transpose and round it on the way into
// LDS, once per block that needs it: right where a layer has few channels and
// large images (each value is needed by one or two blocks), slow where every
// value is needed by many filter tiles and the rows are short. Here one pass
// writes each operand once as fp16 [C / CB][B, H + halo, W + halo][CB] (C
// rounded up to 32; blocks of CB = 64 channels, 32 where C needs it; the halo
// and the added channels zero), after which every pass of the layer is a
// product whose K slices go to LDS by DMA (half_tile.h), with no conversion,
// predicate or register staging:
//   forward   out[n, q] = sum over channel blocks, taps (t, u) and c of
//             x[cb][q + (t, u)][c] * w[n][cb, t, u, c]
//   dX        the same product over dY with the kernel turned around, one
//             phase per residue of the output row / column modulo the stride
//   dW        dW[f][(t, u), c] = sum over pixels q of dY[q][f] * x[q + (t, u)][c]
// A slice of a tile is one run of memory (consecutive pixels, or consecutive
// weight rows). The choice between this path and the direct kernels, with
// times, is in conv.hip.
// Reference: engine_cuda/src/convolution.cu:15-101, 144-366.
#include "conv_packed.h"

#include <algorithm>
#include <type_traits>

#include "half_tile.h"
#include "packed_limits.h"
#include "runtime.h"

namespace seera {
namespace {

int ceil_div(int a, int b) { return (a + b - 1) / b; }

// ---------------------------------------------------------------------------
// Packing: up to two activations and one weight tensor in one launch.
// ---------------------------------------------------------------------------
struct PackAct {
    const float* in;  // [B, C, H, W]
    half_t* out;      // [Cp / CB][B, Hp, Wp][CB]
    float* sums;      // [prow][Cp] sums of `in` over the pixels of a unit row, or nullptr
    int64_t total;    // B * C * H * W
    int B, C, H, W, top, left, Hp, Wp, Cp;
    int lcb;          // log2 CB
    FastDiv by_ncg, by_npg, by_w, by_nh, by_sides;
    int npg;          // 64-pixel groups per image
    int iters;        // groups per wave
    int prow;         // unit rows: ceil(B * npg / iters)
    int block0;       // blocks from here write the pixels,
    int halo0;        // from here the halo's zeros
    int s2d;          // pixels are 2 x 2 blocks of `in`, 16 channels each (below)
    int ph, pw;       // its padding
    FastDiv by_hpwp, by_wp;
};
struct PackWeightPhase {
    int T, U, r0h, r0w, rsh, rsw;  // tap (t, u) is the kernel's (r0h + rsh * t, r0w + rsw * u)
    int off;                       // halves from PackWeights::out
    FastDiv by_u, by_taps;
};
struct PackWeights {
    const float* in;     // [F, C, R, S]
    half_t* out;         // per phase [channel block][tap][n][CB]
    int F, C, RS, S;
    int by_f;            // rows n are filters (k channels) or the reverse
    int N, K, Kp, lcb;   // rows, k, k rounded up, log2 of the k block
    int64_t total;
    int nct;             // 16-channel tiles
    FastDiv by_nct, by_run;
    int nphase, block0;
    PackWeightPhase ph[kMaxPhase];
};
// Space-to-depth weights: [t][n][u * 16 + c2] for the forward, [f block][t][u]
// [c2][CB] with the kernel turned around for dX.
struct PackS2dWeights {
    const float* in;
    half_t* out;
    int F, C, R, S, by_f;
    int Fp, lfb;
    int block0, items;
};
struct PackArgs {
    PackAct act[2];
    PackWeights w;
    PackS2dWeights w2;
    int nact;
};

// A wave takes 32 channels of 64 consecutive pixels of an image at a time: lane
// (4 pixels) x (4 groups of 8 channels), so a load instruction reads 256
// contiguous bytes of each of 4 channels (16 per lane, at whatever 4-byte
// alignment the plane has) and a store writes 64 contiguous bytes of each of
// 16 pixels; the 4 x 8 block turns around in registers.
__device__ __forceinline__ void pack_act(const PackAct& a, int bid) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int unit = (bid - a.block0) * 4 + wave;
    const int prow = a.by_ncg.div(unit), cg = unit - prow * (a.Cp >> 5);
    if (prow >= a.prow) return;
    const int px = (lane & 15) * 4, c0 = cg * 32 + (lane >> 4) * 8;
    const int HpWp = a.Hp * a.Wp, HW = a.H * a.W;
    float s[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) s[j] = 0.f;
    const int g1 = min((prow + 1) * a.iters, a.B * a.npg);
    for (int g = prow * a.iters; g < g1; ++g) {
        const int b = a.by_npg.div(g), p = (g - b * a.npg) * 64 + px;
        // Past the image's last pixel a load may run into the next channel
        // (never past the tensor: make_rsrc_in); those values are not used.
        const rsrc_t rs = make_rsrc_in(a.in, a.total, (int64_t)b * a.C * HW);
        floatx4 v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j)
            v[j] = buf_load4(rs, p < HW && c0 + j < a.C ? (uint32_t)((c0 + j) * HW + p) * 4u : kBufOOB);
        int h = a.by_w.div(p), w = p - h * a.W;
        int pos = (((cg * 32 >> a.lcb) * a.B + b) * HpWp + (h + a.top) * a.Wp + w + a.left);
        const int ce = c0 & ((1 << a.lcb) - 1);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            float x[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) x[j] = v[j][i];
            if (p + i < HW) {
                *reinterpret_cast<half8*>(a.out + (uint32_t)((pos << a.lcb) + ce)) = pack8(x);
#pragma unroll
                for (int j = 0; j < 8; ++j) s[j] += x[j];
            }
            ++pos;
            if (++w == a.W) {
                w = 0;
                pos += a.Wp - a.W;
            }
        }
    }
    if (a.sums) {
#pragma unroll
        for (int m = 1; m < 16; m <<= 1)
#pragma unroll
            for (int j = 0; j < 8; ++j) s[j] += __shfl_xor(s[j], m);
        if (px == 0) {
#pragma unroll
            for (int j = 0; j < 8; ++j) a.sums[(int64_t)prow * a.Cp + c0 + j] = s[j];
        }
    }
}

// The zeros around the images: top and bottom rows, then the sides.
__device__ __forceinline__ void pack_halo(const PackAct& a, int bid) {
    const int HpWp = a.Hp * a.Wp, nh = HpWp - a.H * a.W;
    const int i = (bid - a.halo0) * 256 + (int)threadIdx.x;
    const int r = i >> (a.lcb - 3), k = i - (r << (a.lcb - 3));
    const int img = a.by_nh.div(r);  // image of a channel block
    if (img >= a.B * (a.Cp >> a.lcb)) return;
    const int z = r - img * nh;
    const int tr = a.top * a.Wp, sides = a.Wp - a.W, z1 = z - tr - a.H * sides;
    int p;
    if (z < tr) {
        p = z;
    } else if (z1 < 0) {
        const int row = a.by_sides.div(z - tr), col = (z - tr) - row * sides;
        p = (a.top + row) * a.Wp + (col < a.left ? col : col + a.W);
    } else {
        p = (a.top + a.H) * a.Wp + z1;
    }
    half8 zero;
#pragma unroll
    for (int j = 0; j < 8; ++j) zero[j] = (half_t)0.f;
    *reinterpret_cast<half8*>(a.out + (uint32_t)(((img * HpWp + p) << a.lcb) + k * 8)) = zero;
}

// The space-to-depth form of an image of at most 4 channels, for a 7 x 7 kernel
// at stride 2: pixel (i, j) of the packed image holds x(2 i + dy - ph, 2 j + dx
// - pw) of channel c at (c * 2 + dy) * 2 + dx, zero outside the image and from
// 4 C to 16. Four pixels side by side are one block of 64: the four column
// taps of the kernel's space-to-depth form.
__device__ __forceinline__ void pack_s2d(const PackAct& a, int bid) {
    const int p = (bid - a.block0) * 256 + (int)threadIdx.x;
    const int b = a.by_hpwp.div(p), r = p - b * a.Hp * a.Wp;
    if (b >= a.B) return;
    const int i = a.by_wp.div(r), j = r - i * a.Wp, HW = a.H * a.W;
    const rsrc_t rs = make_rsrc_in(a.in, a.total, (int64_t)b * a.C * HW);
    float v[16];
#pragma unroll
    for (int e = 0; e < 16; ++e) {
        const int c = e >> 2, h = 2 * i + ((e >> 1) & 1) - a.ph, w = 2 * j + (e & 1) - a.pw;
        const bool in = c < a.C && (unsigned)h < (unsigned)a.H && (unsigned)w < (unsigned)a.W;
        v[e] = buf_load1(rs, in ? (uint32_t)(c * HW + h * a.W + w) * 4u : kBufOOB);
    }
    half8* out = reinterpret_cast<half8*>(a.out + (int64_t)p * 16);
    out[0] = pack8(v);
    out[1] = pack8(v + 8);
}

__device__ __forceinline__ void pack_s2d_weights(const PackS2dWeights& w, int bid) {
    const int i = (bid - w.block0) * 256 + (int)threadIdx.x;
    if (i >= w.items) return;
    const int T = (w.R + 1) >> 1;
    auto at = [&](int f, int c2, int t, int u) {
        const int c = c2 >> 2, r = 2 * t + ((c2 >> 1) & 1), q = 2 * u + (c2 & 1);
        return f < w.F && c < w.C && r < w.R && q < w.S ? w.in[((f * w.C + c) * w.R + r) * w.S + q] : 0.f;
    };
    float v[8];
    if (w.by_f) {  // item: 8 of the 64 halves of row (t, f)
        const int k = (i & 7) * 8, f = (i >> 3) % w.F, t = (i >> 3) / w.F;
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = at(f, (k + j) & 15, t, (k + j) >> 4);
    } else {       // item: 8 filters of row (f block, t, u, c2)
        const int q = i & ((1 << (w.lfb - 3)) - 1), n = 4 * w.C;
        int r = i >> (w.lfb - 3);
        const int c2 = r % n;
        r /= n;
        const int u = r & 3, t = (r >> 2) % T, fb = (r >> 2) / T;
        const int f = (fb << w.lfb) + q * 8;
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = at(f + j, c2, T - 1 - t, 3 - u);
    }
    *reinterpret_cast<half8*>(w.out + (int64_t)i * 8) = pack8(v);
}

// A block takes 16 filters x 16 channels with all their taps through LDS: read
// as runs of 16 R S floats, written as 8 consecutive k per thread for every
// tap. (Each value fetched where a tap needs it costs a line per value: 512 x
// 512 3x3 weights took 5 us more.)
__device__ __forceinline__ void pack_weights(const PackWeights& w, int bid, float* lds) {
    const int tile = bid - w.block0, RS = w.RS, tid = threadIdx.x;
    const int fb = w.by_nct.div(tile), cb = tile - fb * w.nct;
    const int f0 = fb * 16, c0 = cb * 16, run = 16 * RS;
    const rsrc_t rs = make_rsrc_in(w.in, w.total, 0);
    const int cmax = (min(w.C, c0 + 16) - c0) * RS;  // values of one filter's run
    for (int i = tid; i < 16 * run; i += 256) {
        const int f = w.by_run.div(i), j = i - f * run;
        lds[i] = buf_load1(rs, f0 + f < w.F && j < cmax ? (uint32_t)(((f0 + f) * w.C + c0) * RS + j) * 4u
                                                        : kBufOOB);
    }
    __syncthreads();
    for (int z = 0; z < w.nphase; ++z) {
        const PackWeightPhase& p = w.ph[z];
        const int taps = p.T * p.U;
        for (int i = tid; i < 32 * taps; i += 256) {  // item: (k half, n of 16, tap)
            const int h = i & 1, n16 = (i >> 1) & 15, tap = i >> 5;
            const int t = p.by_u.div(tap), u = tap - t * p.U;
            const int src = (p.r0h + p.rsh * t) * w.S + p.r0w + p.rsw * u;
            const int n = (w.by_f ? f0 : c0) + n16, k = (w.by_f ? c0 : f0) + 8 * h;
            if (n >= w.N || k >= w.Kp) continue;
            float v[8];
#pragma unroll
            for (int j = 0; j < 8; ++j)
                v[j] = w.by_f ? lds[n16 * run + (8 * h + j) * RS + src] : lds[(8 * h + j) * run + n16 * RS + src];
            const int kb = k >> w.lcb, kr = k & ((1 << w.lcb) - 1);
            *reinterpret_cast<half8*>(w.out + p.off + ((((int64_t)kb * taps + tap) * w.N + n) << w.lcb) + kr) =
                pack8(v);
        }
    }
}

__global__ __launch_bounds__(256) void pack_kernel(const PackArgs a) {
    extern __shared__ __align__(16) float pack_lds[];
    // Weights first: their blocks take longest.
    const int bid = blockIdx.x;
    if (bid < a.act[0].block0) {
        if (bid >= a.w2.block0) return pack_s2d_weights(a.w2, bid);
        return pack_weights(a.w, bid, pack_lds);
    }
    const PackAct& t = a.act[a.nact > 1 && bid >= a.act[1].block0];
    if (t.s2d) return pack_s2d(t, bid);
    if (bid >= t.halo0) return pack_halo(t, bid);
    pack_act(t, bid);
}

// ---------------------------------------------------------------------------
// out[b, n, pixel] = sum over K of w[n][k] * x[pixel row offset + k]
// ---------------------------------------------------------------------------
struct PackedPhase {
    int Ho, Wo;     // output grid of the phase
    int npix;       // B * Ho * Wo
    int T, U;       // kernel rows and columns
    int x0;         // halves from a pixel's row offset to its first tap
    int oph, opw;   // output row = oh * osh + oph
    int64_t woff;   // halves
    FastDiv by_howo, by_wo;
};
struct PackedConvArgs {
    const half_t* x;
    const half_t* w;
    float* out;
    uint32_t x_bytes;
    int pix;              // halves from a pixel to the next (CB, or less where a
                          // block spans several pixels)
    int ncb, plane;       // channel blocks, halves of one
    int Wp, HpWp;         // row and image pitch in pixels
    int N, Hout, Wout;
    int ish, isw, osh, osw;
    int ntn, nblocks, nphase;
    FastDiv by_ntn, by_phase;
    PackedPhase ph[kMaxPhase];
    ConvEpi epi;
    int R, S;             // kS2d*: the kernel's own rows and columns
};

// What the product is of. kS2dForward, kS2dInput: a first layer in
// space-to-depth form, whose 2 T x 8 taps are rounded up from R x S.
enum PackedKind { kPlain, kS2dForward, kS2dInput };

// One sum of a space-to-depth product over the kernel's own taps. The matrix
// cores also multiply the added taps' zero weights, and 0 * inf is NaN where an
// infinite operand is no term of the output: a lane that finds NaN takes the sum
// from here, as far as it stays a number (where all operands are NaN the first
// eight settle it). n: output channel; pi, pj: the output pixel in the phase's grid.
template <int BK, PackedKind KIND>
__device__ __forceinline__ float own_taps_sum(const PackedConvArgs& a, int b, int pi, int pj, int n) {
    const PackedPhase& ph = a.ph[0];
    const int taps = ph.T * ph.U;
    float s = 0.f;
    for (int cb = 0; cb < a.ncb; ++cb)
        for (int tap = 0; tap < taps; ++tap) {
            const int t = tap / ph.U, u = tap - t * ph.U;
            const half8* x = reinterpret_cast<const half8*>(
                a.x + cb * (int64_t)a.plane + ph.x0 +
                (int64_t)(b * a.HpWp + (pi * a.ish + t) * a.Wp + pj * a.isw + u) * a.pix);
            const half8* w = reinterpret_cast<const half8*>(a.w + ph.woff + ((int64_t)(cb * taps + tap) * a.N + n) * BK);
            for (int k = 0; k < BK / 8 && s == s; ++k) {
                const half8 xv = x[k], wv = w[k];
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    // (the forward's slice is a kernel row: 4 columns of 2 x 2 x 4 channels)
                    const int c2 = KIND == kS2dForward ? j : n, col = KIND == kS2dForward ? k >> 1 : 3 - u;
                    const int row = KIND == kS2dForward ? t : ph.T - 1 - t;
                    if (2 * row + ((c2 >> 1) & 1) < a.R && 2 * col + (c2 & 1) < a.S) s += (float)xv[j] * (float)wv[j];
                }
            }
        }
    return s;
}

// BP pixels x BN output channels per block, WP x WN waves, three LDS stages.
template <int BP, int BN, int WP, int WN, int BK>
struct PackedCfg {
    static constexpr int NT = 64 * WP * WN, NS = 3;
    using TX = KcTile<BP, BK, NT>;
    using TW = KcTile<BN, BK, NT>;
    static constexpr int STAGE = TX::HALVES + TW::HALVES;
    static constexpr int LDS_BYTES = NS * STAGE * 2;
    static constexpr int LOADS = TX::PASSES + TW::PASSES;  // DMA instructions per wave and slice
};

// kS2dInput: the output is the space-to-depth form's dX, stored to the image it came
// from: channel (c * 2 + dy) * 2 + dx of pixel (i, j) is pixel (2 i + dy - oph,
// 2 j + dx - opw) of channel c (oph, opw: the padding), where that lies inside.
template <int BP, int BN, int WP, int WN, int BK, PackedKind KIND>
__global__ __launch_bounds__(64 * WP * WN, 1) void packed_conv_kernel(const PackedConvArgs a) {
    using Cfg = PackedCfg<BP, BN, WP, WN, BK>;
    using TX = typename Cfg::TX;
    using TW = typename Cfg::TW;
    constexpr int NT = Cfg::NT, TM = BN / WN / 32, TN = BP / WP / 32;
    extern __shared__ __align__(16) half_t smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int id = xcd_order(blockIdx.x, a.nblocks);
    // The phases of one pixel tile are neighbours: they read the same input, and
    // their stores interleave in the same lines.
    const int pz = a.by_phase.div(id), z = id - pz * a.nphase;
    const int pt = a.by_ntn.div(pz);
    const PackedPhase& ph = a.ph[z];
    const int n0 = (pz - pt * a.ntn) * BN, q0 = pt * BP;
    if (q0 >= ph.npix) return;  // (a phase with fewer tiles than the others)
    const int HoWo = ph.Ho * ph.Wo;
    const int taps = ph.T * ph.U;
    uint32_t xo[TX::PASSES], wo[TW::PASSES];
#pragma unroll
    for (int p = 0; p < TX::PASSES; ++p) {
        int row, chunk;
        TX::item(p * NT + tid, row, chunk);
        const int q = min(q0 + row, ph.npix - 1);
        const int b = ph.by_howo.div(q), r = q - b * HoWo;
        const int oh = ph.by_wo.div(r), ow = r - oh * ph.Wo;
        xo[p] = (uint32_t)((b * a.HpWp + oh * a.ish * a.Wp + ow * a.isw) * a.pix + ph.x0 + chunk * 8) * 2u;
    }
#pragma unroll
    for (int p = 0; p < TW::PASSES; ++p) {
        int row, chunk;
        TW::item(p * NT + tid, row, chunk);
        wo[p] = (uint32_t)(min(n0 + row, a.N - 1) * BK + chunk * 8) * 2u;
    }
    const dma_rsrc_t rx = make_dma_rsrc(a.x, a.x_bytes);
    const dma_rsrc_t rw = make_dma_rsrc(a.w + ph.woff, (uint32_t)((int64_t)a.N * a.ncb * taps * BK * 2));

    const int nslice = a.ncb * taps;
    // Byte steps of the slice offsets: next tap column, next tap row, next
    // channel block, next weight slice.
    const int U = ph.U, T = ph.T;
    const uint32_t du = (uint32_t)a.pix * 2u, dt = (uint32_t)((a.Wp - U) * a.pix) * 2u;
    const uint32_t dc = (uint32_t)(a.plane - T * a.Wp * a.pix) * 2u, dw = (uint32_t)(a.N * BK) * 2u;
    int it = 0, iu = 0;         // tap of the next slice to load
    uint32_t isx = 0, isw = 0;  // its byte offsets
    auto load = [&](int l, half_t* stage) {
        half_t* d = stage + wave * 512 + l * NT * 8;  // the X tile lies behind the W tile
        if (l < TW::PASSES)
            dma16(rw, d, wo[l < TW::PASSES ? l : 0], isw);
        else
            dma16(rx, d, xo[l < TW::PASSES ? 0 : l - TW::PASSES], isx);
        if (l == Cfg::LOADS - 1) {
            isw += dw;
            isx += du;
            if (++iu == U) {
                iu = 0;
                isx += dt;
                if (++it == T) {
                    it = 0;
                    isx += dc;
                }
            }
        }
    };

    floatx16 part[TM][TN], acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) part[i][j][r] = acc[i][j][r] = 0.f;

    const int wn = (wave % WN) * (BN / WN), wp = (wave / WN) * (BP / WP);
    half_pipeline<TW, TX, BK / 16, Cfg::NS, Cfg::LOADS, TM, TN>(smem, Cfg::STAGE, TW::HALVES, wn, wp, 0,
                                                                lane, nslice, part, load, [&](int s) {
                                                                    add_part<768 / BK>(s, part, acc);
                                                                });
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] += part[i][j][r];
    // Lane l holds channels m0 + 32 i + 8 (e / 4) + e % 4 of pixel column l % 32.
    // The bias is in registers before the first store: a load between stores
    // would wait for them.
    const int64_t plane = (int64_t)a.Hout * a.Wout;
    const int m0 = n0 + wn + 4 * (lane >> 5);
    auto chan = [](int i, int e) { return 32 * i + 8 * (e >> 2) + (e & 3); };
    const int act = a.epi.act;
    const float* bp = a.epi.bias;
    float* const mp = a.epi.mask;
    if (bp) {
        float bias[TM][16];
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int e = 0; e < 16; ++e) bias[i][e] = bp[min(m0 + chan(i, e), a.N - 1)];
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int e = 0; e < 16; ++e) acc[i][j][e] += bias[i][e];
    }
    // Stores through a resource over the block's images: a lane past the phase's
    // pixels or the channels gets an offset that the hardware drops.
    const int b0 = ph.by_howo.div(q0), left = a.N - m0;
    const int64_t img = (int64_t)(KIND == kS2dInput ? a.N >> 2 : a.N) * plane;
    const rsrc_t ro = make_rsrc(a.out + b0 * img), rm = make_rsrc((mp ? mp : a.out) + b0 * img);
    const uint32_t step = (uint32_t)plane * 4u;
    static_assert(TM * 16 <= 32, "one bit per sum of a column");
    if constexpr (KIND == kS2dInput) {
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const int q = q0 + wp + 32 * j + (lane & 31);
            const int b = ph.by_howo.div(q), r = q - b * HoWo;
            const int pi = ph.by_wo.div(r), pj = r - pi * ph.Wo;
            const int h0 = 2 * pi - ph.oph, w0 = 2 * pj - ph.opw;
            auto put = [&](int n, float v) {
                const int h = h0 + ((n >> 1) & 1), w = w0 + (n & 1);
                const bool in = q < ph.npix && n < a.N && (unsigned)h < (unsigned)a.Hout &&
                                (unsigned)w < (unsigned)a.Wout;
                const uint32_t o = (uint32_t)((b - b0) * img + (n >> 2) * plane + h * a.Wout + w) * 4u;
                __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), ro, in ? o : kBufOOB, 0, 0);
            };
            uint32_t nan = 0;
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    const float v = acc[i][j][e];
                    put(m0 + chan(i, e), v);
                    nan |= v != v ? 1u << (i * 16 + e) : 0u;
                }
            if (q >= ph.npix) nan = 0;
            for (; nan != 0; nan &= nan - 1) {
                const int k = __builtin_ctz(nan), n = m0 + chan(k >> 4, k & 15);
                if (n < a.N) put(n, own_taps_sum<BK, KIND>(a, b, pi, pj, n));
            }
        }
        return;
    }
    auto store = [&](auto relu, auto mask) {
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const int q = q0 + wp + 32 * j + (lane & 31);
            const int b = ph.by_howo.div(q), r = q - b * HoWo;
            const int oh = ph.by_wo.div(r), ow = r - oh * ph.Wo;
            const uint32_t o = (uint32_t)((b - b0) * img + m0 * plane +
                                          (int64_t)(oh * a.osh + ph.oph) * a.Wout + ow * a.osw +
                                          ph.opw) * 4u;
            const int nl = q < ph.npix ? left : 0;
            auto put = [&](uint32_t at, uint32_t row, float v) {
                const float y = decltype(relu)::value ? (v > 0.f ? v : 0.f) : v;
                __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, y), ro, at, row, 0);
                if (decltype(mask)::value) {
                    const float k = v > 0.f ? 1.f : 0.f;
                    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, k), rm, at, row, 0);
                }
            };
            uint32_t nan = 0;
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    const float v = acc[i][j][e];
                    put(chan(i, e) < nl ? o : kBufOOB, chan(i, e) * step, v);
                    if constexpr (KIND == kS2dForward) nan |= v != v ? 1u << (i * 16 + e) : 0u;
                }
            if constexpr (KIND == kS2dForward) {
                for (; nan != 0; nan &= nan - 1) {
                    const int k = __builtin_ctz(nan), c = chan(k >> 4, k & 15);
                    if (c < nl)
                        put(o + (uint32_t)c * step, 0u,
                            own_taps_sum<BK, KIND>(a, b, oh, ow, m0 + c) + (bp ? bp[m0 + c] : 0.f));
                }
            }
        }
    };
    constexpr std::true_type yes;
    constexpr std::false_type no;
    if (act != kActRelu) store(no, no);
    else if (!mp) store(yes, no);
    else store(yes, yes);
}

// ---------------------------------------------------------------------------
// part[split][f][col] = sum over the split's pixels of dY[q][f] * x[q + tap][c]
// ---------------------------------------------------------------------------
struct PackedWgradArgs {
    const half_t* y;      // dY [B, Hy, Wy, Fp]
    const half_t* x;      // X [B, Hx, Wx, Cp]
    float* part;          // [nsplit][F][L]
    uint32_t y_bytes, x_bytes;
    int F, L, S;          // filters, R * S * Cp columns (tap, c), kernel columns
    int Ho, Wo, npix;
    int Fp, lfb, yplane;             // filters rounded up, log2 of the block, halves of one block
    int Cp, lcb, xplane;             // channels
    int y0, yrow, yimg, ypix;        // halves: dY(0, 0) and its row / image / pixel pitch
    int xrow, ximg, xpix;            // X: the same per output row / column / image
    int xtap, xcol;                  // and per kernel row / column
    int d_b, d_h, d_w;    // BK pixels = d_b images + d_h rows + d_w columns
    int ntf, ntl, nsplit, sps;       // tiles, splits, slices per split
    int nblocks;
    FastDiv by_howo, by_wo, by_cp, by_s;
};

template <int BF, int BL, int WF, int WL, int NS, int KG>
__global__ __launch_bounds__(64 * WF * WL * KG, 1) void packed_wgrad_kernel(const PackedWgradArgs a) {
    constexpr int BK = 64, NT = 64 * WF * WL * KG;
    using TY = McTile<BF, BK, NT>;
    using TXx = McTile<BL, BK, NT>;
    constexpr int STAGE = TY::HALVES + TXx::HALVES, LOADS = TY::PASSES + TXx::PASSES;
    constexpr int TM = BF / WF / 32, TN = BL / WL / 32;
    extern __shared__ __align__(16) half_t smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int id = xcd_order(blockIdx.x, a.nblocks);
    const int tiles = a.ntf * a.ntl, split = id / tiles, tile = id - split * tiles;
    const int f0 = (tile % a.ntf) * BF, l0 = (tile / a.ntf) * BL;

    const int total = (a.npix + BK - 1) / BK;
    const int s0 = split * a.sps, nslice = min(a.sps, total - s0);
    const dma_rsrc_t ry = make_dma_rsrc(a.y, a.y_bytes), rx = make_dma_rsrc(a.x, a.x_bytes);

    // The pixel that a thread loads in each pass, its row and column and the byte
    // offsets of its dY and X rows, moves on by BK pixels per slice: by a fixed
    // step and, at the end of a row or an image, a fixed correction.
    // (Multiplying the place out for every load took as long as the products.)
    struct Pos {
        int q, w, h;
        uint32_t oy, ox;
    };
    const int npix = a.npix, Ho = a.Ho, Wo = a.Wo, d_h = a.d_h, d_w = a.d_w;
    const uint32_t y1 = (uint32_t)(a.d_b * a.yimg + d_h * a.yrow + d_w * a.ypix) * 2u,
                   y2 = (uint32_t)(a.yrow - Wo * a.ypix) * 2u, y3 = (uint32_t)(a.yimg - Ho * a.yrow) * 2u,
                   x1 = (uint32_t)(a.d_b * a.ximg + d_h * a.xrow + d_w * a.xpix) * 2u,
                   x2 = (uint32_t)(a.xrow - Wo * a.xpix) * 2u, x3 = (uint32_t)(a.ximg - Ho * a.xrow) * 2u;
    auto place = [&](int q, int cy, int cx) {
        const int b = a.by_howo.div(q), r = q - b * Ho * Wo;
        Pos p;
        p.q = q;
        p.h = a.by_wo.div(r);
        p.w = r - p.h * Wo;
        p.oy = (uint32_t)(b * a.yimg + p.h * a.yrow + p.w * a.ypix + cy) * 2u;
        p.ox = (uint32_t)(b * a.ximg + p.h * a.xrow + p.w * a.xpix + cx) * 2u;
        return p;
    };
    auto advance = [&](Pos& p) {
        p.q += BK;
        p.w += d_w;
        p.h += d_h;
        p.oy += y1;
        p.ox += x1;
        const bool c = p.w >= Wo;
        p.w -= c ? Wo : 0;
        p.h += c ? 1 : 0;
        p.oy += c ? y2 : 0u;
        p.ox += c ? x2 : 0u;
        const bool d = p.h >= Ho;
        p.h -= d ? Ho : 0;
        p.oy += d ? y3 : 0u;
        p.ox += d ? x3 : 0u;
    };
    auto y_col = [&](int chunk) {  // (past the padded filters: never stored)
        const int f = f0 + chunk * 8;
        return a.y0 + (f < a.Fp ? (f >> a.lfb) * a.yplane + (f & ((1 << a.lfb) - 1)) : 0);
    };
    auto x_col = [&](int chunk) {
        const int col = l0 + chunk * 8, tap = a.by_cp.div(col), c = col - tap * a.Cp;
        const int t = a.by_s.div(tap), u = tap - t * a.S;
        return col < a.L ? (c >> a.lcb) * a.xplane + t * a.xtap + u * a.xcol + (c & ((1 << a.lcb) - 1)) : 0;
    };
    // Tiles of one width load the same pixels in the same passes.
    constexpr bool kSame = BF == BL;
    Pos py[TY::PASSES], px[kSame ? 1 : TXx::PASSES];
#pragma unroll
    for (int p = 0; p < TY::PASSES; ++p) {
        int k, chunk;
        TY::item(p * NT + tid, k, chunk);
        py[p] = place(s0 * BK + k, y_col(chunk), kSame ? x_col(chunk) : 0);
    }
    if constexpr (!kSame) {
#pragma unroll
        for (int p = 0; p < TXx::PASSES; ++p) {
            int k, chunk;
            TXx::item(p * NT + tid, k, chunk);
            px[p] = place(s0 * BK + k, 0, x_col(chunk));
        }
    }
    auto load = [&](int l, half_t* stage) {  // (the X tile lies behind the dY tile)
        half_t* d = stage + wave * 512 + l * NT * 8;
        const bool y = l < TY::PASSES;
        const int i = y ? l : l - TY::PASSES;
        Pos& p = y || kSame ? py[i < TY::PASSES ? i : 0] : px[kSame ? 0 : i];
        dma16(y ? ry : rx, d, p.q < npix ? (y ? p.oy : p.ox) : kBufOOB, 0);
        if (!(y && kSame)) advance(p);
    };

    floatx16 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

    constexpr int GW = WF * WL, KK = BK / 16 / KG;
    const int grp = wave / GW, gw = wave % GW;
    const int wf = (gw % WF) * (BF / WF), wl = (gw / WF) * (BL / WL);
    // Parts of 16 steps, 8 where one wave takes all of a slice and the direct
    // kernels split the pixels finely (few filters). 64 images of 512 channels at
    // 7 x 7: relative error 3.5e-7 in one chain, 1.2e-7 in parts of 16.
    constexpr int kPart = (KG > 1 ? 16 : 8) / KK;
    floatx16 sum[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) sum[i][j] = acc[i][j];
    auto flush = [&](int s) { add_part<kPart>(s, acc, sum); };
    half_pipeline<TY, TXx, KK, NS, LOADS, TM, TN>(smem, STAGE, TY::HALVES, wf, wl, grp * KK, lane,
                                                  nslice, acc, load, flush);
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) sum[i][j][r] += acc[i][j][r];
    sum_groups<KG, GW, TM, TN>(reinterpret_cast<float*>(smem), wave, lane, sum);
    if (grp > 0) return;
    float* out = a.part + (int64_t)split * a.F * a.L;
#pragma unroll
    for (int j = 0; j < TN; ++j) {
        const int col = l0 + wl + 32 * j + (lane & 31);
        if (col >= a.L) continue;
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int f = f0 + wf + 32 * i + 8 * (e >> 2) + 4 * (lane >> 5) + (e & 3);
                if (f < a.F) out[(int64_t)f * a.L + col] = sum[i][j][e];
            }
    }
}

// db[f] = sum over the unit rows of the packing pass's sums: 16 filters a block,
// 32 row classes each added in order and then in a fixed tree.
__device__ __forceinline__ void reduce_db(const float* __restrict__ sums, int prow, int Fp, int F,
                                          float* __restrict__ db, int block, float* red) {
    const int tid = threadIdx.x, f = block * 16 + (tid & 15), g = tid >> 4;
    float s = 0.f;
    if (f < F) {
        int r = g;
        for (; r + 7 * 32 < prow; r += 8 * 32) {
            float v[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) v[i] = sums[(int64_t)(r + 32 * i) * Fp + f];
#pragma unroll
            for (int i = 0; i < 8; ++i) s += v[i];
        }
        for (; r < prow; r += 32) s += sums[(int64_t)r * Fp + f];
    }
    red[tid] = s;
    __syncthreads();
    for (int h = 16; h > 0; h >>= 1) {
        if (g < h) red[tid] += red[tid + 16 * h];
        __syncthreads();
    }
    if (g == 0 && f < F) db[f] = red[tid];
}

// dW[f, c, tap] = sum over splits of part[split][f][tap * Cp + c]: P runs of
// splits each added in order, the runs then in order. Block: one filter, 64 / P
// channels, all taps; the sums through LDS so that the store is contiguous.
// Blocks from nb_w on: db. With many splits (few, small tiles) one run would be
// a chain of memory round trips (49 splits of 64 x 32 3x3 weights: 7.2 -> 6.4 us).
template <int P>
__global__ __launch_bounds__(512) void packed_wgrad_reduce(const float* __restrict__ part,
                                                           float* __restrict__ dW, int F, int C,
                                                           int Cp, int RS, int nsplit,
                                                           int nb_w, const float* __restrict__ sums,
                                                           int prow, int Fp,
                                                           float* __restrict__ db) {
    extern __shared__ __align__(16) float red[];
    const int tid = threadIdx.x;
    if ((int)blockIdx.x >= nb_w) return reduce_db(sums, prow, Fp, F, db, blockIdx.x - nb_w, red);
    constexpr int CG = 64 / P;
    const int ncb = (C + CG - 1) / CG, f = blockIdx.x / ncb, c0 = (blockIdx.x % ncb) * CG;
    const int L = RS * Cp;
    const int64_t stride = (int64_t)F * L;
    const int c = tid & (CG - 1), g = (tid & 63) / CG;
    const int per = (nsplit + P - 1) / P, z1 = min(nsplit, (g + 1) * per);
    for (int tap = tid >> 6; tap < RS; tap += 8) {
        float s = 0.f;
        if (c0 + c < C) {
            const float* src = part + (int64_t)f * L + tap * Cp + c0 + c;
            int z = g * per;
            for (; z + 8 <= z1; z += 8) {
                float v[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) v[i] = src[(z + i) * stride];
#pragma unroll
                for (int i = 0; i < 8; ++i) s += v[i];
            }
            for (; z < z1; ++z) s += src[z * stride];
        }
        red[(c * RS + tap) * P + g] = s;
    }
    __syncthreads();
    const int n = min(CG, C - c0) * RS;
    float* dst = dW + ((int64_t)f * C + c0) * RS;
    for (int i = tid; i < n; i += 512) {
        float s = red[i * P];
#pragma unroll
        for (int k = 1; k < P; ++k) s += red[i * P + k];
        dst[i] = s;
    }
}

// The same for the space-to-depth form: dW[f, c, r, q] = sum over splits of
// part[split][f][(r / 2) * 64 + (q / 2) * 16 + (c * 2 + r % 2) * 2 + q % 2].
// Block: one filter, 64 columns, 8 runs of splits each added in order, the runs
// then in order. Blocks from nb_w on: db as above.
__global__ __launch_bounds__(512) void packed_wgrad_reduce_s2d(const float* __restrict__ part,
                                                               float* __restrict__ dW, int F, int C,
                                                               int R, int S, int L, int nsplit,
                                                               int nb_w, const float* __restrict__ sums,
                                                               int prow, int Fp,
                                                               float* __restrict__ db) {
    __shared__ float red[512];
    if ((int)blockIdx.x >= nb_w) return reduce_db(sums, prow, Fp, F, db, blockIdx.x - nb_w, red);
    const int tid = threadIdx.x, ncol = L >> 6;
    const int f = blockIdx.x / ncol, t = blockIdx.x - f * ncol, col = tid & 63, g = tid >> 6;
    const int64_t stride = (int64_t)F * L;
    const float* src = part + (int64_t)f * L + t * 64 + col;
    const int per = (nsplit + 7) >> 3, z1 = min(nsplit, (g + 1) * per);
    float s = 0.f;
    int z = g * per;
    for (; z + 8 <= z1; z += 8) {
        float v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = src[(z + i) * stride];
#pragma unroll
        for (int i = 0; i < 8; ++i) s += v[i];
    }
    for (; z < z1; ++z) s += src[z * stride];
    red[tid] = s;
    __syncthreads();
    if (g == 0) {
#pragma unroll
        for (int i = 1; i < 8; ++i) s += red[i * 64 + col];
        const int u = col >> 4, c2 = col & 15, c = c2 >> 2;
        const int r = 2 * t + ((c2 >> 1) & 1), q = 2 * u + (c2 & 1);
        if (c < C && r < R && q < S) dW[((f * C + c) * R + r) * S + q] = s;
    }
}

// ---------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------

// One packed activation: geometry and size.
struct Packed {
    int top, left, Hp, Wp, Cp;
    int CB;
    Packed(int top_, int left_, int Hp_, int Wp_, int C, int round = 32)
        : top(top_), left(left_), Hp(Hp_), Wp(Wp_), Cp((C + round - 1) / round * round),
          CB(Cp % 64 == 0 ? 64 : 32) {}
    int lcb() const { return CB == 64 ? 6 : 5; }
    int64_t plane(int B) const { return (int64_t)B * Hp * Wp * CB; }
    int64_t halves(int B) const { return (int64_t)B * Hp * Wp * Cp; }
};

struct Axis {
    int r0, T, q, n;
};
// The kernel taps that reach output residue `phi` of a transposed convolution
// along one axis: taps r0 + s * m (m < T), input row oh + q - m.
Axis dgrad_axis(int phi, int p, int s, int K, int out_len) {
    Axis x;
    x.r0 = (phi + p) % s;
    x.T = K > x.r0 ? (K - x.r0 + s - 1) / s : 0;
    x.q = (phi + p - x.r0) / s;
    x.n = out_len > phi ? (out_len - phi + s - 1) / s : 0;
    return x;
}

// The layer's input as its forward and dW read it.
Packed input_geometry(const Conv& c) { return Packed(c.ph, c.pw, c.H + 2 * c.ph, c.W + 2 * c.pw, c.C); }

// The layer's output (dY) with the halo that the dX phases read.
struct DgradGeometry {
    Axis ah[kMaxPhase], aw[kMaxPhase];
    Packed g;
    explicit DgradGeometry(const Conv& c) : g(0, 0, 0, 0, c.F) {
        auto halo = [](Axis* x, int s, int p, int K, int len, int out, int* before, int* after) {
            *before = *after = 0;
            for (int i = 0; i < s; ++i) {
                x[i] = dgrad_axis(i, p, s, K, len);
                *before = std::max(*before, x[i].T - 1 - x[i].q);
                *after = std::max(*after, x[i].n - 1 + x[i].q - (out - 1));
            }
        };
        int bottom, right;
        halo(ah, c.sh, c.ph, c.R, c.H, c.Ho, &g.top, &bottom);
        halo(aw, c.sw, c.pw, c.S, c.W, c.Wo, &g.left, &right);
        g.Hp = c.Ho + g.top + bottom;
        g.Wp = c.Wo + g.left + right;
    }
};

struct Scratch {
    size_t bytes = 0;
    char* p = nullptr;
    size_t used = 0;
    template <class T>
    void need(int64_t n) {
        bytes += ((size_t)n * sizeof(T) + 255) & ~(size_t)255;
    }
    template <class T>
    T* take(int64_t n) {
        T* r = reinterpret_cast<T*>(p + used);
        used += ((size_t)n * sizeof(T) + 255) & ~(size_t)255;
        return r;
    }
    int get(hipStream_t st, bool* got) {
        void* ws = nullptr;
        SEERA_TRY(staging_workspace_try(std::max<size_t>(bytes, 256), &ws, st, got));
        p = static_cast<char*>(ws);
        return SEERA_OK;
    }
};

// Groups of 64 pixels per wave and unit rows of a packing pass: at most about
// 1024 unit rows, so that the bias gradient's second step stays short.
void pack_split(int B, int HW, int* iters, int* prow) {
    const int64_t groups = (int64_t)B * ceil_div(HW, 64);
    *iters = (int)((groups + 1023) / 1024);
    *prow = (int)((groups + *iters - 1) / *iters);
}

void add_act(PackArgs& pk, int& block, const float* in, half_t* out, int B, int C, int H, int W,
             const Packed& g, float* sums) {
    PackAct& a = pk.act[pk.nact++];
    a.in = in; a.out = out; a.sums = sums;
    a.total = (int64_t)B * C * H * W;
    a.B = B; a.C = C; a.H = H; a.W = W;
    a.top = g.top; a.left = g.left; a.Hp = g.Hp; a.Wp = g.Wp; a.Cp = g.Cp;
    a.lcb = g.lcb();
    a.npg = ceil_div(H * W, 64);
    a.by_ncg = FastDiv(g.Cp / 32);
    a.by_npg = FastDiv(a.npg);
    a.by_w = FastDiv(W);
    a.by_nh = FastDiv(std::max(1, g.Hp * g.Wp - H * W));
    a.by_sides = FastDiv(std::max(1, g.Wp - W));
    pack_split(B, H * W, &a.iters, &a.prow);
    a.block0 = block;
    block += ceil_div(a.prow * (g.Cp / 32), 4);
    a.halo0 = block;
    block += (int)((((int64_t)g.Hp * g.Wp - (int64_t)H * W) * B * (g.Cp / 8) + 255) / 256);
}

// Weights first in the launch (block 0 on); returns their halves.
void add_weights(PackArgs& pk, int& block, const float* in, half_t* out, const Conv& c, bool by_f,
                 const Packed& kg) {
    PackWeights& w = pk.w;
    w.in = in; w.out = out;
    w.F = c.F; w.C = c.C; w.RS = c.R * c.S; w.S = c.S;
    w.by_f = by_f;
    w.N = by_f ? c.F : c.C;
    w.K = by_f ? c.C : c.F;
    w.Kp = kg.Cp;
    w.lcb = kg.lcb();
    w.total = (int64_t)c.F * c.C * w.RS;
    w.nct = ceil_div(by_f ? w.Kp : c.C, 16);
    w.by_nct = FastDiv(w.nct);
    w.by_run = FastDiv(16 * w.RS);
    w.block0 = block;
    block += w.nct * ceil_div(by_f ? c.F : w.Kp, 16);
    pk.w2.block0 = block;
}

int launch_pack(const PackArgs& pk, int blocks, hipStream_t st) {
    hipLaunchKernelGGL(pack_kernel, dim3((unsigned)blocks), dim3(256), 256 * (size_t)pk.w.RS * 4, st, pk);
    SEERA_HIP_TRY(hipGetLastError());
    return SEERA_OK;
}

template <int BP, int BN, int WP, int WN, int BK, PackedKind KIND>
hipError_t launch_conv(PackedConvArgs a, int most, hipStream_t st) {
    using Cfg = PackedCfg<BP, BN, WP, WN, BK>;
    auto kern = packed_conv_kernel<BP, BN, WP, WN, BK, KIND>;
    static_assert(Cfg::LDS_BYTES <= 160 * 1024, "LDS of one CU");
    if (Cfg::LDS_BYTES > 65536) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, Cfg::LDS_BYTES);
        if (e != hipSuccess) return e;
    }
    a.ntn = ceil_div(a.N, BN);
    a.by_ntn = FastDiv(a.ntn);
    a.by_phase = FastDiv(a.nphase);
    a.nblocks = ceil_div(most, BP) * a.ntn * a.nphase;
    hipLaunchKernelGGL(kern, dim3((unsigned)a.nblocks), dim3(Cfg::NT), Cfg::LDS_BYTES, st, a);
    return hipGetLastError();
}

// The largest tile that still gives most CUs a block. A 128 x 128 block takes
// 0.40 us per 64-deep slice on top of about 8 us (launch, first loads, stores),
// whatever the number of blocks up to one per CU: 196 of them run the 14 x 14
// layer at 256 channels (36 slices) in 22 us. us of the forward by tile (pixels
// x channels):     256x128  128x128  64x128  64x64
//   128x256x14x14    51.7     55.5     58.4    60.9
//   64x256x14x14     41.4     33.1     37.4    41.6
//   64x512x7x7       58.0     40.7     38.5    37.6
//   8x256x14x14      31.6     22.7     20.4    18.2
template <int BK, PackedKind KIND = kPlain>
hipError_t launch_conv_bk(const PackedConvArgs& a, hipStream_t st) {
    int most = 0;
    for (int z = 0; z < a.nphase; ++z) most = std::max(most, a.ph[z].npix);
    if (most == 0) return hipSuccess;
    const int n64 = ceil_div(a.N, 64);
    const int64_t tiles = (int64_t)ceil_div(most, 64) * a.nphase * n64;  // of 64 x 64
    if (n64 == 1) {
        // (256 x 64, one block per CU, ran the first layer's forward, 4 slices
        // deep, in 42 us; 128 x 64, two per CU, in 32)
        if (tiles >= 500) return launch_conv<128, 64, 2, 2, BK, KIND>(a, most, st);
        return launch_conv<64, 64, 2, 2, BK, KIND>(a, most, st);
    }
    if (tiles >= 1400) return launch_conv<256, 128, 4, 2, BK, KIND>(a, most, st);
    if (tiles >= 600) return launch_conv<128, 128, 4, 2, BK, KIND>(a, most, st);
    if (tiles >= 300) return launch_conv<64, 128, 2, 2, BK, KIND>(a, most, st);
    return launch_conv<64, 64, 2, 2, BK, KIND>(a, most, st);
}

int run_conv(const PackedConvArgs& a, int CB, hipStream_t st) {
    const hipError_t e = CB == 64 ? launch_conv_bk<64>(a, st) : launch_conv_bk<32>(a, st);
    return e == hipSuccess ? SEERA_OK : fail_hip(e, "packed conv launch");
}

// The forward product over the packed input xp.
int run_fwd(const Conv& c, const Packed& g, const half_t* xp, const half_t* wp, float* out,
            const ConvEpi& epi, hipStream_t st) {
    PackedConvArgs a{};
    a.x = xp; a.w = wp; a.out = out;
    a.x_bytes = (uint32_t)(g.halves(c.B) * 2);
    a.pix = g.CB; a.ncb = g.Cp / g.CB; a.plane = (int)g.plane(c.B);
    a.Wp = g.Wp; a.HpWp = g.Hp * g.Wp;
    a.N = c.F; a.Hout = c.Ho; a.Wout = c.Wo;
    a.ish = c.sh; a.isw = c.sw; a.osh = 1; a.osw = 1;
    a.nphase = 1;
    a.ph[0] = PackedPhase{c.Ho, c.Wo, c.B * c.Ho * c.Wo, c.R, c.S, 0, 0, 0, 0,
                          FastDiv(c.Ho * c.Wo), FastDiv(c.Wo)};
    a.epi = epi;
    return run_conv(a, g.CB, st);
}
void fwd_weights(PackArgs& pk, int& block, const float* W, half_t* wp, const Conv& c, const Packed& g) {
    add_weights(pk, block, W, wp, c, true, g);
    pk.w.nphase = 1;
    pk.w.ph[0] = PackWeightPhase{c.R, c.S, 0, 0, 1, 1, 0, FastDiv(c.S), FastDiv(c.R * c.S)};
}

// The transposed product over the packed output yp: fills `a` and the weights.
void plan_dgrad(const Conv& c, const DgradGeometry& d, const half_t* yp, const half_t* wp, float* out,
                PackedConvArgs& a, PackWeights& w) {
    const Packed& g = d.g;
    a.x = yp; a.w = wp; a.out = out;
    a.x_bytes = (uint32_t)(g.halves(c.B) * 2);
    a.pix = g.CB; a.ncb = g.Cp / g.CB; a.plane = (int)g.plane(c.B);
    a.Wp = g.Wp; a.HpWp = g.Hp * g.Wp;
    a.N = c.C; a.Hout = c.H; a.Wout = c.W;
    a.ish = 1; a.isw = 1; a.osh = c.sh; a.osw = c.sw;
    int64_t off = 0;
    for (int i = 0; i < c.sh; ++i)
        for (int j = 0; j < c.sw; ++j) {
            const Axis &h = d.ah[i], &v = d.aw[j];
            if (h.n == 0 || v.n == 0) continue;
            const int T = v.T == 0 ? 0 : h.T, U = T == 0 ? 0 : v.T;  // (no taps: zeros)
            PackedPhase& p = a.ph[a.nphase];
            p.Ho = h.n; p.Wo = v.n; p.npix = c.B * h.n * v.n;
            p.T = T; p.U = U;
            p.x0 = T == 0 ? 0 : ((h.q - (h.T - 1) + g.top) * g.Wp + (v.q - (v.T - 1) + g.left)) * g.CB;
            p.oph = i; p.opw = j;
            p.woff = off;
            p.by_howo = FastDiv(h.n * v.n);
            p.by_wo = FastDiv(v.n);
            // tap (t, u) reads row oh + q - (T - 1) + t: the kernel's tap
            // r0 + s * (T - 1 - t)
            w.ph[a.nphase] = PackWeightPhase{T, U, h.r0 + c.sh * (h.T - 1), v.r0 + c.sw * (v.T - 1),
                                             -c.sh, -c.sw, (int)off, FastDiv(std::max(U, 1)),
                                             FastDiv(std::max(T * U, 1))};
            off += (int64_t)c.C * T * U * g.Cp;
            ++a.nphase;
        }
    w.nphase = a.nphase;
}

template <int BF, int BL, int WF, int WL, int NS, int KG>
hipError_t launch_wgrad_tile(const PackedWgradArgs& a, hipStream_t st) {
    constexpr int lds = std::max(NS * (BF + BL) * 64 * 2, KG > 1 ? BF * BL * 4 : 0);
    static_assert(lds <= 160 * 1024, "LDS of one CU");
    auto kern = packed_wgrad_kernel<BF, BL, WF, WL, NS, KG>;
    if (lds > 65536) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, lds);
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL(kern, dim3((unsigned)a.nblocks), dim3(64 * WF * WL * KG), lds, st, a);
    return hipGetLastError();
}

// dW over npix pixels of F x L sums. Two wave groups over K on the large tile;
// layers of at most 64 filters on the 64-filter tile, 64 columns wide while
// the wider one would leave CUs without a block. Pixels are split for about
// 256 blocks, of at least 4 slices each.
struct WgradPlan {
    PackedWgradArgs a{};
    int BF, BL;
    WgradPlan(int F, int L, int Ho, int Wo, int B) {
        a.F = F; a.L = L;
        a.Ho = Ho; a.Wo = Wo; a.npix = B * Ho * Wo;
        const int slices = ceil_div(a.npix, 64);
        BF = F > 64 ? 128 : 64;
        BL = L > 64 && (F > 64 || (int64_t)ceil_div(L, 128) * slices >= 8 * 256) ? 128 : 64;
        if (F > 64 && L <= 64) BF = 64;
        a.ntf = ceil_div(F, BF);
        a.ntl = ceil_div(L, BL);
        const int tiles = a.ntf * a.ntl;
        // The 64-filter tiles leave room for two blocks per CU: two rounds of
        // splits where each still has 16 slices (first layer, 6272 slices: 37.8 us
        // with 256 blocks, 28.8 with 512).
        const int blocks = BF == 64 && (int64_t)tiles * slices >= 512 * 16 ? 512 : 256;
        const int want = std::max(1, std::min(blocks / std::max(tiles, 1), slices / 4));
        a.sps = ceil_div(slices, want);
        a.nsplit = ceil_div(slices, a.sps);
        a.nblocks = tiles * a.nsplit;
        a.by_howo = FastDiv(Ho * Wo);
        a.by_wo = FastDiv(Wo);
        a.d_b = 64 / (Ho * Wo);
        const int rem = 64 - a.d_b * Ho * Wo;
        a.d_h = rem / Wo;
        a.d_w = rem - a.d_h * Wo;
    }
    int64_t part_floats() const { return (int64_t)a.nsplit * a.F * a.L; }
    // dY in `g` with `top`, `left` as its halo
    void output(const half_t* yp, const Packed& g, int B) {
        a.y = yp;
        a.y_bytes = (uint32_t)(g.halves(B) * 2);
        a.Fp = g.Cp; a.lfb = g.lcb(); a.yplane = (int)g.plane(B);
        a.ypix = g.CB; a.yrow = g.Wp * g.CB; a.yimg = g.Hp * a.yrow;
        a.y0 = g.top * a.yrow + g.left * a.ypix;
    }
    void input(const half_t* xp, const Packed& g, const Conv& c) {
        a.x = xp;
        a.x_bytes = (uint32_t)(g.halves(c.B) * 2);
        a.Cp = g.Cp; a.lcb = g.lcb(); a.xplane = (int)g.plane(c.B);
        a.xcol = g.CB; a.xtap = g.Wp * g.CB;
        a.xpix = c.sw * a.xcol; a.xrow = c.sh * a.xtap; a.ximg = g.Hp * a.xtap;
        a.S = c.S;
        a.by_cp = FastDiv(g.Cp);
        a.by_s = FastDiv(c.S);
    }
    int run(float* part, hipStream_t st) {
        a.part = part;
        hipError_t e;
        if (BF == 128) e = launch_wgrad_tile<128, 128, 2, 2, 3, 2>(a, st);
        else if (BL == 128) e = launch_wgrad_tile<64, 128, 2, 2, 3, 1>(a, st);
        else e = launch_wgrad_tile<64, 64, 2, 2, 3, 1>(a, st);
        return e == hipSuccess ? SEERA_OK : fail_hip(e, "packed wgrad launch");
    }
};

int run_reduce(const Conv& c, const WgradPlan& wg, int Cp, float* dW, const PackAct& y, float* db,
               hipStream_t st) {
    const bool many = wg.a.nsplit >= 16;
    const int nb_w = c.F * ceil_div(c.C, many ? 16 : 64), nb_db = db ? ceil_div(c.F, 16) : 0;
    const size_t lds = std::max<size_t>(64 * (size_t)c.R * c.S, 512) * 4;
    hipLaunchKernelGGL(many ? packed_wgrad_reduce<4> : packed_wgrad_reduce<1>, dim3((unsigned)(nb_w + nb_db)),
                       dim3(512), lds, st, wg.a.part, dW, c.F, c.C, Cp, c.R * c.S, wg.a.nsplit, nb_w, y.sums,
                       y.prow, wg.a.Fp, db);
    SEERA_HIP_TRY(hipGetLastError());
    return SEERA_OK;
}

bool sizes_ok(const Conv& c, const Packed& x, const Packed& y) {
    return packed_sizes_ok(c, x.halves(c.B), y.halves(c.B));
}

}  // namespace

int packed_conv_fwd(const float* X, const float* Wt, float* Y, int B, int C, int H, int W, int F,
                    int R, int S, int sh, int sw, int ph, int pw, const ConvEpi& epi,
                    hipStream_t st, bool* used) {
    *used = false;
    const Conv c{B, C, H, W, F, R, S, sh, sw, ph, pw, (H + 2 * ph - R) / sh + 1, (W + 2 * pw - S) / sw + 1};
    const Packed g = input_geometry(c);
    if (!sizes_ok(c, g, g)) return SEERA_OK;
    const int64_t xn = g.halves(B), wn = (int64_t)F * R * S * g.Cp;
    Scratch sc;
    sc.need<half_t>(xn);
    sc.need<half_t>(wn);
    bool got = false;
    SEERA_TRY(sc.get(st, &got));
    if (!got) return SEERA_OK;
    half_t* xp = sc.take<half_t>(xn);
    half_t* wp = sc.take<half_t>(wn);
    PackArgs pk{};
    int block = 0;
    fwd_weights(pk, block, Wt, wp, c, g);
    add_act(pk, block, X, xp, B, C, H, W, g, nullptr);
    SEERA_TRY(launch_pack(pk, block, st));
    SEERA_TRY(run_fwd(c, g, xp, wp, Y, epi, st));
    *used = true;
    return SEERA_OK;
}

int packed_conv_bwd(const float* dY, const float* Wt, const float* X, float* dX, float* dW,
                    float* db, int B, int C, int H, int W, int F, int R, int S, int sh, int sw,
                    int ph, int pw, hipStream_t st, bool* used) {
    *used = false;
    const Conv c{B, C, H, W, F, R, S, sh, sw, ph, pw, (H + 2 * ph - R) / sh + 1, (W + 2 * pw - S) / sw + 1};
    if (sh > kMaxPhase || sw > kMaxPhase) return SEERA_OK;
    const Packed gx = input_geometry(c);
    const DgradGeometry d(c);
    if (!sizes_ok(c, gx, d.g)) return SEERA_OK;
    const int64_t xn = gx.halves(B), yn = d.g.halves(B), wn = (int64_t)C * R * S * d.g.Cp;
    WgradPlan wg(F, R * S * gx.Cp, c.Ho, c.Wo, B);
    int iters, prow;
    pack_split(B, c.Ho * c.Wo, &iters, &prow);
    const int64_t sn = db ? (int64_t)prow * d.g.Cp : 0;
    Scratch sc;
    sc.need<half_t>(xn);
    sc.need<half_t>(yn);
    sc.need<half_t>(wn);
    sc.need<float>(wg.part_floats());
    sc.need<float>(sn);
    bool got = false;
    SEERA_TRY(sc.get(st, &got));
    if (!got) return SEERA_OK;
    half_t* xp = sc.take<half_t>(xn);
    half_t* yp = sc.take<half_t>(yn);
    half_t* wp = sc.take<half_t>(wn);
    float* part = sc.take<float>(wg.part_floats());
    float* sums = db ? sc.take<float>(sn) : nullptr;

    PackArgs pk{};
    PackedConvArgs a{};
    int block = 0;
    add_weights(pk, block, Wt, wp, c, false, d.g);
    plan_dgrad(c, d, yp, wp, dX, a, pk.w);
    add_act(pk, block, dY, yp, B, F, c.Ho, c.Wo, d.g, sums);
    add_act(pk, block, X, xp, B, C, H, W, gx, nullptr);
    SEERA_TRY(launch_pack(pk, block, st));
    SEERA_TRY(run_conv(a, d.g.CB, st));
    wg.output(yp, d.g, B);
    wg.input(xp, gx, c);
    SEERA_TRY(wg.run(part, st));
    SEERA_TRY(run_reduce(c, wg, gx.Cp, dW, pk.act[0], db, st));
    *used = true;
    return SEERA_OK;
}

int packed_convT_fwd(const float* X, const float* Wt, float* out, int B, int F, int Hi, int Wi, int C,
                     int H, int W, int R, int S, int sh, int sw, int ph, int pw, hipStream_t st,
                     bool* used) {
    *used = false;
    // (the adjoint of the convolution [B, C, H, W] -> [B, F, Hi, Wi])
    const Conv c{B, C, H, W, F, R, S, sh, sw, ph, pw, Hi, Wi};
    if (sh > kMaxPhase || sw > kMaxPhase) return SEERA_OK;
    const DgradGeometry d(c);
    if (!sizes_ok(c, d.g, d.g)) return SEERA_OK;
    const int64_t yn = d.g.halves(B), wn = (int64_t)C * R * S * d.g.Cp;
    Scratch sc;
    sc.need<half_t>(yn);
    sc.need<half_t>(wn);
    bool got = false;
    SEERA_TRY(sc.get(st, &got));
    if (!got) return SEERA_OK;
    half_t* yp = sc.take<half_t>(yn);
    half_t* wp = sc.take<half_t>(wn);
    PackArgs pk{};
    PackedConvArgs a{};
    int block = 0;
    add_weights(pk, block, Wt, wp, c, false, d.g);
    plan_dgrad(c, d, yp, wp, out, a, pk.w);
    add_act(pk, block, X, yp, B, F, Hi, Wi, d.g, nullptr);
    SEERA_TRY(launch_pack(pk, block, st));
    SEERA_TRY(run_conv(a, d.g.CB, st));
    *used = true;
    return SEERA_OK;
}

int packed_convT_bwd(const float* dY, const float* Wt, const float* X, float* dX, float* dW, int B,
                     int F, int Hi, int Wi, int C, int H, int W, int R, int S, int sh, int sw, int ph,
                     int pw, hipStream_t st, bool* used) {
    *used = false;
    // dX is the convolution of dY [B, C, H, W], dW that convolution's with its
    // output in the place of X [B, F, Hi, Wi].
    const Conv c{B, C, H, W, F, R, S, sh, sw, ph, pw, Hi, Wi};
    const Packed gx = input_geometry(c), gy(0, 0, Hi, Wi, F);
    if (!sizes_ok(c, gx, gy)) return SEERA_OK;
    const int64_t xn = gx.halves(B), yn = gy.halves(B), wn = (int64_t)F * R * S * gx.Cp;
    WgradPlan wg(F, R * S * gx.Cp, Hi, Wi, B);
    Scratch sc;
    sc.need<half_t>(xn);
    sc.need<half_t>(yn);
    sc.need<half_t>(wn);
    sc.need<float>(wg.part_floats());
    bool got = false;
    SEERA_TRY(sc.get(st, &got));
    if (!got) return SEERA_OK;
    half_t* xp = sc.take<half_t>(xn);
    half_t* yp = sc.take<half_t>(yn);
    half_t* wp = sc.take<half_t>(wn);
    float* part = sc.take<float>(wg.part_floats());
    PackArgs pk{};
    int block = 0;
    fwd_weights(pk, block, Wt, wp, c, gx);
    add_act(pk, block, dY, xp, B, C, H, W, gx, nullptr);
    add_act(pk, block, X, yp, B, F, Hi, Wi, gy, nullptr);
    SEERA_TRY(launch_pack(pk, block, st));
    SEERA_TRY(run_fwd(c, gx, xp, wp, dX, ConvEpi{}, st));
    wg.output(yp, gy, B);
    wg.input(xp, gx, c);
    SEERA_TRY(wg.run(part, st));
    SEERA_TRY(run_reduce(c, wg, gx.Cp, dW, pk.act[0], nullptr, st));
    *used = true;
    return SEERA_OK;
}

namespace {

// A first layer in space-to-depth form (pack_s2d): kernel 7 or 8 wide and at
// most 8 high, stride 2, at most 4 channels. As an ordinary packed layer its
// channels would be padded to 32.
bool stem_ok(const Conv& c) {
    return c.C <= 4 && c.sh == 2 && c.sw == 2 && (c.S == 7 || c.S == 8) && c.R >= 2 && c.R <= 8;
}

// X in that form: [B, Ho + T - 1, Wo + 3] pixels of 16 halves.
struct StemInput {
    int T, H2, W2;
    explicit StemInput(const Conv& c) : T((c.R + 1) / 2), H2(c.Ho + T - 1), W2(c.Wo + 3) {}
    int64_t halves(int B) const { return (int64_t)B * H2 * W2 * 16; }
};

void add_stem_act(PackArgs& pk, int& block, const float* X, half_t* out, const Conv& c, const StemInput& g) {
    PackAct& a = pk.act[pk.nact++];
    a.in = X; a.out = out;
    a.total = (int64_t)c.B * c.C * c.H * c.W;
    a.B = c.B; a.C = c.C; a.H = c.H; a.W = c.W;
    a.Hp = g.H2; a.Wp = g.W2;
    a.ph = c.ph; a.pw = c.pw;
    a.s2d = 1;
    a.by_hpwp = FastDiv(g.H2 * g.W2);
    a.by_wp = FastDiv(g.W2);
    a.block0 = block;
    block += (int)(((int64_t)c.B * g.H2 * g.W2 + 255) / 256);
}

void add_stem_weights(PackArgs& pk, int& block, const float* W, half_t* out, const Conv& c, bool by_f,
                      const Packed& gy, int64_t halves) {
    PackS2dWeights& w = pk.w2;
    w.in = W; w.out = out;
    w.F = c.F; w.C = c.C; w.R = c.R; w.S = c.S;
    w.by_f = by_f;
    w.Fp = gy.Cp; w.lfb = gy.lcb();
    w.items = (int)(halves / 8);
    w.block0 = block;
    block += ceil_div(w.items, 256);
}

}  // namespace

int packed_stem_fwd(const float* X, const float* Wt, float* Y, int B, int C, int H, int W, int F,
                    int R, int S, int sh, int sw, int ph, int pw, const ConvEpi& epi,
                    hipStream_t st, bool* used) {
    *used = false;
    const Conv c{B, C, H, W, F, R, S, sh, sw, ph, pw, (H + 2 * ph - R) / sh + 1, (W + 2 * pw - S) / sw + 1};
    if (!stem_ok(c)) return SEERA_OK;
    const StemInput g(c);
    if (!stem_sizes_ok(c, g.halves(B), 0, c.Ho * (int64_t)c.Wo)) return SEERA_OK;
    const int64_t xn = g.halves(B), wn = (int64_t)g.T * F * 64;
    Scratch sc;
    sc.need<half_t>(xn);
    sc.need<half_t>(wn);
    bool got = false;
    SEERA_TRY(sc.get(st, &got));
    if (!got) return SEERA_OK;
    half_t* xp = sc.take<half_t>(xn);
    half_t* wp = sc.take<half_t>(wn);
    PackArgs pk{};
    int block = 0;
    add_stem_weights(pk, block, Wt, wp, c, true, Packed(0, 0, 1, 1, F), wn);
    add_stem_act(pk, block, X, xp, c, g);
    SEERA_TRY(launch_pack(pk, block, st));
    PackedConvArgs a{};
    a.x = xp; a.w = wp; a.out = Y;
    a.x_bytes = (uint32_t)(xn * 2);
    a.pix = 16; a.ncb = 1; a.plane = 0;
    a.Wp = g.W2; a.HpWp = g.H2 * g.W2;
    a.N = F; a.Hout = c.Ho; a.Wout = c.Wo;
    a.ish = 1; a.isw = 1; a.osh = 1; a.osw = 1;
    a.nphase = 1;
    a.ph[0] = PackedPhase{c.Ho, c.Wo, B * c.Ho * c.Wo, g.T, 1, 0, 0, 0, 0, FastDiv(c.Ho * c.Wo), FastDiv(c.Wo)};
    a.epi = epi;
    a.R = R; a.S = S;
    const hipError_t e = launch_conv_bk<64, kS2dForward>(a, st);
    if (e != hipSuccess) return fail_hip(e, "packed conv launch");
    *used = true;
    return SEERA_OK;
}

int packed_stem_bwd(const float* dY, const float* Wt, const float* X, float* dX, float* dW, float* db,
                    int B, int C, int H, int W, int F, int R, int S, int sh, int sw, int ph, int pw,
                    hipStream_t st, bool* used) {
    *used = false;
    const Conv c{B, C, H, W, F, R, S, sh, sw, ph, pw, (H + 2 * ph - R) / sh + 1, (W + 2 * pw - S) / sw + 1};
    if (!stem_ok(c)) return SEERA_OK;
    const StemInput gx(c);
    // The 2 x 2 blocks of the padded image that hold a pixel of the image.
    const int ni = (H - 1 + ph) / 2 + 1, nj = (W - 1 + pw) / 2 + 1;
    const Packed gy(gx.T - 1, 3, gx.T - 1 + std::max(c.Ho, ni), 3 + std::max(c.Wo, nj), F, 64);
    if (!stem_sizes_ok(c, gx.halves(B), gy.halves(B), (int64_t)ni * nj)) return SEERA_OK;
    const int64_t xn = gx.halves(B), yn = gy.halves(B), wn = (int64_t)gx.T * 4 * 4 * C * gy.Cp;
    WgradPlan wg(F, gx.T * 64, c.Ho, c.Wo, B);
    int iters, prow;
    pack_split(B, c.Ho * c.Wo, &iters, &prow);
    const int64_t sn = db ? (int64_t)prow * gy.Cp : 0;
    Scratch sc;
    sc.need<half_t>(xn);
    sc.need<half_t>(yn);
    sc.need<half_t>(wn);
    sc.need<float>(wg.part_floats());
    sc.need<float>(sn);
    bool got = false;
    SEERA_TRY(sc.get(st, &got));
    if (!got) return SEERA_OK;
    half_t* xp = sc.take<half_t>(xn);
    half_t* yp = sc.take<half_t>(yn);
    half_t* wp = sc.take<half_t>(wn);
    float* part = sc.take<float>(wg.part_floats());
    float* sums = db ? sc.take<float>(sn) : nullptr;
    PackArgs pk{};
    int block = 0;
    add_stem_weights(pk, block, Wt, wp, c, false, gy, wn);
    add_act(pk, block, dY, yp, B, F, c.Ho, c.Wo, gy, sums);
    add_stem_act(pk, block, X, xp, c, gx);
    SEERA_TRY(launch_pack(pk, block, st));

    PackedConvArgs a{};
    a.x = yp; a.w = wp; a.out = dX;
    a.x_bytes = (uint32_t)(yn * 2);
    a.pix = gy.CB; a.ncb = gy.Cp / gy.CB; a.plane = (int)gy.plane(B);
    a.Wp = gy.Wp; a.HpWp = gy.Hp * gy.Wp;
    a.N = 4 * C; a.Hout = H; a.Wout = W;
    a.ish = 1; a.isw = 1; a.osh = 1; a.osw = 1;
    a.nphase = 1;
    a.ph[0] = PackedPhase{ni, nj, B * ni * nj, gx.T, 4, 0, ph, pw, 0, FastDiv(ni * nj), FastDiv(nj)};
    a.R = R; a.S = S;
    const hipError_t e = launch_conv<128, 32, 4, 1, 64, kS2dInput>(a, B * ni * nj, st);
    if (e != hipSuccess) return fail_hip(e, "packed conv launch");

    wg.output(yp, gy, B);
    wg.a.x = xp;
    wg.a.x_bytes = (uint32_t)(xn * 2);
    wg.a.Cp = 64; wg.a.lcb = 6; wg.a.xplane = 0;
    wg.a.xcol = 0; wg.a.xtap = gx.W2 * 16;
    wg.a.xpix = 16; wg.a.xrow = wg.a.xtap; wg.a.ximg = gx.H2 * wg.a.xtap;
    wg.a.S = 1;
    wg.a.by_cp = FastDiv(64);
    wg.a.by_s = FastDiv(1);
    SEERA_TRY(wg.run(part, st));
    const int nb_w = F * gx.T, nb_db = db ? ceil_div(F, 16) : 0;
    hipLaunchKernelGGL(packed_wgrad_reduce_s2d, dim3((unsigned)(nb_w + nb_db)), dim3(512), 0, st, part, dW, F, C,
                       R, S, gx.T * 64, wg.a.nsplit, nb_w, sums, pk.act[0].prow, gy.Cp, db);
    SEERA_HIP_TRY(hipGetLastError());
    *used = true;
    return SEERA_OK;
}

}  // namespace seera
