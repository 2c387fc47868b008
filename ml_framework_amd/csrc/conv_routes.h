// conv_routes.h -- which kernels a convolution runs on: operands packed to fp16
// (conv_packed.hip), one pass over fp32 memory for 1x1 layers
// (conv_pointwise.hip), or the kernels that read fp32 NCHW rows directly
// (conv_split.hip, conv_stream.hip, conv_band.hip and the stride-2 ones; below
// "direct"). Host code without HIP, so that the rules are checked on the CPU
// against the times they were taken from (tests/golden/conv_routes.csv: about 600
// layers timed both ways, finite operands: with infinite ones the chip clocks higher).
//
// Packing costs one pass over the operands (4 bytes read, 2 written, at least 64
// per pixel: channels are rounded up to 32) and pays where the direct kernels read
// every value several times over (many filters), have few blocks (many channels
// on small images), widen rows that are not float4s first, or miss their fast
// shapes. Times below are direct -> packed, us, N x C x H x W -> F:
//   3x3 s1  64x256x14x14 -> 256  fwd 63 -> 31, bwd 148 -> 63
//           64x512x7x7 -> 512    fwd 67 -> 37, bwd 224 -> 77
//           64x128x32x32 -> 128  fwd 63 -> 35, bwd 106 -> 78
//           64x64x56x56 -> 128   fwd 51 -> 80, bwd 131 -> 175 (direct)
//   3x3 s2  64x128x28x28 -> 256  fwd 43 -> 25, bwd 114 -> 57
//   1x1     64x256x16x16 -> 256  fwd 35 -> 17, bwd 96 -> 38
//   5x5 s1  32x64x28x28 -> 64    fwd 158 -> 21, bwd 566 -> 51
#pragma once

#include <algorithm>
#include <cstdint>

namespace seera {

// Whether a stride-2 convolution takes the space-to-depth form: a kernel with
// more taps than the direct band kernels hold (16) whose halves fit them.
inline bool s2d_applies(int R, int S, int sh, int sw) {
    return sh == 2 && sw == 2 && R * S > 16 && ((R + 1) / 2) * ((S + 1) / 2) <= 16;
}

// First layers whose space-to-depth form has paths of its own (packed up to 4
// channels, direct up to 8).
inline bool s2d_layer(int C, int R, int S, int sh, int sw) { return s2d_applies(R, S, sh, sw) && C <= 8; }

inline bool is_kernel(int R, int S, int sh, int sw, int ph, int pw, int k, int s, int p) {
    return R == k && S == k && sh == s && sw == s && ph == p && pw == p;
}

// The part of the matrix cores' 64 columns that rows of W pixels fill in column
// tiles of at most 56 (conv_split.hip).
inline double row_fill(int W) { return W / (64.0 * ((W + 55) / 56)); }

// 3x3 stride-1 pad-1 products of 128, 192 or 256 channels to few filters: the
// three-role kernel (conv_split.hip) reads X once per 64 filters and runs once
// per 64 channels, each launch after the first adding to the output. Packing
// reads and writes X again for one column of filter tiles, so it loses from the
// size on where the launches no longer weigh (rows that fill the column tiles
// fully), and in any case where X and its packed copy outgrow the 256 MB cache:
//   32x128x56x56 -> 32 32 -> 40, 64x 47 -> 69, 64x128x112x112 -> 32 184 -> 287
//   12x128x56x56 -> 48 22.4 -> 23.4, 123x128x48x48 -> 8 (fill 0.75, 145 MB) 61 -> 86,
//   64x128x64x64 -> 32 (0.5, 134 MB) 96 -> 80, 32x128x128x128 -> 32 (0.67, 268 MB) 154 -> 174
//   192 channels: 50x56x56 -> 32 65 -> 73; 256: 32x56x56 -> 32 62 -> 66, 64x 94 -> 135
// With 65 to 128 filters (two launches per slice) only where the images' column
// tiles give every CU the same rows and the tensors still stay in the cache:
// 64x128x56x56 -> 128 86 -> 104, 16x112x112 99 -> 104, but 66x56x56 123 -> 106, 32x112x112 223 -> 212.
inline bool channel_slices_pay(int B, int C, int H, int W, int F) {
    const int n = C / 64;
    if (C % 64 != 0 || n < 2 || n > 4) return false;
    const double mb = 4e-6 * B * C * H * W;
    if ((int64_t)C * F <= 128 * 64) {
        if (W % 56 == 0) return mb >= 48 + 72 * (n - 2);
        return mb >= (row_fill(W) >= 0.7 ? 130 + 60 * (n - 2) : 260 + 10 * (n - 2));
    }
    const int64_t tiles = (int64_t)B * (W / 56);
    return C == 128 && F <= 128 && W % 56 == 0 && tiles >= 16 && tiles <= 64 && 256 % tiles == 0 && mb >= 75 &&
           mb <= 130;
}

// A strided product with few filters over an input that, or whose packed copy,
// fills the cache: the direct band kernel reads it once. (3x3 rows of more than
// 112 outputs take several column tiles there, and packing wins.)
//   3x3 s2  64x64x112x112 -> 64 85 -> 99, 64x64x128x128 -> 64 116 -> 148; 5x64x448x448 -> 48 164 -> 136
//   1x1 s2  64x256x56x56 -> 64 61 -> 71, 64x64x112x112 -> 64 60 -> 89; 6x128x448x448 -> 96 187 -> 273
//   2x2 s2  24x320x160x160 -> 64 191 -> 371, 23x64x160x160 -> 64 51 -> 67; 12x512x96x96 -> 16 105 -> 81
//   4x4 s2  23x4x448x448 -> 8 145 -> 285; 28x160x160x224 -> 4 355 -> 383, 126x512x56x56 -> 32 539 -> 453
inline bool strided_past_cache(int B, int C, int H, int W, int F, int R, int S, int sw) {
    const double mb = 1e-6 * B * H * W * std::max(4.0 * C, 64.0 * ((C + 31) / 32));
    if (R * S == 1) return mb > 150 && W >= 48 && F <= (W >= 256 ? 96 : 64);
    if (F > 64) return false;
    if (R <= 2 && S <= 2) return mb > 150 && C <= 320;
    if (R <= 3 && S <= 3) return mb > 190 && W <= 112 * sw;
    return mb > 190 && C <= 16;
}

// The backward of a first layer of one or two channels in space-to-depth form on
// packed operands, where the direct form (fp32 space-to-depth copies) applies:
// not over so many pixels that its 16-channel copies and dY's 64-channel one pass
// the cache several times (32x1x448x448 -> 16 292 -> 360, 16x2x512x512 -> 32 231 -> 249;
// 32x3x224x224 -> 64 334 -> 107).
inline bool packed_stem_bwd_pays(int B, int C, int H, int W, int F, int Wo) {
    return !(C <= 2 && F <= 32 && Wo % 4 == 0 && (int64_t)B * H * W >= 4000000);
}

// The forward on packed operands, with or without bias and activation (the fused
// calls give the unfused ones' bits, so both take one route).
inline bool packed_fwd_pays(int B, int C, int H, int W, int F, int R, int S, int sh, int sw, int ph, int pw) {
    if (s2d_layer(C, R, S, sh, sw)) return false;
    const int64_t pixels = (int64_t)B * H * W;
    // One channel under a large kernel: its columns are a short contraction for
    // the gather GEMM and 32 padded channels here (32x1x32x32 -> 8, 5x5 11.5 ->
    // 23, 9x48x48 -> 64 15 -> 23; 85x56x56 -> 128 100 -> 82).
    if (R * S > 16 && sh == 1 && sw == 1 && (int64_t)C * R * S <= 49 && pixels * F <= 6500000) return false;
    if (W % 4 != 0 || R * S > 16) return true;
    if (is_kernel(R, S, sh, sw, ph, pw, 4, 2, 1)) {
        // conv_stride2.hip on 32 and 64 channels (32x64x16x16 -> 64 11 -> 16 us; other
        // counts 16x128x64x64 -> 128 58 -> 32), and up to 96 channels on small images the
        // band kernel in one launch (32x16x32x32 -> 16 8.7 -> 13, 5x96x56x56 -> 64 17 ->
        // 21; 32x16x64x64 18 -> 16, 58x8x28x28 -> 128 17 -> 15).
        if (C == 32 || C == 64) return false;
        return !(C <= 96 && W <= 56 && pixels <= 40000 && pixels * F <= 2500000) &&
               !strided_past_cache(B, C, H, W, F, R, S, sw);
    }
    if (sh > 1 || sw > 1) {
        if (strided_past_cache(B, C, H, W, F, R, S, sw)) return false;
        // Few channels and filters on mid-sized images (8x3x224x224 -> 16 21 -> 28,
        // 32x128x128 21.5 -> 30; 8x64x64 11.5 -> 9.1, 32x224x224 64 -> 66; 8x3x224x224 -> 32
        // 25 -> 29 but with bias and ReLU 35 -> 32; 2x2 32x16x112x112 -> 16 17 -> 23).
        if (C > 16 || F > 32) return true;
        if (R == 3 && S == 3 && F <= 16 && W <= 240) return !(pixels >= 125000 && pixels <= 530000);
        if (R == 2 && S == 2 && W <= 256) return !(pixels >= 300000 && pixels <= 620000);
        return true;
    }
    // Channels that are not a multiple of 8 (first layers): 39x3x28x28 -> 32
    // 26 -> 13, 8x3x224x224 -> 64 65 -> 42.
    if (C % 8 != 0) return true;
    if (R * S == 1) return F >= 128 && (int64_t)C * F >= 128 * 128;
    if (C <= 64) return false;
    if (is_kernel(R, S, sh, sw, ph, pw, 3, 1, 1)) {
        // Three 32-channel chunks on short rows: one launch (8x96x8x8 -> 96 9.8 -> 13.0,
        // 125x16x16 -> 64 13.7 -> 19.2; 28x28 27 -> 13).
        if (C <= 96 && W <= 16 && F <= 128 && pixels <= 33000) return false;
        // Few filters over an input past the cache, whatever the direct kernel
        // (64x320x64x64 -> 64 208 -> 236, 113x160x64x64 -> 64 201 -> 226, 64x320x56x56 -> 64
        // 152 -> 172, 69x512x56x56 -> 32 227 -> 294; 32x320x64x64 128 -> 101).
        if (F <= 64 && C % 32 == 0 && W <= 112 && 4e-6 * pixels * C >= (W % 56 == 0 ? 250 : 290)) return false;
        return !channel_slices_pay(B, C, H, W, F);
    }
    return true;
}

// The backward (dX and dW, with or without db: the same bits) on packed operands.
inline bool packed_bwd_pays(int B, int C, int H, int W, int F, int R, int S, int sh, int sw, int ph, int pw) {
    if (s2d_layer(C, R, S, sh, sw)) return false;
    const int Wo = (W + 2 * pw - S) / sw + 1;
    const int64_t pixels = (int64_t)B * H * W;
    if (W % 4 != 0 || Wo % 4 != 0 || R * S > 16) return true;
    const bool k3 = is_kernel(R, S, sh, sw, ph, pw, 3, 1, 1);
    // 4x4 at stride 2 has direct kernels (conv_phase2.hip and conv_wgrad_s2.hip).
    const bool k4 = is_kernel(R, S, sh, sw, ph, pw, 4, 2, 1) && F % 32 == 0 && F <= 128 && W % 8 == 0;
    // Few pixels: the direct kernels leave most CUs without a block, whatever
    // the channels (16x32x32x32 -> 32 36 -> 24). Not where the pixels' channels
    // already make packing X the longer part beside at most 64 filters (8x256x56x56 -> 32
    // 41 -> 48, 8x320x56x56 -> 64 49 -> 66; 8x128x28x28 -> 64 35 -> 24, rows of 24 and less
    // 81 -> 51, many images of many channels 32x320x32x32 -> 64 80 -> 73), sooner on the
    // one-pass 64 -> 64 kernel (3x112x112 29 -> 37, 8x64x64 31 -> 34, with db 37 -> 34; 8x56x56
    // 28 -> 31 but with db 32 -> 30).
    if (pixels < 40000) {
        // 4x4 on rows that fill the direct kernels' tiles (12x32x56x56 -> 128 28 -> 36,
        // 4x128x64x64 -> 128 31 -> 37, 4x512x64x64 -> 32 38 -> 46; 4x64x64x64 -> 64 27 -> 23,
        // 3x32x64x64 -> 128 26 -> 26 and db adds 4 to the first, 1x256x160x160 -> 128 60 -> 48).
        if (k4 && pixels >= 16000 && (F >= 96 || C >= 256) && W >= 48 && (W <= 128 || W % 112 == 0)) return false;
        if (!k3 || F < 8 || F > 64 || W < 28 || (C > 256 && B > 16)) return true;
        if (C == 64 && F == 64 && W >= 32) return pixels < 32000;
        return pixels * C < 3500000;
    }
    // Channels not a multiple of 8: 111x3x28x28 -> 8 (87 k) 52 -> 44, 110x3x64x64 -> 8 80 -> 110.
    if (C % 8 != 0 && pixels < 100000) return true;
    // (16x128x64x64 -> 128 50 -> 57)
    if (k4) return false;
    if (sh > 1 || sw > 1) return true;
    // (1x1: 64x64x112x112 -> 128 328 -> 364, 56x56 83 -> 83)
    if (R * S == 1) return F >= 128 && !(C <= 64 && F <= 128 && pixels > 250000);
    if (C < 128 || F < 128) return false;
    // 128 -> 128: the direct passes where 4 or 8 strips of every column tile fill the
    // CUs (64x56x56 189 -> 223, 62x56x56 185 -> 204, 32x112x112 390 -> 437, 8x224x224
    // 400 -> 435; 66x56x56 292 -> 228, 13x112x112 223 -> 176).
    const int64_t tiles = (int64_t)B * (W / 56), strips = tiles <= 32 ? 8 : 4;
    return !(k3 && C == 128 && F == 128 && W % 56 == 0 && pixels >= 100000 && tiles <= 64 && tiles * strips >= 224);
}

// 1x1 stride-1 layers in one pass over fp32 memory (conv_pointwise.hip), which
// takes up to 128 filters (backward 64): the blocks stream tiles of 128 pixels,
// and a long contraction on few tiles leaves CUs without one. Measured, us, with
// the rules above -> in one pass:
//   fwd  64x256x56x56 -> 64 (1600 tiles)  79 -> 62    64x128x56x56 -> 96  91 -> 54
//        64x64x56x56 -> 64   34 -> 27     32x256x28x28 -> 64 (224)  28 -> 18
//        32x128x28x28 -> 64 (224)  11.1 -> 11.7 (not)   32x256x14x14 -> 64 (64)  12 -> 16 (not)
//        32x64x56x56 -> 96 (800)  25 -> 26 (not)        64x192x28x28 -> 80 (448)  30 -> 27
//        64x64x56x56 -> 128 (1600)  34 -> 37, with bias and ReLU 62 -> 49
//        64x32x64x64 -> 96 (2048)  35 -> 38, with bias and ReLU 58 -> 51; 64x112x112 (6272)  147 -> 104
//        30x8x112x112 -> 4 (2940)  16 -> 20 (not)       31x1x128x128 -> 8 (3968)  49 -> 26
//   bwd  64x256x56x56 -> 64  168 -> 126   64x64x28x28 -> 32 (448)  36 -> 20
//        16x64x28x28 -> 64 (112)  18 -> 13              64x128x28x28 -> 64 (448)  39 -> 30
//        32x256x28x28 -> 64 (224)  32 -> 39 (not)       256x256x14x14 -> 64 (512)  59 -> 64 (not)
inline int64_t pixel_tiles(int B, int H, int W) { return (int64_t)B * (((int64_t)H * W + 127) / 128); }

inline bool pointwise_fwd_pays(int B, int C, int H, int W, int F) {
    if (F >= 128 && (int64_t)C * F >= 128 * 128) return false;  // packed
    const int64_t tiles = pixel_tiles(B, H, W);
    if (F > 64) return tiles >= 1200 || (C > 128 && tiles >= 400);
    // (64 channel rows are loaded for 8 or 16)
    if (C % 8 == 0 && C <= 16 && F <= 8 && tiles >= 2000) return false;
    return C <= 64 || tiles >= 800 || (C > 128 && tiles >= 200);
}

inline bool pointwise_bwd_pays(int B, int C, int H, int W) { return C <= 128 || pixel_tiles(B, H, W) >= 800; }

// ConvTranspose2D from F channels of Hi x Wi to C channels. 4x4 at stride 2
// keeps its direct kernels (conv_phase2.hip, conv_stride2.hip) on the channel
// counts they take: 64x128x28x28 -> 64 fwd 33 -> 55, bwd 76 -> 79; others
// 64x256x14x14 -> 128 fwd 55 -> 40, bwd 161 -> 67; 2x2 16x128x16x16 -> 64 fwd 24 -> 12.
// 3x3 at stride 1 is the forward's product with the kernel turned around.
inline bool packed_convT_fwd_pays(int B, int F, int Hi, int Wi, int C, int H, int W, int R, int S, int sh, int sw,
                                  int ph, int pw) {
    if (Wi % 4 != 0) return true;
    if (sh == 1 && sw == 1)
        return F > 64 && (!is_kernel(R, S, sh, sw, ph, pw, 3, 1, 1) ||
                          packed_fwd_pays(B, F, Hi, Wi, C, 3, 3, 1, 1, 1, 1));
    if (R != 4 || S != 4 || sh != 2 || sw != 2) return true;
    // (9x24x4x4 -> 16 8.0 -> 10.5, 38x8x8x8 -> 256 13.5 -> 14.8)
    if (F <= 24 && Hi <= 16 && Wi <= 8 && (int64_t)B * Hi * Wi < 3000) return false;
    return !(F % 32 == 0 && F <= 128 && H % 2 == 0 && W % 8 == 0);
}

inline bool packed_convT_bwd_pays(int B, int F, int Hi, int Wi, int C, int H, int W, int R, int S, int sh, int sw,
                                  int ph, int pw) {
    if (Wi % 4 != 0 || W % 4 != 0) return true;
    const int64_t pixels = (int64_t)B * Hi * Wi;
    if (is_kernel(R, S, sh, sw, ph, pw, 4, 2, 1)) {
        if ((C == 32 || C == 64) && F <= 192) return false;
        // Few images and output channels (4x64x16x16 -> 3 17 -> 22, 1x256x20x20 -> 32 18 ->
        // 25; 28x8x16x16 -> 3 24 -> 21, 2x64x32x32 -> 16 30 -> 21),
        // and few over very many pixels (32x64x112x112 -> 3 167 -> 184).
        return !(C <= 32 && B <= 16 && Hi <= 32 && Wi <= 28 && pixels <= 6500) && !(C <= 4 && pixels >= 380000);
    }
    // Few output channels over many pixels: packing X and dY costs more than the
    // direct passes (3x3: 32x64x56x56 -> 64 45 -> 61, 32x128x112x112 -> 64 200 -> 294,
    // 4x128x64x64 -> 64 33 -> 34; 32x128x64x64 -> 128 144 -> 139. 2x2: 32x64x112x112 -> 3
    // 107 -> 152, 32x64x56x56 -> 64 79 -> 66).
    if (is_kernel(R, S, sh, sw, ph, pw, 3, 1, 1)) {
        if (C == 64 && F == 64) return pixels < 32000;
        return !(C >= 8 && C <= 64 && F <= 192 && pixels >= 90000);
    }
    if (is_kernel(R, S, sh, sw, ph, pw, 2, 2, 0)) return !(C <= 48 && pixels >= 380000);
    return true;
}

}  // namespace seera
