// packed_limits.h -- sizes that the 32-bit offsets of conv_packed.hip hold.
// Host code without HIP, so that the rules are checked on the CPU at sizes that
// no test would run.
#pragma once

#include <algorithm>
#include <cstdint>

namespace seera {

// Offsets from a buffer resource's base stay below this; lanes without work
// carry kBufOOB = 0x7FFFFF00, at which the hardware drops the access.
constexpr int64_t kPackedMost = 0x7F000000ll;
// Pixels of the largest tile of the convolution products.
constexpr int64_t kPackedTilePixels = 256;

// Images of `pixels` pixels each that one tile can touch.
inline int64_t packed_tile_images(int64_t pixels) { return kPackedTilePixels / pixels + 2; }

// Highest channel that a wave adds as its uniform offset, plus one: its rows of
// a tile are 32 channels up to 64 output channels and 64 beyond. Lanes past the
// last channel carry kBufOOB and still add it.
inline int64_t packed_channel_rows(int64_t N) { return N > 64 ? 64 : 32; }

// Whether the offsets of a product's stores hold: N output channels of `plane`
// pixels, tiles over a grid of `pixels` pixels per image (fewer than the plane
// where a launch writes one stride residue of it). A dropped lane's offset must
// not pass 2^32, where it would count from 0 again.
inline bool packed_stores_hold(int64_t N, int64_t plane, int64_t pixels) {
    return plane * 4 * packed_channel_rows(N) < kPackedMost &&
           packed_tile_images(pixels) * N * plane * 4 < kPackedMost;
}

// A convolution [B, C, H, W] -> [B, F, Ho, Wo].
struct Conv {
    int B, C, H, W, F, R, S, sh, sw, ph, pw, Ho, Wo;
};

// Pixels per image of the smallest stride residue of the input's grid.
inline int64_t residue_pixels(const Conv& c) {
    return (int64_t)std::max(1, c.H / c.sh) * std::max(1, c.W / c.sw);
}

// Strides whose residues one launch holds.
constexpr int kMaxPhase = 9;

// The packed tensors (x_halves, y_halves), the images of the fp32 ones as read
// and as stored from the tiles, the weights, and the taps that the weights' LDS
// tile holds.
inline bool packed_sizes_ok(const Conv& c, int64_t x_halves, int64_t y_halves) {
    if ((int64_t)c.R * c.S > 64 || c.sh > kMaxPhase || c.sw > kMaxPhase || c.sh * c.sw > kMaxPhase) return false;
    const int64_t hw = (int64_t)c.H * c.W, out = (int64_t)c.Ho * c.Wo;
    const double wn = ((double)c.F + 31) * ((double)c.C + 31) * c.R * c.S;  // (channels rounded up to 32)
    return x_halves * 2 < kPackedMost && y_halves * 2 < kPackedMost && wn * 4 < (double)kPackedMost &&
           c.B * hw < kPackedMost && packed_stores_hold(c.C, hw, residue_pixels(c)) &&
           packed_stores_hold(c.F, out, out);
}

// The same for a first layer in space-to-depth form (at most 4 channels): Y is
// stored from its own grid; dX from a grid of `blocks` 2 x 2 blocks per image,
// each lane by its whole offset.
inline bool stem_sizes_ok(const Conv& c, int64_t x_halves, int64_t y_halves, int64_t blocks) {
    const int64_t hw = (int64_t)c.H * c.W, out = (int64_t)c.Ho * c.Wo;
    return x_halves * 2 < kPackedMost && y_halves * 2 < kPackedMost && (int64_t)c.F * 8192 < kPackedMost &&
           c.B * hw < kPackedMost && packed_tile_images(blocks) * c.C * hw * 4 < kPackedMost &&
           packed_stores_hold(c.F, out, out);
}

}  // namespace seera
