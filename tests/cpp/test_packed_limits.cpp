// The size rules of the packed convolutions (packed_limits.h) against the
// offsets that their kernels form, in 64 bits.
#include <cstdio>
#include <cstdlib>
#include <random>

#include "packed_limits.h"

using namespace seera;

#define CHECK(c)                                                          \
    do {                                                                  \
        if (!(c)) {                                                       \
            std::fprintf(stderr, "line %d: %s\n", __LINE__, #c);          \
            std::exit(1);                                                 \
        }                                                                 \
    } while (0)

constexpr int64_t kBufOOB = 0x7FFFFF00ll;  // as in mfma_core.h

Conv conv(int B, int C, int H, int W, int F, int k, int s, int p) {
    return Conv{B, C, H, W, F, k, k, s, s, p, p, (H + 2 * p - k) / s + 1, (W + 2 * p - k) / s + 1};
}
int64_t up(int64_t n) { return (n + 31) / 32 * 32; }
int64_t x_halves(const Conv& c) { return (int64_t)c.B * (c.H + 2 * c.ph) * (c.W + 2 * c.pw) * up(c.C); }
int64_t y_halves(const Conv& c) { return (int64_t)c.B * (c.Ho + 2) * (c.Wo + 2) * up(c.F); }
bool ok(const Conv& c) { return packed_sizes_ok(c, x_halves(c), y_halves(c)); }

// The stores of packed_conv_kernel for one grid: N channels of a plane, tiles of
// 256 pixels over `pixels` pixels per image.
void stores(int64_t N, int64_t plane, int64_t pixels) {
    // the tile that touches most images begins at an image's last pixel
    const int64_t images = (pixels - 1 + 255) / pixels + 1;
    CHECK(images * N * plane * 4 <= kBufOOB);  // every stored offset, channel included
    // a wave's highest uniform offset: channel 27 of its 32 rows, 59 of 64
    const int64_t top = N > 64 ? 59 : 27;
    CHECK(kBufOOB + top * plane * 4 < (1ll << 32));
}

int main() {
    // layers that the library runs every day
    CHECK(ok(conv(64, 256, 14, 14, 256, 3, 1, 1)));
    CHECK(ok(conv(64, 128, 28, 28, 256, 3, 2, 1)));
    CHECK(ok(conv(1, 3, 2048, 2048, 3, 3, 1, 1)));
    const Conv stem = conv(32, 3, 224, 224, 64, 7, 2, 3);
    CHECK(stem_sizes_ok(stem, 32ll * 115 * 115 * 16, 32ll * 118 * 118 * 64, 113 * 113));
    // few output channels on planes whose 28th channel row passes 2^32 - kBufOOB
    CHECK(!ok(conv(1, 3, 4480, 4480, 3, 3, 1, 1)));
    const Conv up2 = conv(1, 3, 4480, 4480, 3, 2, 2, 0);  // as a transposed convolution 2240 -> 4480
    CHECK(!packed_sizes_ok(up2, y_halves(up2), y_halves(up2)));
    const Conv big_stem = conv(1, 1, 9000, 9000, 3, 7, 2, 3);
    CHECK(!stem_sizes_ok(big_stem, 4503ll * 4503 * 16, 0, 4500ll * 4500));
    // a stride residue of 4 pixels puts 65 images into a tile
    CHECK(!ok(conv(2, 600000, 4, 4, 1, 1, 2, 0)));

    std::mt19937_64 rng(5);
    auto log_int = [&](double most) { return (int)std::exp(std::uniform_real_distribution<>(0, std::log(most))(rng)); };
    int taken = 0;
    for (int i = 0; i < 2000000; ++i) {
        const int k = 1 + rng() % 5, s = 1 + rng() % 3, p = rng() % k;
        const Conv c = conv(log_int(300), log_int(1 << 20), k + log_int(20000), k + log_int(20000), log_int(1 << 20), k, s, p);
        if (!ok(c)) continue;
        ++taken;
        stores(c.F, (int64_t)c.Ho * c.Wo, (int64_t)c.Ho * c.Wo);
        for (int a = 0; a < s; ++a)
            for (int b = 0; b < s; ++b) {
                const int64_t h = (c.H - a + s - 1) / s, w = (c.W - b + s - 1) / s;  // the residue's grid
                if (h > 0 && w > 0) stores(c.C, (int64_t)c.H * c.W, h * w);
            }
    }
    CHECK(taken > 10000);
    std::puts("all checks passed");
}
