// The dispatch rules (conv_routes.h, gemm_routes.h) against the times they were
// taken from: each row of the tables holds one call and its time, us, on the
// direct kernels and on the path beside them (packed operands; for 1x1 layers with
// few filters the one-pass kernels). argv: the two tables.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <fstream>
#include <sstream>
#include <string>

#include "conv_routes.h"
#include "gemm_routes.h"

using namespace seera;

struct Score {
    double best = 0, chosen = 0;
    int rows = 0, off = 0;
    void add(const std::string& line, bool packed, double direct_us, double packed_us) {
        const double b = std::min(direct_us, packed_us), c = packed ? packed_us : direct_us;
        best += b;
        chosen += c;
        ++rows;
        if (c > 1.15 * b + 3) {
            ++off;
            std::printf("off: %s\n", line.c_str());
        }
    }
};

template <class Choice>
Score run(const char* path, Choice choice) {
    std::ifstream in(path);
    std::string line;
    Score s;
    while (std::getline(in, line)) {
        if (line.empty() || line[0] == '#') continue;
        std::istringstream f(line);
        double t[2];
        const bool packed = choice(f);
        f >> t[0] >> t[1];
        if (!f) {
            std::fprintf(stderr, "bad row: %s\n", line.c_str());
            std::exit(1);
        }
        s.add(line, packed, t[0], t[1]);
    }
    std::printf("%s: %d rows, chosen %.0f us, best %.0f us, %d off\n", path, s.rows, s.chosen, s.best, s.off);
    return s;
}

int main(int, char** argv) {
    const Score conv = run(argv[1], [](std::istringstream& f) {
        std::string kind, pass;
        int B, C, H, W, F, k, s, p;
        f >> kind >> pass >> B >> C >> H >> W >> F >> k >> s >> p;
        const bool fwd = pass == "fwd";
        if (kind == "convt") {
            const int Ho = (H - 1) * s - 2 * p + k, Wo = (W - 1) * s - 2 * p + k;
            return fwd ? packed_convT_fwd_pays(B, C, H, W, F, Ho, Wo, k, k, s, s, p, p)
                       : packed_convT_bwd_pays(B, C, H, W, F, Ho, Wo, k, k, s, s, p, p);
        }
        if (C <= 4 && s == 2 && (k == 7 || k == 8))
            return fwd || packed_stem_bwd_pays(B, C, H, W, F, (W + 2 * p - k) / s + 1);
        if (k == 1 && s == 1 && p == 0 && H * W % 4 == 0) {
            if (fwd && F <= 128 && pointwise_fwd_pays(B, C, H, W, F)) return true;
            if (!fwd && F <= 64 && C <= 512 && pointwise_bwd_pays(B, C, H, W)) return true;
        }
        return fwd ? packed_fwd_pays(B, C, H, W, F, k, k, s, s, p, p)
                   : packed_bwd_pays(B, C, H, W, F, k, k, s, s, p, p);
    });
    const Score gemm = run(argv[2], [](std::istringstream& f) {
        std::string pass;
        int M, N, K;
        f >> pass >> M >> N >> K;
        return pass == "fwd" ? packed_gemm_fwd_pays(true, true, M, N, K) : packed_gemm_bwd_pays(true, true, true, M, N, K);
    });
    // the choices cost at most 2 % over the better path of every row, and few
    // rows more than 15 % and 3 us
    if (conv.rows < 400 || gemm.rows < 100 || conv.chosen > 1.02 * conv.best || gemm.chosen > 1.02 * gemm.best ||
        conv.off * 20 > conv.rows || gemm.off * 20 > gemm.rows)
        return 1;
    std::puts("all checks passed");
}
