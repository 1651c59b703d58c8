// Host-side checks of gemm_lds_plan (csrc/gemm_lds.hip) over the ESM-2
// projections and over the room its caller has for partial sums: splits stay
// within that room, no tile that was meant to run in k-splits is left without
// them, and 128 x 320 tiles fill the CUs as their rule states.
#include <cstdio>

#include "../../codon-infer_amd/csrc/kernels.h"

using namespace cih;

int main() {
    const int dims[6] = {320, 480, 640, 1280, 2560, 96}, hidden[6] = {1280, 1920, 2560, 5120, 10240, 160};
    const int cus = device_cus();
    long plans = 0, split = 0, bad = 0;
    for (int m = 0; m < 6; m++)
        for (int pair = 0; pair < 2; pair++)
            for (int proj = 0; proj < 4; proj++) {  // QKV, Wo, FC1, FC2
                DevMatrix W;
                W.fmt = pair ? WF_F16P : WF_Q8;
                W.N = proj == 0 ? 3 * dims[m] : (proj == 2 ? hidden[m] : dims[m]);
                W.K = proj == 3 ? hidden[m] : dims[m];
                if (pair) {
                    W.kx = W.K;
                    W.K *= 2;
                }
                W.q = W.q16 = reinterpret_cast<unsigned short *>(16);
                const int epi = proj == 0 ? EPI_NONE : (proj == 2 ? EPI_GELU_H2 : EPI_RESIDUAL);
                for (int M = 1; M <= 4200; M += M < 700 ? 1 : 37) {
                    const size_t mn = (size_t)M * W.N;
                    const size_t rooms[9] = {0, mn, 2 * mn, 2 * mn + mn / 2, 3 * mn, 4 * mn, 6 * mn, 8 * mn,
                                             (size_t)4 << 20};
                    LdsPlan none;
                    const bool ok0 = gemm_lds_plan(W, AF_H2, M, epi, 0, none);
                    for (size_t room : rooms) {
                        LdsPlan p;
                        const bool ok = gemm_lds_plan(W, AF_H2, M, epi, room, p);
                        bool good = M > 48 || !ok;
                        if (ok) {
                            plans++;
                            split += p.splits > 1;
                            const long wg = (long)((M + 127) / 128) * ((W.N + 319) / 320) * p.splits;
                            if (p.splits > 1)
                                good = good && p.splits * mn <= room && epi == EPI_RESIDUAL &&
                                       (p.splits - 1) * p.kps < W.K / 32 && p.splits * p.kps >= W.K / 32;
                            if (p.splits > 1 && p.tile == LDS_TILE_128x320)
                                good = good && wg * 10 >= cus * 8 && p.kps >= 40;
                            // unsplit: the tile of a caller without room (64 x 64 tiles: K too short to split)
                            if (p.splits <= 1 && p.tile != LDS_TILE_64x64) good = good && ok0 && p.tile == none.tile;
                        }
                        if (!good && ++bad <= 20)
                            printf("N=%d K=%d pair=%d M=%d room=%zu: tile %d, %d splits of %d (no room: tile %d)\n",
                                   W.N, W.K, pair, M, room, p.tile, p.splits, p.kps, none.tile);
                    }
                }
            }
    printf("%ld plans, %ld split, %ld bad\n", plans, split, bad);
    printf(bad || !split ? "FAILED\n" : "OK\n");
    return bad != 0 || split == 0;
}
