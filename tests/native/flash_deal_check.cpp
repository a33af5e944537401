// Balanced flash grids (csrc/flash_deal.h) over every tail and key range up to
// 160 key tiles: the pieces cover each (query tile, key tile) once, in bounds,
// each in a partial slot of its own, and the slots the combine pass reads for a
// tile are the ones written for it.
#define __host__
#define __device__
#include "flash_deal.h"

#include <cstdio>
#include <vector>

using namespace anima_hip;

int main()
{
    long plans = 0;
    for (int ntail = 1; ntail < kFlashTargetBlocks; ++ntail)
        for (int nk = 2; nk <= 160; ++nk) {
            const int all = ntail * nk;
            const int u = (all + kFlashTargetBlocks - 1) / kFlashTargetBlocks;
            if (u >= nk)
                continue;
            ++plans;
            FlashDeal deal;
            int ng = 0, nshorter = 0;
            deal_pieces(ntail, nk, u, deal, ng, nshorter);
            std::vector<int> seen(all, 0), slot(ntail + ng - 1, -1);
            for (int i = 0; i < ng + nshorter; ++i) {
                const FlashPiece p = flash_piece(i, ntail, nk, u, ng, deal);
                if (p.jn == 0 && i >= ng)
                    continue;
                const bool ok = p.jn > 0 && p.t >= 0 && p.t < ntail && p.g >= 0 && p.g < ng &&
                                p.j0 >= 0 && p.j0 + p.jn <= nk && slot[p.t + p.g] < 0;
                if (!ok) {
                    std::printf("ntail %d nk %d piece %d\n", ntail, nk, i);
                    return 1;
                }
                slot[p.t + p.g] = p.t;
                for (int j = 0; j < p.jn; ++j)
                    ++seen[p.t * nk + p.j0 + j];
            }
            for (int n : seen)
                if (n != 1) {
                    std::printf("ntail %d nk %d: a key tile %d times\n", ntail, nk, n);
                    return 1;
                }
            for (int t = 0; t < ntail; ++t) {
                const int g0 = t * nk / u, g1 = (t * nk + nk - 1) / u;
                for (int s = t + g0; s <= t + g1; ++s)
                    if (slot[s] != t) {
                        std::printf("ntail %d nk %d: slot %d\n", ntail, nk, s);
                        return 1;
                    }
            }
        }
    std::printf("%ld plans\n", plans);
    return plans > 0 ? 0 : 1;
}
