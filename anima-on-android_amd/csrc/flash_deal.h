// Balanced flash grids: how the key tiles of the query tiles that do not come
// out even over the CUs are cut into even shares, and the order in which the
// shares' pieces are launched (FlashPlan in common.h says when).
//
// The list of key tiles, tail tile after tail tile (`ntail` of them, `nk` key
// tiles each), is cut into shares of `u` < nk, so the boundary of a query tile
// cuts a share into at most two pieces.  A piece is a workgroup: first the
// longer piece of every share, then the shorter pieces.
#pragma once

#include <algorithm>
#include <iterator>

namespace anima_hip {

constexpr int kFlashTargetBlocks = 256;  // one flash workgroup per CU of an MI355X
constexpr unsigned kXcds = 8;
constexpr int kNoPart = 255;

// The shares in launch order of their longer pieces; then, for the workgroups
// after those, the tail tile whose beginning cuts the share (kNoPart: nothing
// to do).  Kernel argument of the balanced grids alone (544 bytes more cost the
// smallest launches 0.5 us).
struct FlashDeal {
    unsigned char share[kFlashTargetBlocks];
    unsigned char shorter[kFlashTargetBlocks + 32];
};

// Key tiles [j0, j0 + jn) of tail tile t, in share g; jn == 0: nothing to do.
struct FlashPiece {
    int t, g, j0, jn;
};

// The piece of workgroup i of `ng` shares' pieces.
__host__ __device__ inline FlashPiece flash_piece(int i, int ntail, int nk, int u, int ng,
                                                  const FlashDeal &deal)
{
    int g, cut;  // cut: the tile that begins inside share g
    if (i < ng) {
        g = deal.share[i];
        cut = g * u / nk + 1;
    } else {
        cut = deal.shorter[i - ng];
        if (cut == kNoPart)
            return FlashPiece{0, 0, 0, 0};
        g = cut * nk / u;
    }
    const int lo = g * u, all = ntail * nk, hi = lo + u < all ? lo + u : all;
    const int at = cut * nk < hi ? cut * nk : hi;  // hi: the share is in one piece
    const bool second = (hi - at > at - lo) == (i < ng);
    if (second)
        return FlashPiece{cut, g, 0, hi - at};
    return FlashPiece{cut - 1, g, lo - (cut - 1) * nk, at - lo};
}

// Fills `deal` and counts the shares and the workgroups after them.  Workgroup
// i goes to XCD i % 8 and there to shader engine (i / 8) % 4, in order: one
// that finds no free CU holds up those behind it.  An XCD takes a contiguous
// range of shares (whose K/V its L2 then serves).  Its cut shares are dealt to
// the engines in order of their longer piece, and each engine gets the shorter
// pieces of its own shares in the same order, so the CU that frees first takes
// the piece that makes it end with the others.  (2304 queries and keys, 16
// heads, f32, 21 key tiles a share: shorter pieces placed by XCD alone ran as
// long as 29, 465 us; these 345 us.)
inline void deal_pieces(int ntail, int nk, int u, FlashDeal &deal, int &ng, int &nshorter)
{
    constexpr int X = kXcds, kEngines = 4, kMost = kFlashTargetBlocks / X;
    const int all = ntail * nk;
    ng = (all + u - 1) / u;
    nshorter = 0;
    std::fill(std::begin(deal.shorter), std::end(deal.shorter),
              static_cast<unsigned char>(kNoPart));
    for (int x = 0, g0 = 0; x < X; ++x) {
        const int len = ng / X + (x < ng % X ? 1 : 0);
        struct Cut {
            int longer, g, tile;
        } cuts[kMost];
        int whole[kMost], ncut = 0, nwhole = 0, at = 0;
        for (int g = g0; g < g0 + len; ++g) {
            const int lo = g * u, hi = std::min(lo + u, all);
            const int tile = lo / nk + 1, b = tile * nk;
            if (b < hi)
                cuts[ncut++] = Cut{std::max(b - lo, hi - b), g, tile};
            else
                whole[nwhole++] = g;
        }
        g0 += len;
        std::stable_sort(cuts, cuts + ncut,
                         [](const Cut &a, const Cut &b) { return a.longer < b.longer; });
        for (int c = 0; c < ncut; ++c)
            deal.share[X * at++ + x] = static_cast<unsigned char>(cuts[c].g);
        for (int w = 0; w < nwhole; ++w)
            deal.share[X * at++ + x] = static_cast<unsigned char>(whole[w]);
        int next[kEngines] = {0, 1, 2, 3};
        for (int left = ncut; left > 0; ++at) {
            int &c = next[at % kEngines];
            if (c >= ncut)
                continue;
            const int i = X * at + x - ng;
            deal.shorter[i] = static_cast<unsigned char>(cuts[c].tile);
            nshorter = std::max(nshorter, i + 1);
            c += kEngines;
            --left;
        }
    }
}

}  // namespace anima_hip
