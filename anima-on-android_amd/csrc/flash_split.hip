// The kernel that merges the partial outputs of the D == 128 flash kernels where
// a query tile's keys are shared out over several workgroups (flash_plan.h).
//
// Merging follows from the online-softmax identity the flash kernels already
// use between key tiles (anima_rt/include/cpu/flash_attention.h:145-178 rescales
// the running sum and output when a later key block raises the max): with
// split s holding O_s = sum_j p_j v_j / l_s, p_j = 2^(x_j - m_s), l_s = sum_j p_j,
//   O = sum_s l_s 2^(m_s - M) O_s / sum_s l_s 2^(m_s - M),  M = max_s m_s.
#include "common.h"
#include "flash_tile.h"

#include <algorithm>
#include <cmath>
#include <type_traits>

namespace anima_hip {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kD = kFlashD, kBM8 = kFlashRows8;

struct CombineArgs {
    float *o;
    int64_t ob, oh, os;
    int H, S_q;
    FlashSplitArgs sa;
    TermOut ot;     // set: O as bf16 terms instead of f32 at o
    int64_t total;  // rows * 32 float4 columns
};

// A balanced grid's tail tiles, and the query tiles of a (batch, head).
struct CombineTail {
    FlashTail t;
    int n_qtiles;
};

// One thread per (row, float4 of the head dim).  Tail = CombineTail: the rows are
// those of a balanced grid's tail tiles, whose parts differ in number.  Bound by
// the latency of its loads: a balanced grid's 2304 tokens, B = 2, H = 16 (256 parts
// of 128 KiB at most) 11 us, waves waiting 60 % of them.
template <typename Tail>
__global__ __launch_bounds__(256) void flash_combine_kernel(CombineArgs a, Tail tail)
{
    const int64_t idx = int64_t(blockIdx.x) * 256 + threadIdx.x;
    if (idx >= a.total)
        return;
    int64_t row = idx >> 5;  // bh * S_q + q
    const int c4 = int(idx & 31);
    // Part s of this row is at partial row row0 + s * plane.
    int64_t bh, row0, plane;
    int q, n;
    if constexpr (std::is_same<Tail, CombineTail>::value) {
        const int t = int(row / kBM8), r = int(row - int64_t(t) * kBM8);
        const int tile = tail.t.full + t;
        bh = tile / tail.n_qtiles;
        q = int(tile - bh * tail.n_qtiles) * kBM8 + r;
        const int64_t k0 = int64_t(t) * tail.t.nk;
        const int g0 = int(k0 / tail.t.u), g1 = int((k0 + tail.t.nk - 1) / tail.t.u);
        n = g1 - g0 + 1;
        if (q >= a.S_q)
            return;
        row0 = int64_t(t + g0) * kBM8 + r;
        plane = kBM8;
    } else {
        bh = row / a.S_q;
        q = int(row - bh * a.S_q);
        n = a.sa.n;
        row0 = row;
        plane = a.sa.BH * a.S_q;
    }
    // Groups of kU splits: all loads of a group are issued before any use,
    // so the merge costs a few memory latencies rather than one per split.
    constexpr int kU = 8;
    float mx = -INFINITY;
    for (int s0 = 0; s0 < n; s0 += kU) {
        float2 v[kU];
#pragma unroll
        for (int u = 0; u < kU; ++u)
            v[u] = s0 + u < n ? a.sa.ml[(s0 + u) * plane + row0] : make_float2(0.f, 0.f);
        // A part with l == 0 saw no key (causal) or only masked ones; a NaN l (a
        // NaN score, also where the part's live scores are all NaN and its max is
        // still -inf) joins and makes the row NaN, as in the reference.
#pragma unroll
        for (int u = 0; u < kU; ++u)
            if (v[u].y != 0.0f)
                mx = fmaxf(mx, v[u].x);
    }
    float lsum = 0.0f;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    for (int s0 = 0; s0 < n; s0 += kU) {
        float2 v[kU];
        f32x4 x[kU];
#pragma unroll
        for (int u = 0; u < kU; ++u) {
            const bool in = s0 + u < n;
            const int64_t prow = (s0 + u) * plane + row0;
            v[u] = in ? a.sa.ml[prow] : make_float2(0.f, 0.f);
            x[u] = in ? *reinterpret_cast<const f32x4 *>(a.sa.part + prow * kD + 4 * c4)
                      : f32x4{0.f, 0.f, 0.f, 0.f};
        }
#pragma unroll
        for (int u = 0; u < kU; ++u) {
            if (v[u].y != 0.0f) {
                const float w = v[u].y * exp2f(v[u].x - mx);
                lsum += w;
                acc += w * x[u];
            }
        }
    }
    const float inv = lsum > 0.0f ? 1.0f / lsum : 0.0f;
    if (mx == -INFINITY)  // no part has a score above -inf: zeros (store_o_rows)
        acc = f32x4{0.f, 0.f, 0.f, 0.f};
    const int b = int(bh / a.H), h = int(bh - int64_t(b) * a.H);
    flash_tile::store_out4(acc * inv, a.o + b * a.ob + h * a.oh + q * a.os,
                           a.ot.t ? a.ot.t + b * a.ot.tb + h * a.ot.th + q * a.ot.ts : nullptr,
                           a.ot.lo, 4 * c4);
}

}  // namespace

bool term_out_ok(const TermOut &t)
{
    return (reinterpret_cast<uintptr_t>(t.t) & 15u) == 0 && t.tb % 8 == 0 && t.th % 8 == 0 &&
           t.ts % 8 == 0 && t.lo % 8 == 0 && t.lo >= 0;
}

FlashSplitArgs flash_split_args(const FlashPlan &pl, int64_t BH, int S_q, const FlashScratch &s,
                                FlashShares &sh)
{
    FlashSplitArgs sa;
    sa.BH = BH;
    size_t rows = 0;
    if (pl.u > 0) {
        FlashTail &t = sh.tail;
        t.full = pl.full;
        t.ntail = pl.ntail;
        t.nk = pl.nk;
        t.u = pl.u;
        deal_pieces(pl.ntail, pl.nk, pl.u, sh.deal, t.ng, t.nshorter);
        sa.part = static_cast<float *>(s.balance);
        rows = pl.bytes / kFlashSlotBytes * kBM8;
    } else if (pl.splits > 1) {
        sa.n = pl.splits;
        sa.tiles = pl.tiles;
        sa.part = static_cast<float *>(s.part);
        rows = size_t(pl.splits) * size_t(BH) * size_t(S_q);
    }
    sa.ml = reinterpret_cast<float2 *>(reinterpret_cast<char *>(sa.part) +
                                       flash_round_up256(rows * kD * sizeof(float)));
    return sa;
}

int64_t flash_blocks(const FlashSplitArgs &sa, const FlashWhole &, int64_t BH, int S_q, int BM)
{
    return BH * flash_ceil_div(S_q, BM) * sa.n;
}

int64_t flash_blocks(const FlashSplitArgs &, const FlashShares &sh, int64_t, int, int)
{
    return sh.tail.full + sh.tail.ng + sh.tail.nshorter;
}

bool launch_flash_combine(const FlashProblem &p, const FlashSplitArgs &sa, const FlashTail &tail,
                          hipStream_t st)
{
    const bool bal = tail.u > 0;
    if (sa.n == 1 && !bal)
        return true;
    CombineArgs a;
    a.o = p.o;
    a.ob = p.os.b;
    a.oh = p.os.h;
    a.os = p.os.s;
    a.H = p.H;
    a.S_q = p.S_q;
    a.sa = sa;
    a.ot = p.ot;
    a.total = (bal ? int64_t(tail.ntail) * kBM8 : sa.BH * p.S_q) * (kD / 4);
    const int64_t nblk = flash_ceil_div(a.total, 256);
    if (nblk > INT32_MAX)
        return fail("flash_combine: problem too large for one launch");
    if (bal)
        hipLaunchKernelGGL(flash_combine_kernel<CombineTail>, dim3(unsigned(nblk)), dim3(256), 0,
                           st, a, CombineTail{tail, int(flash_ceil_div(p.S_q, kBM8))});
    else
        hipLaunchKernelGGL(flash_combine_kernel<FlashWhole>, dim3(unsigned(nblk)), dim3(256), 0, st,
                           a, FlashWhole{});
    return hip_ok(hipGetLastError(), "flash_combine_kernel launch");
}

}  // namespace anima_hip
