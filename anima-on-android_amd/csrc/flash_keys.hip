// Flash attention for grids that leave most of the GPU idle: a workgroup's
// waves share the keys of 64 query rows (gfx950, bf16 MFMA, D = 128).
//
// The computation, operands and layouts of flash_bf16.hip (TERMS = 1: bf16 q
// and k rows, packed V^T) and flash_x3.hip (TERMS = 2: [hi | lo] term rows and
// term V^T, every product as hi*hi + hi*lo + lo*hi); anima_rt_run_sdpa_flash
// (anima_rt/src/anima_rt.cpp:147-156 -> anima_rt/include/cpu/flash_attention.h:
// 55-208) without a mask.
//
// Why: those kernels give a wave 32 query rows and walk all keys in series, so
// 256 queries of 16 heads are 32 workgroups of 4 waves on 256 CUs, each with
// one wave per SIMD and every tile's latency in the open; split over more
// workgroups they pay a combine pass.  Here 8 waves are 2 (query rows) x 4
// (keys): wave (r, g) takes rows 32r .. 32r+31 and key tiles g, g + 4, ..., with
// its own running max, sum and O; the four parts of a row are merged through
// LDS at the end.  Four times the workgroups, two waves per SIMD, no second
// launch; each K/V tile serves 64 rows instead of 128 or 256.  Bound by the chain
// of a round, whose copies, products and softmax follow one another between two
// barriers: on its fullest grid (1024 x 1024, 16 heads, f32x3) the MFMA pipes are
// busy 26 % of the cycles and LDS 11 %, waves wait 36 %, and 12 MB come from HBM.
// Whole attention calls on MI355X before and now, 16 heads (f32x3 / bf16): self
// 256 tokens 24.7 -> 22.3 / 17.8 -> 15.5 us, 1024 tokens 50.4 -> 45.6 / 39.1 ->
// 30.3; cached cross-attention, query rows normalised in here, 2 x 256 on 512
// 28.8 -> 17.9 / 20.7 -> 12.0, 1024 x 512 34.5 -> 20.0 / 22.6 -> 12.7.  (Waiting
// for K and V^T with a barrier of its own each, so that more copies are in
// flight, was 3 to 16 % slower.)
//
// Per key group one K tile and one V^T tile (16 KiB each: 32 keys of terms, 64
// of bf16), single-buffered and refilled in turn: V^T lands while the scores
// run, the next K while the softmax and P.V run, one barrier after each.
#include "qrow.h"

#include <cmath>

namespace anima_hip {
namespace {

using namespace flash_tile;

constexpr int kGroups = 4;           // key groups of a workgroup
constexpr int kRowsPerBlock = 64;    // query rows of a workgroup
constexpr int kTileEl = 8192;        // bf16 per K or V^T tile (16 KiB)
constexpr int kPitch = kD + 4;       // floats per merged row (4 against bank conflicts)
constexpr int kRingBytes = kGroups * 2 * kTileEl * 2;
constexpr int kMergeBytes = 8 * 32 * kPitch * 4;

struct KeysArgs {
    const u16 *q, *k, *vt;
    float *o;
    int64_t qb, qh, qs, kb, kh, ks, vb, vh, vd, ob, oh, os;
    int H, S_q, S_kv, n_qtiles;
    float c;    // scale * log2(e), > 0
    int dma32;  // K/V^T tile rows fit 32-bit byte offsets from the tile start
    TermOut ot;
    const float *qx, *qw;  // raw query rows (RawQ, no RoPE) in place of q when qx is set
    int64_t rqb, rqh, rqs, qplane;
    int qparts;
    float eps;
};

// By bits: this file is compiled without NaN comparisons.  A part with any sum but
// zero takes part in the merge, a NaN sum included.
__device__ __forceinline__ bool joins(const float2 &p) { return (__float_as_uint(p.y) << 1) != 0; }
__device__ __forceinline__ bool is_nan(float x) { return (__float_as_uint(x) << 1) > 0xFF000000u; }

// The terms of the workgroup's 64 raw rows, bit for bit those of the row prologue
// (prologue.hip) and q_terms_from_raw: one lane per row adds the squares in
// index order, every thread then scales and splits its own four float4 (row
// tid / 32 + 16 i, columns 4 (tid % 32)), and the waves read their fragments
// back.  (q_terms_from_raw in every wave would do the work of a row four times
// over, once for each key group.)
template <int TERMS>
__device__ __forceinline__ void keys_q_terms(const KeysArgs &a, float *rows, const f32x4 (&v)[4],
                                             int tid, bf16x8 (&qh)[8], bf16x8 (&ql)[8])
{
#pragma clang fp contract(off)
    constexpr int kTermPitch = TERMS * kD + 8;  // 16-bit elements, 16 bytes against conflicts
    __shared__ float inv[kRowsPerBlock];
    if (tid < kRowsPerBlock) {
        const float *row = rows + tid * kPitch;
        float ss = 0.0f;
#pragma unroll 4
        for (int j = 0; j < kD / 4; ++j) {
            const f32x4 x = *reinterpret_cast<const f32x4 *>(row + 4 * j);
            ss = ss + x.x * x.x;
            ss = ss + x.y * x.y;
            ss = ss + x.z * x.z;
            ss = ss + x.w * x.w;
        }
        inv[tid] = inv_rms(ss, kD, a.eps);
    }
    const int c4 = tid & 31;
    f32x4 w = f32x4{1.f, 1.f, 1.f, 1.f};
    if (a.qw)
        w = *reinterpret_cast<const f32x4 *>(a.qw + 4 * c4);
    __syncthreads();  // the sums are there, the rows are read
    u16 *const terms = reinterpret_cast<u16 *>(rows);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int r = (tid >> 5) + 16 * i;
        f32x4 y = v[i] * inv[r];
        if (a.qw)
            y = y * w;
        uint2 th, tl;
        split_terms4(y, th, tl);
        *reinterpret_cast<uint2 *>(terms + r * kTermPitch + 4 * c4) = th;
        if (TERMS == 2)
            *reinterpret_cast<uint2 *>(terms + r * kTermPitch + kD + 4 * c4) = tl;
    }
    __syncthreads();
    const int lane = tid & 63, row = 32 * ((tid >> 6) & 1) + (lane & 31);
    const u16 *src = terms + row * kTermPitch + 64 * (lane >> 5);
#pragma unroll
    for (int t = 0; t < 8; ++t) {
        qh[t] = *reinterpret_cast<const bf16x8 *>(src + 8 * t);
        if (TERMS == 2)
            ql[t] = *reinterpret_cast<const bf16x8 *>(src + kD + 8 * t);
    }
}

template <int TERMS>
__global__ __launch_bounds__(512, 1) void flash_keys_d128(KeysArgs a)
{
    constexpr int KT = 64 / TERMS, NB = KT / 32;   // keys per tile, 32-key blocks
    constexpr int kRow = TERMS * kD, CK = kRow / 8;  // K row: elements, 16-byte chunks
    constexpr int CV = KT / 8;                     // chunks of a V^T row
    constexpr int kCopies = kTileEl / 8 / 128;     // 16-byte copies per thread and tile
    static_assert(KT * kRow == kTileEl, "tile sizes");
    static_assert(kRowsPerBlock * kPitch * 4 <= kGroups * kTileEl * 2, "raw rows fit");

    __shared__ __attribute__((aligned(16))) unsigned char
        smem[kMergeBytes > kRingBytes ? kMergeBytes : kRingBytes];
    __shared__ float2 ml[8][32];  // (max, sum) per wave and row
    __shared__ float sums[8][32];  // sums against the row's max

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 31, half = lane >> 5;
    const int rg = wave & 1, kg = wave >> 1;
    u16 *const ks = reinterpret_cast<u16 *>(smem) + kg * kTileEl;
    u16 *const vs = ks + kGroups * kTileEl;

    const int blk = xcd_major_block();
    const int qt = blk % a.n_qtiles, bh = blk / a.n_qtiles;
    const int b = bh / a.H, h = bh - b * a.H;
    const int q0 = qt * kRowsPerBlock;
    const int qrow = q0 + 32 * rg + col;
    const u16 *kp = a.k + b * a.kb + h * a.kh;
    const u16 *vp = a.vt + b * a.vb + h * a.vh;
    const int ntiles = (a.S_kv + KT - 1) / KT;

    // Copy i of this wave fills the 64 chunks of window w = kCopies*rg + i of its
    // group's tile.  LDS layouts, unpadded, XOR-swizzled so that the 16 lanes a
    // fragment read serves per clock hit 16 bank groups: chunk c of K row r at
    // c ^ (r & 15); of V^T row r at c ^ ((r >> 2) & 3) (four chunks a row) or
    // c ^ ((r >> 1) & 7) (eight).
    auto vswz = [](int r) { return TERMS == 2 ? (r >> 2) & 3 : (r >> 1) & 7; };
    unsigned koff[kCopies], voff[2];
#pragma unroll
    for (int i = 0; i < kCopies; ++i) {
        const int f = (kCopies * rg + i) * 64 + lane, r = f / CK;
        koff[i] = unsigned(r * a.ks + 8 * ((f % CK) ^ (r & 15))) * 2u;
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        // Rows of window i, from row (kCopies*rg) * 64/CV; the swizzle of a
        // window depends on its parity only.
        const int f = (kCopies * rg + i) * 64 + lane, r = f / CV;
        voff[i] = unsigned((lane / CV) * a.vd + 8 * ((f % CV) ^ vswz(r))) * 2u;
    }
    auto dma_k = [&](int t) {
        const int key0 = t * KT;
        if (a.dma32 && key0 + KT <= a.S_kv) {
#pragma unroll
            for (int i = 0; i < kCopies; ++i)
                dma16s(kp + int64_t(key0) * a.ks, koff[i], ks + (kCopies * rg + i) * 512);
        } else {
            // Keys past S_kv copy row S_kv - 1; their scores are masked.
#pragma unroll
            for (int i = 0; i < kCopies; ++i) {
                const int f = (kCopies * rg + i) * 64 + lane, r = f / CK;
                dma16(kp + int64_t(min(key0 + r, a.S_kv - 1)) * a.ks + 8 * ((f % CK) ^ (r & 15)),
                      ks + (kCopies * rg + i) * 512);
            }
        }
    };
    auto dma_v = [&](int t) {
        // V^T is zero-padded in HBM to whole 64-key tiles.
        const u16 *base = vp + t * KT;
#pragma unroll
        for (int i = 0; i < kCopies; ++i) {
            const int win = kCopies * rg + i;
            if (a.dma32)
                dma16s(base + int64_t(win * (64 / CV)) * a.vd, voff[i & 1], vs + win * 512);
            else
                dma16(base + int64_t(win * (64 / CV) + lane / CV) * a.vd +
                          8 * (((win * 64 + lane) % CV) ^ vswz((win * 64 + lane) / CV)),
                      vs + win * 512);
        }
    };
    // Fragments: K key row col + 32*kb, term chunk 8*half + t; V^T row
    // 128*term + 32*blk + col, keys [16i, 16i + 16) (chunk half + 2i).
    auto kfrag = [&](int t, int kb, int term) {
        return *reinterpret_cast<const bf16x8 *>(
            ks + (col + 32 * kb) * kRow + 8 * (16 * term + (((half << 3) | t) ^ (col & 15))));
    };
    auto vfrag = [&](int blk, int i, int term) {
        return *reinterpret_cast<const bf16x8 *>(vs + (128 * term + 32 * blk + col) * KT +
                                                 8 * ((half + 2 * i) ^ vswz(col)));
    };

    if (kg < ntiles)
        dma_k(kg);
    // Q terms: hi Q[qrow][64*half + 8t .. +7], lo 128 elements further.
    bf16x8 qh[8], ql[8];
    if (a.qx) {
        // The 64 raw rows once for the four key groups, through the V^T tiles'
        // space, their planes added in order.
        float *const rows = reinterpret_cast<float *>(smem + kGroups * kTileEl * 2);
        const float *x[4];
        f32x4 v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int f = tid + 512 * i, r = min(q0 + (f >> 5), a.S_q - 1);
            x[i] = a.qx + b * a.rqb + h * a.rqh + int64_t(r) * a.rqs + 4 * (f & 31);
            v[i] = *reinterpret_cast<const f32x4 *>(x[i]);
        }
        for (int p0 = 1; p0 < a.qparts; p0 += 3) {  // three planes' loads in flight
            f32x4 y[3][4];
#pragma unroll
            for (int u = 0; u < 3; ++u)
#pragma unroll
                for (int i = 0; i < 4; ++i)  // past the last plane: read, not added
                    y[u][i] = *reinterpret_cast<const f32x4 *>(
                        x[i] + min(p0 + u, a.qparts - 1) * a.qplane);
#pragma unroll
            for (int u = 0; u < 3; ++u)
                if (p0 + u < a.qparts) {
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        v[i] += y[u][i];
                }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int f = tid + 512 * i;
            *reinterpret_cast<f32x4 *>(rows + (f >> 5) * kPitch + 4 * (f & 31)) = v[i];
        }
        __syncthreads();
        keys_q_terms<TERMS>(a, rows, v, tid, qh, ql);
    } else {
        const u16 *qr = a.q + b * a.qb + h * a.qh + int64_t(min(qrow, a.S_q - 1)) * a.qs;
        const bf16x8 *src = reinterpret_cast<const bf16x8 *>(qr + 64 * half);
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            qh[t] = src[t];
            if (TERMS == 2)
                ql[t] = src[kD / 8 + t];
        }
    }
    f32x16 o[4] = {};
    float m = -INFINITY, l = 0.0f, l2 = 0.0f;
    wait_vmcnt<0>();
    ring_barrier();

    for (int t0 = 0; t0 < ntiles; t0 += kGroups) {
        const int t = t0 + kg;  // this group's tile; none in a ragged last round
        const bool live = t < ntiles;
        f32x16 s[NB] = {};
        if (live) {
            dma_v(t);
            // Scores S^T; with terms the cross products in a chain of their own.
            f32x16 x = {};
#pragma unroll
            for (int i = 0; i < 8; ++i) {
#pragma unroll
                for (int kb = 0; kb < NB; ++kb) {
                    const bf16x8 k0 = kfrag(i, kb, 0);
                    s[kb] = mfma_bf16(k0, qh[i], s[kb]);
                    if (TERMS == 2) {
                        x = mfma_bf16(k0, ql[i], x);
                        x = mfma_bf16(kfrag(i, kb, 1), qh[i], x);
                    }
                }
            }
            if (TERMS == 2)
                s[0] += x;
        }
        wait_vmcnt<0>();
        ring_barrier();  // V^T is there, K is read
        if (t + kGroups < ntiles)
            dma_k(t + kGroups);
        if (live) {
            const int key0 = t * KT;
            if (key0 + KT > a.S_kv) {
#pragma unroll
                for (int kb = 0; kb < NB; ++kb)
#pragma unroll
                    for (int r = 0; r < 16; ++r)
                        if (key0 + 32 * kb + acc_row(r, half) >= a.S_kv)
                            s[kb][r] = -INFINITY;
            }
            float mx = -INFINITY;
#pragma unroll
            for (int kb = 0; kb < NB; ++kb)
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    mx = fmaxf(mx, s[kb][r]);
            // The max on raw scores (c > 0) and the lazy rescale, as in the
            // kernels of whole key ranges.
            const float cand = row_pair_max(mx) * a.c;
            if (__any(cand > m + kRescaleLog2)) {
                const float m_new = fmaxf(m, cand);
                const float alpha =
                    m_new == -INFINITY ? 1.0f : __builtin_amdgcn_exp2f(m - m_new);
                m = m_new;
                l *= alpha;
                l2 *= alpha;
#pragma unroll
                for (int d = 0; d < 4; ++d)
                    o[d] *= alpha;
            }
            const float neg_m = (m == -INFINITY) ? 0.0f : -m;
            // P in chunks of 16 keys, its terms summed as the MFMAs take them.
            float sum = 0.0f, sum2 = 0.0f;
#pragma unroll
            for (int i = 0; i < 2 * NB; ++i) {
                f32x16 &sc = s[i >> 1];
                bf16x8 ph, pl;
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    sc[8 * (i & 1) + e] =
                        __builtin_amdgcn_exp2f(fmaf(sc[8 * (i & 1) + e], a.c, neg_m));
                ph = pack8(sc, 8 * (i & 1));
                sum = row_sum8(ph, sum);
                if (TERMS == 2) {
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        sc[8 * (i & 1) + e] -= float(ph[e]);
                    pl = pack8(sc, 8 * (i & 1));
                    sum2 = row_sum8(pl, sum2);
                }
#pragma unroll
                for (int d = 0; d < 4; ++d) {
                    const bf16x8 v0 = vfrag(d, i, 0);
                    o[d] = mfma_bf16(v0, ph, o[d]);
                    if (TERMS == 2) {
                        o[d] = mfma_bf16(v0, pl, o[d]);
                        o[d] = mfma_bf16(vfrag(d, i, 1), ph, o[d]);
                    }
                }
            }
            l += sum;
            l2 += sum2;
        }
        wait_vmcnt<0>();
        ring_barrier();  // the next K is there, V^T is read
    }

    // Merge the four parts of every row.  A part without a live key has sum 0 and
    // drops out; a NaN sum joins and makes the row NaN, also where all of the
    // part's scores were NaN and its max is still -inf; a row whose every part's
    // max is -inf is zeros, as in the reference (store_o_rows).
    l += l2;
    l += __shfl_xor(l, 32);
    if (half == 0)
        ml[wave][col] = make_float2(m, l);
    __syncthreads();
    float mx = -INFINITY;
#pragma unroll
    for (int g = 0; g < kGroups; ++g) {
        const float2 p = ml[2 * g + rg][col];
        if (joins(p))
            mx = fmaxf(mx, p.x);
    }
    const float w = m == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m - mx);
    if (half == 0)
        sums[wave][col] = mx == -INFINITY ? 0.0f : m == -INFINITY ? l : l * w;
    float *const part = reinterpret_cast<float *>(smem);
#pragma unroll
    for (int d = 0; d < 4; ++d)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            f32x4 v = f32x4{o[d][4 * g], o[d][4 * g + 1], o[d][4 * g + 2], o[d][4 * g + 3]} * w;
            if (m == -INFINITY)
                v = f32x4{0.f, 0.f, 0.f, 0.f};
            *reinterpret_cast<f32x4 *>(part + (wave * 32 + col) * kPitch + 32 * d +
                                       acc_row(4 * g, half)) = v;
        }
    __syncthreads();
#pragma unroll 1
    for (int i = 0; i < kRowsPerBlock * 32 / 512; ++i) {
        const int f = tid + 512 * i, r = f >> 5, c4 = f & 31;
        if (q0 + r >= a.S_q)
            continue;
        const int r0 = r >> 5, rr = r & 31;
        float sum = 0.0f;
        f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int g = 0; g < kGroups; ++g) {
            sum += sums[2 * g + r0][rr];
            v += *reinterpret_cast<const f32x4 *>(part + ((2 * g + r0) * 32 + rr) * kPitch +
                                                  4 * c4);
        }
        v *= is_nan(sum) ? sum : sum > 0.0f ? 1.0f / sum : 0.0f;
        const int q = q0 + r;
        store_out4(v, a.o + b * a.ob + h * a.oh + int64_t(q) * a.os,
                   a.ot.t ? a.ot.t + b * a.ot.tb + h * a.ot.th + int64_t(q) * a.ot.ts : nullptr,
                   a.ot.lo, 4 * c4);
    }
}

}  // namespace

bool launch_flash_keys(const FlashProblem &p, int terms, bool dma32, hipStream_t st)
{
    if (p.rq.freqs)
        return fail("flash_keys: raw query rows with RoPE are not taken");
    const int64_t BH = int64_t(p.B) * p.H;
    KeysArgs a;
    a.q = static_cast<const u16 *>(p.q);
    a.k = static_cast<const u16 *>(p.k);
    a.vt = static_cast<const u16 *>(p.v);
    a.o = p.o;
    a.qb = p.qs.b; a.qh = p.qs.h; a.qs = p.qs.s;
    a.kb = p.ks.b; a.kh = p.ks.h; a.ks = p.ks.s;
    a.vb = p.vs.b; a.vh = p.vs.h; a.vd = vt_padded_len(p.S_kv);
    a.ob = p.os.b; a.oh = p.os.h; a.os = p.os.s;
    a.H = p.H;
    a.S_q = p.S_q;
    a.S_kv = p.S_kv;
    a.n_qtiles = (p.S_q + kRowsPerBlock - 1) / kRowsPerBlock;
    a.c = p.scale * kLog2e;
    a.dma32 = dma32 ? 1 : 0;
    a.ot = p.ot;
    a.qx = p.rq.x;
    a.qw = p.rq.w;
    a.rqb = p.rq.s.b; a.rqh = p.rq.s.h; a.rqs = p.rq.s.s;
    a.qparts = p.rq.parts;
    a.qplane = p.rq.plane;
    a.eps = p.rq.eps;
    const int64_t nblk = BH * a.n_qtiles;
    if (nblk > INT32_MAX)
        return fail("flash_keys: problem too large for one launch");
    if (terms == 2)
        hipLaunchKernelGGL(flash_keys_d128<2>, dim3(unsigned(nblk)), dim3(512), 0, st, a);
    else
        hipLaunchKernelGGL(flash_keys_d128<1>, dim3(unsigned(nblk)), dim3(512), 0, st, a);
    return hip_ok(hipGetLastError(), "flash_keys_d128 launch");
}

}  // namespace anima_hip
