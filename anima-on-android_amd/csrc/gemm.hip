// Linear layer GEMM: C[M,N] = A[M,K] . W[N,K]^T, A f32, W bf16 or f32, f32
// accumulation on v_mfma_f32_32x32x2_f32.
//
// Replaces anima_rt_run_gemm_bf16 / anima_rt_run_gemm_fp32
// (anima_rt/src/gemm_backend.cpp:140-173, row-major C = A @ W^T with W laid
// out [out_features, in_features]); used here for the cross-attention context
// projections k_proj / v_proj (anima_rt/scripts/numpy_dit.py:277-281), whose
// results the context K/V cache keeps for every denoise step.
//
// Two kernels:
//   gemm_tile_kernel  f32 weights, 16-byte aligned rows, K a multiple of 32: the
//                     operands reach LDS by DMA;
//   gemm_kernel       everything else: block tile 128x128, K chunk 32, 4 waves
//                     in a 2x2 grid each owning 64x64 (four 32x32 MFMA
//                     accumulators), operands staged through LDS as f32 element
//                     by element (bf16 weights widened on the way in); every
//                     global access is bounds-checked so any M, N, K and any
//                     leading dimensions are accepted.
#include "flash_tile.h"

namespace anima_hip {
namespace {

using flash_tile::f32x16;
using flash_tile::f32x4;

constexpr int kBM = 128, kBN = 128, kBK = 32;
constexpr int kPitch = kBK + 4;  // floats per LDS row

struct GemmArgs {
    const float *a;
    const void *w;
    float *c;
    int64_t lda, ldw, ldc;
    int M, N, K, w_bf16, n_tiles_n;
};

__device__ __forceinline__ float load_w(const GemmArgs &g, int64_t idx)
{
    if (g.w_bf16) {
        const unsigned short bits = static_cast<const unsigned short *>(g.w)[idx];
        return __uint_as_float(unsigned(bits) << 16);
    }
    return static_cast<const float *>(g.w)[idx];
}

__global__ __launch_bounds__(256) void gemm_kernel(GemmArgs g)
{
    __shared__ __attribute__((aligned(16))) float As[kBM * kPitch];
    __shared__ __attribute__((aligned(16))) float Ws[kBN * kPitch];
    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const int col = lane & 31, half = lane >> 5;
    const int tm = blockIdx.x / g.n_tiles_n, tn = blockIdx.x % g.n_tiles_n;
    const int m0 = tm * kBM, n0 = tn * kBN;
    const int wm = (wave >> 1) * 64, wn = (wave & 1) * 64;

    f32x16 acc[2][2] = {};
    for (int k0 = 0; k0 < g.K; k0 += kBK) {
        // 128 x 32 elements of each operand, 16 per thread, coalesced along K.
#pragma unroll 4
        for (int i = 0; i < 16; ++i) {
            const int e = tid + 256 * i;
            const int r = e >> 5, kk = e & 31;
            const int gm = m0 + r, gn = n0 + r, gk = k0 + kk;
            As[r * kPitch + kk] = (gm < g.M && gk < g.K) ? g.a[gm * g.lda + gk] : 0.0f;
            Ws[r * kPitch + kk] = (gn < g.N && gk < g.K) ? load_w(g, gn * g.ldw + gk) : 0.0f;
        }
        __syncthreads();
        // Lane half h contracts k = 16h + t (t = 0..15) of the chunk, for A
        // and W alike.
#pragma unroll
        for (int t4 = 0; t4 < 4; ++t4) {
            f32x4 av[2], wv[2];
#pragma unroll
            for (int x = 0; x < 2; ++x) {
                av[x] = *reinterpret_cast<const f32x4 *>(
                    &As[(wm + 32 * x + col) * kPitch + 16 * half + 4 * t4]);
                wv[x] = *reinterpret_cast<const f32x4 *>(
                    &Ws[(wn + 32 * x + col) * kPitch + 16 * half + 4 * t4]);
            }
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int x = 0; x < 2; ++x)
#pragma unroll
                    for (int y = 0; y < 2; ++y)
                        acc[x][y] = __builtin_amdgcn_mfma_f32_32x32x2f32(av[x][e], wv[y][e],
                                                                         acc[x][y], 0, 0, 0);
        }
        __syncthreads();
    }
    // acc[x][y] register r, lane l: row 8(r/4) + 4h + (r%4), column l%32.
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int gm = m0 + wm + 32 * x + 8 * (r >> 2) + 4 * half + (r & 3);
                const int gn = n0 + wn + 32 * y + col;
                if (gm < g.M && gn < g.N)
                    g.c[gm * g.ldc + gn] = acc[x][y][r];
            }
}

// C = A . W^T on f32 MFMA from DMA-staged tiles: 64 x 64 of C per workgroup, 4
// waves in a 2x2 grid each owning 32 x 32.  Bound by the f32 MFMA pipe (busy 83 %
// of the cycles at 8192x2048x2048, 74 % at 2400x2048x2048, whose 1216 tiles are
// less than the 1280 that five to a CU make), which takes 64 cycles per 32x32x2
// product: a chunk of 32 k needs 16 bytes per clock from L2 and 32 from LDS,
// inside what a CU gets (35 and 128), so the small tile costs little and comes
// out more even over the CUs.  Two stages of one chunk
// (32 KiB, five workgroups to a CU), one barrier per chunk; other workgroups'
// products fill a wave's waits.  Two accumulators take the products of even and
// odd k: shorter chains, and rounding errors 0.7 times one chain's.
// Whole calls on MI355X, before (gemm_kernel) and now: 2400x2048x2048 785 ->
// 171 us (118 TFLOP/s; up to 187 by box and load), 8192x2048x2048 1061 -> 537
// (128), 512x2048x8192 2575 -> 155, 100x2048x2048 365 -> 40.  Measured beside it
// at the first two shapes in one run that gave it 187 / 537: 128 x 128 tiles, two
// workgroups to a CU 257 / 518 us; three stages and three workgroups 191 / 567;
// one accumulator 188 / 542; no raised priority 191 / 558.
//
// A chunk's row holds 32 k as eight 16-byte pieces; piece c of row r is at
// c ^ ((r >> 1) & 7), so the 16 rows that a fragment read serves per clock fall
// into 16 different bank groups.  Lane half h contracts k = 16h + t (t = 0..15)
// of the chunk, for A and W alike.
struct TileArgs {
    const float *a, *w;
    float *c;
    int64_t lda, ldw, ldc;
    int M, N, chunks, n_tiles_n;
};

constexpr int kT = 64;

__global__ __launch_bounds__(256, 5) void gemm_tile_kernel(TileArgs g)
{
    constexpr int kRows = 2 * kT;             // A rows, then W rows
    constexpr int kCopies = kRows * 8 / 256;  // 16-byte copies per thread and chunk
    __shared__ __attribute__((aligned(16))) float ring[2][kRows * kBK];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 31, half = lane >> 5;
    const int blk = flash_tile::xcd_major_block();
    const int m0 = blk / g.n_tiles_n * kT, n0 = blk % g.n_tiles_n * kT;

    // Copy i of this wave fills pieces (wave*kCopies + i)*64 + lane of the
    // stage; rows past M or N copy the last row (their C is not stored).
    const float *src[kCopies];
#pragma unroll
    for (int i = 0; i < kCopies; ++i) {
        const int f = (wave * kCopies + i) * 64 + lane, r = f >> 3;
        const int c = (f & 7) ^ ((r >> 1) & 7);
        src[i] = (r < kT ? g.a + int64_t(min(m0 + r, g.M - 1)) * g.lda
                         : g.w + int64_t(min(n0 + r - kT, g.N - 1)) * g.ldw) +
                 4 * c;
    }
    auto copy = [&](int chunk) {
#pragma unroll
        for (int i = 0; i < kCopies; ++i)
            flash_tile::dma16(reinterpret_cast<const flash_tile::u16 *>(src[i] + chunk * kBK),
                              reinterpret_cast<flash_tile::u16 *>(
                                  &ring[chunk & 1][(wave * kCopies + i) * 256]));
    };
    copy(0);

    const int wm = (wave >> 1) * 32, wn = (wave & 1) * 32;
    const int sw = (col >> 1) & 7;
    f32x16 acc0 = {}, acc1 = {};
    for (int k = 0; k < g.chunks; ++k) {
        flash_tile::wait_vmcnt<0>();
        flash_tile::ring_barrier();
        // The other stage was read in the previous iteration.
        if (k + 1 < g.chunks)
            copy(k + 1);
        const float *ar = ring[k & 1] + (wm + col) * kBK;
        const float *wr = ring[k & 1] + (kT + wn + col) * kBK;
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int t4 = 0; t4 < 4; ++t4) {
            const int piece = 4 * ((4 * half + t4) ^ sw);
            const f32x4 av = *reinterpret_cast<const f32x4 *>(ar + piece);
            const f32x4 wv = *reinterpret_cast<const f32x4 *>(wr + piece);
            acc0 = __builtin_amdgcn_mfma_f32_32x32x2f32(av.x, wv.x, acc0, 0, 0, 0);
            acc1 = __builtin_amdgcn_mfma_f32_32x32x2f32(av.y, wv.y, acc1, 0, 0, 0);
            acc0 = __builtin_amdgcn_mfma_f32_32x32x2f32(av.z, wv.z, acc0, 0, 0, 0);
            acc1 = __builtin_amdgcn_mfma_f32_32x32x2f32(av.w, wv.w, acc1, 0, 0, 0);
        }
        __builtin_amdgcn_s_setprio(0);
    }
    acc0 += acc1;
    // Register r, lane l: row acc_row(r, half), column l%32.
    const int gn = n0 + wn + col;
    float *c = g.c + int64_t(m0 + wm) * g.ldc + gn;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int row = flash_tile::acc_row(r, half);
        if (m0 + wm + row < g.M && gn < g.N)
            c[row * g.ldc] = acc0[r];
    }
}

bool tile_supported(const float *a, int64_t lda, const void *w, bool w_bf16, int64_t ldw, int K)
{
    return !w_bf16 && K > 0 && K % kBK == 0 && lda % 4 == 0 && ldw % 4 == 0 &&
           flash_tile::aligned(a, 16) && flash_tile::aligned(w, 16);
}

}  // namespace

bool launch_gemm(const float *a, int64_t lda, const void *w, bool w_bf16, int64_t ldw, float *c,
                 int64_t ldc, int M, int N, int K, hipStream_t st)
{
    if (M < 0 || N < 0 || K < 0)
        return fail("gemm: negative dimension");
    if (M == 0 || N == 0)
        return true;  // K == 0 runs the kernel, which then stores zeros
    if (tile_supported(a, lda, w, w_bf16, ldw, K)) {
        const int64_t n_tiles_n = (int64_t(N) + kT - 1) / kT;
        const int64_t nblk = (int64_t(M) + kT - 1) / kT * n_tiles_n;
        if (nblk > INT32_MAX)
            return fail("gemm: problem too large for one launch");
        const TileArgs t{a, static_cast<const float *>(w), c, lda, ldw, ldc, M, N, K / kBK,
                         int(n_tiles_n)};
        hipLaunchKernelGGL(gemm_tile_kernel, dim3(unsigned(nblk)), dim3(256), 0, st, t);
        return hip_ok(hipGetLastError(), "gemm_tile_kernel launch");
    }
    GemmArgs g;
    g.a = a;
    g.w = w;
    g.c = c;
    g.lda = lda;
    g.ldw = ldw;
    g.ldc = ldc;
    g.M = M;
    g.N = N;
    g.K = K;
    g.w_bf16 = w_bf16 ? 1 : 0;
    g.n_tiles_n = (N + kBN - 1) / kBN;
    const int64_t nblk = int64_t((M + kBM - 1) / kBM) * g.n_tiles_n;
    if (nblk > INT32_MAX)
        return fail("gemm: problem too large for one launch");
    hipLaunchKernelGGL(gemm_kernel, dim3(unsigned(nblk)), dim3(256), 0, st, g);
    return hip_ok(hipGetLastError(), "gemm_kernel launch");
}

}  // namespace anima_hip
