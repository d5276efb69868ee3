// The float32 product of many rows, C[M, N] = A[M, K] . B[N, K]^T, on the bfloat16 matrix cores without losing a bit of
// an operand.  A float32 number is the sum of three bfloat16 numbers, x = x1 + x2 + x3 (x1 = x rounded, x2 = what is left
// rounded, x3 = the rest: 3 x 8 significand bits and two signs hold 24), so
//   a b = a1 b1 + (a1 b2 + a2 b1) + (a1 b3 + a2 b2 + a3 b1) + what is below 2^-24 of it (2^-27.5 on average),
// six products of the bfloat16 matrix instruction, each exact, added up in float32: no more is lost than by one float32
// rounding of a b.  The float32 matrix instruction does 157 TFLOP/s, the bfloat16 one 2500, a sixth of which is 417.
#include "common.h"
#include "lds.h"
#include "parts.h"
#include <math.h>

LLE_DEFINE_ERROR_STRING()

typedef bf16_t sbf16x8 __attribute__((ext_vector_type(8)));
typedef float sf32x4 __attribute__((ext_vector_type(4)));
typedef float sf32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t su32x4 __attribute__((ext_vector_type(4)));

#define SG_BK 32      // columns of K per step
#define SG_PIECES 4   // 8-element pieces of a row of a step

// Tiles of 64 TM rows of A x 64 TN rows of B, four wavefronts of 32 TM x 32 TN.  A step of 32 columns is asked for while the
// one before is multiplied, split in registers on its way to LDS (one buffer; two or more workgroups a CU fill each other's
// gaps), its 16-byte pieces XOR-swizzled by the row, so that no read meets a bank conflict.  blockIdx.y: a slice of K, whose
// sums go to C + blockIdx.y * M * N.
//
// Bound by the matrix cores: at 2048 x 24576 x 4096 the 256 x 128 tiles keep them busy 0.77 of the time, at the 1.8 GHz that
// their power leaves: 1800 us, 229 TFLOP/s of float32 product (1.37 PFLOP/s of the instruction); the float32 instruction, in
// 64 x 64 tiles, took 4160 us.  2048 x 4096 x 12288: 965 us against 1774; 2048 x 4096 x 4096: 321 against 590.  The error
// against 64 bits is a tenth smaller (1.0e-6 against 1.1e-6 at K = 4096): fewer, exact products per rounding of a sum.
//
// SPLIT_SILU, SPLIT_CLAMPED: B holds gate rows and then up rows, N of each, and C [M, N] is act(gate) . up.  Of a wavefront's 64 rows of B
// the first 32 are gate rows and the others the up rows that go with them, so a lane holds both sums of a place; the same sums and
// the same bits as the whole product and the activation's pass, without the way of 2 N floats a row to memory and back.
enum SplitOut { SPLIT_PLAIN = 0, SPLIT_SILU, SPLIT_CLAMPED };

template <int OUT, int TM, int TN, int PER_SIMD>
__global__ __launch_bounds__(256, PER_SIMD) void gemm_nt_split_kernel(const float* __restrict__ A, const float* __restrict__ B,
                                                                      float* __restrict__ C, int M, int N, int K, int64_t lda,
                                                                      int64_t ldb, int64_t ldc, int m_tiles, int n_tiles, int slice,
                                                                      const float* __restrict__ bias, float limit) {
    constexpr int BM = 64 * TM, BN = 64 * TN, COLUMNS = OUT == SPLIT_PLAIN ? BN : BN / 2;
    static_assert(OUT == SPLIT_PLAIN || TN == 2, "a gate tile and an up tile for every wavefront");
    extern __shared__ __attribute__((aligned(16))) unsigned char sg_lds[];
    unsigned char* as = sg_lds;                            // [3 parts][BM][4 pieces of 16 bytes]
    unsigned char* bs = sg_lds + 3 * BM * SG_BK * 2;       // [3 parts][BN][4 pieces]
    const int wave = threadIdx.x / LLE_WAVE, lane = threadIdx.x % LLE_WAVE;
    // consecutive workgroups go to different dies: a die takes every eighth column of tiles, all its row tiles one after the
    // other, so that its L2 sees few rows of B at a time
    const int die = blockIdx.x % 8, at = blockIdx.x / 8;
    const int nt = die + 8 * (at / m_tiles), mt = at % m_tiles;
    if (nt >= n_tiles) return;
    const int m0 = mt * BM, n0 = nt * COLUMNS;
    const int k_begin = blockIdx.y * slice, k_end = min(K, k_begin + slice);  // (a slice is a whole number of steps)
    C += (int64_t)blockIdx.y * M * N;
    // the copy: thread -> (row of 64, piece)
    const int lr = threadIdx.x / SG_PIECES, lp = threadIdx.x % SG_PIECES;
    const float *ap[TM], *bp[TN];
#pragma unroll
    for (int i = 0; i < TM; ++i) ap[i] = A + (int64_t)min(m0 + 64 * i + lr, M - 1) * lda;
#pragma unroll
    for (int j = 0; j < TN; ++j) {
        if constexpr (OUT == SPLIT_PLAIN)
            bp[j] = B + (int64_t)min(n0 + 64 * j + lr, N - 1) * ldb;
        else
            bp[j] = B + ((int64_t)min(n0 + 32 * j + lr % 32, N - 1) + (lr < 32 ? 0 : N)) * ldb;
    }
    const int dst = lr * (SG_BK * 2) + ((lp ^ ((lr >> 3) & 3)) * 16);
    sf32x4 ar[TM][2], br[TN][2];
    auto issue = [&](int k0) {
        const int ka = min(k0 + 8 * lp, K - 4), kb = min(k0 + 8 * lp + 4, K - 4);
#pragma unroll
        for (int i = 0; i < TM; ++i) ar[i][0] = *(const sf32x4*)(ap[i] + ka), ar[i][1] = *(const sf32x4*)(ap[i] + kb);
#pragma unroll
        for (int j = 0; j < TN; ++j) br[j][0] = *(const sf32x4*)(bp[j] + ka), br[j][1] = *(const sf32x4*)(bp[j] + kb);
    };
    auto store = [&](unsigned char* base, int rows, int i, const sf32x4* v) {
        su32x4 p1, p2, p3;
#pragma unroll
        for (int h = 0; h < 4; ++h) {
            uint32_t q1, q2, q3;
            split2(v[h / 2][2 * (h % 2)], v[h / 2][2 * (h % 2) + 1], q1, q2, q3);
            p1[h] = q1, p2[h] = q2, p3[h] = q3;
        }
        unsigned char* d = base + 64 * i * (SG_BK * 2) + dst;
        *(su32x4*)d = p1;
        *(su32x4*)(d + rows * SG_BK * 2) = p2;
        *(su32x4*)(d + 2 * rows * SG_BK * 2) = p3;
    };
    const int wm = (wave / 2) * 32 * TM, wn = (wave % 2) * 32 * TN;
    sf32x16 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
    // fragments of 32 rows x 16 columns: lane -> row lane % 32, eight columns from 8 (lane / 32) on
    const int fr = lane % 32, fh = lane / 32;
    const unsigned char* af = as + (wm + fr) * (SG_BK * 2);
    const unsigned char* bf = bs + (wn + fr) * (SG_BK * 2);

    issue(k_begin);
    for (int k0 = k_begin; k0 < k_end; k0 += SG_BK) {
        if (k0 + SG_BK > K) {  // past the end: zeros for A (B's repeated columns then count for nothing)
            const sf32x4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int h = 0; h < 2; ++h)
                    if (k0 + 8 * lp + 4 * h >= K) ar[i][h] = zero;
        }
#pragma unroll
        for (int i = 0; i < TM; ++i) store(as, BM, i, ar[i]);
#pragma unroll
        for (int j = 0; j < TN; ++j) store(bs, BN, j, br[j]);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        issue(k0 + SG_BK);  // on its way while this step is multiplied (past the end: the last columns again)
        __builtin_amdgcn_sched_barrier(0);  // (the compiler would ask for it where it is needed)
        __builtin_amdgcn_s_setprio(1);  // matrix instructions ahead of the other workgroup's splitting: 3 % at 2048 x 24576 x 4096
#pragma unroll
        for (int s = 0; s < SG_BK / 16; ++s) {
            const int piece = ((2 * s + fh) ^ ((fr >> 3) & 3)) * 16;
            sbf16x8 b[TN][3];
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int p = 0; p < 3; ++p) b[j][p] = *(const sbf16x8*)(bf + (p * BN + 32 * j) * SG_BK * 2 + piece);
#pragma unroll
            for (int i = 0; i < TM; ++i) {
                sbf16x8 a[3];
#pragma unroll
                for (int p = 0; p < 3; ++p) a[p] = *(const sbf16x8*)(af + (p * BM + 32 * i) * SG_BK * 2 + piece);
                // the smallest products first
                constexpr int pa[6] = {2, 1, 0, 1, 0, 0}, pb[6] = {0, 1, 2, 0, 1, 0};
#pragma unroll
                for (int q = 0; q < 6; ++q)
#pragma unroll
                    for (int j = 0; j < TN; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[pa[q]], b[j][pb[q]], acc[i][j], 0, 0, 0);
            }
        }
        __builtin_amdgcn_s_setprio(0);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();  // nobody reads this step any more
    }
    // lane holds C[m = 8 (e / 4) + 4 (lane / 32) + e % 4][n = lane % 32] of every 32 x 32 tile
    auto not_finite = [](float v) { return (__builtin_bit_cast(uint32_t, v) & 0x7f800000u) == 0x7f800000u; };
    // the sums of a 32 x 32 tile by the float32 instruction, straight from memory; a_row, b_row: the lane's row of either
    auto plain_sums = [&](const float* a_row, const float* b_row) {
        sf32x16 sum;
#pragma unroll
        for (int e = 0; e < 16; ++e) sum[e] = 0.f;
#pragma unroll 4
        for (int k = k_begin; k < k_end; k += 8) {  // a lane's four columns are its slot of four instructions
            const int at = k + 4 * fh;
            sf32x4 av = {0.f, 0.f, 0.f, 0.f}, bv = av;
            if (at < k_end) av = *(const sf32x4*)(a_row + at), bv = *(const sf32x4*)(b_row + at);
#pragma unroll
            for (int e = 0; e < 4; ++e) sum = __builtin_amdgcn_mfma_f32_32x32x2f32(av[e], bv[e], sum, 0, 0, 0);
        }
        return sum;
    };
    if constexpr (OUT != SPLIT_PLAIN) {
        const int n = n0 + wn / 2 + fr, nb = min(n, N - 1);
        const float b_gate = OUT == SPLIT_CLAMPED && bias ? bias[nb] : 0.f, b_up = OUT == SPLIT_CLAMPED && bias ? bias[N + nb] : 0.f;
#pragma unroll
        for (int i = 0; i < TM; ++i) {
#pragma unroll
            for (int j = 0; j < 2; ++j) {  // (what is not finite is made again, as below)
                bool odd = false;
#pragma unroll
                for (int e = 0; e < 16; ++e) odd |= not_finite(acc[i][j][e]);
                if (__any(odd)) {
                    const sf32x16 sum = plain_sums(A + (int64_t)min(m0 + wm + 32 * i + fr, M - 1) * lda, B + ((int64_t)nb + (j ? N : 0)) * ldb);
#pragma unroll
                    for (int e = 0; e < 16; ++e) acc[i][j][e] = not_finite(acc[i][j][e]) ? sum[e] : acc[i][j][e];
                }
            }
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int m = m0 + wm + 32 * i + 8 * (e / 4) + 4 * fh + e % 4;
                float g = acc[i][0][e], u = acc[i][1][e];
                if constexpr (OUT == SPLIT_CLAMPED) {
                    g = fminf(g + b_gate, limit), u = fminf(fmaxf(u + b_up, -limit), limit);
                    g = g / (1.0f + expf(-1.702f * g)) * (u + 1.0f);
                } else {
                    g = g / (1.0f + expf(-g)) * u;
                }
                if (m < M && n < N) C[m * ldc + n] = g;
            }
        }
        return;
    }
    uint32_t again = 0;  // the tiles with a result that is not finite, the same in all lanes
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            bool odd = false;
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int m = m0 + wm + 32 * i + 8 * (e / 4) + 4 * fh + e % 4, n = n0 + wn + 32 * j + fr;
                const float v = acc[i][j][e];
                odd |= not_finite(v);
                if (m < M && n < N) C[m * ldc + n] = v;
            }
            if (__any(odd)) again |= 1u << (i * TN + j);
        }
    // An infinity has no parts (inf - inf is no number), and numbers within 2^-9 of the largest one round to infinity: such a tile
    // is made again with the float32 instruction, straight from memory.  (A request whose rows are no numbers any more has this
    // in every product of every layer, beside requests that are in order.  2048 x 24576 x 4096, 1.8 ms: with one such row 2.9,
    // with 64 of them 3.7, 72 with a loop over K for every element; with all 2048 rows 8.3.)
    while (again) {
        const int t = __builtin_ctz(again), i = t / TN, j = t % TN;
        again &= again - 1;
        const sf32x16 sum = plain_sums(A + (int64_t)min(m0 + wm + 32 * i + fr, M - 1) * lda, B + (int64_t)min(n0 + wn + 32 * j + fr, N - 1) * ldb);
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const int m = m0 + wm + 32 * i + 8 * (e / 4) + 4 * fh + e % 4, n = n0 + wn + 32 * j + fr;
            if (m >= M || n >= N) continue;
            float* at = C + m * ldc + n;  // (what is finite stays: a row's bits do not depend on its neighbours)
            if (not_finite(*at)) *at = sum[e];
        }
    }
}

template <int OUT, int TM, int TN, int PER_SIMD>
static int launch_split(const float* A, const float* B, float* C, int M, int N, int K, int64_t lda, int64_t ldb, int64_t ldc,
                        int slices, hipStream_t stream, const float* bias = nullptr, float limit = 0.f) {
    constexpr int lds = 3 * 64 * (TM + TN) * SG_BK * 2, columns = OUT == SPLIT_PLAIN ? 64 * TN : 32 * TN;
    const int m_tiles = (M + 64 * TM - 1) / (64 * TM), n_tiles = (N + columns - 1) / columns;
    static std::atomic<uint64_t> granted{0};
    const hipError_t e = lle_grant_lds((const void*)gemm_nt_split_kernel<OUT, TM, TN, PER_SIMD>, lds, granted);
    if (e != hipSuccess) return (int)e;
    const int64_t blocks = (int64_t)8 * m_tiles * ((n_tiles + 7) / 8);
    if (blocks > 0x7fffffff) return (int)hipErrorInvalidValue;
    const int steps = (K + SG_BK - 1) / SG_BK, slice = (steps + slices - 1) / slices * SG_BK;
    gemm_nt_split_kernel<OUT, TM, TN, PER_SIMD><<<dim3((int)blocks, slices), 256, lds, stream>>>(A, B, C, M, N, K, lda, ldb, ldc, m_tiles,
                                                                                              n_tiles, slice, bias, limit);
    LLE_RETURN_LAUNCH_STATUS();
}

// The tiles, and what a step of one costs (us): alone on a CU, and each of several that share one.  Large tiles read less and
// lose where they leave CUs without work; measured over M from 66 to 2048 (see choose).
struct SplitTile {
    int tm, tn;
    float alone, shared;
};
static const SplitTile split_tiles[4] = {{4, 2, 2.70f, 2.35f}, {2, 2, 1.63f, 1.28f}, {2, 1, 1.09f, 0.74f}, {1, 1, 0.70f, 0.43f}};

static int units_of_device() {
    static int units[64] = {0};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
    if (units[dev] == 0 && hipDeviceGetAttribute(&units[dev], hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) units[dev] = 256;
    return units[dev];
}

// The tiles, and the slices of K (up to `most`), that take the least time by the steps of the CU with the most tiles, plus the
// way of the slices' sums to their reader and back at 5 TB/s.
static void choose(int M, int N, int K, int most, int& tiles, int& slices) {
    const int units = units_of_device(), steps = (K + SG_BK - 1) / SG_BK;
    float best = 0.f;
    tiles = 0, slices = 1;
    for (int s = 1; s <= most; ++s)
        for (int t = 0; t < 4; ++t) {
            const SplitTile& v = split_tiles[t];
            const int64_t count = (int64_t)((M + 64 * v.tm - 1) / (64 * v.tm)) * ((N + 64 * v.tn - 1) / (64 * v.tn)) * s;
            const float each = fmaxf(v.alone, (float)((count + units - 1) / units) * v.shared);
            const float us = (float)((steps + s - 1) / s) * each + (s > 1 ? (float)s * M * N * 8 / 5e6f : 0.f);
            if (best == 0.f || us < best) best = us, tiles = t, slices = s;
        }
}

// In how many slices of K (up to 8) a product is taken whose reader adds up partial sums; 1: whole.  Of the weight's sizes
// alone, so that a row's sums are the same whatever else is in the step: the best for SLICES_ROWS rows, half a default
// portion.  By the times above, against the best for each number of rows: 0 to 8 % more at 1000 to 2048 rows (4096 x 12288 at
// 2048 956 against 929 us), up to 18 % at 4096, and up to 14 us more at 65 to 512 (2048 x 2048 at 65 rows 23 against 9).
#define SLICES_ROWS 1024
extern "C" int lle_gemm_nt_f32_slices(int N, int K) {
    int tiles, slices;
    if (N <= 0 || K <= 0) return 1;
    choose(SLICES_ROWS, N, K, 8, tiles, slices);
    return slices;
}

// float32 in, float32 out; K, lda and ldb multiples of 4.  slices > 1: C is [slices][M][N], contiguous, the sums of equal parts
// of K (rounded up to whole steps).  tiles: which of split_tiles, below zero for the one that takes the least time.
extern "C" int lle_gemm_nt_f32(const void* A, const void* B, void* C, int M, int N, int K, int64_t lda, int64_t ldb, int64_t ldc,
                               int slices, int tiles, hipStream_t stream) {
    if (M <= 0 || N <= 0) return 0;
    if (K <= 0 || K % 4 != 0 || lda % 4 != 0 || ldb % 4 != 0 || slices < 1 || slices > 65535) return (int)hipErrorInvalidValue;
    if (slices > 1 && ldc != N) return (int)hipErrorInvalidValue;
    if (tiles < 0) {
        int unused;
        // (a slice's product is as long as a whole one of its part of K)
        choose(M, N * slices, (K + slices - 1) / slices, 1, tiles, unused);
    }
    const float *a = (const float*)A, *b = (const float*)B;
    float* c = (float*)C;
    switch (tiles) {
        case 0: return launch_split<SPLIT_PLAIN, 4, 2, 2>(a, b, c, M, N, K, lda, ldb, ldc, slices, stream);
        case 1: return launch_split<SPLIT_PLAIN, 2, 2, 3>(a, b, c, M, N, K, lda, ldb, ldc, slices, stream);
        case 2: return launch_split<SPLIT_PLAIN, 2, 1, 4>(a, b, c, M, N, K, lda, ldb, ldc, slices, stream);
        case 3: return launch_split<SPLIT_PLAIN, 1, 1, 6>(a, b, c, M, N, K, lda, ldb, ldc, slices, stream);
        default: return (int)hipErrorInvalidValue;
    }
}

// In which tiles (0 or 1 of split_tiles, and one) gate and up, N rows of B together, are taken with their activation, or 0 where the product
// and a pass for the activation, which may take the other tiles, are expected to be faster: by the times above, 4 us for the launch,
// and the pass' bytes and half of the product's result at 4.8 TB/s; and where the tiles are one for a CU at most, whose long end nothing covers
// then.  In a HIP graph, product and pass -> one launch (us; where it is not taken: / one launch):
//   24576 x 4096 at 262 / 512 / 1024 / 2048 rows 431 / 449, 525 -> 508, 1070 -> 959, 1830 -> 1774; 16384 x 2048 at 300 / 512 / 2048 rows 147 / 143,
//   178 -> 167, 629 -> 602; 6144 x 1024 at 512 / 1024 / 2048 rows 52 / 60, 85 -> 75, 145 -> 130; 8192 x 1024 at 400 / 700 / 2048 rows 57 / 62,
//   85 -> 75, 177 -> 159; 51200 x 5120 at 100 / 262 / 700 rows 382 -> 383, 994 -> 959, 2088 -> 1977
extern "C" int lle_gemm_nt_gated_f32_tiles(int M, int N, int K) {
    if (M <= 0 || N <= 0 || N % 2 != 0 || K <= 0 || K % 4 != 0) return 0;
    const int units = units_of_device(), steps = (K + SG_BK - 1) / SG_BK;
    const float pass = 4.f + (float)M * N * 8 / 4.8e6f;
    float best = 0.f;
    int choice = 0;
    for (int t = 0; t < 4; ++t) {
        const SplitTile& v = split_tiles[t];
        const int64_t count = (int64_t)((M + 64 * v.tm - 1) / (64 * v.tm)) * ((N + 64 * v.tn - 1) / (64 * v.tn));
        const bool in_one = t < 2 && count > units;
        const float us = (float)steps * fmaxf(v.alone, (float)((count + units - 1) / units) * v.shared) + (in_one ? 0.f : pass);
        if (t == 0 || us < best) best = us, choice = in_one ? t + 1 : 0;
    }
    return choice;
}

// A [M, K], B [N, K] (gate rows, then up rows), C [M, N / 2], contiguous; N even, K a multiple of 4.  gated 1: silu(gate) . up; gated 2: with bias
// [N] (or null) and limit, g = min(gate + b, limit), u = clamp(up + b, -limit, limit), C = g sigmoid(1.702 g) (u + 1).  tiles: 0 or 1.
extern "C" int lle_gemm_nt_gated_f32(const void* A, const void* B, const void* bias, float limit, void* C, int M, int N, int K, int gated,
                                     int tiles, hipStream_t stream) {
    if (M <= 0 || N <= 0) return 0;
    if (K <= 0 || K % 4 != 0 || N % 2 != 0 || (tiles != 0 && tiles != 1)) return (int)hipErrorInvalidValue;
    const float *a = (const float*)A, *b = (const float*)B;
    float* c = (float*)C;
    const int half = N / 2;
    if (gated == SPLIT_SILU)
        return tiles == 0 ? launch_split<SPLIT_SILU, 4, 2, 2>(a, b, c, M, half, K, K, K, half, 1, stream)
                          : launch_split<SPLIT_SILU, 2, 2, 3>(a, b, c, M, half, K, K, K, half, 1, stream);
    if (gated != SPLIT_CLAMPED || !(limit > 0.f)) return (int)hipErrorInvalidValue;
    return tiles == 0 ? launch_split<SPLIT_CLAMPED, 4, 2, 2>(a, b, c, M, half, K, K, K, half, 1, stream, (const float*)bias, limit)
                      : launch_split<SPLIT_CLAMPED, 2, 2, 3>(a, b, c, M, half, K, K, K, half, 1, stream, (const float*)bias, limit);
}

// ---------------------------------------------------------------------------------
// Up to 64 rows of A against a weight with few rows per CU, whose reader adds up partial sums (o_proj, down_proj): the product
// in slices of K.  What bounds it is what a CU takes in, of A as much as of B: with sixteen rows of B and all of K a workgroup
// reads M / 16 times as many bytes of A as of B.  So a workgroup takes 64 rows of B and a slice of K: four wavefronts (one for
// every 16 rows) read the same pieces of A, which the CU's vector cache hands out; four such groups take every fourth step of
// 32 columns; their sums meet in LDS.  Two sets of operands: the next is on its way while one is multiplied (float32 matrix
// instruction).  (Rows of whole lines go by way of LDS, below.)  Against all of K in one workgroup: 1024 x 3072 at 32 rows 15.4 -> 7.6 us, at 1 row 7.6 -> 4.8;
// 4096 x 12288 at 8 rows 52.0 -> 43.0, at 32 rows 84.6 -> 68.5; 4096 x 4096 at 8 rows 18.7 -> 16.1.
// ---------------------------------------------------------------------------------
#define FS_ROWS 64
#define FS_KW 4      // groups of wavefronts that share a slice
#define FS_STEP 32   // columns of a step: 128 bytes of a row
template <int MT>
__global__ __launch_bounds__(16 * LLE_WAVE) void gemm_slices_f32_kernel(const float* __restrict__ A, const float* __restrict__ B,
                                                                        float* __restrict__ out, int M, int N, int K, int slice_steps) {
    constexpr int U = MT <= 2 ? 2 : 1;  // steps of a set
    __shared__ float red[16][MT][16][17];
    const int wave = threadIdx.x / LLE_WAVE, lane = threadIdx.x % LLE_WAVE;
    const int c = lane / 16, r16 = lane % 16;
    const int tile = wave % 4, kw = wave / 4;
    const int n0 = blockIdx.x * FS_ROWS + 16 * tile;
    const int first = blockIdx.y * slice_steps, last = min((K + FS_STEP - 1) / FS_STEP, first + slice_steps);
    const float* bp = B + (int64_t)min(n0 + r16, N - 1) * K;
    const float* ap[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) ap[mt] = A + (int64_t)min(16 * mt + r16, M - 1) * K;
    struct Set {
        sf32x4 b[U][2], a[U][MT][2];
    };
    auto load = [&](Set& s, int step) {  // (past the slice: its last step again)
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k0 = min(step + u * FS_KW, last - 1) * FS_STEP + 8 * c;
            const int ka = min(k0, K - 4), kb = min(k0 + 4, K - 4);
            s.b[u][0] = *(const sf32x4*)(bp + ka), s.b[u][1] = *(const sf32x4*)(bp + kb);
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) s.a[u][mt][0] = *(const sf32x4*)(ap[mt] + ka), s.a[u][mt][1] = *(const sf32x4*)(ap[mt] + kb);
        }
    };
    sf32x4 acc[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[mt] = sf32x4{0.f, 0.f, 0.f, 0.f};
    auto multiply = [&](Set& s, int step) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int st = step + u * FS_KW;
            if (st >= last) continue;
            if ((st + 1) * FS_STEP > K) {  // past the end of the rows: zeros
                const sf32x4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int h = 0; h < 2; ++h)
                    if (st * FS_STEP + 8 * c + 4 * h >= K) {
                        s.b[u][h] = zero;
#pragma unroll
                        for (int mt = 0; mt < MT; ++mt) s.a[u][mt][h] = zero;
                    }
            }
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int mt = 0; mt < MT; ++mt)
                        acc[mt] = __builtin_amdgcn_mfma_f32_16x16x4f32(s.b[u][h][e], s.a[u][mt][h][e], acc[mt], 0, 0, 0);
        }
    };
    constexpr int STRIDE = U * FS_KW;
    Set s0, s1;
    int step = first + kw;
    load(s0, step);
    for (; step + 2 * STRIDE < last; step += 2 * STRIDE) {
        load(s1, step + STRIDE);
        multiply(s0, step);
        load(s0, step + 2 * STRIDE);
        multiply(s1, step + STRIDE);
    }
    if (step + STRIDE < last) {
        load(s1, step + STRIDE);
        multiply(s0, step);
        multiply(s1, step + STRIDE);
    } else {
        multiply(s0, step);
    }
    // lane holds C^T[n = 4 c + i][m = r16]
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int i = 0; i < 4; ++i) red[wave][mt][4 * c + i][r16] = acc[mt][i];
    __syncthreads();
    float* dst = out + (int64_t)blockIdx.y * M * N;
    for (int idx = threadIdx.x; idx < MT * 16 * FS_ROWS; idx += 16 * LLE_WAVE) {
        const int n = idx % FS_ROWS, m = idx / FS_ROWS;  // consecutive threads: consecutive columns
        const int col = blockIdx.x * FS_ROWS + n;
        if (m >= M || col >= N) continue;
        float sum = 0.f;
#pragma unroll
        for (int g = 0; g < FS_KW; ++g) sum += red[4 * g + n / 16][m / 16][n % 16][m % 16];
        dst[(int64_t)m * N + col] = sum;
    }
}

// The same by way of LDS where rows are whole lines of 128 bytes (K a multiple of 32): the same products and sums in the same order, bit
// for bit.  Loads of operands as the matrix instruction wants them touch sixteen lines for half of each, four cycles of the CU's
// vector cache for every one of them; here a load brings eight whole lines straight into LDS.
// From 17 rows on where a slice is long the rows of X that four wavefronts share come once (gemm_slices_lines_f32_kernel: a stage is a
// step for each of the FS_KW groups, a barrier a stage, as many stages as LDS holds).  Up to 16 rows, and up to 32 in short
// slices, every wavefront brings what it multiplies itself and waits for nobody (gemm_slices_own_f32_kernel): X comes four times, but
// in stages 4096 x 12288 takes 44.9 us at 8 rows against 40.3, 1024 x 2048 in ten slices 6.4 at 32 rows against 5.5 (in long
// slices at 32 rows 48.2 against 53.6).
// In a HIP graph at 1 / 8 / 16 / 32 / 64 rows, operand-shaped -> so (us): 1024 x 2048 4.4 / 5.1 / 5.7 / 7.6 / 10.9 -> 3.9 / 4.1 / 4.4 / 5.5 / 8.1;
// 1024 x 3072 4.8 / 5.4 / 6.3 / 8.1 / 10.9 -> 4.6 / 4.7 / 4.9 / 5.8 / 8.6; 4096 x 4096 15.7 / 16.9 / 19.1 / 25.3 / 41.2 -> 15.1 / 15.3 / 15.9 / 18.5 /
// 24.4; 4096 x 12288 40.5 / 47.0 / 52.8 / 71.0 / 117 -> 39.3 / 40.3 (5.0 TB/s) / 43.0 / 47.4 / 68.3; 5120 x 25600 97 / 114 / 136 / 185 / 313 -> 93 / 94 /
// 104 / 108 / 157.
// LDS of a stage: [step][8 groups of 8 rows of B, then 2 MT groups of X][1 KB]; where piece p of row r lies: p ^ swizzle
#define FS_SWIZZLE(r) ((((r) >> 1) & 7) ^ (((((r) >> 3) ^ ((r) >> 2)) & 1) << 1))
template <int MT, int STAGES>
__global__ __launch_bounds__(16 * LLE_WAVE) void gemm_slices_lines_f32_kernel(const float* __restrict__ A, const float* __restrict__ B,
                                                                              float* __restrict__ out, int M, int N, int K, int slice_steps) {
    constexpr int GROUPS = 8 + 2 * MT, STEP = GROUPS * 1024, STAGE = FS_KW * STEP;
    constexpr int XL = (FS_KW * 2 * MT + 15) / 16, LOADS = 2 + XL;  // a wavefront's loads of a stage: two of B, and of X
    static_assert(STAGES * STAGE <= 160 * 1024 && 16 * MT * 16 * 17 * 4 <= STAGES * STAGE, "the LDS of a CU, and the sums in its place");
    extern __shared__ __attribute__((aligned(16))) unsigned char fs_lds[];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / LLE_WAVE), lane = threadIdx.x % LLE_WAVE;
    const int c = lane / 16, r16 = lane % 16;
    const int tile = wave % 4, kw = wave / 4;
    const int n0 = blockIdx.x * FS_ROWS;
    const int first = blockIdx.y * slice_steps, last = min(K / FS_STEP, first + slice_steps);
    // the wavefront's loads: the 16 rows of B that it multiplies, at its own step; group g of X's of the stage, at step g / (2 MT)
    unsigned offset[LOADS], at[LOADS];
    int step_of[LOADS];
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
        const int g = i < 2 ? 0 : (wave + 16 * (i - 2)) % (FS_KW * 2 * MT), u = i < 2 ? kw : g / (2 * MT);
        const int r = i < 2 ? 16 * tile + 8 * i + lane / 8 : 8 * (g % (2 * MT)) + lane / 8;
        const int row = i < 2 ? min(r, N - 1 - n0) : min(r, M - 1);
        offset[i] = (unsigned)row * (unsigned)(K * 4) + ((lane % 8) ^ FS_SWIZZLE(r % 16)) * 16;
        at[i] = u * STEP + (i < 2 ? 2 * tile + i : 8 + g % (2 * MT)) * 1024;
        step_of[i] = u;
    }
    const float* b = B + (int64_t)n0 * K;
    const unsigned lds_base = (unsigned)(size_t)(__attribute__((address_space(3))) void*)fs_lds;
    auto issue = [&](int step, int buf) {  // (past the slice: its last step again)
#pragma unroll
        for (int i = 0; i < LOADS; ++i)
            load_into_lds(lds_base + buf * STAGE + at[i], offset[i], (i < 2 ? b : A) + min(step + step_of[i], last - 1) * FS_STEP);
    };
    const int at0 = r16 * 128 + ((2 * c) ^ FS_SWIZZLE(r16)) * 16, at1 = r16 * 128 + ((2 * c + 1) ^ FS_SWIZZLE(r16)) * 16;
    sf32x4 acc[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[mt] = sf32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < STAGES - 1; ++s)
        if (first + s * FS_KW < last) issue(first + s * FS_KW, s);
    int buf = 0;
    for (int step = first; step < last; step += FS_KW) {
        // this stage has landed for every wavefront, and nobody reads the buffer any more that the next load takes
        if (step + (STAGES - 2) * FS_KW < last)
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((STAGES - 2) * LOADS) : "memory");
        else
            asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (step + (STAGES - 1) * FS_KW < last) issue(step + (STAGES - 1) * FS_KW, buf == 0 ? STAGES - 1 : buf - 1);
        if (step + kw < last) {
            const unsigned char* from = fs_lds + buf * STAGE + kw * STEP;
            const sf32x4 b0 = *(const sf32x4*)(from + 2 * tile * 1024 + at0), b1 = *(const sf32x4*)(from + 2 * tile * 1024 + at1);
            sf32x4 a0[MT], a1[MT];
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) a0[mt] = *(const sf32x4*)(from + (8 + 2 * mt) * 1024 + at0), a1[mt] = *(const sf32x4*)(from + (8 + 2 * mt) * 1024 + at1);
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int mt = 0; mt < MT; ++mt)
                        acc[mt] = __builtin_amdgcn_mfma_f32_16x16x4f32(h ? b1[e] : b0[e], h ? a1[mt][e] : a0[mt][e], acc[mt], 0, 0, 0);
        }
        buf = buf == STAGES - 1 ? 0 : buf + 1;
    }
    __syncthreads();  // the sums take the operands' place
    // lane holds C^T[n = 4 c + i][m = r16]
    float* red = (float*)fs_lds;  // [16 wavefronts][MT][16 n][17]
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int i = 0; i < 4; ++i) red[((wave * MT + mt) * 16 + 4 * c + i) * 17 + r16] = acc[mt][i];
    __syncthreads();
    float* dst = out + (int64_t)blockIdx.y * M * N;
    for (int idx = threadIdx.x; idx < MT * 16 * FS_ROWS; idx += 16 * LLE_WAVE) {
        const int n = idx % FS_ROWS, m = idx / FS_ROWS;  // consecutive threads: consecutive columns
        const int col = n0 + n;
        if (m >= M || col >= N) continue;
        float sum = 0.f;
#pragma unroll
        for (int g = 0; g < FS_KW; ++g) sum += red[(((4 * g + n / 16) * MT + m / 16) * 16 + n % 16) * 17 + m % 16];
        dst[(int64_t)m * N + col] = sum;
    }
}

// Up to 16 rows, and up to 32 in short slices: a wavefront brings its rows of B and X (8 XH of them) itself, into LDS of its own, DEPTH steps ahead, and waits for
// its own loads alone, without a barrier.
template <int XH>
__global__ __launch_bounds__(16 * LLE_WAVE) void gemm_slices_own_f32_kernel(const float* __restrict__ A, const float* __restrict__ B,
                                                                            float* __restrict__ out, int M, int N, int K, int slice_steps) {
    constexpr int MT = (XH + 1) / 2, LOADS = 2 + XH, STEP = LOADS * 1024, DEPTH = 10 / LOADS, OWN = DEPTH * STEP;
    extern __shared__ __attribute__((aligned(16))) unsigned char fs_lds[];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / LLE_WAVE), lane = threadIdx.x % LLE_WAVE;
    const int c = lane / 16, r16 = lane % 16;
    const int tile = wave % 4, kw = wave / 4;
    const int n0 = blockIdx.x * FS_ROWS;
    const int first = blockIdx.y * slice_steps + kw, last = min(K / FS_STEP, (int)(blockIdx.y + 1) * slice_steps);
    const int steps = (last - first + FS_KW - 1) / FS_KW;  // of this wavefront (none: zero or less)
    unsigned offset[LOADS];
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
        const int r = (i < 2 ? 16 * tile + 8 * i : 8 * (i - 2)) + lane / 8;
        offset[i] = (unsigned)min(r, i < 2 ? N - 1 - n0 : M - 1) * (unsigned)(K * 4) + ((lane % 8) ^ FS_SWIZZLE(r % 16)) * 16;
    }
    const float *b = B + (int64_t)n0 * K + first * FS_STEP, *a = A + first * FS_STEP;
    const unsigned own_at = (unsigned)(size_t)(__attribute__((address_space(3))) void*)fs_lds + wave * OWN;
    const unsigned char* own = fs_lds + wave * OWN;
    auto issue = [&](int step, int buf) {
#pragma unroll
        for (int i = 0; i < LOADS; ++i) load_into_lds(own_at + buf * STEP + i * 1024, offset[i], (i < 2 ? b : a) + step * (FS_KW * FS_STEP));
    };
#pragma unroll
    for (int d = 0; d < DEPTH; ++d)
        if (d < steps) issue(d, d);
    const int xr = XH == 1 ? r16 % 8 : r16;  // (of eight rows: each twice)
    int b_at[2], a_at[2];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
        b_at[e] = r16 * 128 + ((2 * c + e) ^ FS_SWIZZLE(r16)) * 16;
        a_at[e] = 2048 + xr * 128 + ((2 * c + e) ^ FS_SWIZZLE(xr)) * 16;
    }
    sf32x4 acc[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[mt] = sf32x4{0.f, 0.f, 0.f, 0.f};
    int buf = 0;
    for (int step = 0; step < steps; ++step) {
        if (step + DEPTH <= steps)
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"((DEPTH - 1) * LOADS) : "memory");
        else
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        sf32x4 bv[2], av[MT][2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            bv[e] = *(const sf32x4*)(own + buf * STEP + b_at[e]);
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) av[mt][e] = *(const sf32x4*)(own + buf * STEP + mt * 2048 + a_at[e]);
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the buffer has been read
        if (step + DEPTH < steps) issue(step + DEPTH, buf);
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) acc[mt] = __builtin_amdgcn_mfma_f32_16x16x4f32(bv[h][e], av[mt][h][e], acc[mt], 0, 0, 0);
        buf = buf == DEPTH - 1 ? 0 : buf + 1;
    }
    // lane holds C^T[n = 4 c + i][m = r16]; a wavefront's sums take the place of its operands
    float* mine = (float*)(fs_lds + wave * OWN);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int i = 0; i < 4; ++i) mine[(mt * 16 + 4 * c + i) * 17 + r16] = acc[mt][i];
    __syncthreads();
    float* dst = out + (int64_t)blockIdx.y * M * N;
    const int n = threadIdx.x % FS_ROWS, col = n0 + n;  // consecutive threads: consecutive columns
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
        const int m16 = threadIdx.x / FS_ROWS, m = 16 * mt + m16;
        if (m >= M || col >= N) return;
        float sum = 0.f;
#pragma unroll
        for (int g = 0; g < FS_KW; ++g) sum += *(const float*)(fs_lds + (4 * g + n / 16) * OWN + ((mt * 16 + n % 16) * 17 + m16) * 4);
        dst[(int64_t)m * N + col] = sum;
    }
}

template <int XH>
static int launch_slices_own(const float* A, const float* B, float* out, int M, int N, int K, int each, dim3 grid, hipStream_t stream) {
    constexpr int LDS = 16 * (10 / (2 + XH)) * (2 + XH) * 1024;
    static std::atomic<uint64_t> granted{0};
    const hipError_t e = lle_grant_lds((const void*)gemm_slices_own_f32_kernel<XH>, LDS, granted);
    if (e != hipSuccess) return (int)e;
    gemm_slices_own_f32_kernel<XH><<<grid, 16 * LLE_WAVE, LDS, stream>>>(A, B, out, M, N, K, each);
    LLE_RETURN_LAUNCH_STATUS();
}

template <int MT>
static int launch_slices_lines(const float* A, const float* B, float* out, int M, int N, int K, int each, dim3 grid, hipStream_t stream) {
    constexpr int STAGE = FS_KW * (8 + 2 * MT) * 1024, STAGES = 160 * 1024 / STAGE;
    auto kernel = gemm_slices_lines_f32_kernel<MT, STAGES>;
    static std::atomic<uint64_t> granted{0};
    const hipError_t e = lle_grant_lds((const void*)kernel, STAGES * STAGE, granted);
    if (e != hipSuccess) return (int)e;
    kernel<<<grid, 16 * LLE_WAVE, STAGES * STAGE, stream>>>(A, B, out, M, N, K, each);
    LLE_RETURN_LAUNCH_STATUS();
}

// In how many slices of K the product of up to 64 rows is taken: as many workgroups of 64 rows of B as there are CUs, six steps
// for the four wavefronts of a row group at least; 1 where the rows of B alone occupy the CUs, and where K is so short that the
// sums' way to the norm and back costs what the slices gain.  Product and norm, whole / in slices of four steps / so, at 1, 8
// and 32 rows: 512 x 512 5.4, 5.8, 7.1 / 6.7, 7.9, 10.5 us / whole; 512 x 1024 5.8, 6.6, 9.3 / 6.6, 7.5, 10.1 / whole; 1024 x 2048
// 8.3, 9.4, 14.4 / 8.4, 9.3, 12.5 / 7.8, 8.8, 11.4; 1024 x 3072 10.4, 11.3, 18.9 in 16 slices 8.4, 9.3, 12.4.
extern "C" int lle_gemm_slices_f32_count(int N, int K) {
    if (N <= 0 || K < 1536) return 1;
    const int groups = (N + FS_ROWS - 1) / FS_ROWS, steps = (K + FS_STEP - 1) / FS_STEP;
    int slices = units_of_device() / groups;
    if (slices > steps / 6) slices = steps / 6;
    if (slices < 2) return 1;
    const int each = (steps + slices - 1) / slices;
    return (steps + each - 1) / each;  // (none of them empty)
}

// float32, contiguous; out [slices][M][N]; 1 <= M <= 64, K a multiple of 4
extern "C" int lle_gemm_slices_f32(const void* A, const void* B, void* out, int M, int N, int K, int slices, hipStream_t stream) {
    if (M <= 0 || N <= 0) return 0;
    if (M > 64 || K <= 0 || K % 4 != 0 || slices < 1 || slices > 65535) return (int)hipErrorInvalidValue;
    const int steps = (K + FS_STEP - 1) / FS_STEP, each = (steps + slices - 1) / slices;
    if ((int64_t)each * (slices - 1) >= steps) return (int)hipErrorInvalidValue;  // an empty slice
    const dim3 grid((N + FS_ROWS - 1) / FS_ROWS, slices);
    const float *a = (const float*)A, *b = (const float*)B;
    float* o = (float*)out;
    // (by K and the operands' addresses, not by M; a tile's rows in 32-bit offsets)
    if (K % FS_STEP == 0 && (((uintptr_t)A | (uintptr_t)B) & 15) == 0 && (int64_t)FS_ROWS * K * 4 <= 0x7fffffff) switch ((M + 15) / 16) {
        case 1: return M <= 8 ? launch_slices_own<1>(a, b, o, M, N, K, each, grid, stream) : launch_slices_own<2>(a, b, o, M, N, K, each, grid, stream);
        case 2: return each <= 16 ? launch_slices_own<4>(a, b, o, M, N, K, each, grid, stream) : launch_slices_lines<2>(a, b, o, M, N, K, each, grid, stream);
        case 3: return launch_slices_lines<3>(a, b, o, M, N, K, each, grid, stream);
        default: return launch_slices_lines<4>(a, b, o, M, N, K, each, grid, stream);
    }
    switch ((M + 15) / 16) {
        case 1: gemm_slices_f32_kernel<1><<<grid, 16 * LLE_WAVE, 0, stream>>>(a, b, o, M, N, K, each); break;
        case 2: gemm_slices_f32_kernel<2><<<grid, 16 * LLE_WAVE, 0, stream>>>(a, b, o, M, N, K, each); break;
        case 3: gemm_slices_f32_kernel<3><<<grid, 16 * LLE_WAVE, 0, stream>>>(a, b, o, M, N, K, each); break;
        default: gemm_slices_f32_kernel<4><<<grid, 16 * LLE_WAVE, 0, stream>>>(a, b, o, M, N, K, each); break;
    }
    LLE_RETURN_LAUNCH_STATUS();
}
