// bfloat16 products X[M, K] . W[N, K]^T of 33 to 192 rows (gate and up: 256) against weights of up to 48 rows for every CU: gate and up with the activation
// between them (W holds gate rows and then up rows), and whole products.
//
// A workgroup takes all rows of X and `tile_rows` rows of W (or as many gate rows, and the up rows that go with them), so that the
// weight is one round of the CUs and no byte of it is read twice.  Stages of 64 SUB columns go from memory straight into LDS, as many
// ahead as it holds; a barrier a stage, which is why a stage of narrow tiles has more columns.  What bounds it is what a CU takes in: W from
// memory and X from L2 come through one queue in order, 30 B/ns together while W does (24576 x 4096 gated at 64 rows: 786 + 512 KB a
// CU in 43 us, 4.5 TB/s of W).
// In a HIP graph, weights from memory, the library's product (and the activation's pass) -> this kernel (us) at 64 / 128 / 192 rows:
//   24576 x 4096 gated 50.0 / 53.8 / 63.0 -> 45.3 / 49.7 / 54.5; 16384 x 2048 gated 19.9 / 23.0 / 25.3 -> 16.1 / 18.5 / 24.2; 6144 x 1024 gated 14.1 / 15.0 /
//   16.2 -> 6.2 / 8.3 / 10.5; 10240 x 5120 30.5 / 37.1 -> 27.1 / 36.1; 6144 x 4096 17.8 / 25.3 -> 16.9 / 23.8; 8768 x 2048 15.2 / 18.1 -> 12.2 / 16.0;
//   4096 x 2048 12.3 / 14.8 -> 8.7 / 12.2; 4096 x 1024 8.7 / 9.3 -> 4.5 / 6.3
// In tiles of gemm_wide, or the library's product and the pass -> this kernel at 193 / 224 / 256 rows, gated: 24576 x 4096 65.3 / 65.1 / 66.7 -> 57.5 / 60.8 / 61.9;
//   19456 x 2560 43.7 / 45.8 / 50.7 -> 37.5 / 39.3 / 42.2; 6144 x 1024 16.5 / 14.1 / 14.2 -> 11.2 / 11.9 / 12.5; at 262 rows (288 a workgroup) 70.4 -> 68.7, not built
// Whole products of more than 128 rows are the library's, and weights of more than one round (51200 x 5120 gated at 64 rows 104 -> 107).
#include "common.h"
#include "lds.h"
#include <math.h>
#include <algorithm>
#include <type_traits>

LLE_DEFINE_ERROR_STRING()

typedef bf16_t rbf16x8 __attribute__((ext_vector_type(8)));
typedef bf16_t rbf16x4 __attribute__((ext_vector_type(4)));
typedef float rf32x4 __attribute__((ext_vector_type(4)));

#define ROWS_BK 64  // columns of a part of a stage: 128 bytes of a row, eight pieces of 16 bytes
// where piece p of row r lies in its row of LDS (p ^ this): a 16-byte read serves sixteen lanes a cycle, rows with r / 4 in {0, 3} at one piece and
// the others at the next one (or the other way round); this spreads them over all banks
#define ROWS_SWIZZLE(r) ((((r) >> 1) & 7) ^ ((((r) >> 3) ^ ((r) >> 2)) & 1))

enum RowsOut { ROWS_PLAIN = 0, ROWS_SILU, ROWS_CLAMPED };

// MT tiles of 16 rows of X, dealt out to WM wavefronts, times NG tiles of 16 rows of W (gated: and of up rows) to WN; STAGES buffers of LDS,
// STAGES - 1 of them on their way.  bias [N] (or null) and limit: ROWS_CLAMPED.

template <int OUT, int MT, int WM, int NG, int WN, int SUB, int STAGES>
__global__ __launch_bounds__(WM* WN* LLE_WAVE) void gemm_rows_kernel(const bf16_t* __restrict__ X, const bf16_t* __restrict__ W,
                                                                      bf16_t* __restrict__ C, int M, int N, int K, int tile_rows,
                                                                      const bf16_t* __restrict__ bias, float limit) {
    constexpr int NT = OUT == ROWS_PLAIN ? 1 : 2, WAVES = WM * WN, MPW = MT / WM, NPW = NG / WN;
    constexpr int XG = 2 * MT, WG = 2 * NG, GROUPS = XG + NT * WG, LOADS = (GROUPS + WAVES - 1) / WAVES, PART = GROUPS * 1024, STAGE = SUB * PART;
    static_assert(MT % WM == 0 && NG % WN == 0 && GROUPS >= WAVES, "whole tiles for every wavefront, and a load");
    extern __shared__ __attribute__((aligned(16))) unsigned char rows_lds[];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / LLE_WAVE), lane = threadIdx.x % LLE_WAVE;
    const int rows = N / NT, n0 = blockIdx.x * tile_rows, steps = K / (SUB * ROWS_BK);
    // a load brings eight rows of 128 bytes; lane -> row lane / 8, physical piece lane % 8, the logical piece that belongs there (rows
    // behind the last read it again and are dropped)
    const bf16_t* base[LOADS];
    unsigned offset[LOADS];
    int group[LOADS];
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
        int g = wave + WAVES * i;
        if (g >= GROUPS) g -= WAVES;  // (every wavefront has as many loads on their way: some bring a group twice)
        group[i] = g;
        const bool x = g < XG, up = NT == 2 && g >= XG + WG;
        const int r = 8 * (x ? g : up ? g - XG - WG : g - XG) + lane / 8;
        const int row = x ? min(r, M - 1) : min(min(r, tile_rows - 1), rows - 1 - n0);
        base[i] = x ? X : W + (int64_t)(n0 + (up ? rows : 0)) * K;
        offset[i] = (unsigned)row * (unsigned)(K * 2) + ((lane % 8) ^ ROWS_SWIZZLE(r % 16)) * 16;
    }
    const unsigned lds_base = (unsigned)(size_t)(__attribute__((address_space(3))) void*)rows_lds;
    auto issue = [&](int step, int buf) {
#pragma unroll
        for (int u = 0; u < SUB; ++u)
#pragma unroll
            for (int i = 0; i < LOADS; ++i)
                load_into_lds(lds_base + buf * STAGE + u * PART + group[i] * 1024, offset[i], base[i] + (step * SUB + u) * ROWS_BK);
    };
    const int wm = wave / WN, wn = wave % WN, c = lane / 16, r16 = lane % 16;
    const int at0 = r16 * 128 + (c ^ ROWS_SWIZZLE(r16)) * 16;
    rf32x4 acc[NT][NPW][MPW];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int j = 0; j < NPW; ++j)
#pragma unroll
            for (int i = 0; i < MPW; ++i) acc[t][j][i] = rf32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < STAGES - 1; ++s)
        if (s < steps) issue(s, s);
    int buf = 0;
    for (int step = 0; step < steps; ++step) {
        // this stage has landed (what was asked for behind it may stay on its way), for every wavefront; and nobody reads the buffer of
        // the stage before any more, which the next load takes
        if (step + STAGES - 1 <= steps)
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((STAGES - 2) * SUB * LOADS) : "memory");
        else
            asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (step + STAGES - 1 < steps) issue(step + STAGES - 1, buf == 0 ? STAGES - 1 : buf - 1);
#pragma unroll
        for (int u = 0; u < SUB; ++u) {
        const unsigned char* at = rows_lds + buf * STAGE + u * PART;
        rbf16x8 x[2][MPW], w[2][NT][NPW];
#pragma unroll
        for (int k = 0; k < 2; ++k) {
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int j = 0; j < NPW; ++j) w[k][t][j] = *(const rbf16x8*)(at + (XG + t * WG + 2 * (wn * NPW + j)) * 1024 + (at0 ^ (64 * k)));
#pragma unroll
            for (int i = 0; i < MPW; ++i) x[k][i] = *(const rbf16x8*)(at + 2 * (wm * MPW + i) * 1024 + (at0 ^ (64 * k)));
        }
#pragma unroll
        for (int k = 0; k < 2; ++k)
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int j = 0; j < NPW; ++j)
#pragma unroll
                    for (int i = 0; i < MPW; ++i) acc[t][j][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[k][t][j], x[k][i], acc[t][j][i], 0, 0, 0);
        }
        asm volatile("" ::: "memory");
        buf = buf == STAGES - 1 ? 0 : buf + 1;
    }
    // a lane holds four neighbouring columns (4 c ..) of row r16 of every 16 x 16 tile
#pragma unroll
    for (int j = 0; j < NPW; ++j)
#pragma unroll
        for (int i = 0; i < MPW; ++i) {
            const int m = 16 * (wm * MPW + i) + r16, in_tile = 16 * (wn * NPW + j) + 4 * c, n = n0 + in_tile;
            if (m >= M || in_tile >= tile_rows || n >= rows) continue;
            rf32x4 v = acc[0][j][i], u = acc[NT - 1][j][i];
            rbf16x4 out;
            if (OUT == ROWS_CLAMPED && bias) {
                const rbf16x4 bg = *(const rbf16x4*)(bias + n), bu = *(const rbf16x4*)(bias + rows + n);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    v[e] += (float)bg[e];
                    u[e] += (float)bu[e];
                }
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if constexpr (OUT == ROWS_CLAMPED) {
                    const float g = fminf(v[e], limit), w = fminf(fmaxf(u[e], -limit), limit);
                    out[e] = (bf16_t)(g / (1.0f + expf(-1.702f * g)) * (w + 1.0f));
                } else if constexpr (OUT == ROWS_SILU) {
                    out[e] = (bf16_t)(v[e] / (1.0f + expf(-v[e])) * u[e]);
                } else {
                    out[e] = (bf16_t)v[e];
                }
            }
            *(rbf16x4*)(C + (int64_t)m * rows + n) = out;
        }
}

template <int OUT, int MT, int WM, int NG, int WN, int SUB>
static int launch_rows(const void* X, const void* W, const void* bias, float limit, void* C, int M, int N, int K, int tile_rows, hipStream_t stream) {
    constexpr int NT = OUT == ROWS_PLAIN ? 1 : 2, STAGE = SUB * (2 * MT + NT * 2 * NG) * 1024, MOST = 160 * 1024 / STAGE, STAGES = MOST > 8 ? 8 : MOST;
    static_assert(STAGES >= 2, "LDS");
    auto kernel = gemm_rows_kernel<OUT, MT, WM, NG, WN, SUB, STAGES>;
    static std::atomic<uint64_t> granted{0};
    const hipError_t e = lle_grant_lds((const void*)kernel, STAGES * STAGE, granted);
    if (e != hipSuccess) return (int)e;
    kernel<<<(N / NT + tile_rows - 1) / tile_rows, WM * WN * LLE_WAVE, STAGES * STAGE, stream>>>((const bf16_t*)X, (const bf16_t*)W, (bf16_t*)C, M, N, K,
                                                                                            tile_rows, (const bf16_t*)bias, limit);
    LLE_RETURN_LAUNCH_STATUS();
}

// Tiles of up to 16, 32 or 48 rows by up to 64, 128, 192 or (gated, 16 and 48) 256 of X; the shapes of the wavefronts and stages are those that took the least
// time (24576 x 4096 gated at 64 rows, tiles of 48: stages of 64 / 128 columns 46.7 / 45.0 us, at 128 rows 49.8 / 58.5; 6144 x 1024 gated at 64
// rows, tiles of 16: 64 / 128 / 256 columns 6.8 / 6.6 / 6.2).
template <int OUT>
static int launch_rows_form(const void* X, const void* W, const void* bias, float limit, void* C, int M, int N, int K, int tile_rows, hipStream_t stream) {
#define ROWS_CASE(MT, WM, NG, WN, SUB) \
    if (M <= 16 * MT && tile_rows <= 16 * NG) return launch_rows<OUT, MT, WM, NG, WN, SUB>(X, W, bias, limit, C, M, N, K, tile_rows, stream);
    ROWS_CASE(4, 4, 1, 1, 4)
    ROWS_CASE(4, 4, 2, 2, 2)
    ROWS_CASE(4, 2, 3, 3, 2)
    ROWS_CASE(8, 8, 1, 1, 2)
    ROWS_CASE(8, 4, 2, 2, 2)
    ROWS_CASE(8, 4, 3, 3, OUT == ROWS_PLAIN ? 2 : 1)
    ROWS_CASE(12, 4, 1, 1, 1)
    ROWS_CASE(12, 4, 2, 2, 1)
    ROWS_CASE(12, 4, 3, 3, 1)
    if constexpr (OUT != ROWS_PLAIN) {  // (whole products of so many rows are the library's)
        ROWS_CASE(16, 8, 1, 1, 1)
        ROWS_CASE(16, 4, 3, 3, 1)
    }
#undef ROWS_CASE
    return (int)hipErrorInvalidValue;
}

// How many rows of W a workgroup takes (gated: gate rows) where this kernel takes the product on a chip of `units` CUs, 0 where it does not: as
// many, in eights, as make the weight one round of the CUs.  Not where X, which every CU reads whole, is many times the CU's share of W, unless
// the product is short (us, library / so: 2048 x 2048 at 64 / 128 rows 8.9, 8.4 / 6.7, 9.7; 2048 x 4096 at 128 rows 12.7 / 19.5; 4096 x 8192 at 64
// rows 24.0 / 25.3; gated beyond 192 rows the wide tiles are as fast in between, 16384 x 2048 at 208 / 256 26.0, 26.4 / 26.3, 27.3, 12288 x 1536 20.1, 20.6 / 20.4,
// 21.6, 8192 x 2048 19.8, 27.6 / 20.4, 22.3; 7168 x 5120 at 64 / 96 rows 22.4, 28.7 / 24.8, 30.6; 6144 x 4096 17.8, 22.9 / 16.9, 22.5; 10240 x 5120 30.5, 34.1 / 27.1, 32.6).
extern "C" int lle_gemm_rows_tile(int M, int N, int K, int gated, int units) {
    if (M <= 32 || M > (gated ? 256 : 128) || N <= 0 || units <= 0 || K < 1024 || K % 256 != 0 || (int64_t)256 * K * 2 > 0x7fffffff) return 0;
    if (N % (gated ? 8 : 4) != 0) return 0;
    const int rows = gated ? N / 2 : N, share = (rows + units - 1) / units;
    if (share > 48 || K > std::max(M <= 64 ? 4096 : 1024, 176 * share * (gated ? 2 : 1))) return 0;
    if (M > 192 && share <= 32 && (share > 16 || K > 1024)) return 0;
    return (share + 7) / 8 * 8;
}

// X [M, K] and W [N, K] bfloat16, contiguous, 16-byte aligned; C [M, N], or gated [M, N / 2].  gated 1: silu(gate) . up; gated 2: with bias [N]
// (or null) and limit, g = min(gate + b, limit), u = clamp(up + b, -limit, limit), C = g sigmoid(1.702 g) (u + 1).  tile_rows: as above.
extern "C" int lle_gemm_rows_bf16(const void* X, const void* W, const void* bias, float limit, void* C, int M, int N, int K, int gated, int tile_rows,
                                  hipStream_t stream) {
    if (M <= 0 || N <= 0) return 0;
    if (M > (gated ? 256 : 192) || K <= 0 || K % 256 != 0 || (int64_t)256 * K * 2 > 0x7fffffff || N % (gated ? 8 : 4) != 0) return (int)hipErrorInvalidValue;
    if (tile_rows <= 0 || tile_rows > 48 || tile_rows % 4 != 0) return (int)hipErrorInvalidValue;
    if ((((uintptr_t)X | (uintptr_t)W) & 15) || (((uintptr_t)bias | (uintptr_t)C) & 7)) return (int)hipErrorInvalidValue;
    switch (gated) {
        case ROWS_PLAIN: return launch_rows_form<ROWS_PLAIN>(X, W, nullptr, 0.f, C, M, N, K, tile_rows, stream);
        case ROWS_SILU: return launch_rows_form<ROWS_SILU>(X, W, nullptr, 0.f, C, M, N, K, tile_rows, stream);
        case ROWS_CLAMPED:
            if (!(limit > 0.f)) return (int)hipErrorInvalidValue;
            return launch_rows_form<ROWS_CLAMPED>(X, W, bias, limit, C, M, N, K, tile_rows, stream);
        default: return (int)hipErrorInvalidValue;
    }
}
