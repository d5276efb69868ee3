// bfloat16 products X[M, K] . W[N, K]^T whose reader adds up partial sums (o_proj, down_proj), for more rows than the
// weight-streaming kernels take: tiles of up to 256 x 128 and slices of K, so that every CU has a tile where the whole product
// has too few.  A stage of 64 columns goes from memory straight into LDS, two to five stages ahead of the matrix
// instructions; what bounds the kernel is what a CU takes in: 35 to 50 GB/s, less the larger the tiles (fewer bytes on their
// way for one that is multiplied), or W's way from memory.  Measured with the norm that adds the sums up, against the sliced
// kernel of up to 128 rows or the library (batched over slices of K where K >= 2 N):
//   4096 x 12288:   64 rows 33.0 -> 30.2 us, 128 rows 44.3 -> 34.8
//   5120 x 25600:   32 rows 68.4 -> 55.8 us, 64 rows 80.2 -> 57.6, 128 rows 114.3 -> 69.1
//   4096 x 4096:   160 rows 33.5 -> 23.4 us, 512 rows 37.7 -> 35.5
//   1024 x 2048:   209 rows 12.9 -> 11.6 us, 1000 rows 24.1 -> 17.0
// (256 x 256 tiles: 5120 x 8192 at 400 rows 92 us against 63 in 256 x 128.)
// For whole products (gate_up, qkv) the library's tiles are as fast or faster.
#include "common.h"
#include "lds.h"
#include <math.h>

LLE_DEFINE_ERROR_STRING()

typedef bf16_t tbf16x8 __attribute__((ext_vector_type(8)));
typedef float tf32x16 __attribute__((ext_vector_type(16)));

#define BK 64  // columns of K per stage: 128 bytes of a row, eight pieces of 16 bytes
// where piece p of row r lies in its row of LDS (p ^ this): a 16-byte read serves sixteen lanes a cycle (rows 4 q .. 4 q + 3 for q in
// {0, 3, 5, 6} or {1, 2, 4, 7} of a 32-row fragment, the same piece), which this spreads over all banks
#define TILE_SWIZZLE(r) ((((r) >> 1) & 1) | ((((r) >> 3) & 3) << 1))

// WM x WN wavefronts of TM x TN matrix tiles of 32 x 32; STAGES buffers of LDS, STAGES - 1 of them on their way.
// The float32 sums of a slice of K go to C + slice * M * N.
template <int WM, int WN, int TM, int TN, int STAGES>
__global__ __launch_bounds__(WM* WN* LLE_WAVE, 2) void gemm_tile_kernel(const bf16_t* __restrict__ X, const bf16_t* __restrict__ W,
                                                                               float* __restrict__ C, int M, int N, int K, int m_tiles,
                                                                               int n_tiles, int slices, int slice_stages) {
    constexpr int WAVES = WM * WN, BM = 32 * TM * WM, BN = 32 * TN * WN;
    constexpr int PIECES = BK / 8, ROW = BK * 2;  // 16-byte pieces of a row of a stage; its bytes
    constexpr int RPL = 64 / PIECES;         // rows that one wavefront's load brings
    constexpr int GROUPS = (BM + BN) / RPL;
    constexpr int LOADS = GROUPS / WAVES;    // per wavefront and stage
    constexpr int STAGE = (BM + BN) * BK * 2;   // bytes
    static_assert(GROUPS % WAVES == 0 && BM % RPL == 0, "every wavefront loads as much");
    extern __shared__ __attribute__((aligned(16))) unsigned char gb_lds[];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / LLE_WAVE), lane = threadIdx.x % LLE_WAVE;
    // consecutive workgroups go to different dies: a die takes every eighth part of W (a column of tiles in a slice of K), all
    // its row tiles one after the other
    const int die = blockIdx.x % 8, at = blockIdx.x / 8;
    const int part = die + 8 * (at / m_tiles), mt = at % m_tiles;
    if (part >= n_tiles * slices) return;
    const int nt = part % n_tiles, slice = part / n_tiles;
    const int m0 = mt * BM, n0 = nt * BN;
    const int first = slice * slice_stages, steps = min(K / BK - first, slice_stages);
    const bf16_t* xb = X + (int64_t)m0 * K + first * BK;
    const bf16_t* wb = W + (int64_t)n0 * K + first * BK;
    // a load: eight rows of 128 bytes; lane -> row lane / 8, physical piece lane % 8, the logical piece that belongs there
    unsigned offset[LOADS];
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
        const int g = wave + WAVES * i, r = RPL * g + lane / PIECES;
        const int piece = (lane % PIECES) ^ TILE_SWIZZLE(r < BM ? r : r - BM);
        const int64_t row = g < BM / RPL ? min(r, M - 1 - m0) : min(r - BM, N - 1 - n0);
        offset[i] = (unsigned)(row * K * 2 + piece * 16);
    }
    const unsigned lds_base = (unsigned)(size_t)(__attribute__((address_space(3))) void*)gb_lds;
    auto issue = [&](int step, int buf) {
#pragma unroll
        for (int i = 0; i < LOADS; ++i) {
            const int g = wave + WAVES * i;
            const bf16_t* base = (g < BM / RPL ? xb : wb) + step * BK;
            load_into_lds(lds_base + buf * STAGE + g * 1024, offset[i], base);
        }
    };
    const int wm = wave / WN * (32 * TM), wn = wave % WN * (32 * TN);
    const int fr = lane % 32, fh = lane / 32;
    const unsigned char* af = gb_lds + (wm + fr) * ROW;
    const unsigned char* bf = gb_lds + (BM + wn + fr) * ROW;
    tf32x16 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
#pragma unroll
    for (int s = 0; s < STAGES - 1; ++s)
        if (s < steps) issue(s, s);
    int buf = 0;
    for (int step = 0; step < steps; ++step) {
        // this stage has landed (what was asked for behind it may stay on its way), for every wavefront; and nobody reads the
        // buffer of the stage before any more, which the next load takes (lgkmcnt: the reads have arrived, not only been issued)
        if (step + STAGES - 1 <= steps)
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((STAGES - 2) * LOADS) : "memory");
        else
            asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (step + STAGES - 1 < steps) issue(step + STAGES - 1, buf == 0 ? STAGES - 1 : buf - 1);
        const int at_stage = buf * STAGE;
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int s = 0; s < BK / 16; ++s) {
            const int piece = ((2 * s + fh) ^ TILE_SWIZZLE(fr)) * 16;
            tbf16x8 b[TN], a[TM];
#pragma unroll
            for (int j = 0; j < TN; ++j) b[j] = *(const tbf16x8*)(bf + at_stage + 32 * j * ROW + piece);
#pragma unroll
            for (int i = 0; i < TM; ++i) a[i] = *(const tbf16x8*)(af + at_stage + 32 * i * ROW + piece);
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
        }
        __builtin_amdgcn_s_setprio(0);
        asm volatile("" ::: "memory");
        buf = buf == STAGES - 1 ? 0 : buf + 1;
    }
    // lane holds C[m = 8 (e / 4) + 4 (lane / 32) + e % 4][n = lane % 32] of every 32 x 32 tile
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const int m = m0 + wm + 32 * i + 8 * (e / 4) + 4 * fh + e % 4;
            if (m >= M) continue;
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                const int n = n0 + wn + 32 * j + fr;
                if (n < N) C[((int64_t)slice * M + m) * N + n] = acc[i][j][e];
            }
        }
}

template <int WM, int WN, int TM, int TN, int STAGES>
static int launch_tile(const void* X, const void* W, void* C, int M, int N, int K, int slices, hipStream_t stream) {
    constexpr int BM = 32 * TM * WM, BN = 32 * TN * WN, lds = STAGES * (BM + BN) * BK * 2;
    static_assert(lds <= 160 * 1024, "the LDS of a CU");
    const int m_tiles = (M + BM - 1) / BM, n_tiles = (N + BN - 1) / BN;
    auto kernel = gemm_tile_kernel<WM, WN, TM, TN, STAGES>;
    static std::atomic<uint64_t> granted{0};
    const hipError_t e = lle_grant_lds((const void*)kernel, lds, granted);
    if (e != hipSuccess) return (int)e;
    const int64_t blocks = (int64_t)8 * m_tiles * (((int64_t)n_tiles * slices + 7) / 8);
    if (blocks > 0x7fffffff) return (int)hipErrorInvalidValue;
    kernel<<<(int)blocks, WM * WN * LLE_WAVE, lds, stream>>>((const bf16_t*)X, (const bf16_t*)W, (float*)C, M, N, K, m_tiles, n_tiles, slices,
                                                             (K / BK + slices - 1) / slices);
    LLE_RETURN_LAUNCH_STATUS();
}

// The tile shapes, and what a CU takes in of their operands (GB/s).
struct TileShape {
    int bm, bn;
    float intake;
};
static const TileShape tile_shapes[3] = {{64, 128, 50.f}, {128, 128, 44.f}, {256, 128, 37.f}};

static int units_of_device() {
    static int units[64] = {0};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
    if (units[dev] == 0 && hipDeviceGetAttribute(&units[dev], hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) units[dev] = 256;
    return units[dev];
}

// The tiles and the slices of K that take the least time: rounds of workgroups over the CUs of the die that gets most of them (a
// die has whole parts of W, see the kernel: 28 columns of tiles in 3 slices are 11 parts for four dies, 33 workgroups of 129
// rows in tiles of 64 for 32 CUs), each with a start of 3 us and its operands at the shape's rate, but not less than W's way from
// memory (5.2 TB/s into all CUs); the sums' way to their reader and back (5 TB/s), who asks for a slice after the other.
// Measured at 17 to 2048 rows of 73 weights from 512 x 1024 to 8192 x 16384, the choice is 1.6 % slower than the best of
// all tiles and slices, over 10 % in 3 of 100 (with rounds over all CUs alike 3 %, and 8 of 100).
static void choose(int M, int N, int K, int first, int last, int& tiles, int& slices) {
    constexpr int DIES = 8;
    const int units = units_of_device(), per_die = units >= DIES ? units / DIES : 1, stages = K / BK;
    const float from_memory = (float)N * K * 2 / 5.2e6f;
    float best = 0.f;
    tiles = 0, slices = first;
    for (int s = first; s <= last && s <= stages; ++s)
        for (int t = 0; t < 3; ++t) {
            const TileShape& v = tile_shapes[t];
            const int64_t m_tiles = (M + v.bm - 1) / v.bm, parts = (int64_t)((N + v.bn - 1) / v.bn) * s;
            const int64_t rounds = ((parts + DIES - 1) / DIES * m_tiles + per_die - 1) / per_die;
            const float each = (float)((stages + s - 1) / s) * (v.bm + v.bn) * BK * 2 / (v.intake * 1e3f);
            const float memory = from_memory * (float)(rounds * units) / (parts * m_tiles);  // (CUs without a tile take in nothing)
            const float us = fmaxf(rounds * (3.f + each), memory) + (float)s * M * N * 8 / 5e6f + 0.15f * s;
            if (best == 0.f || us < best) best = us, tiles = t, slices = s;
        }
}

// In how many slices of K (up to 16) the product is taken.
extern "C" int lle_gemm_tile_sums_slices(int M, int N, int K) {
    int tiles, slices;
    if (M <= 0 || N <= 0 || K <= 0) return 1;
    choose(M, N, K, 1, 16, tiles, slices);
    return slices;
}

// X [M, K] and W [N, K] bfloat16, contiguous; out float32 [slices][M][N], the sums of equal parts of K (rounded up to whole
// stages); K a multiple of 64.  tiles: which of tile_shapes, below zero for the one that takes the least time.
extern "C" int lle_gemm_tile_sums_bf16(const void* X, const void* W, void* out, int M, int N, int K, int slices, int tiles, hipStream_t stream) {
    if (M <= 0 || N <= 0) return 0;
    if (K <= 0 || K % BK != 0 || slices < 1 || slices > K / BK) return (int)hipErrorInvalidValue;
    if ((int64_t)256 * K * 2 > 0x7fffffff) return (int)hipErrorInvalidValue;  // (a tile's rows in 32-bit offsets)
    if (tiles < 0) {
        int unused;
        choose(M, N, K, slices, slices, tiles, unused);
    }
    switch (tiles) {
        case 0: return launch_tile<2, 4, 1, 1, 6>(X, W, out, M, N, K, slices, stream);
        case 1: return launch_tile<2, 4, 2, 1, 4>(X, W, out, M, N, K, slices, stream);
        case 2: return launch_tile<4, 2, 2, 2, 3>(X, W, out, M, N, K, slices, stream);
        default: return (int)hipErrorInvalidValue;
    }
}
