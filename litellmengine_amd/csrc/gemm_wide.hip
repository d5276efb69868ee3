// bfloat16 products X[M, K] . W[N, K]^T of many rows, gate and up with the activation between them (W holds gate rows and
// then up rows, the result is act(gate) . up).
//
// Tiles of 128 to 288 rows of X by 256 or 128 of W (half of them gate rows, half the up rows that go with them: a lane then holds the
// sums of both for the same places), stages of 64 columns straight into LDS, eight wavefronts in two groups of four that take
// turns: while one group multiplies, the other reads its next operands from LDS and asks for a later stage.  A stage is two such
// turns: the first half of the tile's rows, then the second.  What bounds a stage is LDS (192 KB of operands read, 64 KB
// written, against 2048 cycles of matrix instructions a SIMD), so the reads are dealt evenly to both turns: the second turn also
// reads the first half of the next stage's W, which therefore has three buffers in LDS and two in registers.  With
// all CUs at work the chip's power is the next bound: 4096 x 4096 at 4096 rows takes 96 us, of zeros 72.
// Measured (us; the library's product, with its pass for the activation where it is gated / this kernel):
//   24576 x 4096 gated, 262 / 700 / 1024 / 2048 / 2111 rows: 77 / 159 / 184 / 306 / 369 -> 69 / 128 / 166 / 275 / 322
//   51200 x 5120 gated, 512 / 1024 / 2048 / 2111 rows: 280 / 510 / 895 / 1021 -> 234 / 443 / 780 / 827
//   16384 x 2048 gated, 300 / 2048 rows: 34 / 121 -> 27 / 106; 6144 x 1024 gated, 600 / 2048 rows: 19 / 35 -> 13 / 27
// Whole products in such tiles are the library's: it does between 0.65 and 1.5 PFLOP/s, by no rule that sizes tell (these tiles
// 1.1 to 1.3), and where a model of both took the tiles, 38 of 63 measured products were slower by up to 16 %.
// Tried: all W of a stage read in the first turn, two buffers of everything (24576 x 4096 gated at 1500 rows 236 -> 222, tiles
// of 128 rows 51 -> 46 us a round); 32 x 32 matrix instructions (+10 %); a ring of all 160 KB with loads asked for half a
// stage earlier (+15 %: its bookkeeping stands between the turns).
#include "common.h"
#include "lds.h"
#include <math.h>
#include <type_traits>

LLE_DEFINE_ERROR_STRING()

typedef bf16_t wbf16x8 __attribute__((ext_vector_type(8)));
typedef bf16_t wbf16x4 __attribute__((ext_vector_type(4)));
typedef float wf32x4 __attribute__((ext_vector_type(4)));

#define WIDE_BK 64       // columns of K per stage: 128 bytes of a row, eight pieces of 16 bytes
// where piece p of row r lies in its row of LDS (p ^ this): a 16-byte read serves sixteen lanes a cycle, which are the sixteen rows of
// a fragment, those with r / 4 in {0, 3} at one piece and the others at the next one (or the other way round); this spreads
// them over all banks
#define WIDE_SWIZZLE(r) ((((r) >> 1) & 7) ^ ((((r) >> 3) ^ ((r) >> 2)) & 1))

enum WideOut { WIDE_SILU = 1, WIDE_CLAMPED };

// A tile is 32 I0 + 32 I1 rows, its two halves, by 64 J gate rows and 64 J up rows of W.  bias [N] (or null) and limit: WIDE_CLAMPED.
template <int OUT, int I0, int I1, int J>
__global__ __launch_bounds__(512, 2) void gemm_wide_kernel(const bf16_t* __restrict__ X, const bf16_t* __restrict__ W,
                                                           bf16_t* __restrict__ C, int M, int N, int K, int m_tiles, int n_tiles,
                                                           const bf16_t* __restrict__ bias, float limit) {
    constexpr int ROWS0 = 32 * I0, BM = ROWS0 + 32 * I1;
    extern __shared__ __attribute__((aligned(16))) unsigned char wide_lds[];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / LLE_WAVE), lane = threadIdx.x % LLE_WAVE;
    // Consecutive workgroups go to different dies.  A die takes an eighth of all tiles, neighbours in an order that walks bands of up
    // to eight rows of tiles column by column: what its CUs read at a time are about as many rows as columns, and no die has more
    // than its share (220 tiles in 20 columns: with whole columns for a die 33 tiles for some dies' 32 CUs).
    const int tiles = m_tiles * n_tiles, share = (tiles + 7) / 8, at = blockIdx.x / 8;
    const int id = blockIdx.x % 8 * share + at;
    if (at >= share || id >= tiles) return;
    const int bands = (m_tiles + 7) / 8, band = (m_tiles + bands - 1) / bands;
    const int b = id / (band * n_tiles), in_band = id - b * band * n_tiles;
    const int height = min(band, m_tiles - b * band), nt = in_band / height, mt = b * band + in_band - nt * height;
    const int rows = N / 2;  // of a result
    const int m0 = mt * BM, n0 = nt * (64 * J);
    const int steps = K / WIDE_BK;
    const bf16_t* xb = X + (int64_t)m0 * K;
    const bf16_t* wb0 = W + (int64_t)n0 * K;
    const bf16_t* wb1 = wb0 + (int64_t)rows * K;
    // a load brings eight rows of 128 bytes, the eight wavefronts' 64; lane -> row lane / 8, physical piece lane % 8, the logical
    // piece that belongs there (rows behind the last read it again and are dropped).  Of 32 rows that are left of a half two
    // wavefronts bring the same eight, so that all have as many loads on their way.
    constexpr int LX0 = (I0 + 1) / 2, LX1 = (I1 + 1) / 2;  // a wavefront's loads of the halves
    auto group_of = [&](int rows32, int i) { return wave + 8 * i < 4 * rows32 ? wave + 8 * i : wave + 8 * i - 4; };
    unsigned xo0[LX0], xo1[LX1], wo[J];
#pragma unroll
    for (int i = 0; i < LX0; ++i) {
        const int r = 8 * group_of(I0, i) + lane / 8;
        xo0[i] = (unsigned)min(r, M - 1 - m0) * (unsigned)(K * 2) + ((lane % 8) ^ WIDE_SWIZZLE(r % 16)) * 16;
    }
#pragma unroll
    for (int i = 0; i < LX1; ++i) {
        const int r = 8 * group_of(I1, i) + lane / 8;
        xo1[i] = (unsigned)min(ROWS0 + r, M - 1 - m0) * (unsigned)(K * 2) + ((lane % 8) ^ WIDE_SWIZZLE(r % 16)) * 16;
    }
#pragma unroll
    for (int i = 0; i < J; ++i) {
        const int r = 8 * (wave + 8 * i) + lane / 8;
        wo[i] = (unsigned)min(r, rows - 1 - n0) * (unsigned)(K * 2) + ((lane % 8) ^ WIDE_SWIZZLE(r % 16)) * 16;
    }
    // LDS: two buffers of the first half of X, of the second and of the second half of W; three of the first half of W
    constexpr int X0_BYTES = I0 * 4096, X1_BYTES = I1 * 4096, W_BYTES = J * 8192;
    constexpr int AT_X0 = 0, AT_X1 = 2 * X0_BYTES, AT_W1 = AT_X1 + 2 * X1_BYTES, AT_W0 = AT_W1 + 2 * W_BYTES;
    using Half0 = std::integral_constant<int, 0>;
    using Half1 = std::integral_constant<int, 1>;
    const unsigned lds_base = (unsigned)(size_t)(__attribute__((address_space(3))) void*)wide_lds;
    auto dma = [&](unsigned at_lds, unsigned offset, const bf16_t* base) { load_into_lds(lds_base + at_lds, offset, base); };
    auto issue_x = [&](int step, auto half) {
        constexpr int h = decltype(half)::value;
#pragma unroll
        for (int i = 0; i < (h ? LX1 : LX0); ++i)
            dma((h ? AT_X1 + (step & 1) * X1_BYTES : AT_X0 + (step & 1) * X0_BYTES) + group_of(h ? I1 : I0, i) * 1024,
                h ? xo1[i < LX1 ? i : 0] : xo0[i < LX0 ? i : 0], xb + step * WIDE_BK);
    };
    auto issue_w = [&](int step, int at_lds, auto half) {
        constexpr int h = decltype(half)::value;
#pragma unroll
        for (int i = 0; i < J; ++i) dma(at_lds + (wave + 8 * i) * 1024, wo[i], (h ? wb1 : wb0) + step * WIDE_BK);
    };
    const int group = wave / 4, wn = wave % 4;
    const int c = lane / 16, r16 = lane % 16;
    const int sw = WIDE_SWIZZLE(r16);
    const unsigned char* lane_at[2] = {wide_lds + r16 * 128 + (c ^ sw) * 16, wide_lds + r16 * 128 + ((c ^ sw) ^ 4) * 16};
    constexpr int I = I0 > I1 ? I0 : I1;
    wf32x4 acc[2][2][I][J];
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int i = 0; i < I; ++i)
#pragma unroll
                for (int j = 0; j < J; ++j) acc[a][h][i][j] = wf32x4{0.f, 0.f, 0.f, 0.f};
    wbf16x8 xf[I][2], wf0[2][J][2], wf1[J][2];
    auto read_x = [&](int buf, auto half) {
        constexpr int h = decltype(half)::value, IH = h ? I1 : I0;
#pragma unroll
        for (int i = 0; i < IH; ++i)
#pragma unroll
            for (int k = 0; k < 2; ++k)
                xf[i][k] = *(const wbf16x8*)(lane_at[k] + (h ? AT_X1 + buf * X1_BYTES : AT_X0 + buf * X0_BYTES) + (16 * IH * group + 16 * i) * 128);
    };
    auto read_w = [&](wbf16x8 (&f)[J][2], int at_lds) {
#pragma unroll
        for (int j = 0; j < J; ++j)
#pragma unroll
            for (int k = 0; k < 2; ++k) f[j][k] = *(const wbf16x8*)(lane_at[k] + at_lds + (16 * J * wn + 16 * j) * 128);
    };
    auto multiply = [&](auto half, const wbf16x8 (&w0)[J][2]) {
        constexpr int a = decltype(half)::value;
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int k = 0; k < 2; ++k)
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int j = 0; j < J; ++j)
#pragma unroll
                    for (int i = 0; i < (a ? I1 : I0); ++i)
                        acc[a][h][i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(h ? wf1[j][k] : w0[j][k], xf[i][k], acc[a][h][i][j], 0, 0, 0);
        __builtin_amdgcn_s_setprio(0);
    };
    auto barrier = [&]() {
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_barrier" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    constexpr int BEHIND = LX0 + LX1 + 2 * J;  // a wavefront's loads of a stage
    auto landed = [&](bool whole) {
        if (whole)
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(BEHIND) : "memory");
        else
            asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    };
    issue_w(0, AT_W0, Half0{});
    issue_x(0, Half0{});
    issue_w(0, AT_W1, Half1{});
    issue_x(0, Half1{});
    if (steps > 1) {
        issue_w(1, AT_W0 + W_BYTES, Half0{});
        issue_x(1, Half0{});
        issue_w(1, AT_W1 + W_BYTES, Half1{});
    }
    landed(steps > 1);
    barrier();
    read_w(wf0[0], AT_W0);
    if (group) barrier();
    int w0_read = AT_W0 + W_BYTES, w0_fill = AT_W0 + 2 * W_BYTES;  // of stages t + 1 and t + 2
    auto next_of_three = [](int at_lds) { return at_lds == AT_W0 + 2 * W_BYTES ? AT_W0 : at_lds + W_BYTES; };
    auto stage = [&](int t, auto set) {
        constexpr int cur = decltype(set)::value;
        const int buf = t & 1;
        const bool more = t + 2 < steps;
        read_x(buf, Half0{});
        read_w(wf1, AT_W1 + buf * W_BYTES);
        if (t + 1 < steps) issue_x(t + 1, Half1{});
        if (more) issue_w(t + 2, w0_fill, Half0{});
        landed(more);
        barrier();
        multiply(Half0{}, wf0[cur]);
        barrier();
        read_x(buf, Half1{});
        if (t + 1 < steps) read_w(wf0[cur ^ 1], w0_read);
        if (more) {
            issue_x(t + 2, Half0{});
            issue_w(t + 2, AT_W1 + buf * W_BYTES, Half1{});
        }
        landed(more);
        barrier();
        multiply(Half1{}, wf0[cur]);
        barrier();
        w0_read = next_of_three(w0_read);
        w0_fill = next_of_three(w0_fill);
    };
    for (int t = 0; t < steps; t += 2) {
        stage(t, Half0{});
        if (t + 1 < steps) stage(t + 1, Half1{});
    }
    if (!group) barrier();
    // a lane holds four neighbouring columns (4 c ..) of row r16 of every 16 x 16 tile
    auto put = [&](int m, int n, wf32x4 v, wf32x4 u) {  // (n: of the result's columns; u: the up rows' sums)
        if (m >= M || n >= rows) return;
        wbf16x4 out;
        if (OUT == WIDE_CLAMPED && bias) {
            const wbf16x4 bg = *(const wbf16x4*)(bias + n), bu = *(const wbf16x4*)(bias + rows + n);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                v[e] += (float)bg[e];
                u[e] += (float)bu[e];
            }
        }
        // (The hardware's exponential and reciprocal, each good to a unit in the last place of 32 bits, and the exponent's rounding, 1e-7 of
        // every unit of the gate: what follows is rounded to 16.  A reciprocal below the least normal number comes out as 0, so gates
        // below -87.3 give 0; silu_mul gives the 1e-36 that is due down to -88.7.  Adding up a quarter of the sum keeps those too; it
        // changes the last bits of everything else and measured 0.3 % slower.)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            constexpr float LOG2E = 1.44269504088896340736f;
            if constexpr (OUT == WIDE_CLAMPED) {
                const float g = fminf(v[e], limit), w = fminf(fmaxf(u[e], -limit), limit);
                out[e] = (bf16_t)(g * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(g * (-1.702f * LOG2E))) * (w + 1.0f));
            } else {
                out[e] = (bf16_t)(v[e] * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(v[e] * -LOG2E)) * u[e]);
            }
        }
        *(wbf16x4*)(C + (int64_t)m * rows + n) = out;
    };
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int i = 0; i < (a ? I1 : I0); ++i)
#pragma unroll
            for (int j = 0; j < J; ++j) {
                const int m = m0 + ROWS0 * a + 16 * (a ? I1 : I0) * group + 16 * i + r16, n = n0 + 16 * J * wn + 16 * j + 4 * c;
                put(m, n, acc[a][0][i][j], acc[a][1][i][j]);
            }
}

template <int OUT, int I0, int I1, int J>
static int launch_wide(const void* X, const void* W, const void* bias, float limit, void* C, int M, int N, int K, hipStream_t stream) {
    constexpr int BM = 32 * (I0 + I1), BN = 64 * J, LDS = 8192 * (I0 + I1) + 5 * 8192 * J;
    static_assert(LDS <= 160 * 1024, "the LDS of a CU");
    const int m_tiles = (M + BM - 1) / BM, n_tiles = (N / 2 + BN - 1) / BN;
    const int64_t blocks = ((int64_t)m_tiles * n_tiles + 7) / 8 * 8;
    if (blocks > 0x7fffffff) return (int)hipErrorInvalidValue;
    auto kernel = gemm_wide_kernel<OUT, I0, I1, J>;
    static std::atomic<uint64_t> granted{0};
    const hipError_t e = lle_grant_lds((const void*)kernel, LDS, granted);
    if (e != hipSuccess) return (int)e;
    kernel<<<(int)blocks, 512, LDS, stream>>>((const bf16_t*)X, (const bf16_t*)W, (bf16_t*)C, M, N, K, m_tiles, n_tiles,
                                                   (const bf16_t*)bias, limit);
    LLE_RETURN_LAUNCH_STATUS();
}

// The tiles (rows of X by rows of W), and what a round of one takes: a start, and for every stage of 64 columns `stage` us and
// `full` more with all CUs at work (power, and what the dies read).  Fitted to both sides' times at 129 to 2111 rows of six gated
// weights, 6144 x 1024 to 51200 x 5120, from memory: the choice is 1 % slower than the best of all eleven.
struct WideForm {
    int rows, columns;
    float start, stage, full;
};
static const WideForm wide_forms[11] = {
    {256, 256, 6.5f, 0.97f, 0.36f}, {224, 256, 6.3f, 0.96f, 0.25f}, {192, 256, 4.2f, 0.98f, 0.14f}, {160, 256, 4.1f, 0.93f, 0.07f},
    {128, 256, 3.7f, 0.79f, 0.09f}, {288, 128, 4.4f, 0.84f, 0.10f}, {256, 128, 4.6f, 0.72f, 0.13f}, {224, 128, 5.1f, 0.70f, 0.09f},
    {192, 128, 4.4f, 0.68f, 0.07f}, {160, 128, 2.8f, 0.72f, -0.13f}, {128, 128, 2.1f, 0.67f, -0.16f}};

template <int OUT>
static int launch_wide_form(const void* X, const void* W, const void* bias, float limit, void* C, int M, int N, int K, int form,
                            hipStream_t stream) {
#define WIDE_CASE(F, I0, I1, J) \
    case F: return launch_wide<OUT, I0, I1, J>(X, W, bias, limit, C, M, N, K, stream);
    switch (form) {
        WIDE_CASE(0, 4, 4, 2) WIDE_CASE(1, 4, 3, 2) WIDE_CASE(2, 3, 3, 2) WIDE_CASE(3, 3, 2, 2)
        WIDE_CASE(4, 2, 2, 2) WIDE_CASE(5, 5, 4, 1) WIDE_CASE(6, 4, 4, 1) WIDE_CASE(7, 4, 3, 1)
        WIDE_CASE(8, 3, 3, 1) WIDE_CASE(9, 3, 2, 1) WIDE_CASE(10, 2, 2, 1)
    }
#undef WIDE_CASE
    return (int)hipErrorInvalidValue;
}

// The form in which the product takes the least time (which of wide_forms, and one) on a chip of `units` CUs, or 0 where the library's
// product with the pass of its own that the activation takes is expected to be as fast: 1.0 PFLOP/s (256 CUs) or W at 6 TB/s, 9 us, and
// the activation's 4.8 TB/s; slower than the library is at its best and than this kernel nearly everywhere.  481 sizes of 129 to
// 8192 rows, 120 of them random: of the 429 that are taken 417 are not slower, 12 by 1 to 8 % (36864 x 4608 at 256 and 576 rows, 51200 x
// 5120 at 300 to 384 and 576: the library's tiles happen to fit), all together 0.82 of the library's time.
extern "C" int lle_gemm_wide_form(int M, int N, int K, int units) {
    if (M <= 128 || N <= 0 || K <= 0 || units <= 0 || K % WIDE_BK != 0 || N % 8 != 0 || (int64_t)320 * K * 2 > 0x7fffffff) return 0;
    const float stages = (float)(K / WIDE_BK), gflop = 2e-9f * M * N * K;
    float best = 0.f;
    int choice = 0;
    for (int i = 0; i < 11; ++i) {
        const WideForm& v = wide_forms[i];
        const int64_t tiles = (int64_t)((M + v.rows - 1) / v.rows) * ((N + v.columns - 1) / v.columns), whole = tiles / units;
        const float rest = (float)(tiles - whole * units) / units;
        const float us = whole * (v.start + stages * (v.stage + v.full)) + (rest > 0.f ? v.start + stages * (v.stage + v.full * rest) : 0.f);
        if (choice == 0 || us < best) best = us, choice = i + 1;
    }
    const float library = 0.97f * (fmaxf(gflop * 256.f / units, (float)N * K / 3e6f) + 9.f + (float)M * N / 1.6e6f);
    return best < library ? choice : 0;
}

// X [M, K] and W [N, K] bfloat16, contiguous, 16-byte aligned; K a multiple of 64, N of 8; W is gate rows and then up rows, C [M, N / 2].
// gated 1: silu(gate) . up; gated 2: with bias [N] (or null) and limit, g = min(gate + b, limit), u = clamp(up + b, -limit, limit),
// C = g sigmoid(1.702 g) (u + 1).  form: which of wide_forms.
extern "C" int lle_gemm_wide_bf16(const void* X, const void* W, const void* bias, float limit, void* C, int M, int N, int K, int gated,
                                  int form, hipStream_t stream) {
    if (M <= 0 || N <= 0) return 0;
    if (K <= 0 || K % WIDE_BK != 0 || (int64_t)320 * K * 2 > 0x7fffffff || N % 8 != 0) return (int)hipErrorInvalidValue;
    if ((((uintptr_t)X | (uintptr_t)W) & 15) || (((uintptr_t)bias | (uintptr_t)C) & 7)) return (int)hipErrorInvalidValue;
    switch (gated) {
        case WIDE_SILU: return launch_wide_form<WIDE_SILU>(X, W, nullptr, 0.f, C, M, N, K, form, stream);
        case WIDE_CLAMPED:
            if (!(limit > 0.f)) return (int)hipErrorInvalidValue;
            return launch_wide_form<WIDE_CLAMPED>(X, W, bias, limit, C, M, N, K, form, stream);
        default: return (int)hipErrorInvalidValue;
    }
}
