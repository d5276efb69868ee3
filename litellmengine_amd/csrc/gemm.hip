// Matrix products C[M, N] = A[M, K] . B[N, K]^T (weights are [out, in] row-major
// like the reference's Linear, src/layers/linear.cu:169-215, which calls
// cublasSgemm).  This file holds the 32-bit product for any sizes (plain FMA, no matrix
// cores; the sum over k runs in index order whatever M is, so a row's result does not
// depend on what else is in the batch; gemm_f32.hip has the one for many rows), the bfloat16 weight-streaming product of decoding, and its 32-bit twin (32-bit
// operands through the 32-bit matrix instruction: products and sums in float32).
#include "common.h"
#include "lds.h"
#include <type_traits>

LLE_DEFINE_ERROR_STRING()

#define GT_BM 64
#define GT_BN 64
#define GT_BK 16

template <typename TA, typename TC>
__global__ __launch_bounds__(256) void gemm_nt_simt_kernel(const TA* __restrict__ A, const TA* __restrict__ B,
                                                           TC* __restrict__ C, int M, int N, int K, int64_t lda,
                                                           int64_t ldb, int64_t ldc) {
    __shared__ float As[GT_BK][GT_BM + 4];
    __shared__ float Bs[GT_BK][GT_BN + 4];
    const int tx = threadIdx.x % 16, ty = threadIdx.x / 16;
    const int64_t m0 = (int64_t)blockIdx.y * GT_BM, n0 = (int64_t)blockIdx.x * GT_BN;
    float acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = 0.f;

    for (int k0 = 0; k0 < K; k0 += GT_BK) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int idx = threadIdx.x + 256 * i;
            const int r = idx / GT_BK, c = idx % GT_BK;
            const bool kin = k0 + c < K;
            As[c][r] = (kin && m0 + r < M) ? to_f32<TA>(A[(m0 + r) * lda + k0 + c]) : 0.f;
            Bs[c][r] = (kin && n0 + r < N) ? to_f32<TA>(B[(n0 + r) * ldb + k0 + c]) : 0.f;
        }
        __syncthreads();
#pragma unroll
        for (int kk = 0; kk < GT_BK; ++kk) {
            float a[4], b[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) a[i] = As[kk][ty * 4 + i];
#pragma unroll
            for (int j = 0; j < 4; ++j) b[j] = Bs[kk][tx * 4 + j];
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(a[i], b[j], acc[i][j]);
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int64_t m = m0 + ty * 4 + i;
        if (m >= M) continue;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int64_t n = n0 + tx * 4 + j;
            if (n < N) C[m * ldc + n] = from_f32<TC>(acc[i][j]);
        }
    }
}

// float32 in, float32 out (in_dtype and out_dtype must say so)
extern "C" int lle_gemm_nt_simt(const void* A, const void* B, void* C, int M, int N, int K, int64_t lda,
                                int64_t ldb, int64_t ldc, int in_dtype, int out_dtype, hipStream_t stream) {
    if (M <= 0 || N <= 0) return 0;
    if (in_dtype != LLE_F32 || out_dtype != LLE_F32) return (int)hipErrorInvalidValue;
    dim3 grid((N + GT_BN - 1) / GT_BN, (M + GT_BM - 1) / GT_BM);
    if (grid.y > 65535) return (int)hipErrorInvalidValue;
    gemm_nt_simt_kernel<float, float><<<grid, 256, 0, stream>>>((const float*)A, (const float*)B, (float*)C, M, N, K,
                                                                 lda, ldb, ldc);
    LLE_RETURN_LAUNCH_STATUS();
}

// ---------------------------------------------------------------------------------
// Skinny product for decoding: M <= 64 rows of activations against a weight
// matrix that is read exactly once (gemm_lines_kernel takes what it can of it, see there; this one float32 and
// what has no whole lines, few columns, odd addresses or more rows).  bfloat16 in, 32-bit accumulate, bfloat16 or
// 32-bit out.  HBM-bound: the kernel is shaped to keep whole 128-byte lines of W
// in flight from all CUs.
//   workgroup = 16 rows of W (one matrix-core tile), 16 wavefronts split K:
//   wavefront w takes the 64-element k steps w, w + 16, ... (neighbouring
//   wavefronts read neighbouring 128-byte pieces of the same rows);
//   C^T tile = W tile [16 n x 64 k] . X^T [64 k x 16 m] by two
//   v_mfma_f32_16x16x32_bf16 per 16 rows of X; lane (c = lane / 16, r = lane % 16)
//   loads 32 contiguous bytes W[n0 + r][k0 + 16c .. + 15]; X comes from L2.
//   The 16 partial tiles are added in LDS in wavefront order, so the sum over k
//   has one fixed order for every M.
// ---------------------------------------------------------------------------------
typedef bf16_t gbf16x8 __attribute__((ext_vector_type(8)));
typedef float gf32x4 __attribute__((ext_vector_type(4)));

// An operand type T of the weight-streaming kernels: 16 bytes of it, and the product of 16 rows of W and of X over the columns
// that the lanes hold 16 bytes of each (bfloat16: one instruction; float32: four of the float32 instruction, whose products and
// sums are float32, element e of the lanes in instruction e).  A step is 128 bytes of a row.
template <typename T> struct SkOp;
template <> struct SkOp<bf16_t> {
    typedef gbf16x8 vec;
    static constexpr int E = 8;
    static __device__ __forceinline__ gf32x4 mma(vec w, vec x, gf32x4 acc) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(w, x, acc, 0, 0, 0); }
};
template <> struct SkOp<float> {
    typedef gf32x4 vec;
    static constexpr int E = 4;
    static __device__ __forceinline__ gf32x4 mma(vec w, vec x, gf32x4 acc) {
#pragma unroll
        for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(w[e], x[e], acc, 0, 0, 0);
        return acc;
    }
};
#define SK_KSTEP 64  // elements of a bfloat16 step
// How the wavefronts share the columns of a row, in rounds of 128 bytes a wavefront, each lane two pieces of 16 bytes a round:
// bfloat16 wavefronts take 128 bytes in a row, a lane's pieces side by side; float32 ones 64 bytes of each half of the round,
// as gemm_skinny_f32_kernel does: which of the float32 kernels takes a product follows the number of rows, and a row's sums must
// not.  (The other way round that kernel is slower with few rows: 6144 x 4096 at 1 row 21 us, with 128 bytes in a row 26.  The
// products that go by way of LDS, by K, take 128 bytes in a row whatever the number of rows.)
template <typename T, int WAVES = 16> struct SkShare {
    static constexpr bool HALVES = std::is_same<T, float>::value;
    static constexpr int E = SkOp<T>::E;
    static constexpr int ROUND = 8 * E * WAVES;               // elements of a round
    static constexpr int WAVE = HALVES ? 4 * E : 8 * E;       // from a wavefront's first element to the next one's
    static constexpr int LANE = HALVES ? E : 2 * E;           // from lane group c to c + 1
    static constexpr int SECOND = HALVES ? ROUND / 2 : E;     // from a lane's first piece to its second
    static constexpr int EXTENT = HALVES ? SECOND + WAVE : WAVE;  // from a wavefront's first element to behind its last of a round
};

// What such a launch is made of (in a HIP graph, one after the other): 1.7 us for a kernel that does nothing, 0.9 ns for every
// instruction of a wavefront whose CU holds sixteen, a trip to memory; so reductions stay between registers (common.h), what a
// launch will need is asked for at its start, and rounds that are left over go together.  With four, eight and sixteen
// wavefronts a workgroup: 6144 x 1024 gated at 1 row 5.8, 4.9, 4.9 us, 4096 x 12288 at 8 rows 29.0, 23.3, 22.1.
// Before / after these three (0.6B sizes): qkv at 1 / 32 rows 4.4 / 6.8 -> 4.1 / 6.1 us, gate_up 5.5 / 7.8 -> 4.9 / 7.1,
// down_proj 4.8 / 9.9 -> 4.7 / 9.5.
//
// GATED: W holds gate rows [0, N/2) and then up rows [N/2, N); a workgroup takes 16 gate rows
// and the 16 up rows that go with them (NT = 2) and writes silu(gate) * up, C is [M, N/2].
//
// The RMSNorm between two products can be folded into them (up to 32 rows).  With
//   norm(h)[m][k] = h[m][k] * w[k] * r[m],  r[m] = 1 / sqrt(mean_k h[m][k]^2 + eps)
// the factor r[m] commutes with the product that follows, so
//   RESID (the product before the norm): its result is the delta of the residual stream; the
//     epilogue forms h = hidden + delta in 32-bit, writes it back, writes xw = h * w as the
//     next product's input, and leaves the sums of h^2 over its columns per row in ss_part[16 or 32 rows][parts] (a part a
//     workgroup, or two);
//   SCALED (the product after the norm): adds up the parts, and multiplies its rows by r[m].
struct NormFold {
    float* hidden;          // RESID: residual stream [M, N], read and written
    const void* weight;     // RESID: norm weight [N]
    int weight_dtype;
    void* xw;               // RESID: out, [M, N], of X's type
    float* ss_out;          // RESID: out, [16][parts]; SPLIT: [32][parts] or more
    const float* ss_in;     // SCALED: the same
    int parts;              // SCALED, SPLIT
    int part_rows;          // SPLIT: columns of a part, all of the tile's or half of them
    float eps;              // SCALED
    // GATED: biases [N] (or null) and with act_limit > 0 the clamped activation instead of silu
    const bf16_t* act_bias;
    float act_limit;
};

// what a gated product makes of a gate's and an up row's sums: silu(g) u, or with a limit, g = min(g, limit) and
// u = clamp(u, -limit, limit), g sigmoid(1.702 g) (u + 1)
__device__ __forceinline__ float gated_result(float g, float u, const NormFold& fold, int64_t col, int64_t rows) {
    if (fold.act_limit > 0.f) {  // (the same for the whole launch)
        if (fold.act_bias) {
            g += (float)fold.act_bias[col];
            u += (float)fold.act_bias[rows + col];
        }
        g = fminf(g, fold.act_limit);
        u = fminf(fmaxf(u, -fold.act_limit), fold.act_limit);
        return g / (1.0f + expf(-1.702f * g)) * (u + 1.0f);
    }
    return g / (1.0f + expf(-g)) * u;
}

// What the kernels around a folded norm ask for at their start, and what they do behind their products.
//
// RESID: thread (m, n) of the first 256 owns element [m][n0 + n] of every 16 rows.  What it needs of the residual stream and of the
// norm weight has arrived by the epilogue (all threads ask, for places that are there; the bits of the weight are read as
// they lie and interpreted in the epilogue).
template <int MT>
struct ResidRows {
    float h[MT];
    uint32_t w;
    __device__ __forceinline__ void load(const NormFold& fold, int64_t n0, int tile_rows, int M, int N) {
        const int64_t col = min(n0 + min((int)(threadIdx.x % 16), tile_rows - 1), (int64_t)N - 1);
        if (fold.weight_dtype == LLE_F32)
            w = ((const uint32_t*)fold.weight)[col];
        else
            w = ((const uint16_t*)fold.weight)[col];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) h[mt] = fold.hidden[(int64_t)min(16 * mt + (int)(threadIdx.x / 16) % 16, M - 1) * N + col];
    }
};
// SCALED: wavefront w adds up the parts of the rows w, w + WAVES, ...  The first parts are asked for at the start and added after the
// products.
template <int MT, int WAVES>
struct NormParts {
    static constexpr int EARLY = 4, ROWS = (16 * MT + WAVES - 1) / WAVES;
    float early[ROWS][EARLY];
    __device__ __forceinline__ void load(const NormFold& fold, int wave, int lane, int M) {
#pragma unroll
        for (int j = 0; j < ROWS; ++j)
#pragma unroll
            for (int i = 0; i < EARLY; ++i)  // past the parts: the last one again, dropped below; past the rows likewise
                early[j][i] = fold.ss_in[min(wave + WAVES * j, M - 1) * fold.parts + min(lane + LLE_WAVE * i, fold.parts - 1)];
    }
    template <typename Inv>
    __device__ __forceinline__ void finish(const NormFold& fold, int wave, int lane, int M, int K, const Inv& inv) const {
#pragma unroll
        for (int j = 0; j < ROWS; ++j) {
            const int m = wave + WAVES * j;
            if (m >= M) break;  // (the same for the whole wavefront)
            float part = 0.f;
#pragma unroll
            for (int i = 0; i < EARLY; ++i) part += lane + LLE_WAVE * i < fold.parts ? early[j][i] : 0.f;
            // what is left: four loads at a time (one after the other would each pay the way from memory)
            const float* in = fold.ss_in + (int64_t)m * fold.parts;
            for (int b = lane + LLE_WAVE * EARLY; b < fold.parts; b += 4 * LLE_WAVE) {
                float v[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) v[i] = in[min(b + i * LLE_WAVE, fold.parts - 1)];
#pragma unroll
                for (int i = 0; i < 4; ++i) part += b + i * LLE_WAVE < fold.parts ? v[i] : 0.f;
            }
            part = wave_sum(part);
            if (lane == 0) inv(m) = 1.0f / sqrtf(part / (float)K + fold.eps);
        }
    }
};
// The epilogue: total(nt, mt, n, m) adds up the wavefronts' partial sums in their order; inv(m) is row m's factor.
template <int WAVES, int MT, int NT, bool GATED, bool RESID, bool SCALED, bool SPLIT, typename T, typename TC, typename Total, typename Inv>
__device__ __forceinline__ void finish_skinny(const Total& total, TC* C, int M, int N, int64_t n0, int tile_rows, const NormFold& fold,
                                              const ResidRows<MT>& resid, const Inv& inv) {
    if (GATED) {
        for (int idx = threadIdx.x; idx < MT * 256; idx += WAVES * LLE_WAVE) {
            const int mt = idx / 256, m = (idx / 16) % 16, n = idx % 16;
            const int64_t row = 16 * mt + m, col = n0 + n;
            if (row >= M || col >= N / 2 || n >= tile_rows) continue;
            float g = total(0, mt, n, m), u = total(NT - 1, mt, n, m);
            if (SCALED) {
                g *= inv(16 * mt + m);
                u *= inv(16 * mt + m);
            }
            C[row * (N / 2) + col] = from_f32<TC>(gated_result(g, u, fold, col, N / 2));
        }
        return;
    }
    if (RESID) {  // NT = 1
        if (threadIdx.x < 256) {
            const int n = threadIdx.x % 16;
            const int64_t col = n0 + n;
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                const int m16 = threadIdx.x / 16, m = 16 * mt + m16;
                float sq = 0.f;
                if (m < M && col < N && n < tile_rows) {
                    const float h = resid.h[mt] + total(0, mt, n, m16);
                    fold.hidden[(int64_t)m * N + col] = h;
                    ((T*)fold.xw)[(int64_t)m * N + col] =
                        (T)(h * __uint_as_float(fold.weight_dtype == LLE_F32 ? resid.w : resid.w << 16));
                    sq = h * h;
                }
                if (!SPLIT || fold.part_rows == tile_rows) {  // (the same for the whole launch)
                    sq = row16_sum(sq);
                    if (n == 0) fold.ss_out[(int64_t)m * gridDim.x + blockIdx.x] = sq;
                } else {
                    const float first = row16_sum(n < fold.part_rows ? sq : 0.f), second = row16_sum(n < fold.part_rows ? 0.f : sq);
                    const int part = 2 * blockIdx.x + n;
                    if (n < 2 && part < fold.parts) fold.ss_out[(int64_t)m * fold.parts + part] = n == 0 ? first : second;
                }
            }
        }
        return;
    }
    for (int idx = threadIdx.x; idx < NT * MT * 256; idx += WAVES * LLE_WAVE) {
        const int nt = idx / (MT * 256), mt = (idx / 256) % MT, m = (idx / 16) % 16, n = idx % 16;
        const int64_t row = 16 * mt + m, col = n0 + 16 * nt + n;
        if (row >= M || col >= N || (NT == 1 && n >= tile_rows)) continue;
        float sum = total(nt, mt, n, m);
        if (SCALED) sum *= inv(16 * mt + m);
        C[row * N + col] = from_f32<TC>(sum);
    }
}

// SPLIT (RESID): the rows of X are dealt out sixteen a workgroup, see lle_gemm_skinny_resid_bf16.
template <typename T, int MT, int NT, bool GATED, bool RESID, bool SCALED, typename TC, int SK_WAVES, int UNROLL, bool SPLIT = false>
// one tile of W and up to 16 rows of X: two workgroups of 16 wavefronts a CU (8 wavefronts a SIMD),
// which 64 registers allow; the gated form measured faster with the registers it asks for, and the scaled one has no room in
// 64 for the parts that it asks for at its start (three spilled registers cost a launch 0.9 us)
__global__ __launch_bounds__(SK_WAVES* LLE_WAVE, (MT == 1 && !GATED && !SCALED) ? 8 : 4) void gemm_skinny_kernel(const T* __restrict__ X,
                                                                         const T* __restrict__ W,
                                                                         TC* __restrict__ C, int M, int N, int K,
                                                                         int tile_rows, NormFold fold) {
    using Vec = typename SkOp<T>::vec;
    using Share = SkShare<T, SK_WAVES>;
    constexpr int E = SkOp<T>::E, SECOND = Share::SECOND;
    static_assert(!(RESID || SCALED) || MT <= (std::is_same<T, float>::value ? 4 : 2), "the norm is folded for up to 32 rows, float32 64");
    // `tile_rows` (at most 16) rows of W per tile: fewer than 16 where that makes the number of tiles a
    // multiple of the number of CUs (see skinny_tile_rows); the lanes past them read the tile's last
    // row again, which costs no traffic, and write nothing.  Forms with several tiles of W per
    // workgroup (NT > 1, not gated) keep whole tiles.
    // NT tiles of 16 rows of W per workgroup share the X operands they are multiplied with
    __shared__ float s_acc[SK_WAVES][NT][MT][16][17];
    __shared__ float s_inv[16 * MT];
    // A launch is short: what stands between its start and its first load of W counts.  Forms with a folded norm read all
    // arguments in one go (read where they are first used, each group costs a round trip of its own), and the small loads
    // beside W (parts of the norm's sums, residual stream, norm weight) are asked for without a condition around them, so
    // that nothing waits for them before the loads of W are on their way.  Plain forms read what they need (0.1 us of 4).
    if constexpr (RESID || SCALED)
        asm volatile("" ::"s"(X), "s"(W), "s"(C), "s"(M), "s"(N), "s"(K), "s"(tile_rows), "s"(fold.hidden), "s"(fold.weight),
                     "s"(fold.weight_dtype), "s"(fold.xw), "s"(fold.ss_out), "s"(fold.ss_in), "s"(fold.parts),
                     "s"(fold.eps));
    const int wave = threadIdx.x / LLE_WAVE, lane = threadIdx.x % LLE_WAVE;
    if (SPLIT && blockIdx.y > 0) {
        const int before = 16 * blockIdx.y;
        X += (int64_t)before * K;
        M -= before;
        fold.hidden += (int64_t)before * N;
        fold.xw = (T*)fold.xw + (int64_t)before * N;
        fold.ss_out += (int64_t)before * fold.parts;
    }
    NormParts<MT, SK_WAVES> parts;
    if (SCALED) parts.load(fold, wave, lane, M);
    const int c = lane / 16, r16 = lane % 16;
    const int64_t n0 = (int64_t)blockIdx.x * ((GATED || NT == 1) ? tile_rows : 16 * NT);
    ResidRows<MT> resid;
    if (RESID) resid.load(fold, n0, tile_rows, M, N);
    const T* wp[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        const int rt = min(r16, tile_rows - 1);  // the lane's row of the tile
        const int64_t wrow = GATED ? min(n0 + rt, (int64_t)N / 2 - 1) + nt * ((int64_t)N / 2)
                                   : min(n0 + (NT == 1 ? rt : 16 * nt + r16), (int64_t)N - 1);
        wp[nt] = W + wrow * K + Share::LANE * c;
    }
    // rows of X beyond M are never written back, so their lanes may read any valid row
    const T* xp[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) xp[mt] = X + (int64_t)min(16 * mt + r16, M - 1) * K + Share::LANE * c;
    gf32x4 acc[NT][MT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[nt][mt] = gf32x4{0.f, 0.f, 0.f, 0.f};
    const Vec zero = {};

    int kw = wave * Share::WAVE;
    // R rounds at a time: all their loads are issued before the first product
    auto rounds = [&](auto rounds_c) {
        constexpr int R = decltype(rounds_c)::value;
        Vec w0[R][NT], w1[R][NT], x0[R][MT], x1[R][MT];
#pragma unroll
        for (int u = 0; u < R; ++u) {
            const int k0 = kw + u * Share::ROUND;
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                w0[u][nt] = *(const Vec*)(wp[nt] + k0);
                w1[u][nt] = *(const Vec*)(wp[nt] + k0 + SECOND);
            }
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                x0[u][mt] = *(const Vec*)(xp[mt] + k0);
                x1[u][mt] = *(const Vec*)(xp[mt] + k0 + SECOND);
            }
        }
        if (R < UNROLL) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < R; ++u)
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) {
                    acc[nt][mt] = SkOp<T>::mma(w0[u][nt], x0[u][mt], acc[nt][mt]);
                    acc[nt][mt] = SkOp<T>::mma(w1[u][nt], x1[u][mt], acc[nt][mt]);
                }
        kw += R * Share::ROUND;
    };
    auto whole = [&](int n) { return kw + (n - 1) * Share::ROUND + Share::EXTENT <= K; };
    while (whole(UNROLL)) rounds(std::integral_constant<int, UNROLL>{});
    // what is left of K: whole rounds together (one by one each would pay the way from memory), then a round that may be
    // partial (K is a multiple of E); there both operands are zeroed beyond K so that nothing outside the matrices is read
    // (more rows of X leave no registers for it; a plain product of 17 to 32 rows is 2 to 6 % slower with them)
    if constexpr (UNROLL == 4 && (MT == 1 || (MT == 2 && SCALED))) {
        if (whole(3))
            rounds(std::integral_constant<int, 3>{});
        else if (whole(2))
            rounds(std::integral_constant<int, 2>{});
    }
    for (; kw < K; kw += Share::ROUND) {
        const int k0 = kw;
        const bool in0 = k0 + Share::LANE * c + E <= K, in1 = k0 + SECOND + Share::LANE * c + E <= K;
        Vec x0[MT], x1[MT];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            x0[mt] = in0 ? *(const Vec*)(xp[mt] + k0) : zero;
            x1[mt] = in1 ? *(const Vec*)(xp[mt] + k0 + SECOND) : zero;
        }
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            const Vec w0 = in0 ? *(const Vec*)(wp[nt] + k0) : zero;
            const Vec w1 = in1 ? *(const Vec*)(wp[nt] + k0 + SECOND) : zero;
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                acc[nt][mt] = SkOp<T>::mma(w0, x0[mt], acc[nt][mt]);
                acc[nt][mt] = SkOp<T>::mma(w1, x1[mt], acc[nt][mt]);
            }
        }
    }
    auto inv = [&](int m) -> float& { return s_inv[m]; };
    if (SCALED) parts.finish(fold, wave, lane, M, K, inv);
    // lane holds C^T[n = 4c + i][m = r16]
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int i = 0; i < 4; ++i) s_acc[wave][nt][mt][4 * c + i][r16] = acc[nt][mt][i];
    __syncthreads();
    auto total = [&](int nt, int mt, int n, int m) {
        float sum = 0.f;
#pragma unroll
        for (int w = 0; w < SK_WAVES; ++w) sum += s_acc[w][nt][mt][n][m];
        return sum;
    };
    finish_skinny<SK_WAVES, MT, NT, GATED, RESID, SCALED, SPLIT, T>(total, C, M, N, n0, tile_rows, fold, resid, inv);
}

// ---------------------------------------------------------------------------------
// 17 to 128 rows of X against a weight with few rows per CU (N about 16 rows a CU: o_proj,
// down_proj): the product in SLICES of K.  With one 16-row tile of W per workgroup every
// workgroup reads all of X (at 64 rows four times the bytes of its share of W, through L2), and
// taller tiles leave CUs without work: so a workgroup takes 64 rows of W and one of `slices`
// equal parts of K, a grid of (N / 64) x slices workgroups, and writes its 64 x M partial sums in
// float32: out[slice][m][n].  Whoever reads the result adds up the slices (the residual add that
// follows these products does), in slice order: the sum over k has one order whatever else runs.
// A workgroup walks its part of K in stages of 256 columns:
//   * the sixteen wavefronts are 4 tiles of W rows x the 4 64-element steps of a stage; a
//     wavefront's W operands (the only bytes from HBM) and its share of X[:, stage] are asked for
//     three stages ahead, into registers;
//   * X[:, stage] then goes to LDS (two buffers), its 16-byte pieces XOR-swizzled so that the
//     sixteen lanes that a 16-byte LDS read serves in a cycle hit sixteen different columns of
//     the banks, and every wavefront multiplies its W operands with every 16-row tile of it;
//   * at the end the four steps of a tile are added up in LDS.
// Measured on MI355X against the library: o_proj sizes (4096 x 4096) 11.7 against 15.0 us at
// 64 rows and 15.8 against 24.3 at 128, down_proj sizes (4096 x 12288) 29.5 against 38.7 us and
// 37.2 against 67.6; a CU takes in about 29 GB/s of W and X together whatever the depth of the
// loads on their way, and at 128 rows a workgroup reads twice as much X as W.
// ---------------------------------------------------------------------------------
#define MID_ROWS 64    // rows of W per workgroup
#define MID_STEPS 4    // 64-element steps of K per stage: 4 x MID_STEPS wavefronts a workgroup
#define MID_UNIT_STAGES 4  // a slice of K is a whole number of these many stages (the register sets divide it)
#define MID_STAGE (64 * MID_STEPS)  // columns of K per stage
// The XOR of a 16-byte piece index in row r of a 16-row tile of X.  Lanes (c, r) read the pieces
// 2 c and 2 c + 1 of a step; a cycle serves c0 with r / 4 in {0, 3} and c0 + 1 with r / 4 in
// {1, 2} (or the other way round), whose pieces differ in bit 1: r % 4 goes to bits 2-3 and
// r / 8 to bit 0, which makes the sixteen columns different.
#define MID_SWIZZLE(r) ((((r) & 3) << 2) | (((r) >> 3) & 1))
// BUFFERS: register sets, i.e. the stages on their way from memory plus the one that is multiplied
// (four up to 64 rows of X; two at 128 rows, where a stage of X is four loads a thread and the
// sixteen wavefronts of a workgroup have 128 registers a lane each; one to four measured the same).
template <int M_TILES, int BUFFERS>
__global__ __launch_bounds__(4 * MID_STEPS * LLE_WAVE) void gemm_mid_slices_kernel(const bf16_t* __restrict__ X,
                                                                                  const bf16_t* __restrict__ W,
                                                                                  float* __restrict__ out, int M, int N,
                                                                                  int K, int stages) {
    constexpr int WAVES = 4 * MID_STEPS;
    constexpr int XBUF = 16 * M_TILES * MID_STAGE;                      // elements of a stage of X
    constexpr int XL = XBUF / (WAVES * LLE_WAVE * 8);                   // 16-byte loads of X per thread and stage
    static_assert(XL * WAVES * LLE_WAVE * 8 == XBUF, "a stage of X is a whole number of loads for every thread");
    constexpr int PIECES = MID_STAGE / 8;                               // 16-byte pieces of a row of a stage
    extern __shared__ __attribute__((aligned(16))) unsigned char mid_lds[];
    bf16_t* xs = (bf16_t*)mid_lds;  // [2][16 M_TILES][MID_STAGE], swizzled
    float* red = (float*)mid_lds;   // afterwards: [wavefronts][M_TILES][16 n][17]
    const int wave = threadIdx.x / LLE_WAVE, lane = threadIdx.x % LLE_WAVE;
    const int c = lane / 16, r16 = lane % 16;
    const int tile = wave % 4, step = wave / 4;
    const int64_t n0 = (int64_t)blockIdx.x * MID_ROWS;
    const int k_begin = blockIdx.y * stages * MID_STAGE;
    // W: lane (c, r) holds W[n0 + 16 tile + r][k + 16 c .. + 15] of the wavefront's step of a stage
    const bf16_t* wp = W + min(n0 + 16 * tile + r16, (int64_t)N - 1) * K + k_begin + step * SK_KSTEP + 16 * c;
    // X: thread t copies the pieces t, t + threads, ... of a stage (row = piece / PIECES), through
    // registers; piece p of row m goes to piece p ^ swizzle(m % 16) of the row in LDS
    const bf16_t* xsrc[XL];
    int xdst[XL];
#pragma unroll
    for (int i = 0; i < XL; ++i) {
        const int piece = threadIdx.x + WAVES * LLE_WAVE * i;
        const int m = piece / PIECES, p = piece % PIECES;
        xsrc[i] = X + (int64_t)min(m, M - 1) * K + k_begin + 8 * p;
        xdst[i] = m * MID_STAGE + 8 * (p ^ MID_SWIZZLE(m % 16));
    }
    gbf16x8 w0[BUFFERS], w1[BUFFERS], xr[BUFFERS][XL];
    auto issue = [&](int st, auto buf_c) {
        constexpr int buf = decltype(buf_c)::value;
        w0[buf] = *(const gbf16x8*)(wp + st * MID_STAGE);
        w1[buf] = *(const gbf16x8*)(wp + st * MID_STAGE + 8);
#pragma unroll
        for (int i = 0; i < XL; ++i) xr[buf][i] = *(const gbf16x8*)(xsrc[i] + st * MID_STAGE);
    };
    gf32x4 acc[M_TILES];
#pragma unroll
    for (int mt = 0; mt < M_TILES; ++mt) acc[mt] = gf32x4{0.f, 0.f, 0.f, 0.f};
    const int sw = MID_SWIZZLE(r16);
    const int piece0 = 8 * step + 2 * c;  // logical pieces 2 c and 2 c + 1 of the wavefront's step
    const int x_read0 = r16 * MID_STAGE + 8 * (piece0 ^ sw), x_read1 = r16 * MID_STAGE + 8 * ((piece0 + 1) ^ sw);
    // Stage st waits in register set st % BUFFERS (BUFFERS - 1 stages are on their way from
    // memory while one is multiplied) and is multiplied from LDS buffer st % 2.
    auto run_stage = [&](int st, auto buf_c) {
        constexpr int buf = decltype(buf_c)::value;
        bf16_t* xb = xs + (st % 2) * XBUF;
#pragma unroll
        for (int i = 0; i < XL; ++i) *(gbf16x8*)(xb + xdst[i]) = xr[buf][i];
        // the stores to LDS are waited for by hand and the barrier is the bare instruction: a
        // __syncthreads() would also wait for the loads that are meant to stay on their way
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();  // all of stage st is in LDS, and nobody reads stage st - 1 any more
        // (asked for under no condition, past the end the last stage again: where paths meet the
        // compiler would wait for every load that one of them may have issued)
        issue(min(st + BUFFERS - 1, stages - 1), std::integral_constant<int, (buf + BUFFERS - 1) % BUFFERS>{});
#pragma unroll
        for (int mt = 0; mt < M_TILES; ++mt) {
            const gbf16x8 x0 = *(const gbf16x8*)(xb + 16 * mt * MID_STAGE + x_read0);
            const gbf16x8 x1 = *(const gbf16x8*)(xb + 16 * mt * MID_STAGE + x_read1);
            acc[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w0[buf], x0, acc[mt], 0, 0, 0);
            acc[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w1[buf], x1, acc[mt], 0, 0, 0);
        }
    };
    static_assert(BUFFERS >= 2 && BUFFERS <= 4 && MID_UNIT_STAGES % BUFFERS == 0, "register sets for the stages on their way");
    // the number of stages is a multiple of MID_UNIT_STAGES, and so of BUFFERS (the caller sees to it)
#define MID_FOR_BUFFERS(F) F(0) F(1) F(2) F(3)
#define MID_ISSUE_FIRST(B) if constexpr (B < BUFFERS - 1) issue(min(B, stages - 1), std::integral_constant<int, B % BUFFERS>{});
    MID_FOR_BUFFERS(MID_ISSUE_FIRST)
    for (int st = 0; st < stages; st += BUFFERS) {
#define MID_RUN(B) if constexpr (B < BUFFERS) run_stage(st + B, std::integral_constant<int, B % BUFFERS>{});
        MID_FOR_BUFFERS(MID_RUN)
    }
#undef MID_RUN
#undef MID_ISSUE_FIRST
#undef MID_FOR_BUFFERS
    __syncthreads();  // X is no longer needed: its space takes the partial tiles
    // lane holds C^T[n = 4 c + i][m = r16] of tile `tile`, step `step`
#pragma unroll
    for (int mt = 0; mt < M_TILES; ++mt)
#pragma unroll
        for (int i = 0; i < 4; ++i) red[((wave * M_TILES + mt) * 16 + 4 * c + i) * 17 + r16] = acc[mt][i];
    __syncthreads();
    float* dst = out + (int64_t)blockIdx.y * M * N;
    for (int idx = threadIdx.x; idx < 4 * M_TILES * 256; idx += blockDim.x) {
        const int n = idx % 16, t = (idx / 16) % 4, m = idx / 64;  // consecutive threads: consecutive columns
        const int64_t col = n0 + 16 * t + n;
        if (m >= M || col >= N) continue;
        const int mt = m / 16, m16 = m % 16;
        float sum = 0.f;
#pragma unroll
        for (int ph = 0; ph < MID_STEPS; ++ph) sum += red[(((4 * ph + t) * M_TILES + mt) * 16 + n) * 17 + m16];
        dst[(int64_t)m * N + col] = sum;
    }
}

// out [slices][M][N] float32; M <= 128, N a multiple of 64, K a multiple of slices x 4 stages of 256 columns
extern "C" int lle_gemm_mid_slices_unit(void) { return MID_STAGE * MID_UNIT_STAGES; }
extern "C" int lle_gemm_mid_slices_max_rows(void) { return 128; }

extern "C" int lle_gemm_mid_slices_bf16(const void* X, const void* W, void* out, int M, int N, int K, int slices,
                                        hipStream_t stream) {
    if (M <= 0 || M > 128 || N % MID_ROWS != 0 || slices <= 0 || slices > 65535 || K % (MID_STAGE * MID_UNIT_STAGES * slices) != 0)
        return (int)hipErrorInvalidValue;
    const dim3 grid(N / MID_ROWS, slices);
    const int stages = K / (MID_STAGE * slices);
#define LLE_MID_LAUNCH(T, B)                                                                                          \
    {                                                                                                                 \
        constexpr size_t tiles = (size_t)2 * 16 * T * MID_STAGE * sizeof(bf16_t);                           \
        constexpr size_t sums = (size_t)4 * MID_STEPS * T * 16 * 17 * sizeof(float);                                  \
        constexpr size_t lds = tiles > sums ? tiles : sums;                                                           \
        static std::atomic<uint64_t> granted{0};                                                                      \
        const hipError_t e = lle_grant_lds((const void*)gemm_mid_slices_kernel<T, B>, (int)lds, granted);             \
        if (e != hipSuccess) return (int)e;                                                                           \
        gemm_mid_slices_kernel<T, B><<<grid, 4 * MID_STEPS * LLE_WAVE, lds, stream>>>(                                    \
            (const bf16_t*)X, (const bf16_t*)W, (float*)out, M, N, K, stages);                                        \
    }
    if (M <= 32)
        LLE_MID_LAUNCH(2, 4)
    else if (M <= 64)
        LLE_MID_LAUNCH(4, 4)
    else if (M <= 96)
        LLE_MID_LAUNCH(6, 2)
    else
        LLE_MID_LAUNCH(8, 2)
#undef LLE_MID_LAUNCH
    LLE_RETURN_LAUNCH_STATUS();
}

// CUs of the current device (asked once per device)
static int gemm_compute_units() {
    static int cached[64] = {0};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
    if (cached[dev] == 0) {
        int n = 0;
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
        cached[dev] = n;
    }
    return cached[dev];
}

// Rows of W per tile of the one-tile-per-workgroup kernel: as many as give every CU the same share.
// More 16-row tiles than CUs: as many rows as make the last round full (with 320 tiles of 16 rows on
// 256 CUs a quarter of the CUs reads twice what the others read and the launch lasts as long as two
// rounds, with 512 tiles of 10 rows every CU reads the same).  Fewer tiles than CUs (narrow models):
// lower tiles, down to 4 rows, so that every CU takes part: such a launch is short, and the share of
// W that a workgroup has to wait for is what is left to shorten (measured at 16 rows of X: 1024 x 3072
// 8.4 -> 7.3 us, 2048 x 6144 13.6 -> 12.1, 2560 x 9728 21.1 -> 18.9; tiles of 8 rows no better than of 4).
static int skinny_tile_rows(int rows) {
    const int units = gemm_compute_units();
    const int tiles16 = (rows + 15) / 16;
    if (tiles16 <= units) {
        const int per_unit = (rows + units - 1) / units;
        return per_unit < 4 ? 4 : (per_unit > 16 ? 16 : per_unit);
    }
    const int rounds = (tiles16 + units - 1) / units;
    const int per_tile = (int)(((int64_t)rows + (int64_t)rounds * units - 1) / ((int64_t)rounds * units));
    return per_tile < 1 ? 1 : (per_tile > 16 ? 16 : per_tile);
}


// ---------------------------------------------------------------------------------
// The same by way of LDS: up to 32 rows of X, K a multiple of 64 from 1024 on; float32, plain up to 64 rows, of 32 from 512 on.  In bfloat16 the
// same products and sums in the same order, bit for bit; only the operands' way is another one.
// What bounds gemm_skinny_kernel is a CU's vector cache: a load to registers costs it four cycles for every line of 128 bytes that it
// touches, and loads as the matrix instruction wants its operands touch sixteen lines for half of each (16 bytes a cycle, 38 B/ns
// a CU, for W and for X; whole lines 75), while loads straight into LDS, here eight whole lines at a time, bring 85 to 118
// B/ns.  So every wavefront copies its 64 columns of a step of the tile's rows and of X's into LDS of its own and multiplies
// from there: no barrier, it waits for its own loads.  It has up to DEPTH steps on their way, as many as 160 KB hold; a step's
// buffer takes the next load when it has been read.  The wavefronts' sums take the place of their operands.
// WH, XH: loads of eight rows for a tile of W and for sixteen rows of X (one where there are no more than eight).
// Launches in a HIP graph, weights from memory, gemm_skinny_kernel -> this one in us at 1 / 8 / 16 / 32 rows of X (norm folded as in
// a model): 4096 x 1024 4.3 / 4.5 / 4.9 / 6.3 -> 3.7 / 3.8 / 4.4 / 5.5; 6144 x 1024 gated 5.0 / 5.3 / 6.0 / 7.2 -> 4.7 / 4.9 / 5.2 /
// 6.3; 1024 x 2048 3.9 / 4.6 / 5.4 / 5.7 -> 3.5 / 3.6 / 3.8 / 3.9; 1024 x 3072 5.1 / 5.8 / 6.9 / 7.3 -> 4.1 / 4.3 / 5.1 / 5.4; 2048 x
// 8192 at up to 16 rows 11.1 / 11.9 / 14.7 -> 7.7 / 7.9 / 10.2; 4096 x 4096 8.4 / 9.5 / 12.1 -> 8.2 / 8.3 / 8.8; 4096 x 12288 20.2 / 22.5 /
// 28.8 -> 18.9 / 18.9 / 21.8 (5.3 TB/s); 5120 x 25600 54.8 / 64.8 / 81.3 -> 48.2 / 50.9 / 65.5.
// ---------------------------------------------------------------------------------
// where piece p (16 bytes) of row r lies in its 128 bytes of LDS: p ^ this.  A 16-byte read serves sixteen lanes a cycle, rows with
// r / 4 in {0, 3} at piece 2 c + e and the others at that of the next c (or the other way round): they meet every bank once.
#define LINES_SWIZZLE(r) ((((r) >> 1) & 7) ^ (((((r) >> 3) ^ ((r) >> 2)) & 1) << 1))
#define LINES_LDS(scaled) (160 * 1024 - ((scaled) ? 256 : 0))  // (of a CU, less what the row factors take)

// bytes of LDS of a wavefront
static constexpr int lines_bytes(int loads, int depth, int tiles) {
    const int operands = depth * loads * 1024, sums = tiles * 16 * 17 * 4;
    return operands > sums ? operands : (sums + 1023) / 1024 * 1024;
}

template <typename T, int MT, int NT, bool GATED, bool RESID, bool SCALED, typename TC, int WH, int XH, int DEPTH, bool SPLIT>
__global__ __launch_bounds__(16 * LLE_WAVE) void gemm_lines_kernel(const T* __restrict__ X, const T* __restrict__ W,
                                                                   TC* __restrict__ C, int M, int N, int K, int tile_rows, NormFold fold) {
    using Vec = typename SkOp<T>::vec;
    constexpr int COLUMNS = 8 * SkOp<T>::E;  // of a wavefront's part of a step: 128 bytes
    constexpr int WAVES = 16, LOADS = NT * WH + MT * XH, STEP = LOADS * 1024, OWN = lines_bytes(LOADS, DEPTH, NT * MT);
    static_assert(NT == (GATED ? 2 : 1) && WAVES * OWN <= LINES_LDS(SCALED && MT <= 2) && (MT <= 2 || OWN >= NT * MT * 16 * 17 * 4 + 16), "a tile of W, and of the up rows; the LDS of a CU");
    extern __shared__ __attribute__((aligned(16))) unsigned char lines_lds[];
    __shared__ float s_inv[MT <= 2 ? 16 * MT : 1];
    if constexpr (RESID || SCALED)  // (all arguments in one go, as gemm_skinny_kernel)
        asm volatile("" ::"s"(X), "s"(W), "s"(C), "s"(M), "s"(N), "s"(K), "s"(tile_rows), "s"(fold.hidden), "s"(fold.weight),
                     "s"(fold.weight_dtype), "s"(fold.xw), "s"(fold.ss_out), "s"(fold.ss_in), "s"(fold.parts),
                     "s"(fold.eps));
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / LLE_WAVE), lane = threadIdx.x % LLE_WAVE;
    if (SPLIT && blockIdx.y > 0) {
        const int before = 16 * blockIdx.y;
        X += (int64_t)before * K;
        M -= before;
        fold.hidden += (int64_t)before * N;
        fold.xw = (T*)fold.xw + (int64_t)before * N;
        fold.ss_out += (int64_t)before * fold.parts;
    }
    const int64_t n0 = (int64_t)blockIdx.x * tile_rows;
    const int rows = GATED ? N / 2 : N;
    // a load: lane -> row lane / 8, physical piece lane % 8, the logical piece that belongs there; rows behind the tile's and X's last
    // one read it again and are dropped
    unsigned wo[WH], xo[MT][XH];
#pragma unroll
    for (int h = 0; h < WH; ++h) {
        const int r = 8 * h + lane / 8;
        wo[h] = (unsigned)min(min(r, tile_rows - 1), rows - 1 - (int)n0) * (unsigned)(K * sizeof(T)) + ((lane % 8) ^ LINES_SWIZZLE(r)) * 16;
    }
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int h = 0; h < XH; ++h) {
            const int r = 8 * h + lane / 8;
            xo[mt][h] = (unsigned)min(16 * mt + r, M - 1) * (unsigned)(K * sizeof(T)) + ((lane % 8) ^ LINES_SWIZZLE(r)) * 16;
        }
    unsigned char* own = lines_lds + wave * OWN;
    const unsigned own_at = (unsigned)(size_t)(__attribute__((address_space(3))) void*)lines_lds + wave * OWN;
    const T *wb = W + n0 * K + wave * COLUMNS, *xb = X + wave * COLUMNS;
    auto issue = [&](int step, int buf) {
        const int64_t k = (int64_t)step * (COLUMNS * WAVES);
        const unsigned at = own_at + buf * STEP;
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int h = 0; h < WH; ++h) load_into_lds(at + (nt * WH + h) * 1024, wo[h], wb + k + (nt ? (int64_t)rows * K : 0));
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int h = 0; h < XH; ++h) load_into_lds(at + (NT * WH + mt * XH + h) * 1024, xo[mt][h], xb + k);
    };
    NormParts<MT, WAVES> parts;
    if (SCALED) parts.load(fold, wave, lane, M);
    ResidRows<MT> resid;
    if (RESID) resid.load(fold, n0, tile_rows, M, N);
    const int steps = (K / COLUMNS - wave + WAVES - 1) / WAVES;  // of this wavefront: DEPTH or more
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) issue(d, d);
    // lane (c, r) reads pieces 2 c and 2 c + 1 of row r (of eight rows: each twice)
    const int c = lane / 16, r16 = lane % 16;
    int w_at[2], x_at[2];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
        const int wr = WH == 1 ? r16 % 8 : r16, xr = XH == 1 ? r16 % 8 : r16;
        w_at[e] = wr * 128 + ((2 * c + e) ^ LINES_SWIZZLE(wr)) * 16;
        x_at[e] = xr * 128 + ((2 * c + e) ^ LINES_SWIZZLE(xr)) * 16;
    }
    gf32x4 acc[NT][MT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[nt][mt] = gf32x4{0.f, 0.f, 0.f, 0.f};
    int buf = 0;
    // the next step: `behind` steps have been asked for after it
    auto multiply = [&](auto behind) {
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(decltype(behind)::value * LOADS) : "memory");
        const unsigned char* at = own + buf * STEP;
        Vec w[NT][2], x[MT][2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) w[nt][e] = *(const Vec*)(at + nt * WH * 1024 + w_at[e]);
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) x[mt][e] = *(const Vec*)(at + (NT * WH + mt * XH) * 1024 + x_at[e]);
        }
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                for (int e = 0; e < 2; ++e) acc[nt][mt] = SkOp<T>::mma(w[nt][e], x[mt][e], acc[nt][mt]);
    };
    auto next = [&]() { buf = buf == DEPTH - 1 ? 0 : buf + 1; };
    for (int step = 0; step + DEPTH < steps; ++step, next()) {
        multiply(std::integral_constant<int, DEPTH - 1>{});
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the buffer has been read
        issue(step + DEPTH, buf);
    }
    if constexpr (DEPTH >= 5) multiply(std::integral_constant<int, 4>{}), next();
    if constexpr (DEPTH >= 4) multiply(std::integral_constant<int, 3>{}), next();
    if constexpr (DEPTH >= 3) multiply(std::integral_constant<int, 2>{}), next();
    if constexpr (DEPTH >= 2) multiply(std::integral_constant<int, 1>{}), next();
    multiply(std::integral_constant<int, 0>{});
    // (three and four tiles of X's rows take all of LDS: a wavefront keeps its rows' factors behind what its sums will take)
    auto inv = [&](int m) -> float& {
        if constexpr (MT <= 2) return s_inv[m];
        else return *(float*)(lines_lds + m % 16 * OWN + OWN - 16 + m / 16 * 4);
    };
    if (SCALED) parts.finish(fold, wave, lane, M, K, inv);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    // lane holds C^T[n = 4c + i][m = r16]
    float* mine = (float*)own;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int i = 0; i < 4; ++i) mine[((nt * MT + mt) * 16 + 4 * c + i) * 17 + r16] = acc[nt][mt][i];
    __syncthreads();
    auto total = [&](int nt, int mt, int n, int m) {
        const unsigned char* at = lines_lds + (((nt * MT + mt) * 16 + n) * 17 + m) * 4;
        float sum = 0.f;
#pragma unroll
        for (int w = 0; w < WAVES; ++w) sum += *(const float*)(at + w * OWN);
        return sum;
    };
    finish_skinny<WAVES, MT, NT, GATED, RESID, SCALED, SPLIT, T>(total, C, M, N, n0, tile_rows, fold, resid, inv);
}

// DEPTH: the most steps that LDS holds, up to 5, and up to what the wavefront with the fewest has.
template <typename T, int MT, int NT, bool GATED, bool RESID, bool SCALED, typename TC, int WH, int XH, bool SPLIT, int DEPTH>
static hipError_t launch_lines_depth(const T* X, const T* W, TC* C, int M, int N, int K, int tile_rows, const NormFold& fold, int blocks,
                                     hipStream_t stream) {
    constexpr int LDS = 16 * lines_bytes(NT * WH + MT * XH, DEPTH, NT * MT);
    if constexpr (LDS > LINES_LDS(SCALED && MT <= 2)) {
        return launch_lines_depth<T, MT, NT, GATED, RESID, SCALED, TC, WH, XH, SPLIT, DEPTH - 1>(X, W, C, M, N, K, tile_rows, fold, blocks, stream);
    } else if (DEPTH > 1 && K / (16 * 8 * SkOp<T>::E) < DEPTH) {
        return launch_lines_depth<T, MT, NT, GATED, RESID, SCALED, TC, WH, XH, SPLIT, DEPTH == 1 ? 1 : DEPTH - 1>(X, W, C, M, N, K, tile_rows, fold, blocks, stream);
    } else {
        auto kernel = gemm_lines_kernel<T, MT, NT, GATED, RESID, SCALED, TC, WH, XH, DEPTH, SPLIT>;
        static std::atomic<uint64_t> granted{0};
        const hipError_t e = lle_grant_lds((const void*)kernel, LDS, granted);
        if (e != hipSuccess) return e;
        kernel<<<dim3(blocks, SPLIT ? (M + 15) / 16 : 1), 16 * LLE_WAVE, LDS, stream>>>(X, W, C, M, N, K, tile_rows, fold);
        return hipGetLastError();
    }
}

// Whether gemm_lines_kernel takes a product of up to 32 rows (a plain one of float32 64): whole lines, all wavefronts with a step, operands
// that a load into LDS can take (16 bytes).
template <typename T>
static bool lines_fit(const T* X, const T* W, int K) {
    return K % (8 * SkOp<T>::E) == 0 && K >= 16 * 8 * SkOp<T>::E && (int64_t)64 * K * sizeof(T) <= 0x7fffffff && (((uintptr_t)X | (uintptr_t)W) & 15) == 0;
}
template <int MT, int NT, bool GATED, bool RESID, bool SCALED, typename TC, bool SPLIT = false, typename T>
static int launch_lines(const T* X, const T* W, TC* C, int M, int N, int K, int tile_rows, const NormFold& fold, int blocks,
                        hipStream_t stream) {
    if constexpr (MT == 1 && !SPLIT) {
        if (M <= 8)
            return (int)(tile_rows <= 8 ? launch_lines_depth<T, 1, NT, GATED, RESID, SCALED, TC, 1, 1, false, 5>(X, W, C, M, N, K, tile_rows, fold, blocks, stream)
                                        : launch_lines_depth<T, 1, NT, GATED, RESID, SCALED, TC, 2, 1, false, 5>(X, W, C, M, N, K, tile_rows, fold, blocks, stream));
    }
    return (int)(tile_rows <= 8 ? launch_lines_depth<T, MT, NT, GATED, RESID, SCALED, TC, 1, 2, SPLIT, 5>(X, W, C, M, N, K, tile_rows, fold, blocks, stream)
                                : launch_lines_depth<T, MT, NT, GATED, RESID, SCALED, TC, 2, 2, SPLIT, 5>(X, W, C, M, N, K, tile_rows, fold, blocks, stream));
}

// ---------------------------------------------------------------------------------
// The product as a STREAM by way of LDS, for K = 64 * 16 * XS (XS steps a wavefront, all of X that it needs held in registers)
// and up to 16 rows of X, or 32 (MT = 2); plain or gated, with or without the row factors of a folded norm.
// The chip reads fastest when every CU has the same share of W.  There is one workgroup per CU, and it takes `share` rows of W
// (share = rows / CUs, rounded up) in tiles of 16, the last of which may be lower: tile t of all workgroups together is one
// block of consecutive rows (the memory channels see what they see of a plain sweep over W), of which workgroup b takes the
// b-th piece.  The lanes of a tile that is not full read its last row again, which costs no traffic.
// A wavefront's loads are pieces of sixteen rows of 128 bytes, two loads of whole lines into LDS of its own (gemm_lines_kernel says
// why), DEPTH pieces on their way: first its part of X, which goes to registers, then its parts of the tiles one after the other, also
// across the end of a tile, where the partial tiles are added up in LDS between barriers that wait for no load.
// In a HIP graph, weights from memory, with operand-shaped loads to registers -> so, at 1 / 8 / 16 / 32 rows of X (us): 6144 x 4096
// 12.5 / 12.7 / 14.8 -> 11.3 / 11.3 / 11.9 (norm folded); 24576 x 4096 gated 35.1 / 36.5 / 38.2 -> 35.7 / 35.7 / 36.0, plain at 32 rows
// 41.6 -> 37.8; 51200 x 5120 gated 101 / 104 / 109 -> 91 / 92 / 95 (5.7 TB/s); 8768 x 2048 8.9 / 9.2 / 10.3 / 12.6 -> 9.0 / 9.0 / 9.5 /
// 10.6; 12288 x 2048 gated 11.9 / 12.5 / 13.6 / 16.6 -> 11.8 / 11.9 / 12.0 / 13.9; 151936 x 1024 59.7 / 64.4 / 63.1 / 69.0 -> 54.7 / 57.8 /
// 60.9 / 65.2.  What is left is the launch, 2 us, and memory.
// ---------------------------------------------------------------------------------
template <typename T, bool GATED, bool SCALED, int XS, typename TC, int MT, int DEPTH>
__global__ __launch_bounds__(16 * LLE_WAVE) void gemm_lines_stream_kernel(const T* __restrict__ X, const T* __restrict__ W, TC* __restrict__ C, int M,
                                                                          int N, int share, NormFold fold) {
    using Vec = typename SkOp<T>::vec;
    constexpr int WAVES = 16, NT = GATED ? 2 : 1, E = SkOp<T>::E, COLUMNS = 8 * E, K = XS * WAVES * COLUMNS, PIECE = 2048;
    constexpr int ACC = NT * MT * 16 * 17 * 4, OWN = DEPTH * PIECE + ACC;
    extern __shared__ __attribute__((aligned(16))) unsigned char lines_lds[];
    __shared__ float s_inv[16 * MT];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / LLE_WAVE), lane = threadIdx.x % LLE_WAVE;
    const int c = lane / 16, r16 = lane % 16;
    const int rows = GATED ? N / 2 : N;
    const int tiles = (share + 15) / 16;
    // rows [tile_begin(t), tile_end(t)) of this workgroup's tile t; none where W ends before them
    auto tile_begin = [&](int t) { return (int)gridDim.x * 16 * t + (int)blockIdx.x * min(16, share - 16 * t); };
    auto tile_end = [&](int t) { return min(rows, tile_begin(t) + min(16, share - 16 * t)); };
    // wavefront's LDS: the pieces [DEPTH][16 rows][128 bytes], and its sums (all wavefronts' sums one behind the other)
    unsigned char* pieces = lines_lds + wave * (DEPTH * PIECE);
    const unsigned pieces_at = (unsigned)(size_t)(__attribute__((address_space(3))) void*)lines_lds + wave * (DEPTH * PIECE);
    float* sums = (float*)(lines_lds + WAVES * DEPTH * PIECE);  // [wavefronts][NT][MT][16 n][17]
    float* mine = sums + wave * (ACC / 4);
    // a load: eight rows of 128 bytes; lane -> row lane / 8, physical piece lane % 8, the logical piece that belongs there
    const unsigned in_row = (unsigned)(lane % 8) * 16, at_wave = (unsigned)wave * 128;
    auto offset = [&](int row, int r) { return (unsigned)row * (unsigned)(K * sizeof(T)) + (in_row ^ (LINES_SWIZZLE(r) * 16)); };
    const int lr0 = lane / 8, lr1 = 8 + lane / 8;
    int fill = 0;  // the buffer that is asked for next
    auto ask = [&](unsigned o0, unsigned o1, const void* base) {
        load_into_lds(pieces_at + fill * PIECE, o0, base);
        load_into_lds(pieces_at + fill * PIECE + 1024, o1, base);
        fill = fill == DEPTH - 1 ? 0 : fill + 1;
    };
    // the cursor over W's pieces: tile, step, and gate or up rows
    int load_tile = 0, load_step = 0, load_up = 0;
    unsigned wo0, wo1;
    const unsigned char* wb;
    auto aim = [&]() {
        const int first = tile_begin(load_tile), last = max(0, tile_end(load_tile) - 1 - first);  // (a tile without rows reads rows that are there)
        wo0 = offset(min(lr0, last), lr0), wo1 = offset(min(lr1, last), lr1);
        wb = (const unsigned char*)(W + (int64_t)min(first, rows - 1) * K) + at_wave;
    };
    auto ask_w = [&]() {
        ask(wo0, wo1, wb + load_step * (WAVES * 128) + (GATED && load_up ? (int64_t)rows * K * sizeof(T) : 0));
        if (GATED && !load_up) {
            load_up = 1;
            return;
        }
        load_up = 0;
        if (++load_step == XS) {
            load_step = 0;
            if (++load_tile < tiles) aim();
        }
    };
    // SCALED: the parts of the norm's sums of rows wave and 16 + wave, four bytes a lane, where the wavefront's sums will be
    if constexpr (SCALED) {
        const unsigned at = (unsigned)(size_t)(__attribute__((address_space(3))) void*)mine;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                load_word_into_lds(at + (mt * 4 + i) * 256, (unsigned)min(lane + i * LLE_WAVE, fold.parts - 1) * 4,
                                   fold.ss_in + (int64_t)min(16 * mt + wave, M - 1) * fold.parts);
    }
    constexpr int XP = XS * MT;  // pieces of X
    auto ask_x = [&](int q) {
        const int mt = q / XS, step = q % XS;
        ask(offset(min(16 * mt + lr0, M - 1), lr0), offset(min(16 * mt + lr1, M - 1), lr1),
            (const unsigned char*)X + at_wave + step * (WAVES * 128));
    };
    aim();
    auto ask_next = [&](int q) {  // piece q, X's first
        if (q < XP) ask_x(q);
        else ask_w();
    };
#pragma unroll
    for (int q = 0; q < DEPTH; ++q) ask_next(q);  // (W has DEPTH pieces or more)
    // lane (c, r) reads pieces 2 c and 2 c + 1 of row r
    const int at0 = r16 * 128 + ((2 * c) ^ LINES_SWIZZLE(r16)) * 16, at1 = r16 * 128 + ((2 * c + 1) ^ LINES_SWIZZLE(r16)) * 16;
    int buf = 0;
    auto take = [&](Vec& v0, Vec& v1) {
        const unsigned char* at = pieces + buf * PIECE;
        v0 = *(const Vec*)(at + at0);
        v1 = *(const Vec*)(at + at1);
        buf = buf == DEPTH - 1 ? 0 : buf + 1;
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the buffer has been read
    };
    auto landed = [&]() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"((DEPTH - 1) * 2) : "memory"); };
    Vec x0[MT][XS], x1[MT][XS];
#pragma unroll
    for (int q = 0; q < XP; ++q) {
        landed();
        take(x0[q / XS][q % XS], x1[q / XS][q % XS]);
        ask_next(q + DEPTH);
    }
    if constexpr (SCALED) {  // (older than the pieces: landed with the first)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            float v[4], part = 0.f;
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] = mine[(mt * 4 + i) * 64 + lane];
#pragma unroll
            for (int i = 0; i < 4; ++i) part += lane + i * LLE_WAVE < fold.parts ? v[i] : 0.f;
            const float* in = fold.ss_in + (int64_t)min(16 * mt + wave, M - 1) * fold.parts;
            for (int b = lane + 4 * LLE_WAVE; b < fold.parts; b += 4 * LLE_WAVE) {
#pragma unroll
                for (int i = 0; i < 4; ++i) v[i] = in[min(b + i * LLE_WAVE, fold.parts - 1)];
#pragma unroll
                for (int i = 0; i < 4; ++i) part += b + i * LLE_WAVE < fold.parts ? v[i] : 0.f;
            }
            part = wave_sum(part);
            if (lane == 0) s_inv[16 * mt + wave] = 1.0f / sqrtf(part / (float)K + fold.eps);
        }
    }
    int left = tiles * XS * NT - DEPTH;  // pieces that have not been asked for
    for (int tile = 0; tile < tiles; ++tile) {
        gf32x4 acc[NT][MT];
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) acc[nt][mt] = gf32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < XS; ++j)
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                if (left >= 0)
                    landed();
                else
                    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                Vec w0, w1;
                take(w0, w1);
                if (left > 0) ask_w();
                --left;
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) {
                    acc[nt][mt] = SkOp<T>::mma(w0, x0[mt][j], acc[nt][mt]);
                    acc[nt][mt] = SkOp<T>::mma(w1, x1[mt][j], acc[nt][mt]);
                }
            }
        // the tile's sums: nobody adds up the last tile's any more (barriers that wait for no load)
        if (tile > 0) {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
        }
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                for (int i = 0; i < 4; ++i) mine[((nt * MT + mt) * 16 + 4 * c + i) * 17 + r16] = acc[nt][mt][i];
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (threadIdx.x < 256 * MT) {
            const int m = threadIdx.x / 16, n = threadIdx.x % 16;
            const int64_t col = (int64_t)tile_begin(tile) + n;
            if (m < M && col < tile_end(tile)) {
                float g = 0.f, u = 0.f;
#pragma unroll
                for (int w = 0; w < WAVES; ++w) {
                    g += sums[w * (ACC / 4) + ((m / 16) * 16 + n) * 17 + m % 16];
                    if (GATED) u += sums[w * (ACC / 4) + ((MT + m / 16) * 16 + n) * 17 + m % 16];
                }
                if (SCALED) {
                    g *= s_inv[m];
                    u *= s_inv[m];
                }
                C[(int64_t)m * rows + col] = from_f32<TC>(GATED ? gated_result(g, u, fold, col, rows) : g);
            }
        }
    }
}

// TILES: as many as every workgroup has at least.
template <typename T, bool GATED, bool SCALED, int XS, typename TC, int MT, int TILES>
static int launch_lines_stream_depth(const T* X, const T* W, TC* C, int M, int N, int share, int blocks, const NormFold& fold, hipStream_t stream) {
    constexpr int NT = GATED ? 2 : 1, ACC = NT * MT * 16 * 17 * 4, MOST = (LINES_LDS(true) / 16 - ACC) / 2048;
    constexpr int DEPTH = MOST < TILES * XS * NT ? MOST : TILES * XS * NT, LDS = 16 * (DEPTH * 2048 + ACC);
    auto kernel = gemm_lines_stream_kernel<T, GATED, SCALED, XS, TC, MT, DEPTH>;
    static std::atomic<uint64_t> granted{0};
    const hipError_t e = lle_grant_lds((const void*)kernel, LDS, granted);
    if (e != hipSuccess) return (int)e;
    kernel<<<blocks, 16 * LLE_WAVE, LDS, stream>>>(X, W, C, M, N, share, fold);
    return (int)hipGetLastError();
}
template <typename T, bool GATED, bool SCALED, int XS, typename TC, int MT>
static int launch_lines_stream(const T* X, const T* W, TC* C, int M, int N, int share, int blocks, const NormFold& fold, hipStream_t stream) {
    if (XS == 1 && !GATED && share > 48)  // (short rows, an output head: 151936 x 1024 at 8 rows 61.1 us with two pieces on their way, 57.8 with four)
        return launch_lines_stream_depth<T, GATED, SCALED, XS, TC, MT, XS == 1 && !GATED ? 4 : 2>(X, W, C, M, N, share, blocks, fold, stream);
    return launch_lines_stream_depth<T, GATED, SCALED, XS, TC, MT, 2>(X, W, C, M, N, share, blocks, fold, stream);  // (a share is more than a tile)
}

// The streaming kernel takes the product when K is a number of whole rounds of its 16 wavefronts
// (1024 elements a round, 512 of float32) that its registers hold (up to 32 rows of X: fewer rounds
// beyond 16), and W has more than one tile of rows for every CU.
template <typename T, bool GATED, bool SCALED, typename TC>
static bool launch_skinny_stream(const T* X, const T* W, TC* C, int M, int N, int K, const NormFold& fold, hipStream_t stream, hipError_t& e) {
    e = hipSuccess;
    constexpr int ROUND = SkShare<T>::ROUND;
    if (M > 32 || K % ROUND != 0) return false;
    const int rows = GATED ? N / 2 : N;
    const int units = gemm_compute_units();
    const int share = (rows + units - 1) / units;
    if (share <= 16) return false;
    const int blocks = (rows + share - 1) / share;
    if (((uintptr_t)X | (uintptr_t)W) & 15) return false;  // (what no load into LDS takes is gemm_skinny_kernel's)
#define LLE_STREAM_CASE(XSV, MTV)                                                                                                 \
    case XSV:                                                                                                                     \
        e = (hipError_t)launch_lines_stream<T, GATED, SCALED, XSV, TC, MTV>(X, W, C, M, N, share, blocks, fold, stream);          \
        return true;
    if (M > 16) {  // two tiles of X rows: while all of X that a wavefront needs fits its registers
        switch (K / ROUND) {
            LLE_STREAM_CASE(1, 2)
            LLE_STREAM_CASE(2, 2)
        }
        if constexpr (!GATED) switch (K / ROUND) {
            LLE_STREAM_CASE(3, 2)
            LLE_STREAM_CASE(4, 2)
        }
        return false;
    }
    switch (K / ROUND) {
        LLE_STREAM_CASE(1, 1)
        LLE_STREAM_CASE(2, 1)
        LLE_STREAM_CASE(3, 1)
        LLE_STREAM_CASE(4, 1)
        LLE_STREAM_CASE(5, 1)
    }
    // (gated float32 at 8 rows, the plain product and a launch for the activation -> so: 24576 x 4096 75.8 -> 73.2 us, 16384 x 4096 52.8 -> 49.9, 12288 x
    // 3072 30.3 -> 28.9)
    if constexpr (!GATED || std::is_same<T, float>::value) switch (K / ROUND) {
        LLE_STREAM_CASE(6, 1)
        LLE_STREAM_CASE(8, 1)
    }
    return false;
#undef LLE_STREAM_CASE
}


// parts of lle_gemm_skinny_resid_bf16's sums of squares for a weight of N rows (its tiles at up to 16 rows of X): the second size of
// its ss_part
extern "C" int lle_gemm_skinny_resid_parts(int N) {
    if (N <= 0) return 0;
    const int tr = skinny_tile_rows(N);
    return (N + tr - 1) / tr;
}

template <typename T, typename TC, int NT, bool GATED>
static int launch_skinny(const T* X, const T* W, TC* C, int M, int N, int K, hipStream_t stream, const NormFold& none = {}) {
    constexpr int WAVES = 16, UNROLL = 4 / NT;
    const int rows = GATED ? N / 2 : N;
    const int tile_rows = skinny_tile_rows(rows), blocks = (rows + tile_rows - 1) / tile_rows;
    const int mt = (M + 15) / 16;
    if (lines_fit(X, W, K)) {
        if (mt == 1) return launch_lines<1, NT, GATED, false, false>(X, W, C, M, N, K, tile_rows, none, blocks, stream);
        if (mt == 2) return launch_lines<2, NT, GATED, false, false>(X, W, C, M, N, K, tile_rows, none, blocks, stream);
    }
    switch (mt) {
        case 1: gemm_skinny_kernel<T, 1, NT, GATED, false, false, TC, WAVES, UNROLL><<<blocks, WAVES * LLE_WAVE, 0, stream>>>(X, W, C, M, N, K, tile_rows, none); break;
        case 2: gemm_skinny_kernel<T, 2, NT, GATED, false, false, TC, WAVES, UNROLL><<<blocks, WAVES * LLE_WAVE, 0, stream>>>(X, W, C, M, N, K, tile_rows, none); break;
        case 3: gemm_skinny_kernel<T, 3, NT, GATED, false, false, TC, WAVES, UNROLL><<<blocks, WAVES * LLE_WAVE, 0, stream>>>(X, W, C, M, N, K, tile_rows, none); break;
        case 4: gemm_skinny_kernel<T, 4, NT, GATED, false, false, TC, WAVES, UNROLL><<<blocks, WAVES * LLE_WAVE, 0, stream>>>(X, W, C, M, N, K, tile_rows, none); break;
        default: return (int)hipErrorInvalidValue;
    }
    return (int)hipGetLastError();
}

// X [M, K] and W [N, K] bfloat16, contiguous; 1 <= M <= 64; K a multiple of 8.
extern "C" int lle_gemm_skinny_bf16(const void* X, const void* W, void* C, int M, int N, int K, int out_dtype,
                                    hipStream_t stream) {
    if (M <= 0 || N <= 0) return 0;
    if (M > 64 || K % 8 != 0 || K <= 0) return (int)hipErrorInvalidValue;
    const bf16_t* x = (const bf16_t*)X;
    const bf16_t* w = (const bf16_t*)W;
    hipError_t e;
    // one tile of W rows per workgroup measured best up to 16 rows of X (two tiles share the X
    // operands but halve the number of workgroups; they only pay off from 16 rows on)
    if (out_dtype == LLE_F32) {
        if (launch_skinny_stream<bf16_t, false, false, float>(x, w, (float*)C, M, N, K, NormFold{}, stream, e)) return (int)e;
        return launch_skinny<bf16_t, float, 1, false>(x, w, (float*)C, M, N, K, stream);
    }
    if (out_dtype == LLE_BF16) {
        if (launch_skinny_stream<bf16_t, false, false, bf16_t>(x, w, (bf16_t*)C, M, N, K, NormFold{}, stream, e)) return (int)e;
        return launch_skinny<bf16_t, bf16_t, 1, false>(x, w, (bf16_t*)C, M, N, K, stream);
    }
    return (int)hipErrorInvalidValue;
}

// The gated feed-forward's first half in one launch: W [2I, K] holds the gate rows and then the
// up rows; C [M, I] = silu(X gate^T) * (X up^T), the activation in 32-bit.  1 <= M <= 32.
extern "C" int lle_gemm_skinny_gated_bf16(const void* X, const void* W, void* C, int M, int N2, int K,
                                          hipStream_t stream) {
    if (M <= 0 || N2 <= 0) return 0;
    if (M > 32 || K % 8 != 0 || K <= 0 || N2 % 2 != 0) return (int)hipErrorInvalidValue;
    hipError_t e;
    if (launch_skinny_stream<bf16_t, true, false, bf16_t>((const bf16_t*)X, (const bf16_t*)W, (bf16_t*)C, M, N2, K, NormFold{}, stream, e))
        return (int)e;
    return launch_skinny<bf16_t, bf16_t, 2, true>((const bf16_t*)X, (const bf16_t*)W, (bf16_t*)C, M, N2, K, stream);
}

// The same with biases [N2] (or null) and the clamped activation: g = min(gate + b, limit), u = clamp(up + b, -limit, limit),
// C = g sigmoid(1.702 g) (u + 1).
extern "C" int lle_gemm_skinny_clamped_bf16(const void* X, const void* W, const void* bias, float limit, void* C, int M, int N2, int K,
                                            hipStream_t stream) {
    if (M <= 0 || N2 <= 0) return 0;
    if (M > 32 || K % 8 != 0 || K <= 0 || N2 % 2 != 0 || !(limit > 0.f)) return (int)hipErrorInvalidValue;
    NormFold fold = {};
    fold.act_bias = (const bf16_t*)bias;
    fold.act_limit = limit;
    hipError_t e;
    if (launch_skinny_stream<bf16_t, true, false, bf16_t>((const bf16_t*)X, (const bf16_t*)W, (bf16_t*)C, M, N2, K, fold, stream, e))
        return (int)e;
    return launch_skinny<bf16_t, bf16_t, 2, true>((const bf16_t*)X, (const bf16_t*)W, (bf16_t*)C, M, N2, K, stream, fold);
}

// The product BEFORE a folded norm: delta = X W^T [M, N] is added into `hidden` (float32 [M, N],
// in place), xw = hidden * norm_weight goes to `xw` (bfloat16 [M, N]) and the sums of squares of
// the new hidden over each part's columns to ss_part [16 or 32][lle_gemm_skinny_resid_parts(N)]
// (32 rows when M > 16).  1 <= M <= 32.
template <typename T>
static int launch_resid(const T* x, const T* w, void* hidden, const void* norm_weight, int weight_dtype, void* xw, void* ss_part, int M, int N, int K,
                        hipStream_t stream) {
    NormFold fold = {};
    fold.hidden = (float*)hidden;
    fold.weight = norm_weight;
    fold.weight_dtype = weight_dtype;
    fold.xw = xw;
    fold.ss_out = (float*)ss_part;
    // From 17 rows of X on a workgroup takes sixteen of them and, of a narrow model, tiles of W twice as high (two parts of the sums):
    // with all 32 rows a workgroup of the 0.6B sizes reads eight times as much X as W, every CU all of X (1024 x 3072: 24 + 196 KB,
    // so 48 + 98).  1024 x 2048 at 17 / 32 rows 5.9 / 7.2 -> 5.5 / 5.6 us, 1024 x 3072 7.3 / 9.5 -> 7.0 / 7.2.
    // (float32: only where both parts are added up in the same tree, so that a row's sums are the same whatever the number of rows)
    fold.part_rows = skinny_tile_rows(N);
    fold.parts = (N + fold.part_rows - 1) / fold.part_rows;
    const bool high = fold.part_rows <= 8 && (std::is_same<T, bf16_t>::value || (fold.part_rows & (fold.part_rows - 1)) == 0);
    const int tr = M <= 16 || !high ? fold.part_rows : 2 * fold.part_rows, blocks = (N + tr - 1) / tr;
    T* none = nullptr;
    if (lines_fit(x, w, K))
        return M <= 16 ? launch_lines<1, 1, false, true, false>(x, w, none, M, N, K, tr, fold, blocks, stream)
                       : launch_lines<1, 1, false, true, false, T, true>(x, w, none, M, N, K, tr, fold, blocks, stream);
    if (M <= 16)
        gemm_skinny_kernel<T, 1, 1, false, true, false, T, 16, 4><<<blocks, 16 * LLE_WAVE, 0, stream>>>(x, w, none, M, N, K, tr, fold);
    else
        gemm_skinny_kernel<T, 1, 1, false, true, false, T, 16, 4, true><<<dim3(blocks, (M + 15) / 16), 16 * LLE_WAVE, 0, stream>>>(x, w, none, M, N, K, tr, fold);
    LLE_RETURN_LAUNCH_STATUS();
}
extern "C" int lle_gemm_skinny_resid_bf16(const void* X, const void* W, void* hidden, const void* norm_weight,
                                          int weight_dtype, void* xw, void* ss_part, int M, int N, int K,
                                          hipStream_t stream) {
    if (M <= 0 || N <= 0) return 0;
    if (M > 32 || K % 8 != 0 || K <= 0) return (int)hipErrorInvalidValue;
    return launch_resid((const bf16_t*)X, (const bf16_t*)W, hidden, norm_weight, weight_dtype, xw, ss_part, M, N, K, stream);
}
// The same in float32 (xw too), up to 64 rows (ss_part: whole sixteens of them), K a multiple of 4.
extern "C" int lle_gemm_skinny_resid_f32(const void* X, const void* W, void* hidden, const void* norm_weight, int weight_dtype, void* xw,
                                         void* ss_part, int M, int N, int K, hipStream_t stream) {
    if (M <= 0 || N <= 0) return 0;
    if (M > 64 || K % 4 != 0 || K <= 0) return (int)hipErrorInvalidValue;
    return launch_resid((const float*)X, (const float*)W, hidden, norm_weight, weight_dtype, xw, ss_part, M, N, K, stream);
}

// The product AFTER a folded norm: X is the xw of lle_gemm_skinny_resid_bf16 and ss_part its
// (16 or 32) x `parts` sums; the rows of the result are scaled by 1 / sqrt(sum / K + eps).
// gated != 0: W is [2 I, K] and C [M, I] = silu(gate) * up as in lle_gemm_skinny_gated_bf16.
// C is bfloat16, or float32 for a product that is not gated (an output head).  1 <= M <= 32.
#ifndef SCALED_TILES_AT_32_ROWS
#define SCALED_TILES_AT_32_ROWS 4
#endif
template <typename TC>
static int launch_skinny_scaled(const bf16_t* x, const bf16_t* w, TC* c, int M, int N, int K, const NormFold& fold,
                                 hipStream_t stream) {
    hipError_t e;
    if (launch_skinny_stream<bf16_t, false, true, TC>(x, w, c, M, N, K, fold, stream, e)) return (int)e;
    const int threads = 16 * LLE_WAVE;
    const int tr = skinny_tile_rows(N), blocks = (N + tr - 1) / tr;
    if (lines_fit(x, w, K) && (M <= 16 || N < 16 * SCALED_TILES_AT_32_ROWS * gemm_compute_units()))
        return M <= 16 ? launch_lines<1, 1, false, false, true>(x, w, c, M, N, K, tr, fold, blocks, stream)
                       : launch_lines<2, 1, false, false, true>(x, w, c, M, N, K, tr, fold, blocks, stream);
    if (M <= 16) {
        gemm_skinny_kernel<bf16_t, 1, 1, false, false, true, TC, 16, 4><<<blocks, threads, 0, stream>>>(x, w, c, M, N, K, tr, fold);
    } else if (N >= 16 * SCALED_TILES_AT_32_ROWS * gemm_compute_units()) {
        // 17 to 32 rows of X are twice the bytes of a tile of W: with one tile a workgroup a product
        // with many tiles (an output head) spends its time on X; several tiles share what they read of it
        // (the head of the 0.6B sizes, 151936 x 1024, at 32 rows: 137.6 us with one tile, 126.8 with two, 112.1 with four)
        constexpr int NT = SCALED_TILES_AT_32_ROWS;
        gemm_skinny_kernel<bf16_t, 2, NT, false, false, true, TC, 16, 4 / NT>
            <<<(N + 16 * NT - 1) / (16 * NT), threads, 0, stream>>>(x, w, c, M, N, K, 16, fold);
    } else {
        gemm_skinny_kernel<bf16_t, 2, 1, false, false, true, TC, 16, 4><<<blocks, threads, 0, stream>>>(x, w, c, M, N, K, tr, fold);
    }
    return (int)hipGetLastError();
}

extern "C" int lle_gemm_skinny_scaled_bf16(const void* X, const void* W, void* C, const void* ss_part, int parts,
                                           float eps, int M, int N, int K, int gated, int out_dtype,
                                           hipStream_t stream) {
    if (M <= 0 || N <= 0) return 0;
    if (M > 32 || K % 8 != 0 || K <= 0 || parts <= 0 || (gated && N % 2 != 0)) return (int)hipErrorInvalidValue;
    if (out_dtype != LLE_BF16 && !(out_dtype == LLE_F32 && !gated)) return (int)hipErrorInvalidValue;
    NormFold fold = {};
    fold.ss_in = (const float*)ss_part;
    fold.parts = parts;
    fold.eps = eps;
    const bf16_t* x = (const bf16_t*)X;
    const bf16_t* w = (const bf16_t*)W;
    bf16_t* c = (bf16_t*)C;
    const int threads = 16 * LLE_WAVE;
    hipError_t e;
    if (!gated) {
        if (out_dtype == LLE_F32)
            return launch_skinny_scaled<float>(x, w, (float*)C, M, N, K, fold, stream);
        return launch_skinny_scaled<bf16_t>(x, w, c, M, N, K, fold, stream);
    } else if (launch_skinny_stream<bf16_t, true, true, bf16_t>(x, w, c, M, N, K, fold, stream, e)) {
        return (int)e;
    } else {
        const int rows = N / 2;
        const int tr = skinny_tile_rows(rows), blocks = (rows + tr - 1) / tr;
        if (lines_fit((const bf16_t*)X, (const bf16_t*)W, K))
            return M <= 16 ? launch_lines<1, 2, true, false, true>(x, w, c, M, N, K, tr, fold, blocks, stream)
                           : launch_lines<2, 2, true, false, true>(x, w, c, M, N, K, tr, fold, blocks, stream);
        if (M <= 16)
            gemm_skinny_kernel<bf16_t, 1, 2, true, false, true, bf16_t, 16, 2><<<blocks, threads, 0, stream>>>(x, w, c, M, N, K, tr, fold);
        else
            gemm_skinny_kernel<bf16_t, 2, 2, true, false, true, bf16_t, 16, 2><<<blocks, threads, 0, stream>>>(x, w, c, M, N, K, tr, fold);
    }
    LLE_RETURN_LAUNCH_STATUS();
}

// ---------------------------------------------------------------------------------
// The same for float32 operands that do not go by way of LDS (few columns, no whole lines, odd addresses).  W is read once;
// v_mfma_f32_16x16x4_f32 multiplies and adds in float32 (no reduced-precision mode).
// Lane (c, r) loads 16 contiguous bytes W[n0 + r][k0 + 4c .. + 3]; its four values are the
// k slot c of four instructions, and the X operand is laid out the same way.
// ---------------------------------------------------------------------------------
#define SKF_KSTEP 16
template <int MT, int SK_WAVES, int UNROLL>
__global__ __launch_bounds__(SK_WAVES* LLE_WAVE) void gemm_skinny_f32_kernel(const float* __restrict__ X,
                                                                             const float* __restrict__ W,
                                                                             float* __restrict__ C, int M, int N, int K,
                                                                             int tile_rows) {
    // `tile_rows` (at most 16) rows of W per workgroup, as in the bfloat16 kernel (skinny_tile_rows):
    // the lanes past them read the tile's last row again and write nothing
    __shared__ float s_acc[SK_WAVES][MT][16][17];
    const int wave = threadIdx.x / LLE_WAVE, lane = threadIdx.x % LLE_WAVE;
    const int c = lane / 16, r16 = lane % 16;
    const int64_t n0 = (int64_t)blockIdx.x * tile_rows;
    const float* wp = W + min(n0 + min(r16, tile_rows - 1), (int64_t)N - 1) * K + 4 * c;
    // rows of X beyond M are never written back, so their lanes may read any valid row
    const float* xp[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) xp[mt] = X + (int64_t)min(16 * mt + r16, M - 1) * K + 4 * c;
    gf32x4 acc[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[mt] = gf32x4{0.f, 0.f, 0.f, 0.f};

    const int full_steps = K / SKF_KSTEP;
    int ss = wave;
    for (; ss + (UNROLL - 1) * SK_WAVES < full_steps; ss += UNROLL * SK_WAVES) {
        gf32x4 w[UNROLL], x[UNROLL][MT];
#pragma unroll
        for (int u = 0; u < UNROLL; ++u) {
            const int k0 = (ss + u * SK_WAVES) * SKF_KSTEP;
            w[u] = *(const gf32x4*)(wp + k0);
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) x[u][mt] = *(const gf32x4*)(xp[mt] + k0);
        }
#pragma unroll
        for (int u = 0; u < UNROLL; ++u)
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    acc[mt] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[u][j], x[u][mt][j], acc[mt], 0, 0, 0);
    }
    // what is left of K: single steps, the last one may be partial (K is a multiple of 4)
    const int all_steps = (K + SKF_KSTEP - 1) / SKF_KSTEP;
    const gf32x4 zero = {0.f, 0.f, 0.f, 0.f};
    for (; ss < all_steps; ss += SK_WAVES) {
        const int k0 = ss * SKF_KSTEP;
        const bool in = k0 + 4 * c + 4 <= K;
        const gf32x4 w = in ? *(const gf32x4*)(wp + k0) : zero;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            const gf32x4 x = in ? *(const gf32x4*)(xp[mt] + k0) : zero;
#pragma unroll
            for (int j = 0; j < 4; ++j) acc[mt] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[j], x[j], acc[mt], 0, 0, 0);
        }
    }
    // lane holds C^T[n = 4c + i][m = r16]
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int i = 0; i < 4; ++i) s_acc[wave][mt][4 * c + i][r16] = acc[mt][i];
    __syncthreads();
    for (int idx = threadIdx.x; idx < MT * 256; idx += blockDim.x) {
        const int mt = idx / 256, m = (idx / 16) % 16, n = idx % 16;
        const int64_t row = 16 * mt + m, col = n0 + n;
        if (row >= M || col >= N || n >= tile_rows) continue;
        float sum = 0.f;
#pragma unroll
        for (int w = 0; w < SK_WAVES; ++w) sum += s_acc[w][mt][n][m];
        C[row * N + col] = sum;
    }
}

// The product after a folded norm in float32 (lle_gemm_skinny_resid_f32): up to 64 rows, gated up to 32; K a multiple of 4.  By way of LDS
// where K and the operands' addresses let it (then the sums are those of lle_gemm_skinny_f32 and its gated form).
extern "C" int lle_gemm_skinny_scaled_f32(const void* X, const void* W, void* C, const void* ss_part, int parts, float eps, int M, int N, int K,
                                          int gated, hipStream_t stream) {
    if (M <= 0 || N <= 0) return 0;
    const float *x = (const float*)X, *w = (const float*)W;
    float* c = (float*)C;
    if (M > (gated ? 32 : 64) || K <= 0 || parts <= 0 || (gated && N % 2 != 0) || K % 4 != 0) return (int)hipErrorInvalidValue;
    NormFold fold = {};
    fold.ss_in = (const float*)ss_part;
    fold.parts = parts;
    fold.eps = eps;
    const int rows = gated ? N / 2 : N, tr = skinny_tile_rows(rows), blocks = (rows + tr - 1) / tr;
    const int mt = (M + 15) / 16, threads = 16 * LLE_WAVE;
    hipError_t e;
    if (!lines_fit(x, w, K)) {
#define LLE_SCALED_F32(MT, NT, G, U) gemm_skinny_kernel<float, MT, NT, G, false, true, float, 16, U><<<blocks, threads, 0, stream>>>(x, w, c, M, N, K, tr, fold)
        if (gated) {
            if (mt == 1) LLE_SCALED_F32(1, 2, true, 2);
            else LLE_SCALED_F32(2, 2, true, 2);
        } else switch (mt) {
            case 1: LLE_SCALED_F32(1, 1, false, 4); break;
            case 2: LLE_SCALED_F32(2, 1, false, 4); break;
            case 3: LLE_SCALED_F32(3, 1, false, 2); break;
            default: LLE_SCALED_F32(4, 1, false, 2); break;
        }
#undef LLE_SCALED_F32
        LLE_RETURN_LAUNCH_STATUS();
    }
    if (gated) {
        if (launch_skinny_stream<float, true, true, float>(x, w, c, M, N, K, fold, stream, e)) return (int)e;
        return mt == 1 ? launch_lines<1, 2, true, false, true>(x, w, c, M, N, K, tr, fold, blocks, stream)
                       : launch_lines<2, 2, true, false, true>(x, w, c, M, N, K, tr, fold, blocks, stream);
    }
    if (launch_skinny_stream<float, false, true, float>(x, w, c, M, N, K, fold, stream, e)) return (int)e;
    switch (mt) {
        case 1: return launch_lines<1, 1, false, false, true>(x, w, c, M, N, K, tr, fold, blocks, stream);
        case 2: return launch_lines<2, 1, false, false, true>(x, w, c, M, N, K, tr, fold, blocks, stream);
        case 3: return launch_lines<3, 1, false, false, true>(x, w, c, M, N, K, tr, fold, blocks, stream);
        default: return launch_lines<4, 1, false, false, true>(x, w, c, M, N, K, tr, fold, blocks, stream);
    }
}

// X [M, K] and W [N, K] float32, contiguous; C [M, N] float32; 1 <= M <= 64; K a multiple of 4.
// K a multiple of 32 from 512 on goes by way of LDS whatever the number of rows (one of them decides the order of a row's sums, so K has to),
// as bfloat16 does; in a HIP graph, before -> so, at 1 / 8 / 17 / 32 / 64 rows (us): 4096 x 1024 5.6 / 6.7 / 8.0 / 9.2 / 13.6 -> 5.0 / 5.3 /
// 6.3 / 7.2 / 9.6; 6144 x 4096 22.4 / 28.5 / 37.4 / 48.2 / 80.2 -> 21.9 / 21.9 / 26.5 / 31.4 / 46.5; 24576 x 4096 gated 80.2 / 83.2 / 107 / 121 /
// 255 -> 75.2 / 75.1 / 82.7 / 84.6 / 148; 151936 x 4096 444 / 450 / 725 / 933 / 1540 -> 413 / 424 / 529 / 615 / 860.  The errors against 64 bits are
// the same (1.6e-7 at K = 1024, 3.0e-7 at 4096).
extern "C" int lle_gemm_skinny_f32(const void* X, const void* W, void* C, int M, int N, int K, hipStream_t stream) {
    if (M <= 0 || N <= 0) return 0;
    if (M > 64 || K % 4 != 0 || K <= 0) return (int)hipErrorInvalidValue;
    const float* x = (const float*)X;
    const float* w = (const float*)W;
    float* c = (float*)C;
    hipError_t e;
    if (launch_skinny_stream<float, false, false, float>(x, w, c, M, N, K, NormFold{}, stream, e)) return (int)e;
    const int tr = skinny_tile_rows(N), blocks = (N + tr - 1) / tr;
    if (lines_fit(x, w, K)) switch ((M + 15) / 16) {
        case 1: return launch_lines<1, 1, false, false, false>(x, w, c, M, N, K, tr, NormFold{}, blocks, stream);
        case 2: return launch_lines<2, 1, false, false, false>(x, w, c, M, N, K, tr, NormFold{}, blocks, stream);
        case 3: return launch_lines<3, 1, false, false, false>(x, w, c, M, N, K, tr, NormFold{}, blocks, stream);
        default: return launch_lines<4, 1, false, false, false>(x, w, c, M, N, K, tr, NormFold{}, blocks, stream);
    }
    switch ((M + 15) / 16) {
        case 1: gemm_skinny_f32_kernel<1, 16, 4><<<blocks, 16 * LLE_WAVE, 0, stream>>>(x, w, c, M, N, K, tr); break;
        case 2: gemm_skinny_f32_kernel<2, 16, 4><<<blocks, 16 * LLE_WAVE, 0, stream>>>(x, w, c, M, N, K, tr); break;
        case 3: gemm_skinny_f32_kernel<3, 16, 2><<<blocks, 16 * LLE_WAVE, 0, stream>>>(x, w, c, M, N, K, tr); break;
        default: gemm_skinny_f32_kernel<4, 16, 2><<<blocks, 16 * LLE_WAVE, 0, stream>>>(x, w, c, M, N, K, tr); break;
    }
    LLE_RETURN_LAUNCH_STATUS();
}

// silu(X gate^T) * (X up^T) as lle_gemm_skinny_gated_bf16; 1 <= M <= 32, K a multiple of 4.
extern "C" int lle_gemm_skinny_gated_f32(const void* X, const void* W, void* C, int M, int N2, int K, hipStream_t stream) {
    if (M <= 0 || N2 <= 0) return 0;
    if (M > 32 || K % 4 != 0 || K <= 0 || N2 % 2 != 0) return (int)hipErrorInvalidValue;
    const float *x = (const float*)X, *w = (const float*)W;
    hipError_t e;
    if (launch_skinny_stream<float, true, false, float>(x, w, (float*)C, M, N2, K, NormFold{}, stream, e)) return (int)e;
    return launch_skinny<float, float, 2, true>(x, w, (float*)C, M, N2, K, stream);
}
