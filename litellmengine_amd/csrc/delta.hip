// The gated delta rule: a matrix state per head that is decayed, then corrected towards the new value.
//
//   c = silu(conv(u))                     per channel over time, J taps, the request's last J - 1 rows kept    delta_conv
//   q, k <- every head of c's q and k parts as a unit vector (x / sqrt(sum x^2 + unit_eps)), q times q_scale
//   beta = sigmoid(b),  g = exp(-exp(A_log) softplus(a + dt_bias))     one of each per token and head         delta_scan
//   S <- g S;  w = beta (v - S^T k);  S <- S + k w^T;  o = S^T q       S [key, value] float32, per head
//   y = o / rms(o) * norm_w * act(gate)   per head, eps inside the root, act silu or sigmoid                  delta_out_norm
// The decay may also be one of every key channel, g = exp(-exp(A_log) softplus(z + dt_bias)) with z and dt_bias
// [head][channel]: it then acts on the rows of S, S <- diag(g) S, and is made ahead of the walk              low_rank_gates
//
// Value head h reads the q and k of head h / (H / G).  Every value channel of a head is a recurrence of its
// own over a vector of `dim` numbers (the column S[:, j]): a thread owns KI key channels of one column, the
// DELTA_IG = 16 threads of a column are neighbours in a wavefront and add up their shares of S^T k and S^T q
// through the lanes' cross-bar (no LDS, no barrier inside a token).  The state lies transposed in its row,
// [head][value][key], so a wavefront reads and writes one stretch of memory.
// All of it is 32-bit in every mode; only u, gate and y have the activation type.
#include "common.h"

LLE_DEFINE_ERROR_STRING()

#define DELTA_IG 16   // threads that share a column of the state
#define DELTA_TC 16   // tokens staged at a time
#define DELTA_THREADS 256
#define DELTA_VB (DELTA_THREADS / DELTA_IG)  // value channels of a workgroup
static_assert(DELTA_VB * DELTA_TC == DELTA_THREADS, "a chunk's values are one element a thread");

__device__ __forceinline__ float delta_silu(float x) { return x / (1.0f + expf(-x)); }

// ---------------------------------------------------------------------------------
// Convolution, silu, unit vectors.  A row of u holds q [G dim], k [G dim], v [H vdim].  grid = (tokens,
// units / 4): a wavefront per unit (a q head, a k head or a v head), a lane keeps up to four elements.
// `state` rows hold the last J - 1 rows of u of earlier steps, oldest first (float32); zeros at admission
// stand for the zeros before a request's start.
// ADVANCE (steps of single tokens only): the kept rows move on by the token in the same launch; every element's
// rows are read and written by the one lane that owns it.
// ---------------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(256) void delta_conv_kernel(const T* __restrict__ u, int cols, const float* __restrict__ taps,
                                                          int J, const float* __restrict__ state, int64_t state_stride,
                                                          const int32_t* __restrict__ token_seq,
                                                          const int32_t* __restrict__ cu_tokens,
                                                          const int32_t* __restrict__ seq_slots, float* __restrict__ q,
                                                          float* __restrict__ k, float* __restrict__ v, int G, int dim, int H,
                                                          int vdim, float unit_eps, float q_scale) {
    const int64_t n = blockIdx.x;
    const int unit = blockIdx.y * 4 + threadIdx.x / LLE_WAVE, lane = threadIdx.x % LLE_WAVE;
    if (unit >= 2 * G + H) return;
    const int seq = token_seq[n];
    const int before = (int)(n - cu_tokens[seq]);  // rows of this request in this step ahead of row n
    const float* kept = J > 1 ? state + (int64_t)seq_slots[seq] * state_stride : nullptr;
    int col0, width;
    float* dst;
    if (unit < G) {
        col0 = unit * dim, width = dim, dst = q + n * G * dim + unit * dim;
    } else if (unit < 2 * G) {
        col0 = unit * dim, width = dim, dst = k + n * G * dim + (unit - G) * dim;
    } else {
        col0 = 2 * G * dim + (unit - 2 * G) * vdim, width = vdim, dst = v + n * H * vdim + (unit - 2 * G) * vdim;
    }
    float y[4];
    float ss = 0.f;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int e = lane + LLE_WAVE * r;
        y[r] = 0.f;
        if (e < width) {
            const int c = col0 + e;
            float acc = 0.f;
            for (int j = 0; j < J; ++j) {
                const int back = J - 1 - j;  // how many tokens back this tap reaches
                const float x = back <= before ? to_f32<T>(u[(n - back) * cols + c])
                                               : kept[(int64_t)(J - 1 - (back - before)) * cols + c];
                acc = fmaf(taps[(int64_t)c * J + j], x, acc);
            }
            y[r] = delta_silu(acc);
            ss = fmaf(y[r], y[r], ss);
        }
    }
    float f = 1.0f;
    if (unit < 2 * G) {
        ss = wave_sum(ss);
        f = 1.0f / sqrtf(ss + unit_eps);
        if (unit < G) f *= q_scale;
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int e = lane + LLE_WAVE * r;
        if (e < width) dst[e] = y[r] * f;
    }
}

// The same for runs of consecutive tokens: a wavefront walks `run` tokens of one unit with the taps and the last
// J - 1 inputs of its elements in registers, so a token costs one new load per element whatever J (a workgroup a
// token re-reads J rows and the taps for every token: 61 against 25 us for 2048 tokens of 4096 channels and four
// taps).  Where the request changes inside a run the window is filled anew.
template <typename T, int J, bool ADVANCE>
__global__ __launch_bounds__(256) void delta_conv_run_kernel(const T* __restrict__ u, int cols, const float* __restrict__ taps,
                                                              float* state, int64_t state_stride,
                                                              const int32_t* __restrict__ token_seq,
                                                              const int32_t* __restrict__ cu_tokens,
                                                              const int32_t* __restrict__ seq_slots, float* __restrict__ q,
                                                              float* __restrict__ k, float* __restrict__ v, int N, int run, int G,
                                                              int dim, int H, int vdim, float unit_eps, float q_scale) {
    constexpr int W = J > 1 ? J - 1 : 1;
    const int unit = blockIdx.y * 4 + threadIdx.x / LLE_WAVE, lane = threadIdx.x % LLE_WAVE;
    if (unit >= 2 * G + H) return;
    const int n0 = blockIdx.x * run, n1 = min(N, n0 + run);
    int col0, width, out_cols, out0;
    float* dst;
    if (unit < G) {
        col0 = unit * dim, width = dim, dst = q, out_cols = G * dim, out0 = unit * dim;
    } else if (unit < 2 * G) {
        col0 = unit * dim, width = dim, dst = k, out_cols = G * dim, out0 = (unit - G) * dim;
    } else {
        col0 = 2 * G * dim + (unit - 2 * G) * vdim, width = vdim, dst = v, out_cols = H * vdim, out0 = (unit - 2 * G) * vdim;
    }
    float tp[4][J], win[4][W];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int e = lane + LLE_WAVE * r;
#pragma unroll
        for (int j = 0; j < J; ++j) tp[r][j] = e < width ? taps[(int64_t)(col0 + e) * J + j] : 0.f;
#pragma unroll
        for (int m = 0; m < W; ++m) win[r][m] = 0.f;
    }
    int seq_before = -1;
    for (int n = n0; n < n1; ++n) {
        const int seq = token_seq[n];
        if (J > 1 && seq != seq_before) {  // (the same for the whole wavefront) the J - 1 inputs ahead of this token
            const int before = n - cu_tokens[seq];
            const float* kept = state + (int64_t)seq_slots[seq] * state_stride;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int e = lane + LLE_WAVE * r;
                if (e < width) {
#pragma unroll
                    for (int m = 0; m < W; ++m) {  // (the rows of earlier steps, then those of this one)
                        const int back = J - 1 - m;
                        win[r][m] = back <= before ? to_f32<T>(u[(int64_t)(n - back) * cols + col0 + e])
                                                   : kept[(int64_t)(J - 1 - (back - before)) * cols + col0 + e];
                    }
                }
            }
        }
        seq_before = seq;
        float y[4], ss = 0.f;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int e = lane + LLE_WAVE * r;
            y[r] = 0.f;
            if (e < width) {
                const float x = to_f32<T>(u[(int64_t)n * cols + col0 + e]);
                float acc = 0.f;
                if (J > 1) {
#pragma unroll
                    for (int m = 0; m < W; ++m) acc = fmaf(tp[r][m], win[r][m], acc);
#pragma unroll
                    for (int m = 0; m + 1 < W; ++m) win[r][m] = win[r][m + 1];
                    win[r][W - 1] = x;
                    if (ADVANCE) {
                        float* kept = state + (int64_t)seq_slots[seq] * state_stride;
#pragma unroll
                        for (int m = 0; m < W; ++m) kept[(int64_t)m * cols + col0 + e] = win[r][m];
                    }
                }
                acc = fmaf(tp[r][J - 1], x, acc);
                y[r] = delta_silu(acc);
                ss = fmaf(y[r], y[r], ss);
            }
        }
        float f = 1.0f;
        if (unit < 2 * G) {
            ss = wave_sum(ss);
            f = 1.0f / sqrtf(ss + unit_eps);
            if (unit < G) f *= q_scale;
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int e = lane + LLE_WAVE * r;
            if (e < width) dst[(int64_t)n * out_cols + out0 + e] = y[r] * f;
        }
    }
}

template <typename T, bool ADVANCE>
static bool delta_conv_runs(const void* u, int cols, const void* taps, int J, void* state, int64_t state_stride,
                            const void* token_seq, const void* cu_tokens, const void* seq_slots, void* q, void* k, void* v, int N,
                            int G, int dim, int H, int vdim, float unit_eps, float q_scale, hipStream_t stream) {
    const int blocks = (2 * G + H + 3) / 4;
    // runs long enough that taps and windows are loaded seldom, short enough that a prompt fills the chip
    int run = (int)((int64_t)N * blocks / 2048);
    run = run < 1 ? 1 : run > 16 ? 16 : run;
    const dim3 grid((N + run - 1) / run, blocks);
#define DELTA_CONV_CASE(JJ)                                                                                                   \
    case JJ:                                                                                                                  \
        delta_conv_run_kernel<T, JJ, ADVANCE><<<grid, 256, 0, stream>>>(                                                      \
            (const T*)u, cols, (const float*)taps, (float*)state, state_stride, (const int32_t*)token_seq,                    \
            (const int32_t*)cu_tokens, (const int32_t*)seq_slots, (float*)q, (float*)k, (float*)v, N, run, G, dim, H, vdim,   \
            unit_eps, q_scale);                                                                                               \
        return true;
    switch (J) {
        DELTA_CONV_CASE(1)
        DELTA_CONV_CASE(2)
        DELTA_CONV_CASE(3)
        DELTA_CONV_CASE(4)
        DELTA_CONV_CASE(5)
        DELTA_CONV_CASE(6)
        DELTA_CONV_CASE(7)
        DELTA_CONV_CASE(8)
    }
#undef DELTA_CONV_CASE
    return false;  // more taps: a workgroup a token
}

extern "C" int lle_delta_conv_max_advance(void) { return 8; }

// `advance` != 0: every request of the step has one token, and its kept rows move on (J up to lle_delta_conv_max_advance)
extern "C" int lle_delta_conv(const void* u, int cols, const void* taps, int J, void* state, int64_t state_stride,
                              const void* token_seq, const void* cu_tokens, const void* seq_slots, void* q, void* k, void* v,
                              int N, int G, int dim, int H, int vdim, float unit_eps, float q_scale, int advance, int dtype,
                              hipStream_t stream) {
    if (N <= 0) return 0;
    if (advance && J > 8) return (int)hipErrorInvalidValue;
    if (J < 1 || (J > 1 && state == nullptr) || G <= 0 || H <= 0 || dim <= 0 || vdim <= 0 || dim > 4 * LLE_WAVE ||
        vdim > 4 * LLE_WAVE || cols != 2 * G * dim + H * vdim || (2 * G + H + 3) / 4 > 65535)
        return (int)hipErrorInvalidValue;
    auto runs = [&](auto kernel) {
        return kernel(u, cols, taps, J, state, state_stride, token_seq, cu_tokens, seq_slots, q, k, v, N, G, dim, H, vdim, unit_eps,
                      q_scale, stream);
    };
    if (dtype == LLE_F32 ? (advance ? runs(delta_conv_runs<float, true>) : runs(delta_conv_runs<float, false>))
                         : (advance ? runs(delta_conv_runs<bf16_t, true>) : runs(delta_conv_runs<bf16_t, false>)))
        LLE_RETURN_LAUNCH_STATUS();
    const dim3 grid(N, (2 * G + H + 3) / 4);
    if (dtype == LLE_F32)
        delta_conv_kernel<float><<<grid, 256, 0, stream>>>((const float*)u, cols, (const float*)taps, J, (const float*)state,
                                                            state_stride, (const int32_t*)token_seq, (const int32_t*)cu_tokens,
                                                            (const int32_t*)seq_slots, (float*)q, (float*)k, (float*)v, G, dim,
                                                            H, vdim, unit_eps, q_scale);
    else
        delta_conv_kernel<bf16_t><<<grid, 256, 0, stream>>>((const bf16_t*)u, cols, (const float*)taps, J,
                                                             (const float*)state, state_stride, (const int32_t*)token_seq,
                                                             (const int32_t*)cu_tokens, (const int32_t*)seq_slots, (float*)q,
                                                             (float*)k, (float*)v, G, dim, H, vdim, unit_eps, q_scale);
    LLE_RETURN_LAUNCH_STATUS();
}

// ---------------------------------------------------------------------------------
// The walk.
// ---------------------------------------------------------------------------------
struct DeltaArgs {
    const float* q;        // [N, G dim]
    const float* k;        // [N, G dim]
    const float* v;        // [N, H vdim]
    const float* ba;       // rows of ba_cols: beta's input of every head, then (one decay per head) the decay's
    int ba_cols;
    const float* a_log;    // [H]
    const float* dt_bias;  // [H]
    float* state;          // rows of state_stride floats: [H][vdim][dim]
    int64_t state_stride;
    const int32_t* seq_slots;
    const int32_t* cu_tokens;
    float* out;            // [N, H vdim]
    int H, G, dim, vdim;
    const float* gates;    // [N, 2 H]: decay and beta of every token and head, made ahead (or null: made in the walk)
    const float* decay;    // [N, H dim]: the decays of every key channel (or null: one per head, as above)
    int S;
    int most, few;         // requests of more than `most` tokens go in chunks where there are no more than `few` of them
};

// Whether request s of a step goes in chunks (few: not at all), the same for every wavefront that asks
__device__ __forceinline__ bool delta_in_chunks(const DeltaArgs& a, int tokens) {
    if (tokens <= a.most || a.few <= 0) return false;
    int count = 0;
    for (int s0 = 0; s0 < a.S; s0 += LLE_WAVE) {
        const int s = min(s0 + (int)threadIdx.x % LLE_WAVE, a.S - 1);
        count += __popcll(__ballot(s0 + (int)threadIdx.x % LLE_WAVE < a.S && a.cu_tokens[s + 1] - a.cu_tokens[s] > a.most));
    }
    return count <= a.few;
}

// decay and beta of every token and head, for the walks of long portions: in the walk itself the exponentials and the
// logarithm of a chunk's sixteen tokens are one wavefront's work while the other three wait (a ninth of the walk's time)
__global__ __launch_bounds__(256) void delta_gates_kernel(const float* __restrict__ ba, int ba_cols, const float* __restrict__ a_log,
                                                           const float* __restrict__ dt_bias, float* __restrict__ gates,
                                                           int64_t total, int H) {
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= total) return;
    const int64_t n = idx / H;
    const int h = (int)(idx - n * H);
    const float x = ba[n * ba_cols + H + h] + dt_bias[h];
    const float softplus = fmaxf(x, 0.f) + log1pf(expf(-fabsf(x)));
    gates[n * 2 * H + h] = expf(-expf(a_log[h]) * softplus);
    gates[n * 2 * H + H + h] = 1.0f / (1.0f + expf(-ba[n * ba_cols + h]));
}

template <int CTRL>
__device__ __forceinline__ float delta_lanes(float x) {  // x of the lane that the pattern names
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, 0xf, 0xf, true));
}

// the sum over the 16 lanes of a column, in every one of them (each step adds the same two numbers in both lanes)
__device__ __forceinline__ float delta_row_sum(float x) {
    x += delta_lanes<0x140>(x);  // the row of sixteen mirrored
    x += delta_lanes<0x141>(x);  // every eight mirrored
    x += delta_lanes<0x4E>(x);   // lanes 2 3 0 1 of every four
    x += delta_lanes<0xB1>(x);   // lanes 1 0 3 2 of every four
    return x;
}

// The same sums for sixteen tokens at once, token t's in lane t: at every step a lane hands the half
// of its sums that it does not end with to the lane that does, so 15 exchanges do for 16 tokens what 64 do one by one.
template <int CTRL, int M>
__device__ __forceinline__ void delta_fold(float (&r)[DELTA_TC], bool upper) {
#pragma unroll
    for (int t = 0; t < M; ++t) r[t] = (upper ? r[t + M] : r[t]) + delta_lanes<CTRL>(upper ? r[t] : r[t + M]);
}
__device__ __forceinline__ float delta_row_sums(float (&r)[DELTA_TC], int ig) {
    delta_fold<0x140, 8>(r, ig & 8);
    delta_fold<0x141, 4>(r, ig & 4);
    delta_fold<0x4E, 2>(r, ig & 2);
    delta_fold<0xB1, 1>(r, ig & 1);
    return r[0];
}

// What a thread reads of one staged token: its share of k and q (CHANNEL: and of the channels' decays).
template <int KI, bool CHANNEL>
struct DeltaToken {
    float kk[KI], qq[KI], gg[CHANNEL ? KI : 1];
};

template <int N, int STEP = 4>
__device__ __forceinline__ void delta_copy(float* d, const float* __restrict__ p) {  // N aligned floats, four by four STEP apart
    typedef float vec __attribute__((ext_vector_type(N < 4 ? N : 4)));
#pragma unroll
    for (int i = 0; i < N; i += 4) {
        const vec x = *(const vec*)(p + i / 4 * STEP);
        if constexpr (N == 1) d[0] = ((const float*)p)[0];
        else
#pragma unroll
            for (int e = 0; e < (N < 4 ? N : 4); ++e) d[i + e] = x[e];
    }
}

// kt, qt, gt: where the lane's share begins (KI <= 2: q lies right behind k, one load for both)
template <int KI, bool CHANNEL>
__device__ __forceinline__ void delta_read(DeltaToken<KI, CHANNEL>& d, const float* __restrict__ kt, const float* __restrict__ qt,
                                           const float* __restrict__ gt) {
    if constexpr (CHANNEL) delta_copy<KI, 4 * DELTA_IG>(d.gg, gt);
    if constexpr (KI <= 2) {
        float both[2 * KI];
        delta_copy<2 * KI>(both, kt);
#pragma unroll
        for (int ii = 0; ii < KI; ++ii) d.kk[ii] = both[ii], d.qq[ii] = both[KI + ii];
    } else {
        delta_copy<KI, 4 * DELTA_IG>(d.kk, kt);
        delta_copy<KI, 4 * DELTA_IG>(d.qq, qt);
    }
}

// One token of the walk for this thread's share of column j: the sum over the key channels, the lanes' exchange, the
// correction; returns the thread's share of the read-out.
template <int KI, bool CHANNEL>
__device__ __forceinline__ float delta_token(float (&S)[KI], const DeltaToken<KI, CHANNEL>& d, float g, float beta, float v) {
    float p = 0.f, r = 0.f;
#pragma unroll
    for (int ii = 0; ii < KI; ++ii) {
        S[ii] *= CHANNEL ? d.gg[ii] : g;  // (CHANNEL: the rows of S decay each at their own rate)
        p = fmaf(S[ii], d.kk[ii], p);
    }
    const float w = beta * (v - delta_row_sum(p));
#pragma unroll
    for (int ii = 0; ii < KI; ++ii) {
        S[ii] = fmaf(d.kk[ii], w, S[ii]);
        r = fmaf(S[ii], d.qq[ii], r);
    }
    return r;
}

// grid = (blocks of DELTA_VB value channels, heads, requests): neighbouring workgroups, which go to the dies in turn, are one request's (with the
// requests in front, one of 256 tokens behind 31 single ones had all its workgroups on one die and took 172 us instead of 42).  Thread (jl, ig) = (tid / 16, tid % 16) owns KI key channels
// of column j = block DELTA_VB + jl, four neighbours of every 64 (fewer than four: ig KI + 0 .. KI - 1), so that a wavefront's
// 16-byte loads of k, q, decays and state lie one beside the other: no bank is asked twice, the state's lines are read whole.
// The tokens pass through LDS DELTA_TC at a time, in two buffers (one for heads over 128 channels): the next chunk goes to LDS
// and the one behind it is asked for before the current chunk is walked, one barrier a chunk, and inside a chunk every token's
// operands leave LDS one token ahead of their use.  The read-outs of a chunk are added over the lanes together, at its end, and
// leave from the registers, the lane's whose number the token has.
// Long requests go in chunks instead where they are few (below).  What bounds a long walk is the chain of a token (the four exchanges of S^T k and what stands around them, 101 ns) in the
// two wavefronts that 32 heads of 64 x 64 leave a CU.  Measured with a decay per channel, 32 heads of 64 x 64: 2048 tokens
// 237 -> 207 us, single tokens of 8 requests 5.0 -> 4.05, of 64 26.0 -> 21.6; one decay a head, 32 heads of 128 x 128: 2048
// tokens 301 -> 285, single tokens of 8 requests 23.3 -> 10.8, of 32 83.5 -> 34.4; 16 of 256 x 128: 2048 tokens 586 -> 452,
// single tokens of 32 requests 112 -> 32, against every read-out added up by itself and a thread's channels in one stretch.
// Tried and not kept: three barriers a chunk and k . q made ahead of the walk; operands read two or three tokens ahead, or all
// of them at a chunk's start; 32 lanes a column (heads of 64: 265 us, of 256: 381 us, but their single tokens 47).
template <int KI, bool CHANNEL>
__global__ __launch_bounds__(DELTA_THREADS) void delta_scan_kernel(DeltaArgs a) {
    constexpr int KD = KI * DELTA_IG;
    constexpr int PER = DELTA_TC * KD / DELTA_THREADS;  // elements of q (and of k) of a chunk that a thread fetches
    static_assert(DELTA_TC * KD % DELTA_THREADS == 0, "a chunk's q and k are dealt to the threads in equal shares");
    static_assert(KI >= 4 || PER < 4, "heads whose k and q lie beside each other are staged one by one");
    static_assert(DELTA_TC == DELTA_IG, "every lane of a column takes one token's read-out");
    constexpr int BUFS = KD <= 128 ? 2 : 1;
    constexpr bool BOTH = KI <= 2;  // k and q lie lane by lane beside each other
    __shared__ __attribute__((aligned(16))) float s_kq[BUFS][DELTA_TC][2 * KD];
    __shared__ __attribute__((aligned(16))) float s_g[CHANNEL ? BUFS : 1][CHANNEL ? DELTA_TC : 1][CHANNEL ? KD : 4];
    __shared__ __attribute__((aligned(16))) float s_par[BUFS][2][DELTA_TC];  // betas, decays of the staged tokens
    __shared__ __attribute__((aligned(16))) float s_v[BUFS][DELTA_VB][DELTA_TC + 4];
    const int s = blockIdx.z, h = blockIdx.y;
    const int tid = threadIdx.x, jl = tid / DELTA_IG, ig = tid % DELTA_IG;
    const int j0 = blockIdx.x * DELTA_VB, j = j0 + jl;
    const int dim = a.dim, vdim = a.vdim, H = a.H;
    const int hk = h / (H / a.G), GD = a.G * dim, HV = H * vdim;
    [[maybe_unused]] const int HD = H * dim;
    const int q0 = a.cu_tokens[s], q1 = a.cu_tokens[s + 1];
    if (q1 <= q0 || delta_in_chunks(a, q1 - q0)) return;
    float* col = a.state + (int64_t)a.seq_slots[s] * a.state_stride + ((int64_t)h * vdim + j) * dim;
    const bool live = j < vdim;
    constexpr int AT = KI < 4 ? KI : 4, STEP = 4 * DELTA_IG;  // a thread's key channels are m STEP + ig AT + 0 .. AT - 1
    const bool whole = KI >= 4 && dim == KD && a.state_stride % 4 == 0 && ((uintptr_t)a.state & 15) == 0;  // 16 bytes a load
    float S[KI];
    if (whole && live) {
        delta_copy<KI, STEP>(S, col + ig * AT);
    } else {
#pragma unroll
        for (int ii = 0; ii < KI; ++ii) {
            const int i = ii / 4 * STEP + ig * AT + ii % 4;
            S[ii] = (live && i < dim) ? col[i] : 0.f;
        }
    }
    const float decay_rate = CHANNEL ? 0.f : expf(a.a_log[h]), dt_bias = CHANNEL ? 0.f : a.dt_bias[h];

    float fq[PER], fk[PER], fg[CHANNEL ? PER : 1], fv = 0.f, fb = 0.f, fa = 0.f;  // the chunk that is on its way
    const bool wide = PER % 4 == 0 && dim == KD;  // whole heads of a multiple of 64 channels: 16 bytes a load and a store
    auto fetch = [&](int c0, int nt) {
        if (wide) {
#pragma unroll
            for (int r = 0; r + 3 < PER; r += 4) {
                const int e = (tid + DELTA_THREADS * (r / 4)) * 4, t = e / KD, i = e - t * KD;
                float4 x = float4{0.f, 0.f, 0.f, 0.f}, y = x;
                if constexpr (CHANNEL) {
                    float4 z = x;
                    if (t < nt) z = *(const float4*)(a.decay + (int64_t)(c0 + t) * HD + h * dim + i);
                    fg[r] = z.x, fg[r + 1] = z.y, fg[r + 2] = z.z, fg[r + 3] = z.w;
                }
                if (t < nt) {
                    const int64_t at = (int64_t)(c0 + t) * GD + hk * dim + i;
                    x = *(const float4*)(a.q + at);
                    y = *(const float4*)(a.k + at);
                }
                fq[r] = x.x, fq[r + 1] = x.y, fq[r + 2] = x.z, fq[r + 3] = x.w;
                fk[r] = y.x, fk[r + 1] = y.y, fk[r + 2] = y.z, fk[r + 3] = y.w;
            }
        } else {
#pragma unroll
            for (int r = 0; r < PER; ++r) {
                const int e = tid + DELTA_THREADS * r, t = e / KD, i = e - t * KD;
                const bool there = t < nt && i < dim;
                const int64_t at = (int64_t)(c0 + t) * GD + hk * dim + i;
                fq[r] = there ? a.q[at] : 0.f;
                fk[r] = there ? a.k[at] : 0.f;
                if constexpr (CHANNEL) fg[r] = there ? a.decay[(int64_t)(c0 + t) * HD + h * dim + i] : 0.f;
            }
        }
        {  // the chunk's values of the workgroup's columns: one element a thread (one load a lane and token, sixteen
           // lanes asking for the same word, kept the memory pipeline busy for longer than the walk itself)
            const int t = tid / DELTA_VB, e = tid % DELTA_VB;
            fv = (t < nt && j0 + e < vdim) ? a.v[(int64_t)(c0 + t) * HV + h * vdim + j0 + e] : 0.f;
        }
        if (tid < nt) {  // (with gates made ahead: beta, then the decay itself)
            if constexpr (CHANNEL) {
                fb = a.ba[(int64_t)(c0 + tid) * a.ba_cols + h];
            } else {
                const float* ba = a.gates ? a.gates + (int64_t)(c0 + tid) * 2 * H : a.ba + (int64_t)(c0 + tid) * a.ba_cols;
                fb = a.gates ? ba[H + h] : ba[h];
                fa = a.gates ? ba[h] : ba[H + h];
            }
        }
    };
    auto stage = [&](int buf, int nt) {  // what was fetched goes to LDS
        if (wide) {
#pragma unroll
            for (int r = 0; r + 3 < PER; r += 4) {
                const int e = (tid + DELTA_THREADS * (r / 4)) * 4, t = e / KD, i = e - t * KD;
                float* kq = s_kq[buf][t];
                *(float4*)(kq + i) = float4{fk[r], fk[r + 1], fk[r + 2], fk[r + 3]};
                *(float4*)(kq + KD + i) = float4{fq[r], fq[r + 1], fq[r + 2], fq[r + 3]};
                if constexpr (CHANNEL) *(float4*)&s_g[buf][t][i] = float4{fg[r], fg[r + 1], fg[r + 2], fg[r + 3]};
            }
        } else {
#pragma unroll
            for (int r = 0; r < PER; ++r) {
                const int e = tid + DELTA_THREADS * r, t = e / KD, i = e - t * KD;
                const int at = BOTH ? i / KI * 2 * KI + i % KI : i;
                s_kq[buf][t][at] = fk[r];
                s_kq[buf][t][at + (BOTH ? KI : KD)] = fq[r];
                if constexpr (CHANNEL) s_g[buf][t][i] = fg[r];
            }
        }
        if (tid < nt) {
            float2 par = {1.0f, 0.f};
            if (CHANNEL) {
                par.y = 1.0f / (1.0f + expf(-fb));
            } else if (a.gates) {
                par = float2{fa, fb};
            } else {
                const float x = fa + dt_bias;
                const float softplus = fmaxf(x, 0.f) + log1pf(expf(-fabsf(x)));
                par = float2{expf(-decay_rate * softplus), 1.0f / (1.0f + expf(-fb))};
            }
            s_par[buf][0][tid] = par.y;
            s_par[buf][1][tid] = par.x;
        }
        s_v[buf][tid % DELTA_VB][tid / DELTA_VB] = fv;
    };
    auto count = [&](int c0) { return min(DELTA_TC, q1 - c0); };
    fetch(q0, count(q0));
    stage(0, count(q0));
    if (q0 + DELTA_TC < q1) fetch(q0 + DELTA_TC, count(q0 + DELTA_TC));
    __syncthreads();

    int buf = 0;
    for (int c0 = q0; c0 < q1; c0 += DELTA_TC) {
        const int nt = count(c0), c1 = c0 + DELTA_TC, c2 = c1 + DELTA_TC;
        if (BUFS == 2 && c1 < q1) {
            stage(buf ^ 1, count(c1));
            if (c2 < q1) fetch(c2, count(c2));
        }
        float vv[DELTA_TC], beta[DELTA_TC], g[DELTA_TC];
        delta_copy<DELTA_TC>(vv, s_v[buf][jl]);
        delta_copy<DELTA_TC>(beta, s_par[buf][0]);
        if constexpr (!CHANNEL) delta_copy<DELTA_TC>(g, s_par[buf][1]);
        else
#pragma unroll
            for (int t = 0; t < DELTA_TC; ++t) g[t] = 1.f;
        const float* kt = &s_kq[buf][0][ig * AT * (BOTH ? 2 : 1)];
        const float* qt = kt + KD;  // (not BOTH)
        constexpr int GS = CHANNEL ? KD : 0, KS = 2 * KD;
        const float* gt = CHANNEL ? &s_g[buf][0][ig * AT] : &s_g[0][0][0];
        float out = 0.f;  // of token ig
        if (nt == DELTA_TC) {  // a whole chunk: nothing under a condition, every token's operands read a token ahead
            DeltaToken<KI, CHANNEL> cur, nxt;
            float r[DELTA_TC];
            delta_read<KI, CHANNEL>(cur, kt, qt, gt);
#pragma unroll
            for (int t = 0; t < DELTA_TC; ++t) {
                if (t + 1 < DELTA_TC) delta_read<KI, CHANNEL>(nxt, kt + (t + 1) * KS, qt + (t + 1) * KS, gt + (t + 1) * GS);
                r[t] = delta_token<KI, CHANNEL>(S, cur, g[t], beta[t], vv[t]);
                cur = nxt;
            }
            out = delta_row_sums(r, ig);
        } else {
#pragma unroll
            for (int t = 0; t < DELTA_TC; ++t) {
                if (t < nt) {
                    DeltaToken<KI, CHANNEL> cur;
                    delta_read<KI, CHANNEL>(cur, kt + t * KS, qt + t * KS, gt + t * GS);
                    const float o = delta_row_sum(delta_token<KI, CHANNEL>(S, cur, g[t], beta[t], vv[t]));
                    out = ig == t ? o : out;
                }
            }
        }
        if (ig < nt && live) a.out[(int64_t)(c0 + ig) * HV + h * vdim + j] = out;
        __syncthreads();  // this chunk has been read, and the next one is in LDS
        if (BUFS == 2) {
            buf ^= 1;
        } else if (c1 < q1) {
            stage(0, count(c1));
            if (c2 < q1) fetch(c2, count(c2));
            __syncthreads();
        }
    }
    if (whole && live) {
#pragma unroll
        for (int ii = 0; ii + 3 < KI; ii += 4) *(float4*)(col + ii / 4 * STEP + ig * AT) = float4{S[ii], S[ii + 1], S[ii + 2], S[ii + 3]};
    } else if (live) {
#pragma unroll
        for (int ii = 0; ii < KI; ++ii) {
            const int i = ii / 4 * STEP + ig * AT + ii % 4;
            if (i < dim) col[i] = S[ii];
        }
    }
}

#define DELTA_MAX_DIM (16 * DELTA_IG)
#define DELTA_GRID_Z 65535  // most requests of a launch
extern "C" int lle_delta_max_dim(void) { return DELTA_MAX_DIM; }

// q, k float32 [N, G dim] (unit vectors, q scaled), v float32 [N, H vdim], ba float32 [N, 2 H], a_log and dt_bias
// float32 [H]; state float32 rows of `state_stride` floats whose first H vdim dim hold the heads' states transposed;
// out float32 [N, H vdim]; `gates` (or null) scratch float32 [N, 2 H] for the decays and betas made ahead of the walk.
// Where there are `few` requests of more than `most` tokens or fewer, they are left alone: lle_delta_chunks takes them (few = 0: it is not called).
// `decay` float32 [N, H dim] (or null): the decays of every key channel; then ba (rows of ba_cols floats) holds beta's
// inputs alone, and a_log, dt_bias and gates are not used.
extern "C" int lle_delta_scan(const void* q, const void* k, const void* v, const void* ba, int ba_cols, const void* decay,
                              const void* a_log, const void* dt_bias, void* state, int64_t state_stride, const void* seq_slots,
                              const void* cu_tokens, void* out, int S, int H, int G, int dim, int vdim, void* gates, int N, int most, int few,
                              hipStream_t stream) {
    if (S <= 0 || H <= 0) return 0;
    if (G <= 0 || H % G || dim <= 0 || dim > DELTA_MAX_DIM || vdim <= 0 || H > 65535 || (few > 0 && S > DELTA_GRID_Z))
        return (int)hipErrorInvalidValue;
    if (ba_cols < (decay ? H : 2 * H)) return (int)hipErrorInvalidValue;
    DeltaArgs a{(const float*)q, (const float*)k, (const float*)v, (const float*)ba, ba_cols, (const float*)a_log,
                (const float*)dt_bias, (float*)state, state_stride, (const int32_t*)seq_slots, (const int32_t*)cu_tokens,
                (float*)out, H, G, dim, vdim, (const float*)gates, (const float*)decay, S, most, few};
    if (gates != nullptr && decay == nullptr) {  // scratch float32 [N, 2 H], given for steps with long portions
        const int64_t total = (int64_t)N * H;
        delta_gates_kernel<<<(int)((total + 255) / 256), 256, 0, stream>>>((const float*)ba, ba_cols, (const float*)a_log,
                                                                            (const float*)dt_bias, (float*)gates, total, H);
    }
    auto launch = [&](auto kernel) {  // (more requests than the grid's third dimension holds: one launch after the other)
        for (int s0 = 0; s0 < S; s0 += DELTA_GRID_Z) {
            a.seq_slots = (const int32_t*)seq_slots + s0;
            a.cu_tokens = (const int32_t*)cu_tokens + s0;
            a.S = min(DELTA_GRID_Z, S - s0);
            kernel<<<dim3((vdim + DELTA_VB - 1) / DELTA_VB, H, a.S), DELTA_THREADS, 0, stream>>>(a);
        }
        LLE_RETURN_LAUNCH_STATUS();
    };
#define DELTA_CASE(KI) \
    if (dim <= KI * DELTA_IG) return decay ? launch(delta_scan_kernel<KI, true>) : launch(delta_scan_kernel<KI, false>);
    DELTA_CASE(1)
    DELTA_CASE(2)
    DELTA_CASE(4)
    DELTA_CASE(8)
    DELTA_CASE(16)
#undef DELTA_CASE
    return (int)hipErrorInvalidValue;
}

// ---------------------------------------------------------------------------------
// Long portions: the same recurrence in chunks of sixteen tokens.  With c_t the product of a chunk's decays up to token t (per key
// channel), S the state before the chunk and r(t, j) = g_{j+1} ... g_t,
//   L[t][j] = k_t . (r(t, j) k_j)  (j < t),   A[t][j] = q_t . (r(t, j) k_j)  (j <= t)
//   w_t = beta_t (v_t - (c_t k_t)^T S - sum_{j < t} L[t][j] w_j)
//   o_t = (c_t q_t)^T S + sum_{j <= t} A[t][j] w_j,   S <- diag(c_16) S + sum_j (r(16, j) k_j) w_j^T
// The w_t are linear in S, so everything that does not need S is made by one launch for all chunks at once
// (delta_chunk_kernel): X and U with w = U - X S, row t of both by the forward substitution of the line for w_t.  What is
// left to walk is a chunk at a time, three small products (delta_chunk_walk_kernel).  Products of decays are taken as they are, never as
// quotients: a decay of 0 is as good as any.  All of it in 32 bits, the products on the float32 matrix instruction.
//
// A chunk's unit in `work`, float32: X [16][dim], c q [16][dim], r(16, j) k_j [dim][16], A [16][16], c_16 [dim], U [columns][16] (whole
// sixteens of value channels).  Request s has the chunks cu_tokens[s] / 16 + s and on, so that every request's are found without
// a table.
// ---------------------------------------------------------------------------------
typedef float delta_vec4 __attribute__((ext_vector_type(4)));

static constexpr int delta_unit_floats(int dim, int vdim) { return 3 * DELTA_TC * dim + DELTA_TC * DELTA_TC + dim + DELTA_TC * ((vdim + 15) / 16 * 16); }

// grid = (chunks, heads).  Thread (j, ig) = (tid / 16, tid % 16) follows r(t, j) k_j over its 4 KT channels through the chunk's tokens; its
// shares of L[., j] and A[., j] are added over the row of sixteen lanes in one go.  Then a thread a column of X and of U.
template <int KT, bool CHANNEL>
__global__ __launch_bounds__(DELTA_THREADS) void delta_chunk_kernel(DeltaArgs a, int chunks, float* __restrict__ work) {
    constexpr int KD = 64 * KT, TC = DELTA_TC;
    __shared__ __attribute__((aligned(16))) float s_k[TC][KD], s_q[TC][KD], s_g[CHANNEL ? TC : 1][CHANNEL ? KD : TC];
    __shared__ __attribute__((aligned(16))) float s_l[TC][TC], s_beta[TC], s_kd[KD][TC + 1];
    const int h = blockIdx.y, tid = threadIdx.x;
    int s = 0;  // the last request whose chunks begin here or before
    for (int high = a.S - 1; s < high;) {
        const int mid = (s + high + 1) / 2;
        if (a.cu_tokens[mid] / TC + mid <= (int)blockIdx.x) s = mid;
        else high = mid - 1;
    }
    const int q0 = a.cu_tokens[s], q1 = a.cu_tokens[s + 1], c0 = q0 + ((int)blockIdx.x - q0 / TC - s) * TC;
    if (c0 >= q1 || !delta_in_chunks(a, q1 - q0)) return;
    const int nt = min(TC, q1 - c0), hk = h / (a.H / a.G), GD = a.G * KD, HV = a.H * a.vdim;
    // behind the last token: k, q and beta 0, decays 1
#pragma unroll
    for (int r = 0; r < KT; ++r) {
        const int e = (tid + DELTA_THREADS * r) * 4, t = e / KD, i = e - t * KD;
        float4 x = float4{0.f, 0.f, 0.f, 0.f}, y = x, z = float4{1.f, 1.f, 1.f, 1.f};
        if (t < nt) {
            const int64_t at = (int64_t)(c0 + t) * GD + hk * KD + i;
            x = *(const float4*)(a.q + at);
            y = *(const float4*)(a.k + at);
            if constexpr (CHANNEL) z = *(const float4*)(a.decay + (int64_t)(c0 + t) * a.H * KD + h * KD + i);
        }
        *(float4*)&s_q[t][i] = x;
        *(float4*)&s_k[t][i] = y;
        if constexpr (CHANNEL) *(float4*)&s_g[t][i] = z;
    }
    if (tid < TC) {
        const float* ba = a.ba + (int64_t)(c0 + min(tid, nt - 1)) * a.ba_cols;
        s_beta[tid] = tid < nt ? 1.0f / (1.0f + expf(-ba[h])) : 0.f;
        if constexpr (!CHANNEL) {
            const float x = ba[a.H + h] + a.dt_bias[h], softplus = fmaxf(x, 0.f) + log1pf(expf(-fabsf(x)));
            s_g[0][tid] = tid < nt ? expf(-expf(a.a_log[h]) * softplus) : 1.f;
        }
    }
    // from here on thread c makes column c of X (c < KD) or column c - KD of U, which begins with v: asked for ahead of everything
    const int column = __builtin_amdgcn_readfirstlane(tid / LLE_WAVE) * LLE_WAVE < KD ? tid : tid - KD;
    const bool of_x = __builtin_amdgcn_readfirstlane(tid / LLE_WAVE) * LLE_WAVE < KD, of_u = !of_x && column < (a.vdim + 15) / 16 * 16;
    float y[TC];
    if (of_u) {
        const float* v = a.v + (int64_t)c0 * HV + h * a.vdim + min(column, a.vdim - 1);
#pragma unroll
        for (int t = 0; t < TC; ++t) y[t] = v[(int64_t)min(t, nt - 1) * HV];
    }
    float* unit = work + ((int64_t)h * chunks + blockIdx.x) * delta_unit_floats(KD, a.vdim);
    float *out_x = unit, *out_q = unit + TC * KD, *out_k = unit + 2 * TC * KD, *out_a = unit + 3 * TC * KD, *out_c = out_a + TC * TC, *out_u = out_c + KD;
    __syncthreads();
    {
        const int j = tid / TC, ig = tid % TC;
        delta_vec4 r[KT];
        float l[TC], p[TC];
#pragma unroll
        for (int m = 0; m < KT; ++m) r[m] = *(const delta_vec4*)&s_k[j][64 * m + 4 * ig];
#pragma unroll
        for (int t = 0; t < TC; ++t) {
            l[t] = p[t] = 0.f;
            if (t < tid / LLE_WAVE * 4) continue;  // (the wavefront's four j come later)
            float dl = 0.f, dp = 0.f;
#pragma unroll
            for (int m = 0; m < KT; ++m) {
                const delta_vec4 k = *(const delta_vec4*)&s_k[t][64 * m + 4 * ig], q = *(const delta_vec4*)&s_q[t][64 * m + 4 * ig];
                delta_vec4 g;
                if constexpr (CHANNEL) g = *(const delta_vec4*)&s_g[t][64 * m + 4 * ig];
                else g = delta_vec4{s_g[0][t], s_g[0][t], s_g[0][t], s_g[0][t]};
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    r[m][e] *= t > j ? g[e] : 1.f;
                    dl = fmaf(r[m][e], k[e], dl);
                    dp = fmaf(r[m][e], q[e], dp);
                }
            }
            l[t] = t > j ? dl : 0.f;
            p[t] = t >= j ? dp : 0.f;
        }
        s_l[ig][j] = delta_row_sums(l, ig);
        out_a[ig * TC + j] = delta_row_sums(p, ig);
#pragma unroll
        for (int m = 0; m < KT; ++m)
#pragma unroll
            for (int e = 0; e < 4; ++e) s_kd[64 * m + 4 * ig + e][j] = r[m][e];
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 4 * KT; ++r) {
        const int e = tid + DELTA_THREADS * r;
        out_k[e] = s_kd[e / TC][e % TC];
    }
    auto substitute = [&]() {
#pragma unroll
        for (int t = 0; t < TC; ++t) {
            float sum = y[t];
#pragma unroll
            for (int i = 0; i < t; ++i) sum = fmaf(-s_l[t][i], y[i], sum);
            y[t] = s_beta[t] * sum;
        }
    };
    if (of_x) {
        float cum = 1.f;
#pragma unroll
        for (int t = 0; t < TC; ++t) {
            if constexpr (CHANNEL) cum *= s_g[t][column];
            else cum *= s_g[0][t];
            y[t] = cum * s_k[t][column];
            out_q[t * KD + column] = cum * s_q[t][column];
        }
        out_c[column] = cum;
        substitute();
#pragma unroll
        for (int t = 0; t < TC; ++t) out_x[t * KD + column] = y[t];
    } else if (of_u) {
#pragma unroll
        for (int t = 0; t < TC; ++t) y[t] = t < nt && column < a.vdim ? y[t] : 0.f;
        substitute();
#pragma unroll
        for (int t = 0; t < TC; t += 4) *(float4*)(out_u + column * TC + t) = float4{y[t], y[t + 1], y[t + 2], y[t + 3]};
    }
}

// grid = (sixteens of value channels, heads, requests).  The first NW wavefronts carry the state, one for every sixteen key channels: it keeps
// its tile of S, rows 4 c + e and column r in lane (c, r), element e, which is the operand of a product over the key channels as it
// lies; so are the w_t for one over the tokens.  Their shares of X S meet in LDS (two buffers, one barrier a chunk), AHEAD chunks of operands are
// on their way.  The other NW wavefronts take the read-outs of every NW-th chunk each, a tile of S in the time of a chunk: a wavefront issues
// in order, so what is not on the chain S -> X S -> LDS -> w -> S is not in the chain's wavefronts.
// What bounds it is that chain, 0.48 us a chunk (16 of the float32 matrix instruction's 32 cycles, a barrier, the trip through LDS): with
// every wavefront taking its share of the read-outs 0.53, with a barrier that waits for loads 0.74; operands that are never
// further than L2 change nothing.  32 heads of 64 x 64 with a decay per channel: the chunks' launch 29 us and this one 59 for 2048 tokens (31 and
// 72 behind a prompt's other launches, which leave no operand in a cache), walked 207.  A chunk whose corrections are not finite has its rows made one after the other.
template <int NW, int AHEAD>
__global__ __launch_bounds__(2 * NW * LLE_WAVE, NW / 2) void delta_chunk_walk_kernel(DeltaArgs a, int chunks, const float* __restrict__ work) {
    constexpr int KD = 16 * NW, TC = DELTA_TC;
    __shared__ __attribute__((aligned(16))) float s_p[2][NW][256], s_s[2][NW][256];  // X S of every sixteen key channels, S
    const int s = blockIdx.z, h = blockIdx.y;
    const int q0 = a.cu_tokens[s], q1 = a.cu_tokens[s + 1];
    if (!delta_in_chunks(a, q1 - q0)) return;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / LLE_WAVE), lane = threadIdx.x % LLE_WAVE, c = lane / 16, r = lane % 16;
    const int j = blockIdx.x * 16 + r;
    const int unit = delta_unit_floats(KD, a.vdim), n = (q1 - q0 + TC - 1) / TC;
    // (a buffer's address and the chunk's offset are the wavefront's, so that a load takes no additions of 64 bits)
    const __amdgpu_buffer_rsrc_t units =
        __builtin_amdgcn_make_buffer_rsrc((void*)(work + ((int64_t)h * chunks + q0 / TC + s) * unit), 0, 4 * unit * n, 0x00020000);
    auto load = [&](int i, unsigned at) {  // (behind the last chunk: the last one again)
        return __builtin_bit_cast(delta_vec4, __builtin_amdgcn_raw_buffer_load_b128(units, 4 * at, 4 * unit * min(i, n - 1), 0));
    };
    const unsigned in_row = r * KD + 4 * c, in_k = 2 * TC * KD + (16 * wave + r) * TC + 4 * c, in_a = 3 * TC * KD + r * TC + 4 * c;
    const unsigned in_g = 3 * TC * KD + TC * TC + 16 * wave + 4 * c, in_u = 3 * TC * KD + TC * TC + KD + j * TC + 4 * c;
    auto meet = [&]() {  // (waits for no load on its way)
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    auto corrections = [&](const delta_vec4& u, int i) {  // w of chunk i
        delta_vec4 part[NW];
#pragma unroll
        for (int v = 0; v < NW; ++v) part[v] = *(const delta_vec4*)&s_p[i & 1][v][lane * 4];
#pragma unroll
        for (int v = 1; v < NW; ++v) part[0] += part[v];
        return u - part[0];
    };
    if (wave < NW) {
        const bool live = j < a.vdim;
        float* at = a.state + (int64_t)a.seq_slots[s] * a.state_stride + ((int64_t)h * a.vdim + min(j, a.vdim - 1)) * KD + 16 * wave + 4 * c;
        delta_vec4 St;
#pragma unroll
        for (int e = 0; e < 4; ++e) St[e] = at[e];
        struct Operands {
            delta_vec4 x, k, u, g;
        } ops[AHEAD];
        auto ask = [&](Operands& o, int i) {
            o.x = load(i, in_row + 16 * wave);
            o.u = load(i, in_u);
            o.g = load(i, in_g);
            o.k = load(i, in_k);
        };
        auto chunk = [&](Operands& now, int i) {
            delta_vec4 p = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int e = 0; e < 4; ++e) p = __builtin_amdgcn_mfma_f32_16x16x4f32(now.x[e], St[e], p, 0, 0, 0);
            *(delta_vec4*)&s_s[i & 1][wave][lane * 4] = St;
            St *= now.g;
            *(delta_vec4*)&s_p[i & 1][wave][lane * 4] = p;
            meet();
            const delta_vec4 w = corrections(now.u, i);
#pragma unroll
            for (int e = 0; e < 4; ++e) St = __builtin_amdgcn_mfma_f32_16x16x4f32(now.k[e], w[e], St, 0, 0, 0);
            ask(now, i + AHEAD);
        };
#pragma unroll
        for (int i = 0; i < AHEAD; ++i) ask(ops[i], i);
        int i0 = 0;
        for (; i0 + AHEAD <= n; i0 += AHEAD)
#pragma unroll
            for (int b = 0; b < AHEAD; ++b) chunk(ops[b], i0 + b);
#pragma unroll
        for (int b = 0; b < AHEAD - 1; ++b)
            if (i0 + b < n) chunk(ops[b], i0 + b);
        if (live)
#pragma unroll
            for (int e = 0; e < 4; ++e) at[e] = St[e];
        return;
    }
    const int mine = wave - NW;
    const int64_t HV = (int64_t)a.H * a.vdim;
    float* to = a.out + (q0 + mine * TC + 4 * c) * HV + h * a.vdim + j;
    for (int i = 0; i < min(mine, n); ++i) meet();
    for (int i = mine; i < n; i += NW) {
        delta_vec4 q[NW], S[NW];
#pragma unroll
        for (int v = 0; v < NW; ++v) q[v] = load(i, TC * KD + in_row + 16 * v);
        const delta_vec4 t = load(i, in_a), u = load(i, in_u);
        meet();
#pragma unroll
        for (int v = 0; v < NW; ++v) S[v] = *(const delta_vec4*)&s_s[i & 1][v][lane * 4];
        const delta_vec4 w = corrections(u, i);
        delta_vec4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int v = 0; v < NW; ++v) {
            if (v > 0 && i + v < n) meet();
#pragma unroll
            for (int e = 0; e < 4; ++e) o = __builtin_amdgcn_mfma_f32_16x16x4f32(q[v][e], S[v][e], o, 0, 0, 0);
        }
        bool odd = false;
#pragma unroll
        for (int e = 0; e < 4; ++e) odd = odd || !(fabsf(w[e]) < INFINITY);
        if (!__any(odd)) {
#pragma unroll
            for (int e = 0; e < 4; ++e) o = __builtin_amdgcn_mfma_f32_16x16x4f32(t[e], w[e], o, 0, 0, 0);
        } else {  // 0 times a later token's infinity would be NaN: row after row, without what the row does not see
            const delta_vec4 before = o;
#pragma unroll 1
            for (int row = 0; row < TC; ++row) {
                delta_vec4 all = before;
#pragma unroll
                for (int e = 0; e < 4; ++e) all = __builtin_amdgcn_mfma_f32_16x16x4f32(t[e], 4 * c + e <= row ? w[e] : 0.f, all, 0, 0, 0);
#pragma unroll
                for (int e = 0; e < 4; ++e) o[e] = 4 * c + e == row ? all[e] : o[e];
            }
        }
        const int left = q1 - (q0 + i * TC + 4 * c);
        if (j < a.vdim) {
            if (i < n - 1) {  // (the same for the wavefront: a whole chunk)
#pragma unroll
                for (int e = 0; e < 4; ++e) to[e * HV] = o[e];
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (e < left) to[e * HV] = o[e];
            }
        }
        to += NW * TC * HV;
    }
}

// Floats of `work` for a step of N tokens of S requests, or 0 where no chunks are made of such heads or of so many tokens.
extern "C" int lle_delta_chunk_floats(int N, int S, int H, int dim, int vdim) {
    if (N <= 0 || S <= 0 || S > DELTA_GRID_Z || H <= 0 || H > 65535 || vdim <= 0 || (dim != 64 && dim != 128) || dim + vdim > DELTA_THREADS) return 0;
    const int64_t floats = (int64_t)(N / DELTA_TC + S) * H * delta_unit_floats(dim, vdim);
    return floats <= 0x7fffffff ? (int)floats : 0;
}

// The requests of more than `most` tokens of lle_delta_scan (its arguments), where they are `few` or fewer; `work` float32 of lle_delta_chunk_floats, q, k, decay
// and work at 16 bytes.
extern "C" int lle_delta_chunks(const void* q, const void* k, const void* v, const void* ba, int ba_cols, const void* decay,
                                const void* a_log, const void* dt_bias, void* state, int64_t state_stride, const void* seq_slots,
                                const void* cu_tokens, void* out, int S, int H, int G, int dim, int vdim, int N, int most, int few, void* work,
                                hipStream_t stream) {
    if (S <= 0 || H <= 0 || N <= 0) return 0;
    if (lle_delta_chunk_floats(N, S, H, dim, vdim) == 0 || G <= 0 || H % G || ba_cols < (decay ? H : 2 * H) || most < 0 ||
        (((uintptr_t)q | (uintptr_t)k | (uintptr_t)decay | (uintptr_t)work) & 15))
        return (int)hipErrorInvalidValue;
    const DeltaArgs a{(const float*)q, (const float*)k, (const float*)v, (const float*)ba, ba_cols, (const float*)a_log,
                      (const float*)dt_bias, (float*)state, state_stride, (const int32_t*)seq_slots, (const int32_t*)cu_tokens,
                      (float*)out, H, G, dim, vdim, nullptr, (const float*)decay, S, most, few};
    const int chunks = N / DELTA_TC + S;
    const dim3 all(chunks, H), walk((vdim + 15) / 16, H, S);
    float* w = (float*)work;
    if (dim == 64) {
        if (decay) delta_chunk_kernel<1, true><<<all, DELTA_THREADS, 0, stream>>>(a, chunks, w);
        else delta_chunk_kernel<1, false><<<all, DELTA_THREADS, 0, stream>>>(a, chunks, w);
        delta_chunk_walk_kernel<4, 4><<<walk, 8 * LLE_WAVE, 0, stream>>>(a, chunks, w);
    } else {
        if (decay) delta_chunk_kernel<2, true><<<all, DELTA_THREADS, 0, stream>>>(a, chunks, w);
        else delta_chunk_kernel<2, false><<<all, DELTA_THREADS, 0, stream>>>(a, chunks, w);
        delta_chunk_walk_kernel<8, 4><<<walk, 16 * LLE_WAVE, 0, stream>>>(a, chunks, w);
    }
    LLE_RETURN_LAUNCH_STATUS();
}

// ---------------------------------------------------------------------------------
// What a delta rule with a decay per key channel makes of two small projections, each through a narrow middle:
//   decay[n][c] = exp(-exp(a_log[c / dim]) softplus(z + dt_bias[c])),  z = sum_r low[n][a_col + r] a2[c][r]
//   gate[n][c]  = sum_r low[n][g_col + r] g2[c][r]                     (its sigmoid is taken by the output norm)
// low float32 [N, low_cols], a2 float32 [CA, RA], g2 float32 [CG, RG]: RA and RG multiples of 16 (weights and the
// columns of `low` padded with zeros), every row 16-byte aligned.  Everything in 32-bit, on the 32-bit matrix
// instruction: a wavefront takes 16 tokens and NT tiles of 16 channels.  A lane (c, r) loads four neighbouring
// elements of the contraction of token r (channel r); element e is slot c of instruction e.  The result tile leaves it
// with token r and channels 4 c .. 4 c + 3.
// ---------------------------------------------------------------------------------
typedef float delta_f32x4 __attribute__((ext_vector_type(4)));

struct LowRankArgs {
    const float* low;
    int low_cols, a_col, g_col;
    const float* a2;
    int RA, CA;
    const float* g2;
    int RG, CG;
    const float* a_log;
    const float* dt_bias;
    int dim;
    float* decay;
    float* gate;
    int N;
};

// exp(-rate softplus(z)) in base 2: softplus(z) log2 e = max(z, 0) log2 e + log2(1 + x), x = e^-|z|; a small x takes the
// first terms of the series (1 + x would round them away)
__device__ __forceinline__ float delta_decay_of(float z, float rate) {
    const float x = __builtin_amdgcn_exp2f(-fabsf(z) * 1.44269504088896340736f);
    const float series = x * (1.f - x * (0.5f - x * 0.33333333333f)) * 1.44269504088896340736f;
    const float log2_1px = x < 0.01f ? series : __builtin_amdgcn_logf(1.0f + x);
    return __builtin_amdgcn_exp2f(-rate * fmaf(fmaxf(z, 0.f), 1.44269504088896340736f, log2_1px));
}

// grid = (blocks of channels: those of the decays, then those of the gates; tiles of 16 tokens in fours); a wavefront
// of the four has a token tile of its own
template <int NT>
__global__ __launch_bounds__(256) void low_rank_gates_kernel(LowRankArgs a) {
    const int wave = threadIdx.x / LLE_WAVE, lane = threadIdx.x % LLE_WAVE, c = lane / 16, r = lane % 16;
    const int n0 = (blockIdx.y * 4 + wave) * 16;
    if (n0 >= a.N) return;
    const int a_blocks = (a.CA + 16 * NT - 1) / (16 * NT);
    const bool decays = (int)blockIdx.x < a_blocks;
    const int c0 = (decays ? blockIdx.x : blockIdx.x - a_blocks) * 16 * NT;
    const int R = decays ? a.RA : a.RG, C = decays ? a.CA : a.CG;
    const float* w = decays ? a.a2 : a.g2;
    const float* x = a.low + (int64_t)min(n0 + r, a.N - 1) * a.low_cols + (decays ? a.a_col : a.g_col) + 4 * c;
    const float* wr[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n) wr[n] = w + (int64_t)min(c0 + 16 * n + r, C - 1) * R + 4 * c;
    delta_f32x4 acc[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n) acc[n] = delta_f32x4{0.f, 0.f, 0.f, 0.f};
    // (the next sixteen of the contraction are asked for before these are multiplied; past the end: the last ones again)
    delta_f32x4 xv = *(const delta_f32x4*)x, wv[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n) wv[n] = *(const delta_f32x4*)wr[n];
    for (int k = 0; k < R; k += 16) {
        const int next = min(k + 16, R - 16);
        const delta_f32x4 xn = *(const delta_f32x4*)(x + next);
        delta_f32x4 wn[NT];
#pragma unroll
        for (int n = 0; n < NT; ++n) wn[n] = *(const delta_f32x4*)(wr[n] + next);
#pragma unroll
        for (int n = 0; n < NT; ++n)
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[n] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[n][e], xv[e], acc[n], 0, 0, 0);
        xv = xn;
#pragma unroll
        for (int n = 0; n < NT; ++n) wv[n] = wn[n];
    }
    if (n0 + r >= a.N) return;
    float* dst = (decays ? a.decay : a.gate) + (int64_t)(n0 + r) * C;
#pragma unroll
    for (int n = 0; n < NT; ++n) {
        const int ch = c0 + 16 * n + 4 * c;
        float y[4];
        if (decays) {
            // four neighbouring channels of one head share its rate
            const int h = min(ch, C - 1) / a.dim;
            const float rate = expf(a.a_log[h]);
            const bool one_head = a.dim % 4 == 0;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int at = min(ch + e, C - 1);
                y[e] = delta_decay_of(acc[n][e] + a.dt_bias[at], one_head ? rate : expf(a.a_log[at / a.dim]));
            }
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) y[e] = acc[n][e];
        }
        if (C % 4 == 0) {
            if (ch < C) *(float4*)(dst + ch) = make_float4(y[0], y[1], y[2], y[3]);
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (ch + e < C) dst[ch + e] = y[e];
        }
    }
}

extern "C" int lle_low_rank_gates(const void* low, int low_cols, int a_col, int g_col, const void* a2, int RA, int CA,
                                  const void* g2, int RG, int CG, const void* a_log, const void* dt_bias, int dim, void* decay,
                                  void* gate, int N, hipStream_t stream) {
    if (N <= 0) return 0;
    if (low_cols % 4 || a_col % 4 || g_col % 4 || RA <= 0 || RA % 16 || RG % 16 || RG < 0 || CA <= 0 || CG < 0 || dim <= 0 ||
        CA % dim || a_col < 0 || g_col < 0 || a_col + RA > low_cols || g_col + RG > low_cols || (CG > 0 && RG == 0))
        return (int)hipErrorInvalidValue;
    const LowRankArgs a{(const float*)low, low_cols, a_col, g_col, (const float*)a2, RA, CA, (const float*)g2, RG, CG,
                        (const float*)a_log, (const float*)dt_bias, dim, (float*)decay, (float*)gate, N};
    const int rows = (N + 63) / 64;
    if (rows > 65535) return (int)hipErrorInvalidValue;
    // few tokens: a tile of channels a wavefront (more of them); many: four, which share the tokens' operands
    if (N <= 64) low_rank_gates_kernel<1><<<dim3((CA + 15) / 16 + (CG + 15) / 16, rows), 256, 0, stream>>>(a);
    else low_rank_gates_kernel<4><<<dim3((CA + 63) / 64 + (CG + 63) / 64, rows), 256, 0, stream>>>(a);
    LLE_RETURN_LAUNCH_STATUS();
}

// ---------------------------------------------------------------------------------
// y[n, h, :] = o / sqrt(mean(o^2) + eps) * norm_w * act(gate): a wavefront per (token, head);
// grid = (tokens, heads / 4).  norm_w [vdim] is one weight for all heads.  act: silu, or (SIGMOID) the sigmoid.
// ---------------------------------------------------------------------------------
template <typename T, typename TG, bool SIGMOID>
__global__ __launch_bounds__(256) void delta_out_norm_kernel(const float* __restrict__ o, const TG* __restrict__ gate,
                                                              const void* __restrict__ norm_w, int norm_dtype, float eps,
                                                              T* __restrict__ out, int H, int vdim) {
    const int64_t n = blockIdx.x;
    const int h = blockIdx.y * 4 + threadIdx.x / LLE_WAVE, lane = threadIdx.x % LLE_WAVE;
    if (h >= H) return;
    const int64_t at = (n * H + h) * vdim;
    float ss = 0.f;
    for (int e = lane; e < vdim; e += LLE_WAVE) ss = fmaf(o[at + e], o[at + e], ss);
    const float inv = 1.0f / sqrtf(wave_sum(ss) / (float)vdim + eps);
    for (int e = lane; e < vdim; e += LLE_WAVE) {
        const float z = to_f32<TG>(gate[at + e]);
        const float g = SIGMOID ? 1.0f / (1.0f + expf(-z)) : delta_silu(z);
        out[at + e] = from_f32<T>(o[at + e] * inv * load_as_f32(norm_w, e, norm_dtype) * g);
    }
}

// `gate_dtype`: the output's type, or float32; `sigmoid` != 0: the gate is its sigmoid, else its silu
extern "C" int lle_delta_out_norm(const void* o, const void* gate, int gate_dtype, int sigmoid, const void* norm_w, int norm_dtype,
                                  float eps, void* out, int N, int H, int vdim, int dtype, hipStream_t stream) {
    if (N <= 0 || H <= 0) return 0;
    if (vdim <= 0 || (H + 3) / 4 > 65535 || (gate_dtype != dtype && gate_dtype != LLE_F32)) return (int)hipErrorInvalidValue;
    const dim3 grid(N, (H + 3) / 4);
#define DELTA_OUT(T, TG, SIG)                                                                                                \
    delta_out_norm_kernel<T, TG, SIG><<<grid, 256, 0, stream>>>((const float*)o, (const TG*)gate, norm_w, norm_dtype, eps,   \
                                                                (T*)out, H, vdim)
    if (dtype == LLE_F32) {
        if (sigmoid) DELTA_OUT(float, float, true); else DELTA_OUT(float, float, false);
    } else if (gate_dtype == LLE_F32) {
        if (sigmoid) DELTA_OUT(bf16_t, float, true); else DELTA_OUT(bf16_t, float, false);
    } else {
        if (sigmoid) DELTA_OUT(bf16_t, bf16_t, true); else DELTA_OUT(bf16_t, bf16_t, false);
    }
#undef DELTA_OUT
    LLE_RETURN_LAUNCH_STATUS();
}
