// The state-space recurrence of Mamba-2: a matrix state per head with one decay per token and head.
//
//   c = silu(conv(u) + b)               per channel over time, J taps, the request's last J - 1 rows kept     ssd_conv
//   x, B, C = c's parts                 x [H vdim], B and C [G N]; head h reads group h / (H / G)
//   dt = softplus(d + dt_bias),  a = -exp(A_log) dt                 one of each per token and head            ssd_scan
//   S <- exp(a_t) S + dt_t B_t x_t^T;   y_t = S^T C_t + D x_t       S [N, vdim] float32, per head
//   out = norm(y * silu(z)) * w         the root mean square over each of `groups` equal parts of a row       ssd_gate_norm
//
// The state lies transposed in its row, [head][value j][state n].  Everything that enters the recurrence is 32-bit in
// every mode; u, z and out have the activation type.
//
// A request with few tokens in a step (SSD_WALK at most: decoded tokens, short portions) is walked token by token from
// its state.  A longer one is cut into chunks of SSD_CHUNK tokens that are worked on side by side.  With l_t the sum of
// a over the chunk's tokens up to t,
//   pass 1  every chunk's own contribution to the state, sum_s exp(l_last - l_s) dt_s B_s x_s^T, and exp(l_last)
//   carry   a short walk over the chunks leaves every chunk's entry state, and the request's state behind the last
//   pass 2  y_t = exp(l_t) S_entry^T C_t + sum_(s <= t) exp(l_t - l_s) (C_t . B_s) dt_s x_s + D x_t
// All exponents are at most zero.  The sums l are kept as two floats, so that the difference of two neighbours deep in
// a chunk is as exact as if it had been added up on its own.  The products are taken on the 32-bit matrix instruction.
#include "common.h"
#include <type_traits>

LLE_DEFINE_ERROR_STRING()

#define SSD_CHUNK 64
#define SSD_WALK 32
#define SSD_HEADS 32
typedef float ssd_f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float ssd_silu(float x) { return x / (1.0f + expf(-x)); }
__device__ __forceinline__ float ssd_softplus(float x) { return fmaxf(x, 0.f) + log1pf(expf(-fabsf(x))); }

// ---------------------------------------------------------------------------------
// Convolution and silu.  The channels are the columns col0 .. col0 + CC - 1 of u; a thread walks `run` tokens of one
// channel with its taps and the last J - 1 inputs in registers; where the request changes inside a run the window is
// filled anew.  `state` rows hold the last J - 1 inputs of earlier steps, oldest first (float32); zeros at admission
// stand for the zeros before a request's start.  ADVANCE (steps of single tokens only): the kept rows move on by the
// token in the same launch.  grid = (runs, blocks of 256 channels)
// ---------------------------------------------------------------------------------
struct SsdConvArgs {
    const void* u;
    int cols, col0;
    const float* taps;  // [CC, J]
    const float* bias;  // [CC] or null
    float* state;
    int64_t state_stride;
    const int32_t *token_seq, *cu_tokens, *seq_slots;
    float* out;  // [N, CC]
    int N, CC, J, run;
    // steps of single tokens: workgroups behind the convolution's make the step sizes' product, dt = x dt_w^T
    const void* x;     // [N, K] or null
    const void* dt_w;  // [H, K]
    float* dt;         // [N, H]
    int K, H, conv_blocks;
};

// dt[n, h] = sum_k x[n, k] dt_w[h, k] in 32-bit: a wavefront has one head and up to SSD_DT_TOKENS tokens
#define SSD_DT_TOKENS 4
template <typename T>
__device__ __forceinline__ void ssd_step_products(const SsdConvArgs& a, int block) {
    const int wave = block * 4 + threadIdx.x / LLE_WAVE, lane = threadIdx.x % LLE_WAVE;
    const int h = wave % a.H, n0 = wave / a.H * SSD_DT_TOKENS;
    if (n0 >= a.N) return;
    const T* w = (const T*)a.dt_w + (int64_t)h * a.K;
    const T* x = (const T*)a.x;
    float acc[SSD_DT_TOKENS];
#pragma unroll
    for (int t = 0; t < SSD_DT_TOKENS; ++t) acc[t] = 0.f;
#pragma unroll 4
    for (int k = lane; k < a.K; k += LLE_WAVE) {
        const float wv = to_f32<T>(w[k]);
#pragma unroll
        for (int t = 0; t < SSD_DT_TOKENS; ++t) acc[t] = fmaf(to_f32<T>(x[(int64_t)min(n0 + t, a.N - 1) * a.K + k]), wv, acc[t]);
    }
#pragma unroll
    for (int t = 0; t < SSD_DT_TOKENS; ++t) {
        const float sum = wave_sum(acc[t]);
        if (lane == 0 && n0 + t < a.N) a.dt[(int64_t)(n0 + t) * a.H + h] = sum;
    }
}

template <typename T, int J, bool ADVANCE>
__global__ __launch_bounds__(256) void ssd_conv_run_kernel(SsdConvArgs a) {
    constexpr int W = J > 1 ? J - 1 : 1;
    if (ADVANCE && (int)blockIdx.y >= a.conv_blocks) {
        ssd_step_products<T>(a, (blockIdx.y - a.conv_blocks) * gridDim.x + blockIdx.x);
        return;
    }
    const int ch = blockIdx.y * 256 + threadIdx.x;
    if (ch >= a.CC) return;
    const int n0 = blockIdx.x * a.run, n1 = min(a.N, n0 + a.run);
    const T* u = (const T*)a.u + a.col0 + ch;
    float tp[J], win[W];
#pragma unroll
    for (int j = 0; j < J; ++j) tp[j] = a.taps[(int64_t)ch * J + j];
#pragma unroll
    for (int m = 0; m < W; ++m) win[m] = 0.f;
    const float bias = a.bias ? a.bias[ch] : 0.f;
    int seq_before = -1;
    for (int n = n0; n < n1; ++n) {
        const int seq = a.token_seq[n];
        float* kept = J > 1 ? a.state + (int64_t)a.seq_slots[seq] * a.state_stride : nullptr;
        if (J > 1 && seq != seq_before) {  // (the same for the whole wavefront) the J - 1 inputs ahead of this token
            const int before = n - a.cu_tokens[seq];
#pragma unroll
            for (int m = 0; m < W; ++m) {
                const int back = J - 1 - m;
                win[m] = back <= before ? to_f32<T>(u[(int64_t)(n - back) * a.cols]) : kept[(int64_t)(J - 1 - (back - before)) * a.CC + ch];
            }
        }
        seq_before = seq;
        const float x = to_f32<T>(u[(int64_t)n * a.cols]);
        float acc = bias;
        if (J > 1) {
#pragma unroll
            for (int m = 0; m < W; ++m) acc = fmaf(tp[m], win[m], acc);
#pragma unroll
            for (int m = 0; m + 1 < W; ++m) win[m] = win[m + 1];
            win[W - 1] = x;
            if (ADVANCE) {
#pragma unroll
                for (int m = 0; m < W; ++m) kept[(int64_t)m * a.CC + ch] = win[m];
            }
        }
        a.out[(int64_t)n * a.CC + ch] = ssd_silu(fmaf(tp[J - 1], x, acc));
    }
}

// any number of taps: a thread a channel and token
template <typename T>
__global__ __launch_bounds__(256) void ssd_conv_kernel(SsdConvArgs a) {
    const int64_t n = blockIdx.x;
    const int ch = blockIdx.y * 256 + threadIdx.x;
    if (ch >= a.CC) return;
    const T* u = (const T*)a.u + a.col0 + ch;
    const int seq = a.token_seq[n], before = (int)(n - a.cu_tokens[seq]);
    const float* kept = a.state + (int64_t)a.seq_slots[seq] * a.state_stride;
    float acc = a.bias ? a.bias[ch] : 0.f;
    for (int j = 0; j < a.J; ++j) {
        const int back = a.J - 1 - j;
        const float x = back <= before ? to_f32<T>(u[(n - back) * a.cols]) : kept[(int64_t)(a.J - 1 - (back - before)) * a.CC + ch];
        acc = fmaf(a.taps[(int64_t)ch * a.J + j], x, acc);
    }
    a.out[n * a.CC + ch] = ssd_silu(acc);
}

// state row of every request <- the last J - 1 of (what it held, then the request's inputs of this step)
template <typename T>
__global__ __launch_bounds__(256) void ssd_conv_state_kernel(SsdConvArgs a) {
    const int s = blockIdx.x, ch = blockIdx.y * 256 + threadIdx.x;
    if (ch >= a.CC) return;
    const int q0 = a.cu_tokens[s], len = a.cu_tokens[s + 1] - q0, kept = a.J - 1;
    if (len <= 0) return;
    float* row = a.state + (int64_t)a.seq_slots[s] * a.state_stride + ch;
    const T* u = (const T*)a.u + a.col0 + ch;
    for (int m = 0; m < kept; ++m) {  // (row m takes what lies `len` rows further on: never a row written before it)
        const int from = m + len - kept;  // index among this step's inputs, below zero: a kept row
        row[(int64_t)m * a.CC] = from >= 0 ? to_f32<T>(u[(int64_t)(q0 + from) * a.cols]) : row[(int64_t)(m + len) * a.CC];
    }
}

template <typename T>
static bool ssd_conv_runs(SsdConvArgs a, bool advance, hipStream_t stream) {
    const int blocks = (a.CC + 255) / 256;
    int run = (int)((int64_t)a.N * blocks / 2048);  // runs that load taps and windows seldom, and fill the chip
    a.run = run < 1 ? 1 : run > 16 ? 16 : run;
    dim3 grid((a.N + a.run - 1) / a.run, blocks);
    a.conv_blocks = blocks;
    if (advance && a.x) {
        const int waves = a.H * ((a.N + SSD_DT_TOKENS - 1) / SSD_DT_TOKENS);
        grid.y += ((waves + 3) / 4 + grid.x - 1) / grid.x;
    }
#define SSD_CONV_CASE(JJ)                                                             \
    case JJ:                                                                          \
        if (advance) ssd_conv_run_kernel<T, JJ, true><<<grid, 256, 0, stream>>>(a);   \
        else ssd_conv_run_kernel<T, JJ, false><<<grid, 256, 0, stream>>>(a);          \
        return true;
    switch (a.J) {
        SSD_CONV_CASE(1) SSD_CONV_CASE(2) SSD_CONV_CASE(3) SSD_CONV_CASE(4)
        SSD_CONV_CASE(5) SSD_CONV_CASE(6) SSD_CONV_CASE(7) SSD_CONV_CASE(8)
    }
#undef SSD_CONV_CASE
    return false;
}

// u [N, cols] in `dtype`; taps float32 [CC, J], bias float32 [CC] or null; state rows of state_stride floats whose first
// (J - 1) CC hold the kept rows; out float32 [N, CC].  The state is advanced: by this launch where every request of the
// step has one token (`single` != 0), else by one behind it.  With `single` and J <= 8 the launch also makes dt = x dt_w^T
// (x [N, K] and dt_w [H, K] in `dtype`, dt float32 [N, H]) where x is given.
extern "C" int lle_ssd_conv(const void* u, int cols, int col0, const void* taps, int J, const void* bias, void* state,
                            int64_t state_stride, const void* token_seq, const void* cu_tokens, const void* seq_slots, void* out,
                            int N, int S, int CC, int single, const void* x, const void* dt_w, void* dt, int K, int H, int dtype,
                            hipStream_t stream) {
    if (N <= 0 || CC <= 0) return 0;
    if (J < 1 || (J > 1 && !state) || col0 < 0 || col0 + CC > cols || (CC + 255) / 256 > 65535 || S <= 0) return (int)hipErrorInvalidValue;
    if (x && (!single || J > 8 || !dt_w || !dt || K <= 0 || H <= 0)) return (int)hipErrorInvalidValue;
    const SsdConvArgs a{u, cols, col0, (const float*)taps, (const float*)bias, (float*)state, state_stride, (const int32_t*)token_seq,
                        (const int32_t*)cu_tokens, (const int32_t*)seq_slots, (float*)out, N, CC, J, 1, x, dt_w, (float*)dt, K, H, 0};
    const bool advance = single && J <= 8;
    const bool done = dtype == LLE_F32 ? ssd_conv_runs<float>(a, advance, stream) : ssd_conv_runs<bf16_t>(a, advance, stream);
    const int blocks = (CC + 255) / 256;
    if (!done) {
        if (dtype == LLE_F32) ssd_conv_kernel<float><<<dim3(N, blocks), 256, 0, stream>>>(a);
        else ssd_conv_kernel<bf16_t><<<dim3(N, blocks), 256, 0, stream>>>(a);
    }
    if (J > 1 && !advance) {
        if (dtype == LLE_F32) ssd_conv_state_kernel<float><<<dim3(S, blocks), 256, 0, stream>>>(a);
        else ssd_conv_state_kernel<bf16_t><<<dim3(S, blocks), 256, 0, stream>>>(a);
    }
    LLE_RETURN_LAUNCH_STATUS();
}

// ---------------------------------------------------------------------------------
// The recurrence.
// ---------------------------------------------------------------------------------
struct SsdArgs {
    const float* c;  // [N, CC]: x [H vdim], B [G N], C [G N]
    int CC;
    const float* dt_in;  // rows of dt_cols floats: a head's step size before its bias
    int dt_cols;
    const float *dt_bias, *a_log, *D;  // [H]
    float* state;                      // rows of state_stride floats: [H][vdim][N]
    int64_t state_stride;
    const int32_t *seq_slots, *cu_tokens;
    float* y;  // [N, H vdim]
    int H, G, vdim, n;
    int heads_a_group;   // pass 2: heads of one group that a workgroup takes one after the other
    int pieces;          // chunks of the longest request
    float* part;         // [chunk slots][H][vdim n]: a chunk's own contribution, then its entry state
    float* part_decay;   // [chunk slots][H]
    bool state_wide;     // the state rows start at multiples of 16 bytes
};

// where a request's chunks lie in `part`: requests one after the other, never two in one slot
__device__ __forceinline__ int64_t ssd_slot(int q0, int s) { return (int64_t)(q0 / SSD_CHUNK) + s; }

template <int CTRL>
__device__ __forceinline__ float ssd_lanes(float x) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, 0xf, 0xf, false));
}
// the sum over the 16 lanes of a row, in every one of them
__device__ __forceinline__ float ssd_row_sum(float x) {
    x += ssd_lanes<0xB1>(x);
    x += ssd_lanes<0x4E>(x);
    x += ssd_lanes<0x141>(x);
    x += ssd_lanes<0x140>(x);
    return x;
}

// Requests of at most SSD_WALK tokens.  grid = (requests, heads, blocks of 16 value channels), 256 threads: thread
// (jl, ig) = (tid / 16, tid % 16) owns KI state channels of column j = block 16 + jl, four neighbours of every 64 (fewer than
// four: ig KI + 0 .. KI - 1), so that a wavefront's loads lie one beside the other in memory and in LDS; the sixteen
// threads of a column are neighbours in a wavefront and add their shares of S^T C up through the lanes' cross-bar.  The
// tokens pass through LDS SSD_TC at a time.  What bounds it: the states, read and written once.  Single tokens of Rorevik's
// mid sizes (64 heads of 64 x 128): 1 request 4.0 -> 3.7 us, 8 8.9 -> 7.9, 32 27.5 -> 25.6, 128 105 -> 102 (in a graph), against a
// thread's channels in one stretch.
#define SSD_TC 8
template <int KI>
__global__ __launch_bounds__(256) void ssd_walk_kernel(SsdArgs a) {
    constexpr int KN = KI * 16;
    __shared__ __attribute__((aligned(16))) float s_B[SSD_TC][KN], s_C[SSD_TC][KN];
    __shared__ float s_x[SSD_TC][16], s_g[SSD_TC], s_dt[SSD_TC];
    const int s = blockIdx.x, h = blockIdx.y, tid = threadIdx.x, jl = tid / 16, ig = tid % 16;
    const int n = a.n, vdim = a.vdim, j0 = blockIdx.z * 16, j = j0 + jl;
    const int q0 = a.cu_tokens[s], q1 = a.cu_tokens[s + 1];
    if (q1 <= q0 || q1 - q0 > SSD_WALK) return;
    const int grp = h / (a.H / a.G), inner = a.H * vdim;
    float* col = a.state + (int64_t)a.seq_slots[s] * a.state_stride + ((int64_t)h * vdim + j) * n;
    const bool live = j < vdim;
    constexpr int AT = KI < 4 ? KI : 4;
    auto channel = [&](int i) { return i / 4 * 64 + ig * AT + i % 4; };
    float S[KI];
    if (KI % 4 == 0 && n == KN && a.state_wide) {  // (rows of a multiple of 64 channels: 16 bytes a load)
#pragma unroll
        for (int i = 0; i + 3 < KI; i += 4) {
            const float4 v = live ? *(const float4*)(col + channel(i)) : float4{0.f, 0.f, 0.f, 0.f};
            S[i] = v.x, S[i + 1] = v.y, S[i + 2] = v.z, S[i + 3] = v.w;
        }
    } else {
#pragma unroll
        for (int i = 0; i < KI; ++i) S[i] = (live && channel(i) < n) ? col[channel(i)] : 0.f;
    }
    const float rate = expf(a.a_log[h]), dt_bias = a.dt_bias[h], D = a.D[h];
    for (int c0 = q0; c0 < q1; c0 += SSD_TC) {
        const int nt = min(SSD_TC, q1 - c0);
        if (c0 > q0) __syncthreads();  // (the chunk before has been read)
        // R times 256 places, asked for together (in a loop each would wait for the one before) and without a condition: past the
        // last token that one's again, which nobody reads, past the last channel zeros.  Portions of 8 / 16 / 32 tokens of one
        // request of 64 heads of 64 x 128: 6.2 / 9.1 / 15.0 us in a loop, 5.4 / 7.4 / 11.7 so.
        auto stage = [&](auto rounds) {
            constexpr int R = decltype(rounds)::value;
            float vb[R], vc[R];
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const int e = tid + 256 * r, t = e / KN, i = e - t * KN;
                const float* row = a.c + (int64_t)(c0 + min(t, nt - 1)) * a.CC + inner + grp * n + min(i, n - 1);
                vb[r] = row[0];
                vc[r] = row[a.G * n];
            }
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const int e = tid + 256 * r, t = e / KN, i = e - t * KN;
                if (SSD_TC * KN >= 256 || e < SSD_TC * KN) s_B[t][i] = i < n ? vb[r] : 0.f, s_C[t][i] = i < n ? vc[r] : 0.f;
            }
        };
        if (nt * KN <= 256) stage(std::integral_constant<int, 1>{});
        else stage(std::integral_constant<int, (SSD_TC * KN + 255) / 256>{});
        if (tid < SSD_TC * 16) {
            const int t = tid / 16, e = tid % 16;
            s_x[t][e] = (t < nt && j0 + e < vdim) ? a.c[(int64_t)(c0 + t) * a.CC + h * vdim + j0 + e] : 0.f;
        } else if (tid >= 192 && tid - 192 < nt) {
            const float dt = ssd_softplus(a.dt_in[(int64_t)(c0 + tid - 192) * a.dt_cols + h] + dt_bias);
            s_dt[tid - 192] = dt;
            s_g[tid - 192] = expf(-rate * dt);
        }
        __syncthreads();
#pragma unroll
        for (int t = 0; t < SSD_TC; ++t) {
            if (t < nt) {
                const float g = s_g[t], x = s_x[t][jl], xdt = x * s_dt[t];
                float o = 0.f;
#pragma unroll
                for (int i = 0; i < KI; ++i) {
                    S[i] = fmaf(s_B[t][channel(i)], xdt, g * S[i]);
                    o = fmaf(S[i], s_C[t][channel(i)], o);
                }
                o = ssd_row_sum(o);
                if (ig == 0 && live) a.y[(int64_t)(c0 + t) * inner + h * vdim + j] = fmaf(D, x, o);
            }
        }
    }
    if (!live) return;
    if (KI % 4 == 0 && n == KN && a.state_wide) {
#pragma unroll
        for (int i = 0; i + 3 < KI; i += 4) *(float4*)(col + channel(i)) = float4{S[i], S[i + 1], S[i + 2], S[i + 3]};
    } else {
#pragma unroll
        for (int i = 0; i < KI; ++i)
            if (channel(i) < n) col[channel(i)] = S[i];
    }
}

// One wavefront: step sizes of a chunk's tokens (a token a lane; past the last one: 0) and the sums l of the logarithms
// of their decays up to each token, as two floats (the second is what the first has rounded away).
__device__ __forceinline__ void ssd_chunk_steps(const SsdArgs& a, int h, int t0, int nt, float& dt, float& l_hi, float& l_lo) {
    const int lane = threadIdx.x % LLE_WAVE;
    dt = lane < nt ? ssd_softplus(a.dt_in[(int64_t)(t0 + lane) * a.dt_cols + h] + a.dt_bias[h]) : 0.f;
    double l = -(double)expf(a.a_log[h]) * (double)dt;
#pragma unroll
    for (int o = 1; o < LLE_WAVE; o <<= 1) {
        const double before = __shfl_up(l, o, LLE_WAVE);
        if (lane >= o) l += before;
    }
    l_hi = (float)l;
    l_lo = (float)(l - (double)l_hi);
}

// four consecutive elements of a row of `n`, zeros past its end
template <bool WIDE>
__device__ __forceinline__ ssd_f32x4 ssd_quad(const float* row, int i, int n) {
    ssd_f32x4 v = {0.f, 0.f, 0.f, 0.f};
    if (WIDE) {  // (n a multiple of 4, rows aligned)
        if (i < n) v = *(const ssd_f32x4*)(row + i);
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (i + e < n) v[e] = row[i + e];
    }
    return v;
}

// x of a chunk and head on its way to LDS: thread `tid` has the quads tid, tid + 256 .. of [SSD_CHUNK][VX 64]
template <int VX, bool WIDE>
struct SsdX {
    ssd_f32x4 v[4 * VX];
    __device__ __forceinline__ void load(const float* rows, int CC, int h, int vdim, int nt) {
#pragma unroll
        for (int k = 0; k < 4 * VX; ++k) {
            const int e = k * 256 + threadIdx.x, t = e / (16 * VX), i = (e - t * (16 * VX)) * 4;
            v[k] = ssd_quad<WIDE>(rows + (int64_t)min(t, nt - 1) * CC + h * vdim, i, vdim);
        }
    }
    // (tokens past the chunk's last one have a factor of 0, but another token's x: they are left out)
    __device__ __forceinline__ void store(float* s_x, int XS, const float* factor, int nt) const {
#pragma unroll
        for (int k = 0; k < 4 * VX; ++k) {
            const int e = k * 256 + threadIdx.x, t = e / (16 * VX), i = (e - t * (16 * VX)) * 4;
            *(ssd_f32x4*)(s_x + t * XS + i) = t < nt ? v[k] * factor[t] : ssd_f32x4{0.f, 0.f, 0.f, 0.f};
        }
    }
};

// Pass 1.  grid = (requests x pieces, heads / heads_a_group), 256 threads.  A wavefront has NT tiles of 16 state channels;
// their B stays in its registers for all heads that the workgroup takes.  x times its factor waits in LDS, two buffers: the
// next head's is asked for before this one's is multiplied, one barrier a head.  The contribution, [vdim, n] as the state
// lies, is taken in 16 x 16 tiles, four tokens an instruction: a lane (c, r) gives token 4 k + c of row (column) r and
// gets four neighbouring state channels of a value channel.  A row stride of 16 modulo 64 words spreads the four tokens
// over the banks.  What bounds it: the part's 32 KB a chunk and head of 64 x 128 that are written.
// 2048 tokens of 64 heads of 64 x 128, four heads a workgroup: 61 us with a workgroup a head, B in LDS beside x; 39 so.
template <int NT, int VX, bool WIDE>
__global__ __launch_bounds__(256) void ssd_chunk_state_kernel(SsdArgs a) {
    constexpr int XS = VX * 64 + 16;
    extern __shared__ float lds[];
    const int s = blockIdx.x / a.pieces, piece = blockIdx.x % a.pieces, h0 = blockIdx.y * a.heads_a_group;
    const int q0 = a.cu_tokens[s], len = a.cu_tokens[s + 1] - q0;
    if (len <= SSD_WALK || piece * SSD_CHUNK >= len) return;
    const int t0 = q0 + piece * SSD_CHUNK, nt = min(SSD_CHUNK, len - piece * SSD_CHUNK);
    const int n = a.n, vdim = a.vdim, grp = h0 / (a.H / a.G), inner = a.H * vdim;
    float* s_x = lds;                        // [2][SSD_CHUNK][XS]
    float* s_f = s_x + 2 * SSD_CHUNK * XS;   // [heads][SSD_CHUNK] exp(l_last - l_s) dt_s
    const int wave = threadIdx.x / LLE_WAVE, lane = threadIdx.x % LLE_WAVE, c = lane / 16, r = lane % 16;
    const int64_t slot = ssd_slot(q0, s) + piece;
    const float* rows = a.c + (int64_t)t0 * a.CC;
    SsdX<VX, WIDE> x;
    x.load(rows, a.CC, h0, vdim, nt);
    float B[NT][SSD_CHUNK / 4];
#pragma unroll
    for (int q = 0; q < NT; ++q) {
        const int i = (wave * NT + q) * 16 + r;
        const float* col = rows + inner + grp * n + min(i, n - 1);
#pragma unroll
        for (int k = 0; k < SSD_CHUNK / 4; ++k) {
            const float v = col[(int64_t)min(4 * k + c, nt - 1) * a.CC];
            B[q][k] = (i < n && 4 * k + c < nt) ? v : 0.f;
        }
    }
    for (int hh = wave; hh < a.heads_a_group; hh += 4) {  // a wavefront a head
        float dt, hi, lo;
        ssd_chunk_steps(a, h0 + hh, t0, nt, dt, hi, lo);
        const float hi_last = __shfl(hi, LLE_WAVE - 1, LLE_WAVE), lo_last = __shfl(lo, LLE_WAVE - 1, LLE_WAVE);
        s_f[hh * SSD_CHUNK + lane] = expf((hi_last - hi) + (lo_last - lo)) * dt;
        if (lane == 0) a.part_decay[slot * a.H + h0 + hh] = expf(hi_last);
    }
    __syncthreads();
    const int j_tiles = (vdim + 15) / 16;
    for (int hh = 0; hh < a.heads_a_group; ++hh) {
        float* own_x = s_x + (hh & 1) * SSD_CHUNK * XS;
        x.store(own_x, XS, s_f + hh * SSD_CHUNK, nt);
        __syncthreads();  // (and the buffer that the next head writes has been read)
        if (hh + 1 < a.heads_a_group) x.load(rows, a.CC, h0 + hh + 1, vdim, nt);
        float* out = a.part + (slot * a.H + h0 + hh) * (int64_t)vdim * n;
        auto tiles = [&](auto jt_, int jt0) {  // so many tiles of value channels side by side
            constexpr int JT = decltype(jt_)::value;
            ssd_f32x4 acc[NT][JT];
#pragma unroll
            for (int q = 0; q < NT; ++q)
#pragma unroll
                for (int p = 0; p < JT; ++p) acc[q][p] = ssd_f32x4{0.f, 0.f, 0.f, 0.f};
            // (value channels past the last tile lie in the padding of the row, as zeros)
#pragma unroll
            for (int k = 0; k < SSD_CHUNK / 4; ++k) {
                const float* xk = own_x + (4 * k + c) * XS + jt0 * 16 + r;
#pragma unroll
                for (int p = 0; p < JT; ++p) {
                    const float xv = xk[p * 16];
#pragma unroll
                    for (int q = 0; q < NT; ++q) acc[q][p] = __builtin_amdgcn_mfma_f32_16x16x4f32(B[q][k], xv, acc[q][p], 0, 0, 0);
                }
            }
#pragma unroll
            for (int q = 0; q < NT; ++q) {
                const int i = (wave * NT + q) * 16 + 4 * c;
#pragma unroll
                for (int p = 0; p < JT; ++p) {
                    const int j = (jt0 + p) * 16 + r;
                    if (j >= vdim) continue;
                    if (WIDE) {
                        if (i < n) *(ssd_f32x4*)(out + (int64_t)j * n + i) = acc[q][p];
                    } else {
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            if (i + e < n) out[(int64_t)j * n + i + e] = acc[q][p][e];
                    }
                }
            }
        };
        if (j_tiles == 1) tiles(std::integral_constant<int, 1>{}, 0);
        else if (j_tiles == 2) tiles(std::integral_constant<int, 2>{}, 0);
        else
            for (int jt0 = 0; jt0 < j_tiles; jt0 += 4) tiles(std::integral_constant<int, 4>{}, jt0);
    }
}

// grid = (requests, heads, blocks of 256 state elements): a thread walks one element through the chunks and leaves every
// chunk's entry state in the place of its contribution, the state behind the last chunk in the request's row
__global__ __launch_bounds__(256) void ssd_carry_kernel(SsdArgs a) {
    const int s = blockIdx.x, h = blockIdx.y, elems = a.vdim * a.n;
    const int e = blockIdx.z * 256 + threadIdx.x;
    const int q0 = a.cu_tokens[s], len = a.cu_tokens[s + 1] - q0;
    if (e >= elems || len <= SSD_WALK) return;
    const int live = (len + SSD_CHUNK - 1) / SSD_CHUNK;
    const int64_t slot0 = ssd_slot(q0, s), stride = (int64_t)a.H * elems;
    float* base = a.part + (slot0 * a.H + h) * elems + e;
    const float* decay = a.part_decay + slot0 * a.H + h;
    float* own = a.state + (int64_t)a.seq_slots[s] * a.state_stride + (int64_t)h * elems + e;
    float S = *own;
    for (int p0 = 0; p0 < live; p0 += 8) {
        float A[8], B[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) {  // (asked for together)
            const int p = min(p0 + k, live - 1);
            B[k] = base[p * stride];
            A[k] = decay[(int64_t)p * a.H];
        }
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            if (p0 + k < live) {
                base[(p0 + k) * stride] = S;
                S = fmaf(A[k], S, B[k]);
            }
        }
    }
    *own = S;
}

// Pass 2.  grid = (requests x pieces, heads / heads_a_group), 256 threads; wavefront w has the chunk's tokens
// 16 w .. 16 w + 15, and the products C_t . B_s of its rows stay in registers for all heads that the workgroup takes.
// A lane (c, r) loads four neighbouring elements of a contraction of row r; element e is slot c of instruction e:
//   M^T = B C^T: the result leaves the lane with token t = r and keys s = 4 c .. 4 c + 3 of a tile: the second operand of
//   Y^T += (x dt)^T M^T (contraction over s), whose first operand comes from LDS, and of
//   Y^T += S C^T (contraction over n) with the entry state's rows straight from memory.
// The entry state's rows of the next tile of value channels are on their way while this one's are multiplied (states of up
// to 128 channels: two sets of registers; wider ones: one, asked for again behind the products), also over the end of a
// head; so is the next head's x, and the step sizes of all heads are made at the start, a wavefront a head.
// LDS: x dt [SSD_CHUNK][XS], XS = 4 modulo 64 words: the rows 4 c + e of an instruction lie in different banks.
// Bounded by the products (19 us at the matrix instruction's rate) and what four wavefronts read of the entry state, each for
// itself: at the sizes above 79 us with one set of registers and each head's x and step sizes made at its start; 64 so.
template <int NQ, int VX, bool WIDE>
__global__ __launch_bounds__(256) void ssd_chunk_out_kernel(SsdArgs a) {
    constexpr int XS = VX * 64 + 4, SETS = NQ <= 8 ? 2 : 1;
    extern __shared__ float lds[];
    const int s = blockIdx.x / a.pieces, piece = blockIdx.x % a.pieces, h0 = blockIdx.y * a.heads_a_group;
    const int q0 = a.cu_tokens[s], len = a.cu_tokens[s + 1] - q0;
    if (len <= SSD_WALK || piece * SSD_CHUNK >= len) return;
    const int t0 = q0 + piece * SSD_CHUNK, nt = min(SSD_CHUNK, len - piece * SSD_CHUNK);
    const int n = a.n, vdim = a.vdim, grp = h0 / (a.H / a.G), inner = a.H * vdim;
    float* s_x = lds;
    float* s_dt = s_x + SSD_CHUNK * XS;                    // [heads][SSD_CHUNK]
    float* s_hi = s_dt + a.heads_a_group * SSD_CHUNK;      // likewise
    float* s_lo = s_hi + a.heads_a_group * SSD_CHUNK;
    const int wave = threadIdx.x / LLE_WAVE, lane = threadIdx.x % LLE_WAVE, c = lane / 16, r = lane % 16;
    const int64_t slot = ssd_slot(q0, s) + piece;
    const float* rows = a.c + (int64_t)t0 * a.CC;
    const int tok = wave * 16 + r;  // this lane's token of the chunk
    const int j_tiles = (vdim + 15) / 16;
    ssd_f32x4 sv[SETS][NQ];
    auto entry_rows = [&](int set, int h, int jt) {
        const float* row = a.part + (slot * a.H + h) * (int64_t)vdim * n + (int64_t)min(jt * 16 + r, vdim - 1) * n;
#pragma unroll
        for (int q = 0; q < NQ; ++q) sv[set][q] = ssd_quad<WIDE>(row, 16 * q + 4 * c, n);
    };
    SsdX<VX, WIDE> x;
    x.load(rows, a.CC, h0, vdim, nt);
    ssd_f32x4 C[NQ], cb[4];
    {
        const float* crow = rows + (int64_t)min(tok, nt - 1) * a.CC + inner + (a.G + grp) * n;
#pragma unroll
        for (int q = 0; q < NQ; ++q) C[q] = ssd_quad<WIDE>(crow, 16 * q + 4 * c, n);
    }
    for (int hh = wave; hh < a.heads_a_group; hh += 4) {
        float dt, hi, lo;  // of token `lane` of the chunk
        ssd_chunk_steps(a, h0 + hh, t0, nt, dt, hi, lo);
        s_dt[hh * SSD_CHUNK + lane] = dt;
        s_hi[hh * SSD_CHUNK + lane] = hi;
        s_lo[hh * SSD_CHUNK + lane] = lo;
    }
#pragma unroll
    for (int st = 0; st < 4; ++st) {
        cb[st] = ssd_f32x4{0.f, 0.f, 0.f, 0.f};
        if (st <= wave) {
            const float* brow = rows + (int64_t)min(st * 16 + r, nt - 1) * a.CC + inner + grp * n;
#pragma unroll
            for (int q = 0; q < NQ; ++q) {
                const ssd_f32x4 b = ssd_quad<WIDE>(brow, 16 * q + 4 * c, n);
#pragma unroll
                for (int e = 0; e < 4; ++e) cb[st] = __builtin_amdgcn_mfma_f32_16x16x4f32(b[e], C[q][e], cb[st], 0, 0, 0);
            }
        }
    }
    entry_rows(0, h0, 0);
    ssd_f32x4 m[4];
    float entry = 0.f, D = 0.f;
    // a tile of value channels of head h0 + hh; `set`: where its entry rows are
    auto tile = [&](auto set_, int hh, int jt) {
        constexpr int SET = decltype(set_)::value, OTHER = SETS - 1 - SET;
        const int h = h0 + hh;
        const bool last = jt + 1 == j_tiles;
        const bool more = !last || hh + 1 < a.heads_a_group;
        const int j = jt * 16 + 4 * c;
        const ssd_f32x4 xj = ssd_quad<WIDE>(rows + (int64_t)min(tok, nt - 1) * a.CC + h * vdim, j, vdim);
        if (SETS == 2 && more) entry_rows(OTHER, last ? h + 1 : h, last ? 0 : jt + 1);
        // (two chains of sums: a product waits for the one before it in its own chain only)
        ssd_f32x4 acc = {0.f, 0.f, 0.f, 0.f}, acc2 = acc;
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
#pragma unroll
            for (int e = 0; e < 4; e += 2) {
                acc = __builtin_amdgcn_mfma_f32_16x16x4f32(sv[SET][q][e], C[q][e], acc, 0, 0, 0);
                acc2 = __builtin_amdgcn_mfma_f32_16x16x4f32(sv[SET][q][e + 1], C[q][e + 1], acc2, 0, 0, 0);
            }
        }
        if (SETS == 1 && more) entry_rows(0, last ? h + 1 : h, last ? 0 : jt + 1);
        acc = (acc + acc2) * entry;
        acc2 = ssd_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int st = 0; st < 4; ++st) {
            if (st <= wave) {  // (the same for the whole wavefront)
#pragma unroll
                for (int e = 0; e < 4; e += 2) {
                    const float* x2 = s_x + (st * 16 + 4 * c + e) * XS + jt * 16 + r;
                    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(x2[0], m[st][e], acc, 0, 0, 0);
                    acc2 = __builtin_amdgcn_mfma_f32_16x16x4f32(x2[XS], m[st][e + 1], acc2, 0, 0, 0);
                }
            }
        }
        acc += acc2;
        if (tok < nt) {
            float* y = a.y + (int64_t)(t0 + tok) * inner + h * vdim;
            if (WIDE) {
                if (j < vdim) *(ssd_f32x4*)(y + j) = xj * D + acc;
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (j + e < vdim) y[j + e] = fmaf(D, xj[e], acc[e]);
            }
        }
    };
    using First = std::integral_constant<int, 0>;
    using Second = std::integral_constant<int, SETS - 1>;
    for (int hh = 0; hh < a.heads_a_group; ++hh) {
        __syncthreads();  // (step sizes are there; the head before has been read)
        x.store(s_x, XS, s_dt + hh * SSD_CHUNK, nt);
        __syncthreads();
        if (hh + 1 < a.heads_a_group) x.load(rows, a.CC, h0 + hh + 1, vdim, nt);
        const float *hi = s_hi + hh * SSD_CHUNK, *lo = s_lo + hh * SSD_CHUNK;
        const float hi_t = hi[tok], lo_t = lo[tok];
#pragma unroll
        for (int st = 0; st < 4; ++st) {
            const ssd_f32x4 hi_s = *(const ssd_f32x4*)(hi + st * 16 + 4 * c), lo_s = *(const ssd_f32x4*)(lo + st * 16 + 4 * c);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int key = st * 16 + 4 * c + e;
                // (later keys weigh nothing; their exponent would be above zero)
                m[st][e] = key <= tok ? cb[st][e] * expf((hi_t - hi_s[e]) + (lo_t - lo_s[e])) : 0.f;
            }
        }
        entry = expf(hi_t);
        D = a.D[h0 + hh];
        for (int jt = 0; jt < j_tiles; jt += 2) {
            tile(First{}, hh, jt);
            if (jt + 1 < j_tiles) {
                tile(Second{}, hh, jt + 1);
            } else if (SETS == 2) {
#pragma unroll
                for (int q = 0; q < NQ; ++q) sv[0][q] = sv[SETS - 1][q];
            }
        }
    }
}

// ---------------------------------------------------------------------------------
// States of 128 channels and value channels in sixteens: the chunks one after the other, the state in registers, so that no chunk's
// contribution or entry state goes through memory (written twice and read twice, 32 KB a chunk and head of 64 x 128 each time).
//   ssd_pairs_kernel  for every chunk at once: the step sizes and the sums l of its heads, C, B and the products C_t . B_s of its groups in the
//     order in which the other kernel's lanes take them
//   ssd_stream_kernel grid = (sixteens of value channels, heads, requests), four wavefronts.  Wavefront w keeps the state channels 32 w .. 32 w + 31:
//     two tiles, lane (c, r), element e: channel 32 w + 8 c + 2 e + tile of value channel r, which is the operand of the products with C as
//     it lies.  A chunk: the wavefront's share of C S for all 64 tokens and its tiles of the products of tokens within the chunk meet
//     the others' in LDS (two buffers, one barrier a chunk), S moves on by the chunk's B x.  Every operand of the next chunk is asked
//     for as soon as its place is free.
// 64 heads of 64 x 128, a chunk's three passes through memory -> so, in us: one request of 64, 512, 2048 tokens 33 -> 17, 54 -> 41, 120 -> 107; 8 of 64,
// 256, 512 tokens 82 -> 44, 134 -> 95, 234 -> 160.  A workgroup's chunk takes a CU 2.5 us: 1.0 of the float32 matrix instruction, 0.8 of loads (74 KB,
// shared by four workgroups and 32 heads only in L2), the rest a wavefront or two a SIMD that nothing covers.  With eight wavefronts of 16 channels
// each one request of 2048 tokens takes 100, eight of 64 55; with loads from the rows themselves, sixteen lines each, 112 and 49.
// ---------------------------------------------------------------------------------
#define SSD_N 128
#define SSD_OF_B (SSD_CHUNK * SSD_N)
#define SSD_OF_PAIRS (2 * SSD_CHUNK * SSD_N)
#define SSD_OPERANDS (2 * SSD_CHUNK * SSD_N + 10 * 256)
#define SSD_STREAM_CC (0x7fffffff / (4 * SSD_CHUNK))  // widest row of c: a chunk's bytes are counted in 32 bits
struct SsdStream {
    float* operands;  // [chunk slots][G]: C, B and the ten tiles of C_t . B_s, s <= t, all lane by lane (SSD_OPERANDS floats)
    float* steps;  // [chunk slots][H][5][64]: dt, l's two floats, exp(l_last - l) dt, exp(l)
};

// grid = (chunk slots, groups + ceil(heads / 4)), 256 threads
__global__ __launch_bounds__(256) void ssd_pairs_kernel(SsdArgs a, SsdStream p, int S) {
    int s = 0;  // the last request whose chunks begin here or before
    for (int high = S - 1; s < high;) {
        const int mid = (s + high + 1) / 2;
        if (ssd_slot(a.cu_tokens[mid], mid) <= (int64_t)blockIdx.x) s = mid;
        else high = mid - 1;
    }
    const int q0 = a.cu_tokens[s], len = a.cu_tokens[s + 1] - q0, piece = (int)(blockIdx.x - ssd_slot(q0, s));
    if (len <= SSD_WALK || piece * SSD_CHUNK >= len) return;
    const int t0 = q0 + piece * SSD_CHUNK, nt = min(SSD_CHUNK, len - piece * SSD_CHUNK);
    const int wave = threadIdx.x / LLE_WAVE, lane = threadIdx.x % LLE_WAVE, c = lane / 16, r = lane % 16;
    if ((int)blockIdx.y >= a.G) {  // a wavefront a head
        const int h = ((int)blockIdx.y - a.G) * 4 + wave;
        if (h >= a.H) return;
        float dt, hi, lo;
        ssd_chunk_steps(a, h, t0, nt, dt, hi, lo);
        const float hi_last = __shfl(hi, LLE_WAVE - 1, LLE_WAVE), lo_last = __shfl(lo, LLE_WAVE - 1, LLE_WAVE);
        float* out = p.steps + ((int64_t)blockIdx.x * a.H + h) * 5 * SSD_CHUNK + lane;
        out[0] = dt;
        out[SSD_CHUNK] = hi;
        out[2 * SSD_CHUNK] = lo;
        out[3 * SSD_CHUNK] = expf((hi_last - hi) + (lo_last - lo)) * dt;
        out[4 * SSD_CHUNK] = expf(hi);
        return;
    }
    // wavefront w: tokens 16 w .. 16 w + 15 with all keys up to them
    const int inner = a.H * a.vdim, g = blockIdx.y, tok = wave * 16 + r;
    const float* rows = a.c + (int64_t)t0 * a.CC + inner + g * SSD_N;
    const float* crow = rows + (int64_t)min(tok, nt - 1) * a.CC + a.G * SSD_N;
    float* out = p.operands + ((int64_t)blockIdx.x * a.G + g) * SSD_OPERANDS;
    ssd_f32x4 C[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) C[q] = *(const ssd_f32x4*)(crow + 16 * q + 4 * c);
    for (int st = 0; st <= wave; ++st) {
        const float* brow = rows + (int64_t)min(st * 16 + r, nt - 1) * a.CC;
        ssd_f32x4 B[8], acc = {0.f, 0.f, 0.f, 0.f}, acc2 = acc;
#pragma unroll
        for (int q = 0; q < 8; ++q) B[q] = *(const ssd_f32x4*)(brow + 16 * q + 4 * c);
#pragma unroll
        for (int q = 0; q < 8; ++q)
#pragma unroll
            for (int e = 0; e < 4; e += 2) {
                acc = __builtin_amdgcn_mfma_f32_16x16x4f32(B[q][e], C[q][e], acc, 0, 0, 0);
                acc2 = __builtin_amdgcn_mfma_f32_16x16x4f32(B[q][e + 1], C[q][e + 1], acc2, 0, 0, 0);
            }
        *(ssd_f32x4*)(out + SSD_OF_PAIRS + (wave * (wave + 1) / 2 + st) * 256 + lane * 4) = acc + acc2;
    }
    // C and B as ssd_stream_kernel's wavefront w takes them, zeros behind the last token: C of token 16 tt + r and channels 32 w + 8 c + 4 half,
    // B of the tokens 4 k + c, k = 2 m and 2 m + 1, and channels 32 w + 2 r
    const float* brows = rows + 32 * wave + 2 * r;
    const float* crows = rows + a.G * SSD_N + 32 * wave + 8 * c;
#pragma unroll
    for (int tt = 0; tt < 4; ++tt)
#pragma unroll
        for (int half = 0; half < 2; ++half) {
            const ssd_f32x4 v = *(const ssd_f32x4*)(crows + (int64_t)min(16 * tt + r, nt - 1) * a.CC + 4 * half);
            *(ssd_f32x4*)(out + ((wave * 4 + tt) * 2 + half) * 256 + lane * 4) = 16 * tt + r < nt ? v : ssd_f32x4{0.f, 0.f, 0.f, 0.f};
        }
#pragma unroll
    for (int m = 0; m < 8; ++m) {
        ssd_f32x4 v;
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const int t = 4 * (2 * m + k) + c;
            const float* row = brows + (int64_t)min(t, nt - 1) * a.CC;
            v[2 * k] = t < nt ? row[0] : 0.f;
            v[2 * k + 1] = t < nt ? row[1] : 0.f;
        }
        *(ssd_f32x4*)(out + SSD_OF_B + (wave * 8 + m) * 256 + lane * 4) = v;
    }
}

// e^x for x <= 0 to two ulps, as x log2 e in two floats (expf's way to large and odd arguments is half of a tile's instructions).  Results below
// 2^-126 are 0; so are those of what is below -1000, whose product with log2 e may be an infinity; NaN stays.
__device__ __forceinline__ float ssd_exp(float x) {
    x = x < -1000.f ? -1000.f : x;
    const float p = x * 1.44269502162933349609f;
    const float rest = fmaf(x, 1.92596302e-8f, fmaf(x, 1.44269502162933349609f, -p));
    const float y = __builtin_amdgcn_exp2f(p);
    return fmaf(y * 0.69314718f, rest, y);
}

__global__ __launch_bounds__(256, 2) void ssd_stream_kernel(SsdArgs a, SsdStream p) {
    constexpr int XS = 20;  // words of a row of x in LDS: four rows apart meet every bank once
    __shared__ __attribute__((aligned(16))) float s_x[2][SSD_CHUNK][XS], s_xf[2][SSD_CHUNK][XS];  // x, x times its factor
    __shared__ __attribute__((aligned(16))) float s_y[2][4][4][256];                                // [wavefront][tile of tokens]
    __shared__ __attribute__((aligned(16))) float s_step[2][4][SSD_CHUNK];                          // dt, l's two floats, exp(l)
    const int s = blockIdx.z, h = blockIdx.y, j0 = blockIdx.x * 16;
    const int q0 = a.cu_tokens[s], len = a.cu_tokens[s + 1] - q0;
    if (len <= SSD_WALK) return;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / LLE_WAVE), lane = tid % LLE_WAVE, c = lane / 16, r = lane % 16;
    const int grp = h / (a.H / a.G), inner = a.H * a.vdim, live = (len + SSD_CHUNK - 1) / SSD_CHUNK;
    const int64_t slot0 = ssd_slot(q0, s);
    const float* rows = a.c + (int64_t)q0 * a.CC;
    const float D = a.D[h];
    float* own = a.state + (int64_t)a.seq_slots[s] * a.state_stride + ((int64_t)h * a.vdim + j0 + r) * SSD_N + 32 * wave + 8 * c;
    ssd_f32x4 S[2];
#pragma unroll
    for (int e = 0; e < 4; ++e) S[0][e] = own[2 * e], S[1][e] = own[2 * e + 1];
    // The operands that are on their way: C, B and the products C . B of the wavefront's tiles as the lanes take them, four x of token tid / 4,
    // the steps of token tid.
    ssd_f32x4 B[8], C[4][2], cb[3], x;
    float step = 0.f, f = 0.f;
    const int first[4] = {0, 1, 3, 5}, second[4] = {6, 2, 4, 9}, third[4] = {7, 8, 0, 0};
    const int tile_at[3] = {first[wave], second[wave], third[wave]};  // the wavefront's tiles, of the ten
    const int of_lane = 16 * lane, of_x = 4 * (tid / 4 * a.CC + h * a.vdim + j0 + 4 * (tid % 4));
    auto four = [&](__amdgpu_buffer_rsrc_t unit, int floats) {
        return __builtin_bit_cast(ssd_f32x4, __builtin_amdgcn_raw_buffer_load_b128(unit, of_lane, 4 * floats, 0));
    };
    auto unit_of = [&](int i) {
        return __builtin_amdgcn_make_buffer_rsrc((void*)(p.operands + ((slot0 + min(i, live - 1)) * a.G + grp) * SSD_OPERANDS), 0, 4 * SSD_OPERANDS, 0x00020000);
    };
    auto ask_b = [&](int i) {
        const auto unit = unit_of(i);
#pragma unroll
        for (int m = 0; m < 8; ++m) B[m] = four(unit, SSD_OF_B + (wave * 8 + m) * 256);
    };
    auto ask_c = [&](int i) {
        const auto unit = unit_of(i);
#pragma unroll
        for (int tt = 0; tt < 4; ++tt)
#pragma unroll
            for (int half = 0; half < 2; ++half) C[tt][half] = four(unit, ((wave * 4 + tt) * 2 + half) * 256);
    };
    auto ask_cb = [&](int i) {
        const auto unit = unit_of(i);
#pragma unroll
        for (int n = 0; n < 3; ++n) cb[n] = four(unit, SSD_OF_PAIRS + tile_at[n] * 256);
    };
    auto ask_x = [&](int i) {
        // (a buffer that ends with the chunk's last token: tokens past it are zeros; a chunk's bytes fit 32 bits, a long request's of wide rows do not)
        const auto chunk = __builtin_amdgcn_make_buffer_rsrc((void*)(rows + (int64_t)min(i, live - 1) * SSD_CHUNK * a.CC), 0,
                                                             i < live ? min(SSD_CHUNK, len - i * SSD_CHUNK) * a.CC * 4 : 0, 0x00020000);
        x = __builtin_bit_cast(ssd_f32x4, __builtin_amdgcn_raw_buffer_load_b128(chunk, of_x, 0, 0));
        const auto steps = __builtin_amdgcn_make_buffer_rsrc((void*)(p.steps + ((slot0 + min(i, live - 1)) * a.H + h) * (5 * SSD_CHUNK)), 0, 20 * SSD_CHUNK, 0x00020000);
        auto word = [&](int at) { return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(steps, 4 * at, 0, 0)); };
        f = word(3 * SSD_CHUNK + tid / 4);
        step = word((wave == 3 ? 4 : wave) * SSD_CHUNK + lane);  // (a wavefront an array)
    };
    auto stage = [&](int i) {
        const int b = i & 1;
        *(ssd_f32x4*)&s_x[b][tid / 4][4 * (tid % 4)] = x;
        *(ssd_f32x4*)&s_xf[b][tid / 4][4 * (tid % 4)] = x * f;
        s_step[b][wave][lane] = step;
    };
    auto meet = [&]() {  // (waits for no load on its way)
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    ask_x(0);
    ask_c(0);
    ask_cb(0);
    ask_b(0);
    stage(0);
    ask_x(1);
    meet();
    for (int i = 0; i < live; ++i) {
        const int b = i & 1;
        ssd_f32x4 y[4];
        // every token's share of C S, times exp(l_t)
#pragma unroll
        for (int tt = 0; tt < 4; ++tt) y[tt] = ssd_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int e = 0; e < 8; ++e)
#pragma unroll
            for (int tt = 0; tt < 4; ++tt) y[tt] = __builtin_amdgcn_mfma_f32_16x16x4f32(C[tt][e / 4][e % 4], S[e % 2][e / 2], y[tt], 0, 0, 0);
        ask_c(i + 1);
#pragma unroll
        for (int tt = 0; tt < 4; ++tt) y[tt] *= *(const ssd_f32x4*)&s_step[b][3][16 * tt + 4 * c];
        // the chunk's tokens among each other
        auto among = [&](auto tt_, auto st_, const ssd_f32x4& v) {
            constexpr int tt = decltype(tt_)::value, st = decltype(st_)::value;
            const float hi_t = s_step[b][1][16 * tt + r], lo_t = s_step[b][2][16 * tt + r];
            const ssd_f32x4 dt_s = *(const ssd_f32x4*)&s_step[b][0][16 * st + 4 * c], hi_s = *(const ssd_f32x4*)&s_step[b][1][16 * st + 4 * c],
                            lo_s = *(const ssd_f32x4*)&s_step[b][2][16 * st + 4 * c];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                // (later keys weigh nothing; their exponent would be above zero)
                const float m = tt > st || 4 * c + e <= r ? v[e] * ssd_exp((hi_t - hi_s[e]) + (lo_t - lo_s[e])) * dt_s[e] : 0.f;
                y[tt] = __builtin_amdgcn_mfma_f32_16x16x4f32(m, s_x[b][16 * st + 4 * c + e][r], y[tt], 0, 0, 0);
            }
        };
        using T0 = std::integral_constant<int, 0>;
        using T1 = std::integral_constant<int, 1>;
        using T2 = std::integral_constant<int, 2>;
        using T3 = std::integral_constant<int, 3>;
        switch (wave) {  // three, three, two and two of the ten tiles (tile_at)
            case 0: among(T0{}, T0{}, cb[0]), among(T3{}, T0{}, cb[1]), among(T3{}, T1{}, cb[2]); break;
            case 1: among(T1{}, T0{}, cb[0]), among(T1{}, T1{}, cb[1]), among(T3{}, T2{}, cb[2]); break;
            case 2: among(T2{}, T0{}, cb[0]), among(T2{}, T1{}, cb[1]); break;
            default: among(T2{}, T2{}, cb[0]), among(T3{}, T3{}, cb[1]); break;
        }
        ask_cb(i + 1);
#pragma unroll
        for (int tt = 0; tt < 4; ++tt) *(ssd_f32x4*)&s_y[b][wave][tt][lane * 4] = y[tt];
        // the state behind the chunk
        const float keep = s_step[b][3][SSD_CHUNK - 1];
        S[0] *= keep;
        S[1] *= keep;
#pragma unroll
        for (int k = 0; k < 16; ++k) {
            const float xf = s_xf[b][4 * k + c][r];
            S[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(B[k / 2][k % 2 * 2], xf, S[0], 0, 0, 0);
            S[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(B[k / 2][k % 2 * 2 + 1], xf, S[1], 0, 0, 0);
        }
        ask_b(i + 1);
        stage(i + 1);
        ask_x(i + 2);
        meet();
        // four value channels of token tid / 4
        const int t = tid / 4, tok = i * SSD_CHUNK + t;
        ssd_f32x4 sum;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int at = (t % 16 / 4 * 16 + 4 * (tid % 4) + e) * 4 + t % 4;
            sum[e] = ((s_y[b][0][t / 16][at] + s_y[b][1][t / 16][at]) + s_y[b][2][t / 16][at]) + s_y[b][3][t / 16][at];
        }
        const ssd_f32x4 xt = *(const ssd_f32x4*)&s_x[b][t][4 * (tid % 4)];
        if (tok < len) *(ssd_f32x4*)(a.y + (int64_t)(q0 + tok) * inner + h * a.vdim + j0 + 4 * (tid % 4)) = xt * D + sum;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) own[2 * e] = S[0][e], own[2 * e + 1] = S[1][e];
}

extern "C" int lle_ssd_max_dim(void) { return 256; }
extern "C" int lle_ssd_chunk(void) { return SSD_CHUNK; }
extern "C" int lle_ssd_walk(void) { return SSD_WALK; }

// Floats of `part` where the chunks go one after the other (ssd_stream_kernel), for a step of N tokens of S requests
extern "C" int64_t lle_ssd_stream_floats(int N, int S, int H, int G) {
    return (int64_t)(N / SSD_CHUNK + S) * (G * SSD_OPERANDS + H * 5 * SSD_CHUNK);
}

// c float32 [N, CC], CC = H vdim + 2 G n; dt_in float32 rows of dt_cols; dt_bias, a_log, D float32 [H]; state rows of
// state_stride floats that begin with [H][vdim][n]; y float32 [N, H vdim].  `walk`: some request has at most SSD_WALK
// tokens; `pieces` > 0: chunks of the longest request (0: no request has more), with `part` float32
// [(N / SSD_CHUNK + S) H vdim n] and `part_decay` [(N / SSD_CHUNK + S) H].  heads_a_group divides H / G.
// stream_floats > 0: requests of more tokens go chunk after chunk; `part` holds so many floats (lle_ssd_stream_floats), part_decay nothing.
extern "C" int lle_ssd_scan(const void* c, int CC, const void* dt_in, int dt_cols, const void* dt_bias, const void* a_log,
                            const void* D, void* state, int64_t state_stride, const void* seq_slots, const void* cu_tokens, void* y,
                            int S, int H, int G, int vdim, int n, int walk, int pieces, int heads_a_group, void* part,
                            void* part_decay, int N, int64_t stream_floats, hipStream_t stream) {
    if (S <= 0 || H <= 0) return 0;
    if (G <= 0 || H % G || vdim <= 0 || vdim > 256 || n <= 0 || n > 256 || H > 65535 || CC != H * vdim + 2 * G * n || dt_cols < H ||
        pieces < 0 || heads_a_group <= 0 || (H / G) % heads_a_group || (int64_t)S * (pieces > 0 ? pieces : 1) > 0x7fffffff ||
        (pieces > 0 && (!part || (!part_decay && stream_floats == 0))))
        return (int)hipErrorInvalidValue;
    // LDS holds the step sizes of a workgroup's heads: at most SSD_HEADS of them
    for (int k = SSD_HEADS; heads_a_group > SSD_HEADS; --k)
        if (heads_a_group % k == 0) heads_a_group = k;
    const SsdArgs a{(const float*)c, CC, (const float*)dt_in, dt_cols, (const float*)dt_bias, (const float*)a_log, (const float*)D,
                    (float*)state, state_stride, (const int32_t*)seq_slots, (const int32_t*)cu_tokens, (float*)y, H, G, vdim, n,
                    heads_a_group, pieces, (float*)part, (float*)part_decay, (uintptr_t)state % 16 == 0 && state_stride % 4 == 0};
    if (walk) {
        const dim3 grid(S, H, (vdim + 15) / 16);
        if (n <= 16) ssd_walk_kernel<1><<<grid, 256, 0, stream>>>(a);
        else if (n <= 32) ssd_walk_kernel<2><<<grid, 256, 0, stream>>>(a);
        else if (n <= 64) ssd_walk_kernel<4><<<grid, 256, 0, stream>>>(a);
        else if (n <= 128) ssd_walk_kernel<8><<<grid, 256, 0, stream>>>(a);
        else ssd_walk_kernel<16><<<grid, 256, 0, stream>>>(a);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess || pieces == 0) return (int)e;
    }
    if (pieces == 0) return 0;
    if (stream_floats > 0) {
        const int chunks = N / SSD_CHUNK + S;
        if (n != SSD_N || vdim % 16 != 0 || S > 65535 || CC > SSD_STREAM_CC || stream_floats < lle_ssd_stream_floats(N, S, H, G) || (((uintptr_t)c | (uintptr_t)y | (uintptr_t)part) & 15))
            return (int)hipErrorInvalidValue;
        const SsdStream p{(float*)part, (float*)part + (int64_t)chunks * G * SSD_OPERANDS};
        ssd_pairs_kernel<<<dim3(chunks, G + (H + 3) / 4), 256, 0, stream>>>(a, p, S);
        ssd_stream_kernel<<<dim3(vdim / 16, H, S), 256, 0, stream>>>(a, p);
        LLE_RETURN_LAUNCH_STATUS();
    }
    const bool wide = n % 4 == 0 && vdim % 4 == 0;  // (then CC and every column offset are multiples of 4 too)
    const dim3 grid(S * pieces, H / heads_a_group);
    auto go = [&](auto kernel, size_t lds) {
        if (lds > 64 * 1024) {
            const hipError_t e = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
            if (e != hipSuccess) return e;
        }
        kernel<<<grid, 256, lds, stream>>>(a);
        return hipGetLastError();
    };
    const int VX = (vdim + 63) / 64;
    auto by_width = [&](auto launch) {  // launch(how many times 64 value channels, whether 16 bytes a load)
        using No = std::false_type;
        using Yes = std::true_type;
        switch (VX) {
            case 1: return wide ? launch(std::integral_constant<int, 1>{}, Yes{}) : launch(std::integral_constant<int, 1>{}, No{});
            case 2: return wide ? launch(std::integral_constant<int, 2>{}, Yes{}) : launch(std::integral_constant<int, 2>{}, No{});
            case 3: return wide ? launch(std::integral_constant<int, 3>{}, Yes{}) : launch(std::integral_constant<int, 3>{}, No{});
            default: return wide ? launch(std::integral_constant<int, 4>{}, Yes{}) : launch(std::integral_constant<int, 4>{}, No{});
        }
    };
    hipError_t e = by_width([&](auto vx, auto w) {
        constexpr int V = decltype(vx)::value;
        constexpr bool W = decltype(w)::value;
        const size_t lds = ((size_t)2 * SSD_CHUNK * (V * 64 + 16) + heads_a_group * SSD_CHUNK) * sizeof(float);
        if (n <= 64) return go(ssd_chunk_state_kernel<1, V, W>, lds);
        if (n <= 128) return go(ssd_chunk_state_kernel<2, V, W>, lds);
        return go(ssd_chunk_state_kernel<4, V, W>, lds);
    });
    if (e != hipSuccess) return (int)e;
    ssd_carry_kernel<<<dim3(S, H, (vdim * n + 255) / 256), 256, 0, stream>>>(a);
    e = hipGetLastError();
    if (e != hipSuccess) return (int)e;
    return (int)by_width([&](auto vx, auto w) {
        constexpr int V = decltype(vx)::value;
        constexpr bool W = decltype(w)::value;
        const size_t lds = ((size_t)SSD_CHUNK * (V * 64 + 4) + 3 * heads_a_group * SSD_CHUNK) * sizeof(float);
#define SSD_OUT_CASE(NQ) \
    if (n <= 16 * NQ) return go(ssd_chunk_out_kernel<NQ, V, W>, lds);
        SSD_OUT_CASE(1)
        SSD_OUT_CASE(2)
        SSD_OUT_CASE(3)
        SSD_OUT_CASE(4)
        SSD_OUT_CASE(6)
        SSD_OUT_CASE(8)
        SSD_OUT_CASE(12)
        SSD_OUT_CASE(16)
#undef SSD_OUT_CASE
        return hipErrorInvalidValue;
    });
}

// ---------------------------------------------------------------------------------
// out[n, :] = (y silu(z)) / rms(its part) * w: a row is cut into `groups` equal parts, each divided by its own root mean
// square.  z: the columns z0 .. of u.  A workgroup of 256 threads a (token, part); a thread keeps its share of the part in
// registers, in pieces of V elements (parts up to 256 x SSD_PER; wider ones are made twice).
// ---------------------------------------------------------------------------------
#define SSD_PER 32
template <typename T, int V>
__global__ __launch_bounds__(256) void ssd_gate_norm_kernel(const float* __restrict__ y, const T* __restrict__ u, int cols, int z0,
                                                             const float* __restrict__ w, float eps, T* __restrict__ out, int inner,
                                                             int width) {
    __shared__ float red[16];
    const int64_t n = blockIdx.x;
    const int p0 = blockIdx.y * width;
    const float* yr = y + n * inner + p0;
    const T* zr = u + n * cols + z0 + p0;
    T* dst = out + n * inner + p0;
    typedef T piece_t __attribute__((ext_vector_type(V)));
    typedef float fpiece_t __attribute__((ext_vector_type(V)));
    float keep[SSD_PER], ss = 0.f;
    const bool fits = width <= 256 * SSD_PER;
    if (fits) {
#pragma unroll
        for (int k = 0; k < SSD_PER; k += V) {
            const int i = (k / V * 256 + threadIdx.x) * V;
            if (k * 256 >= width) break;  // (the same for every thread)
            if (i < width) {  // (V divides the width and every offset)
                const fpiece_t yv = *(const fpiece_t*)(yr + i);
                const piece_t zv = *(const piece_t*)(zr + i);
#pragma unroll
                for (int e = 0; e < V; ++e) {
                    const float z = to_f32<T>(zv[e]);
                    keep[k + e] = yv[e] * z * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(z * -1.44269504088896340736f));
                    ss = fmaf(keep[k + e], keep[k + e], ss);
                }
            }
        }
    } else {
        for (int i = threadIdx.x; i < width; i += 256) {
            const float v = yr[i] * ssd_silu(to_f32<T>(zr[i]));
            ss = fmaf(v, v, ss);
        }
    }
    const float inv = 1.0f / sqrtf(block_sum(ss, red) / (float)width + eps);
    if (fits) {
#pragma unroll
        for (int k = 0; k < SSD_PER; k += V) {
            const int i = (k / V * 256 + threadIdx.x) * V;
            if (k * 256 >= width) break;
            if (i < width) {
                const fpiece_t wv = *(const fpiece_t*)(w + p0 + i);
                piece_t o;
#pragma unroll
                for (int e = 0; e < V; ++e) o[e] = from_f32<T>(keep[k + e] * inv * wv[e]);
                *(piece_t*)(dst + i) = o;
            }
        }
    } else {
        for (int i = threadIdx.x; i < width; i += 256)
            dst[i] = from_f32<T>(yr[i] * ssd_silu(to_f32<T>(zr[i])) * inv * w[p0 + i]);
    }
}

extern "C" int lle_ssd_gate_norm(const void* y, const void* u, int cols, int z0, const void* w, float eps, void* out, int N, int inner,
                                 int groups, int dtype, hipStream_t stream) {
    if (N <= 0 || inner <= 0) return 0;
    if (groups <= 0 || inner % groups || groups > 65535 || z0 < 0 || z0 + inner > cols) return (int)hipErrorInvalidValue;
    const dim3 grid(N, groups);
    const bool wide = (inner / groups) % 4 == 0 && cols % 4 == 0 && z0 % 4 == 0;
#define SSD_GATE(T, V)                                                                                                         \
    ssd_gate_norm_kernel<T, V><<<grid, 256, 0, stream>>>((const float*)y, (const T*)u, cols, z0, (const float*)w, eps, (T*)out, inner, \
                                                         inner / groups)
    if (dtype == LLE_F32) {
        if (wide) SSD_GATE(float, 4); else SSD_GATE(float, 1);
    } else {
        if (wide) SSD_GATE(bf16_t, 4); else SSD_GATE(bf16_t, 1);
    }
#undef SSD_GATE
    LLE_RETURN_LAUNCH_STATUS();
}
