// Paged grouped-query attention over the cache, for any mix of prompt portions
// and single decoded tokens in one step.
//
// The reference has three kernels, none of which covers a prompt portion after
// a past: flash_attention_kernel (prefill of one request over its own K/V,
// src/ops/attention.cu:320-426), flash_attention_kv_cache_kernel (:429-535) and
// flash_attention_paged_kv_cache_batch_kernel (:537-669, decode rows through a
// block table packed and uploaded per layer and step, :959-1020).  Here the K/V
// of the step's tokens are already in their pages, the block tables live on the
// device, and every query token attends through them:
//   query at cache position p (= kv_len - q_len + its index in the portion)
//   sees keys lo..p,  lo = max(0, p - window + 1) with a window, else 0, and with `keep_first`
//   also the first keys, 0 .. min(keep_first, lo) - 1: every kernel walks that range first, with
//   the same running maximum and sums, then lo..p
//   score_j = (q . k_j) * scale, with a cap then cap * tanh(score_j / cap);  softmax over j streamed in 32-bit (m, l, acc)
//   kv head of q head h = h / (nq / nkv)                  (:577-668 for the maths)
// A cache page holds K as [nkv][page_size][d], then V as [nkv][d][page_size].
//
// Kernels:
//  * paged_attention_generic_kernel: any type, head size <= 256, page size,
//    window; one workgroup per (token, q head).  The 32-bit path and odd sizes.
//  * mfma_decode_kernel (+ mfma_combine_kernel): bfloat16, head size a multiple of
//    32, page size a multiple of 16.  One workgroup per (request, kv head, key
//    split); the q heads of the group (and up to 16 / group tokens) are the 16
//    columns of v_mfma_f32_16x16x32_bf16 tiles, so every K/V byte is read once
//    per group; the four wavefronts take every fourth 32-key step, their loads
//    two steps ahead; partial (m, l, acc) of the splits are merged by the combine
//    kernel.  In decode steps it can also do what comes before it: the q/k norm,
//    the rotation and the write of the new K and V (FusedQKV).
//  * mfma_prefill_kernel: same tile code, 32 rows (token, head) per wavefront,
//    all keys up to each row's own position; the four wavefronts of a workgroup
//    share the K/V tiles through LDS, two workgroups share a CU.
#include "common.h"
#include "lds.h"
#include "parts.h"
#include <type_traits>
#include <mutex>

LLE_DEFINE_ERROR_STRING()

#define ATT_WAVES 4
#define ATT_MAX_R 4  // head_dim <= 256
#define ATT_KEYS 4   // keys a wavefront works on at a time

template <typename T>
__global__ __launch_bounds__(ATT_WAVES* LLE_WAVE) void paged_attention_generic_kernel(
    const T* __restrict__ q, const T* __restrict__ kv_layer, const int32_t* __restrict__ block_tables,
    const int32_t* __restrict__ seq_slots, const int32_t* __restrict__ cu_tokens,
    const int32_t* __restrict__ kv_lens, const int32_t* __restrict__ token_seq, T* __restrict__ out, int nq,
    int nkv, int d, int page_size, int64_t page_stride, int max_pages, int window, int keep_first, float scale,
    const float* __restrict__ sinks, float softcap) {
    __shared__ float s_m[ATT_WAVES], s_l[ATT_WAVES];
    __shared__ float s_acc[ATT_WAVES][ATT_MAX_R * LLE_WAVE];

    const int64_t tok = blockIdx.x;
    const int h = blockIdx.y;
    const int wave = threadIdx.x / LLE_WAVE, lane = threadIdx.x % LLE_WAVE;
    const int s = token_seq[tok];
    const int kv_len = kv_lens[s];
    const int q_start = cu_tokens[s];
    const int q_len = cu_tokens[s + 1] - q_start;
    const int query_pos = kv_len - q_len + (int)(tok - q_start);
    const int query_lo = window > 0 ? max(0, query_pos - window + 1) : 0;
    const int kept = min(keep_first, query_lo);
    const int kvh = h / (nq / nkv);
    const int32_t* table = block_tables + (int64_t)seq_slots[s] * max_pages;

    float qv[ATT_MAX_R], acc[ATT_MAX_R];
#pragma unroll
    for (int r = 0; r < ATT_MAX_R; ++r) {
        const int e = lane + LLE_WAVE * r;
        qv[r] = e < d ? to_f32<T>(q[(tok * nq + h) * d + e]) : 0.f;
        acc[r] = 0.f;
    }
    float m = -FLT_MAX, l = 0.f;
    const int64_t v_base = ((int64_t)nkv + kvh) * page_size * d;
    // A wavefront takes ATT_KEYS consecutive keys at a time, so that the loads of several keys
    // are on their way together (one key after the other, each would wait for its own K row and
    // then for its own V row).  Which keys share a step depends on (lo, pos) only.
    // (keys j0 .. j0 + ATT_KEYS - 1 lie in one page, side by side, when the steps start at a
    // multiple of ATT_KEYS and pages hold a multiple of it; the last step of a row may reach
    // past `pos`, but not past its page)
    for (int range = kept > 0 ? 0 : 1; range < 2; ++range) {
    const int lo = range == 0 ? 0 : query_lo, pos = range == 0 ? kept - 1 : query_pos;
    const bool keys_in_one_piece = lo % ATT_KEYS == 0 && page_size % ATT_KEYS == 0;
    for (int j0 = lo + wave * ATT_KEYS; j0 <= pos; j0 += ATT_WAVES * ATT_KEYS) {
        const T* vp[ATT_KEYS];
        float dot[ATT_KEYS];
#pragma unroll
        for (int i = 0; i < ATT_KEYS; ++i) {
            const int j = min(j0 + i, pos);  // past the row's last key: that key again, weighted 0 below
            const int lp = j / page_size;
            const int off = j - lp * page_size;
            // the same for the whole wavefront: a scalar load
            const T* page = kv_layer + (int64_t)table[__builtin_amdgcn_readfirstlane(lp)] * page_stride;
            const T* kp = page + ((int64_t)kvh * page_size + off) * d;
            vp[i] = page + v_base + off;  // element e of the value row at vp[e * page_size]
            dot[i] = 0.f;
#pragma unroll
            for (int r = 0; r < ATT_MAX_R; ++r) {
                const int e = lane + LLE_WAVE * r;
                if (e < d) dot[i] += qv[r] * to_f32<T>(kp[e]);
            }
        }
        float vals[ATT_KEYS][ATT_MAX_R];
        if (keys_in_one_piece) {
            // the ATT_KEYS values of an element lie side by side in the page: one load for all of them
            typedef T piece_t __attribute__((ext_vector_type(ATT_KEYS)));
#pragma unroll
            for (int r = 0; r < ATT_MAX_R; ++r) {
                const int e = lane + LLE_WAVE * r;
                if (e < d) {
                    const piece_t piece = *(const piece_t*)(vp[0] + (int64_t)e * page_size);
#pragma unroll
                    for (int i = 0; i < ATT_KEYS; ++i)  // what lies past `pos` was never written: not even times 0
                        vals[i][r] = j0 + i <= pos ? to_f32<T>(piece[i]) : 0.f;
                } else {
#pragma unroll
                    for (int i = 0; i < ATT_KEYS; ++i) vals[i][r] = 0.f;
                }
            }
        } else {
#pragma unroll
            for (int i = 0; i < ATT_KEYS; ++i)
#pragma unroll
                for (int r = 0; r < ATT_MAX_R; ++r) {
                    const int e = lane + LLE_WAVE * r;
                    vals[i][r] = e < d ? to_f32<T>(vp[i][(int64_t)e * page_size]) : 0.f;
                }
        }
        float score[ATT_KEYS];
        float new_m = m;
#pragma unroll
        for (int i = 0; i < ATT_KEYS; ++i) {
            score[i] = wave_sum(dot[i]) * scale;
            if (softcap > 0.f) score[i] = softcap * tanhf(score[i] / softcap);
            if (j0 + i <= pos) new_m = fmaxf(new_m, score[i]);
        }
        const float alpha = expf(m - new_m);
        float beta[ATT_KEYS];
        l *= alpha;
#pragma unroll
        for (int i = 0; i < ATT_KEYS; ++i) {
            beta[i] = j0 + i <= pos ? expf(score[i] - new_m) : 0.f;
            l += beta[i];
        }
#pragma unroll
        for (int r = 0; r < ATT_MAX_R; ++r) {
            float a = acc[r] * alpha;
#pragma unroll
            for (int i = 0; i < ATT_KEYS; ++i) a += beta[i] * vals[i][r];
            acc[r] = a;
        }
        m = new_m;
    }
    }
    if (lane == 0) {
        s_m[wave] = m;
        s_l[wave] = l;
    }
#pragma unroll
    for (int r = 0; r < ATT_MAX_R; ++r) s_acc[wave][lane + LLE_WAVE * r] = acc[r];
    __syncthreads();
    float big = s_m[0];
    for (int w = 1; w < ATT_WAVES; ++w) big = fmaxf(big, s_m[w]);
    // a sink: one more place in the softmax's sum, with a score of its own and no value
    const float sink_share = sinks ? expf(sinks[h] - big) : 0.f;
    for (int e = threadIdx.x; e < d; e += blockDim.x) {
        float num = 0.f, den = sink_share;
        for (int w = 0; w < ATT_WAVES; ++w) {
            const float f = expf(s_m[w] - big);  // a wavefront without keys has l = 0, acc = 0
            num += s_acc[w][e] * f;
            den += s_l[w] * f;
        }
        out[(tok * nq + h) * d + e] = from_f32<T>(num / den);
    }
}

extern "C" int lle_paged_attention_generic(const void* q, const void* kv_layer, const void* block_tables,
                                           const void* seq_slots, const void* cu_tokens, const void* kv_lens,
                                           const void* token_seq, void* out, int N, int nq, int nkv, int d,
                                           int page_size, int64_t page_stride, int max_pages, int window,
                                           int keep_first, float scale, int dtype, const void* sinks, float softcap,
                                           hipStream_t stream) {
    if (N <= 0) return 0;
    if (keep_first < 0 || d > ATT_MAX_R * LLE_WAVE) return (int)hipErrorInvalidValue;
    dim3 grid(N, nq);
    if (dtype == LLE_F32)
        paged_attention_generic_kernel<float><<<grid, ATT_WAVES * LLE_WAVE, 0, stream>>>(
            (const float*)q, (const float*)kv_layer, (const int32_t*)block_tables, (const int32_t*)seq_slots,
            (const int32_t*)cu_tokens, (const int32_t*)kv_lens, (const int32_t*)token_seq, (float*)out, nq, nkv, d,
            page_size, page_stride, max_pages, window, keep_first, scale, (const float*)sinks, softcap);
    else
        paged_attention_generic_kernel<bf16_t><<<grid, ATT_WAVES * LLE_WAVE, 0, stream>>>(
            (const bf16_t*)q, (const bf16_t*)kv_layer, (const int32_t*)block_tables, (const int32_t*)seq_slots,
            (const int32_t*)cu_tokens, (const int32_t*)kv_lens, (const int32_t*)token_seq, (bf16_t*)out, nq, nkv,
            d, page_size, page_stride, max_pages, window, keep_first, scale, (const float*)sinks, softcap);
    LLE_RETURN_LAUNCH_STATUS();
}

// ---------------------------------------------------------------------------------
// matrix-core kernels (bfloat16)
// ---------------------------------------------------------------------------------
typedef bf16_t bf16x8 __attribute__((ext_vector_type(8)));
typedef bf16_t bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

#define NEG_BIG (-1.0e30f)
#define LAZY_MAX 8.0f  // a row's reference maximum may lag its true one by this much (base 2)
#define KSTEP 32  // keys per step: two 16-key tiles; pages hold a multiple of 16 keys
#define KEY_OF_ROW(r, x) (8 * ((r) / 4) + 4 * (x) + (r) % 4)
// LDS tiles of the prompt kernel.  LDS has 64 banks of 4 bytes; a 16-byte read of a wavefront
// is served sixteen lanes a cycle, and the sixteen are not consecutive (measured: a cycle takes
// lanes 0-3, 12-15, 20-23, 24-27, the next 4-11, 16-19, 28-31, then the same of the upper 32).
// With lane = (c, r) = (lane / 16, lane % 16) a cycle holds c0 with r / 4 in {0, 3} and c0 + 1
// with r / 4 in {1, 2}, or the other way round, r % 4 taking all its values.  The tiles have no
// padding; a lane reads 16-byte piece (logical piece) ^ swizzle of its row instead, and the
// swizzle is such that a cycle's sixteen lanes hit the sixteen 16-byte columns of the banks:
//   Q4(q) for q = r / 4: 0, 2, 3, 1, so that c ^ Q4 differs between the four (c, r / 4) of a cycle;
//   V^T rows are 64 bytes (32 keys): element e uses Q4((e / 4) % 4); e % 4 picks the columns 4 (e % 4) ..
//   K rows are 64 DK bytes, key j = 8 (r / 4) + 4 x + r % 4 of the step: the low bits of j
//   choose among what the row's own offset leaves the same: none for odd DK (rows 64 bytes
//   apart mod 256), bit 1 for DK = 2, 6 (128 bytes), bits 1 and 0 for DK = 4, 8 (0 bytes).
#define Q4(q) ((((q) >> 1) & 1) | ((((q) ^ ((q) >> 1)) & 1) << 1))
#define K_SWIZZLE(j, DK) ((Q4(((j) >> 3) & 3) | ((((j) >> 1) & 1) << 2) | (((j) & 1) << 3)) & ((DK) % 4 == 0 ? 15 : (DK) % 2 == 0 ? 7 : 3))
#define V_SWIZZLE(e) Q4(((e) >> 2) & 3)

// What one lane knows about the query row it serves (row = lane % 16 of a 16-row tile).
struct RowInfo {
    const bf16_t* q;  // start of the row's head in q, or nullptr for a row that does not exist
    int pos;          // last key the row sees
    int lo;           // first key the row sees
};

// One wavefront runs `RT` tiles of 16 query rows over the 32-key steps
// step_begin, step_begin + step_stride, ... < step_end.  Products:
//   S^T = K Q^T   (A = K tile [16 keys x 32], B = Q^T [32 x 16 rows])
//   O^T += V^T P^T (A = V^T tile [16 d x 32 keys], B = P^T [32 keys x 16 rows])
// With v_mfma_f32_16x16x32_bf16 a lane (c = lane / 16, r = lane % 16) holds, of a
// result tile, column r and rows 4c..4c+3: for S^T that is query row r and four keys
// — exactly what the B operand of the second product wants, so P never leaves
// registers, and the softmax state of row r sits in the lanes r + 16c.
// Which key a row of a K tile stands for is free.  The two tiles of a step take the keys
//   row r of tile x  <->  key 8 (r / 4) + 4 x + r % 4   of the step        (KEY_OF_ROW)
// so that a lane's eight scores (rows 4c..4c+3 of both tiles) are the CONSECUTIVE keys
// 8c..8c+7: the V^T operand of the second product is then one 16-byte piece per lane
// (keys 8c..8c+7 of one value element), inside one page.
template <int DK, int RT>
struct RowState {
    bf16x8 qv[RT][DK];             // Q^T operands of the lane's row
    int open_lo[RT], open_hi[RT];  // steps with open_lo <= j0 and j0 + 31 <= open_hi need no mask
    f32x4 o[RT][2 * DK];           // O^T tiles: value elements 16 n + 4 c .. + 3 of row r16
    float m[RT], l[RT];            // running maximum (base 2) and this lane's share of the sum
};

// the steps that every row of a tile sees whole (the rows' lo and pos are what they see of the range walked now)
template <int DK, int RT>
__device__ __forceinline__ void set_open_range(RowState<DK, RT>& st, const RowInfo (&row)[RT]) {
#pragma unroll
    for (int t = 0; t < RT; ++t) {
        int lo_max = row[t].q ? row[t].lo : 0, pos_min = row[t].q ? row[t].pos : 0x7fffffff;
#pragma unroll
        for (int off = 1; off < LLE_WAVE; off <<= 1) {
            lo_max = max(lo_max, __shfl_xor(lo_max, off, LLE_WAVE));
            pos_min = min(pos_min, __shfl_xor(pos_min, off, LLE_WAVE));
        }
        // (the same in every lane: kept in scalar registers, so that the test is a scalar branch)
        st.open_lo[t] = __builtin_amdgcn_readfirstlane(lo_max);
        st.open_hi[t] = __builtin_amdgcn_readfirstlane(pos_min == 0x7fffffff ? -1 : pos_min);
    }
}

// LOAD_Q = false: the caller has filled st.qv itself; FIND_OPEN = false: st.open_lo and st.open_hi, too
template <int DK, int RT, bool LOAD_Q = true, bool FIND_OPEN = true>
__device__ __forceinline__ void init_rows(RowState<DK, RT>& st, const RowInfo (&row)[RT]) {
    const int c = (threadIdx.x % LLE_WAVE) / 16;
#pragma unroll
    for (int t = 0; t < RT; ++t) {
        if (LOAD_Q) {
#pragma unroll
            for (int ks = 0; ks < DK; ++ks) {
                if (row[t].q) {
                    st.qv[t][ks] = *(const bf16x8*)(row[t].q + 32 * ks + 8 * c);
                } else {
#pragma unroll
                    for (int i = 0; i < 8; ++i) st.qv[t][ks][i] = (bf16_t)0.0f;
                }
            }
        }
#pragma unroll
        for (int n = 0; n < 2 * DK; ++n) st.o[t][n] = f32x4{0.f, 0.f, 0.f, 0.f};
        st.m[t] = NEG_BIG;
        st.l[t] = 0.f;
    }
    if constexpr (FIND_OPEN) set_open_range<DK, RT>(st, row);
    // The rows of Q are waited for here, once.  Left pending, their first use lies inside the
    // key loop, where the wait for them also waits for the K/V loads just issued for a later
    // step: the loop would run at the latency of memory.
    if (LOAD_Q) {
#pragma unroll
        for (int t = 0; t < RT; ++t)
#pragma unroll
            for (int ks = 0; ks < DK; ++ks) asm volatile("" : "+v"(st.qv[t][ks]));
    }
}

// The largest of eight scores, none of which is a NaN (masked scores are NEG_BIG, not infinite).
// Written with the instruction itself: from fmaxf the compiler first passes every operand that a
// select may have produced through an instruction of its own (x = max(x, x), which quiets a
// signalling NaN), 8 + 7 instructions for what takes 4.
__device__ __forceinline__ float max3(float a, float b, float c) {
    float r;
    asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}
__device__ __forceinline__ float max_of_8(const float (&x)[8]) {
    const float a = max3(x[0], x[1], x[2]), b = max3(x[3], x[4], x[5]);
    return max3(max3(x[6], x[7], a), b, b);
}

// One 32-key step for RT tiles of 16 rows.  load_k(x, ks): for lane (c, r16) key
// KEY_OF_ROW(r16, x) of the step, elements 32 ks + 8 c .. + 7.  load_v(n): value element
// 16 n + r16, keys 8c..8c+7 of the step.  Each operand is fetched once and used by all row tiles.
// No row sees a key outside [seen_lo, seen_hi].
// CAP: the scores pass through cap * tanh(score / cap).  In the base-2 domain that is C (1 - 2 / (1 + 2^(s k))) with
// C = cap log2 e (`cap_log2`) and k = 2 log2 e scale / cap, which the caller hands in for the scale; either end of the
// exponential's range gives the right limit.
template <int DK, int RT, bool CAP, typename LoadK, typename LoadV>
__device__ __forceinline__ void tile_step(RowState<DK, RT>& st, const RowInfo (&row)[RT], LoadK load_k,
                                          LoadV load_v, int j0, int seen_lo, int seen_hi, float scale_log2, float cap_log2) {
    const int c = (threadIdx.x % LLE_WAVE) / 16;
    f32x4 s[RT][2];
#pragma unroll
    for (int t = 0; t < RT; ++t) s[t][0] = s[t][1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int ks = 0; ks < DK; ++ks) {
            const bf16x8 k = load_k(x, ks);
#pragma unroll
            for (int t = 0; t < RT; ++t)
                s[t][x] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k, st.qv[t][ks], s[t][x], 0, 0, 0);
        }
    // the value operands are asked for before the softmax, whose arithmetic covers their way
    // from LDS; asked for one by one between the products, each would be waited for in turn
    bf16x8 vv[2 * DK];
#pragma unroll
    for (int n = 0; n < 2 * DK; ++n) vv[n] = load_v(n);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (CAP) {
#pragma unroll
        for (int t = 0; t < RT; ++t)
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const float e = __builtin_amdgcn_exp2f(s[t][i / 4][i % 4] * scale_log2);
                s[t][i / 4][i % 4] = fmaf(-2.f * cap_log2, __builtin_amdgcn_rcpf(1.f + e), cap_log2);
            }
        scale_log2 = 1.f;
    }
    // Scores relative to the row's reference m, in the base-2 domain: x = s * scale - m.  The
    // reference only has to be near the row's maximum, not equal to it: while no x exceeds
    // LAZY_MAX the weights are exp2(x) <= 2^LAZY_MAX and nothing else is touched.  Only when
    // some row of the wavefront goes beyond (the first keys of a row always do: m starts at
    // NEG_BIG) the maxima are agreed on between the four lanes of each row and m, l and the
    // accumulators are moved; that is rare after a row's first steps.
    float x[RT][8];
    bool raise = false;
#pragma unroll
    for (int t = 0; t < RT; ++t) {
#pragma unroll
        for (int i = 0; i < 8; ++i) x[t][i] = fmaf(s[t][i / 4][i % 4], scale_log2, -st.m[t]);
        if (!(j0 >= st.open_lo[t] && j0 + KSTEP - 1 <= st.open_hi[t])) {  // same for the whole wavefront
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int j = j0 + 8 * c + i;  // score i of the lane: tile i / 4, row 4 c + i % 4
                if (j < row[t].lo || j > row[t].pos) x[t][i] = NEG_BIG;
            }
            if (t == 0 && (j0 < seen_lo || j0 + KSTEP - 1 > seen_hi)) drop_values(vv, j0 + 8 * c, seen_lo, seen_hi);
        }
        raise = raise || max_of_8(x[t]) > LAZY_MAX;
    }
    if (__builtin_amdgcn_ballot_w64(raise) != 0) {
#pragma unroll
        for (int t = 0; t < RT; ++t) {
            // absolute scores again (x has lost them where m was still NEG_BIG)
            float sc[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) sc[i] = x[t][i] <= NEG_BIG ? NEG_BIG : s[t][i / 4][i % 4] * scale_log2;
            float tile_max = max_of_8(sc);
            tile_max = column_max(tile_max);
            const float new_m = fmaxf(st.m[t], tile_max);
            // while the row has seen no key new_m is NEG_BIG as its masked scores are, and
            // exp2(0) = 1 would count them: shift such rows so that they give 0
            const float base = new_m <= NEG_BIG ? 0.f : new_m;
            const float alpha = __builtin_amdgcn_exp2f(st.m[t] - base);
            st.m[t] = new_m;
            st.l[t] *= alpha;
#pragma unroll
            for (int n = 0; n < 2 * DK; ++n) st.o[t][n] *= alpha;
#pragma unroll
            for (int i = 0; i < 8; ++i) x[t][i] = sc[i] - base;
        }
    }
    bf16x8 pb[RT];
#pragma unroll
    for (int t = 0; t < RT; ++t) {
        // two chains of additions instead of one: a dependent addition waits for the one before it
        float psum[2] = {0.f, 0.f};
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float p = __builtin_amdgcn_exp2f(x[t][i]);
            psum[i % 2] += p;
            pb[t][i] = (bf16_t)p;
        }
        st.l[t] += psum[0] + psum[1];
    }
#pragma unroll
    for (int n = 0; n < 2 * DK; ++n) {
#pragma unroll
        for (int t = 0; t < RT; ++t)
            st.o[t][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vv[n], pb[t], st.o[t][n], 0, 0, 0);
    }
}

// the partial sums of a row sit in the four lanes r16 + 16 c
template <int DK, int RT>
__device__ __forceinline__ void finish_rows(RowState<DK, RT>& st) {
#pragma unroll
    for (int t = 0; t < RT; ++t) {
        st.l[t] = column_sum(st.l[t]);
    }
}

// Positions into pages: a shift for the usual powers of two (a division by a number known at run time is some thirty
// instructions, and a decode launch makes half a dozen before its first load of a key)
struct PageSize {
    int P, log2;
    __device__ __forceinline__ explicit PageSize(int P) : P(P), log2((P & (P - 1)) == 0 ? 31 - __clz(P) : -1) {}
    __device__ __forceinline__ int of(int position) const { return log2 >= 0 ? position >> log2 : position / P; }
};

// The operands of one 32-key step as a wavefront loads them straight from the pages.
template <int DK>
struct StepOperands {
    bf16x8 k[2][DK];
    bf16x8 v[2 * DK];
};

// The steps step_begin, step_begin + step_stride, ... < step_end with the operands loaded by
// each wavefront straight from the pages, two steps ahead of their use: while one step is
// multiplied the loads of the next two are on their way.  No load stands under a condition (a
// load under a condition makes the compiler wait for every load where the paths meet again):
// loads past the end go to a page that is there.  The loop is left as soon as its last step is
// multiplied: a wavefront alone issues an instruction in four to eight cycles, so a step that
// is masked out whole would be half a microsecond for nothing.
// `before_keys()` runs when the first table lookup is on its way and no operand is asked for yet:
// what the caller loads there travels beside the lookup, what it stores there is stored before
// this wavefront reads any key.  `after_first_loads()` runs once the first two steps are asked for.
// A second range of keys is walked by a call with FIRST = false (the rows' lo and pos are the range's
// then, what the first call has summed up stays); all calls but the last have LAST = false.
template <int DK, int RT, bool LOAD_Q = true, bool FIRST = true, bool LAST = true, bool CAP = false, bool FIND_OPEN = true,
          typename BeforeKeys, typename AfterFirstLoads>
__device__ __forceinline__ void attend_rows(RowState<DK, RT>& st, const RowInfo (&row)[RT],
                                            const bf16_t* kv_layer, const int32_t* __restrict__ table,
                                            int kvh, int nkv, int P, int64_t page_stride, int step_begin,
                                            int step_end, int step_stride, int lo_min, int hi, float scale_log2,
                                            BeforeKeys before_keys, AfterFirstLoads after_first_loads,
                                            float cap_log2 = 0.f) {
    constexpr int D = DK * 32;
    const int lane = threadIdx.x % LLE_WAVE;
    const int c = lane / 16, r16 = lane % 16;
    if constexpr (FIRST) init_rows<DK, RT, LOAD_Q, FIND_OPEN>(st, row);
    else set_open_range<DK, RT>(st, row);
    // the lane's keys of tile x lie in the 16-key half r16 / 8 of the step, its eight V keys in half c / 2
    const int k_half = r16 / 8, v_half = c / 2;
    const int64_t k_lane[2] = {(int64_t)kvh * P * D + (int64_t)(KEY_OF_ROW(r16, 0) % 16) * D + 8 * c,
                               (int64_t)kvh * P * D + (int64_t)(KEY_OF_ROW(r16, 1) % 16) * D + 8 * c};
    const int64_t v_lane = ((int64_t)nkv + kvh) * P * D + (int64_t)r16 * P + 8 * (c % 2);
    // Page and offset of a step's first key are carried from step to step instead of divided
    // out each time (the page size is no constant), and the table is read one load ahead.  A
    // half wholly outside [lo_min, hi] may lie in a page that is not there: the page index is
    // clamped to those of keys that are.
    const PageSize pages(P);
    const int page_lo = pages.of(lo_min), page_hi = pages.of(hi);
    const int adv_pages = pages.of(step_stride * KSTEP), adv_off = step_stride * KSTEP - adv_pages * P;
    int look_page = pages.of(step_begin * KSTEP), look_off = step_begin * KSTEP - look_page * P;
    int page_id[2], page_off[2];
    auto lookup = [&]() {
        const bool next_page = look_off + 16 == P;  // pages hold a multiple of 16 keys
        const int pg[2] = {look_page, next_page ? look_page + 1 : look_page};
        page_off[0] = look_off;
        page_off[1] = next_page ? 0 : look_off + 16;
#pragma unroll
        for (int x = 0; x < 2; ++x)  // the same for the whole wavefront: a scalar load, which no vector load waits for
            page_id[x] = table[__builtin_amdgcn_readfirstlane(min(max(pg[x], page_lo), page_hi))];
        look_page += adv_pages;
        look_off += adv_off;
        if (look_off >= P) {
            look_off -= P;
            ++look_page;
        }
    };
    auto load = [&](StepOperands<DK>& op) {
        const bf16_t* half0 = kv_layer + (int64_t)page_id[0] * page_stride;
        const bf16_t* half1 = kv_layer + (int64_t)page_id[1] * page_stride;
        const bf16_t* kpage = (k_half ? half1 : half0) + (int64_t)(k_half ? page_off[1] : page_off[0]) * D;
        const bf16_t* vp = (v_half ? half1 : half0) + v_lane + (v_half ? page_off[1] : page_off[0]);
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
            for (int ks = 0; ks < DK; ++ks) op.k[x][ks] = *(const bf16x8*)(kpage + k_lane[x] + 32 * ks);
#pragma unroll
        for (int n = 0; n < 2 * DK; ++n) op.v[n] = *(const bf16x8*)(vp + (int64_t)16 * n * P);
        lookup();
    };
    auto multiply = [&](const StepOperands<DK>& op, int step) {
        tile_step<DK, RT, CAP>(
            st, row, [&](int x, int ks) { return op.k[x][ks]; }, [&](int n) { return op.v[n]; }, step * KSTEP,
            lo_min, hi, scale_log2, cap_log2);
    };
    StepOperands<DK> even, odd;
    lookup();
    before_keys();
    load(even);
    load(odd);
    after_first_loads();
    for (int step = step_begin; step < step_end; step += step_stride) {
        multiply(even, step);
        step += step_stride;
        if (step >= step_end) break;
        load(even);
        multiply(odd, step);
        if (step + step_stride >= step_end) break;
        load(odd);
    }
    if constexpr (LAST) finish_rows<DK, RT>(st);
}

// row `r` of the (token, head-in-group) rows of one request and kv head
__device__ __forceinline__ RowInfo make_row(const bf16_t* q, int r, int nrows, int G, int q_start, int past, int nq,
                                            int kvh, int D, int window) {
    RowInfo info;
    if (r < nrows) {
        const int t = nrows == G ? 0 : r / G, g = r - t * G;
        info.q = q + ((int64_t)(q_start + t) * nq + kvh * G + g) * D;
        info.pos = past + t;
        info.lo = window > 0 ? max(0, info.pos - window + 1) : 0;
    } else {
        info.q = nullptr;
        info.pos = -1;
        info.lo = 0;
    }
    return info;
}

// What the decode kernel needs to do the step before it as well: the RMSNorm of each q and k
// head, the rotation over the whole head, and the write of the new K and V into the pages.
// (Decode steps are short and every launch has a price; the prompt path keeps its own kernel.)
struct FusedQKV {
    const bf16_t* qkv;      // [N, (nq + 2 nkv) * D] as the projection left it
    const int32_t* slots;   // [N] place of each token in the pages (page * P + offset), < 0: not written
    const void* q_weight;   // [D] or nullptr: no norm
    const void* k_weight;
    int weight_dtype;
    const float* cos_sin;   // [N, D / 2, 2]
    float eps;
    int write_kv;
    const int32_t* order;   // the requests, longest first (lle_decode_order), or nullptr: as they come
    // short_decode_kernel, PAIRS: a row of qkv has `cols` columns (q, k, v, others), no norms; the first `rot` elements (a multiple
    // of 8) of every q and k head turn in neighbouring pairs by cos_sin [N, rot / 2, 2].  CAP: see tile_step.
    int cols, rot;
    float cap_log2;
};

// Eight consecutive norm weights (float32 or bfloat16) as they lie in memory; what they mean is
// decided by weights8_as_f32 AFTER the loads have met again.  (Converted inside the branch that
// knows the type, every load would be waited for on the spot, one memory latency each.)
struct RawWeights8 {
    uint32_t bits[8];  // bfloat16: the first four words hold the eight values
};
__device__ __forceinline__ void load_raw_weights8(const void* w, int e, int dtype, RawWeights8& out) {
    if (dtype == LLE_F32) {
        const uint4 a = *(const uint4*)((const float*)w + e), b = *(const uint4*)((const float*)w + e + 4);
        out.bits[0] = a.x, out.bits[1] = a.y, out.bits[2] = a.z, out.bits[3] = a.w;
        out.bits[4] = b.x, out.bits[5] = b.y, out.bits[6] = b.z, out.bits[7] = b.w;
    } else {
        const uint4 a = *(const uint4*)((const bf16_t*)w + e);
        out.bits[0] = a.x, out.bits[1] = a.y, out.bits[2] = a.z, out.bits[3] = a.w;
        out.bits[4] = out.bits[5] = out.bits[6] = out.bits[7] = 0u;
    }
}
__device__ __forceinline__ float weights8_as_f32(const RawWeights8& raw, int i, bool is_f32) {
    const uint32_t word = raw.bits[i / 2];
    const uint32_t as_bf16 = (i % 2) ? (word & 0xffff0000u) : (word << 16);
    return __uint_as_float(is_f32 ? raw.bits[i] : as_bf16);
}
// one weight: the word it lies in (a bfloat16 value in the low half), read by weight_as_f32
__device__ __forceinline__ uint32_t load_raw_weight(const void* w, int e, int dtype) {
    if (dtype == LLE_F32) return ((const uint32_t*)w)[e];
    return ((const uint16_t*)w)[e];
}
__device__ __forceinline__ float weight_as_f32(uint32_t raw, bool is_f32) {
    return __uint_as_float(is_f32 ? raw : raw << 16);
}

// Q^T operands of the lane's row from the raw projection: norm over the head (its 4 * DK * 8
// elements sit in the four lanes r16 + 16 c), weight, rotation.  Element 32 ks + 8 c + i and its
// partner D / 2 further on are both in this lane (DK is even).  Rounded to bfloat16 as the
// separate kernel rounds q.  Everything is ASKED FOR in one go (load) and worked on later
// (finish): a load that followed the arithmetic on another would cost the memory's latency again.
// WEIGHTS: their type where the launch is made for it, -1 where only FusedQKV::weight_dtype knows.
template <int DK, int WEIGHTS = -1>
struct FusedQRow {
    static_assert(DK % 2 == 0, "rotation partners lie in one lane only for an even number of 32-element blocks");
    typedef float4 Table[DK / 2][4];  // cos, sin of element 2 i, then of 2 i + 1
    bf16x8 raw[DK];
    RawWeights8 w[DK];

    // `src`: the head of a row that exists (lanes of rows that do not exist read another row's and drop it)
    __device__ __forceinline__ void load(const bf16_t* src, const void* weight, int weight_dtype) {
        const int c = (threadIdx.x % LLE_WAVE) / 16;
#pragma unroll
        for (int ks = 0; ks < DK; ++ks) raw[ks] = *(const bf16x8*)(src + 32 * ks + 8 * c);
        if (weight) {
#pragma unroll
            for (int ks = 0; ks < DK; ++ks) load_raw_weights8(weight, 32 * ks + 8 * c, WEIGHTS < 0 ? weight_dtype : WEIGHTS, w[ks]);
        }
    }
    static __device__ __forceinline__ void load_table(Table& tab, const FusedQKV& f, int64_t tok) {
        constexpr int D = DK * 32;
        const int c = (threadIdx.x % LLE_WAVE) / 16;
#pragma unroll
        for (int ks = 0; ks < DK / 2; ++ks) {
            const float4* t = (const float4*)(f.cos_sin + (tok * (D / 2) + 32 * ks + 8 * c) * 2);
#pragma unroll
            for (int i = 0; i < 4; ++i) tab[ks][i] = t[i];
        }
    }

    // PAIRS: elements that turn come eight at a time (the others read what is there and are left as they are)
    static __device__ __forceinline__ void load_pair_table(Table& tab, const FusedQKV& f, int64_t tok) {
        const int c = (threadIdx.x % LLE_WAVE) / 16;
        if (f.rot <= 0) return;  // (the same for the whole launch)
#pragma unroll
        for (int ks = 0; ks < DK; ++ks) {
            const float4* t = (const float4*)(f.cos_sin + tok * f.rot + min(32 * ks + 8 * c, f.rot - 8));
            tab[ks / 2][2 * (ks % 2)] = t[0];
            tab[ks / 2][2 * (ks % 2) + 1] = t[1];
        }
    }
    __device__ __forceinline__ void finish_pairs(bf16x8 (&qv)[DK], const Table& tab, const FusedQKV& f) const {
        const int c = (threadIdx.x % LLE_WAVE) / 16;
#pragma unroll
        for (int ks = 0; ks < DK; ++ks) {
            const float4 t0 = tab[ks / 2][2 * (ks % 2)], t1 = tab[ks / 2][2 * (ks % 2) + 1];
            const float cs[4] = {t0.x, t0.z, t1.x, t1.z}, sn[4] = {t0.y, t0.w, t1.y, t1.w};
            bf16x8 turned;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float a = (float)raw[ks][2 * i], b = (float)raw[ks][2 * i + 1];
                turned[2 * i] = (bf16_t)(a * cs[i] - b * sn[i]);
                turned[2 * i + 1] = (bf16_t)(b * cs[i] + a * sn[i]);
            }
            qv[ks] = 32 * ks + 8 * c < f.rot ? turned : raw[ks];
        }
    }

    __device__ __forceinline__ void finish(bf16x8 (&qv)[DK], const Table& tab, const FusedQKV& f, bool normed) const {
        constexpr int D = DK * 32;
        float x[DK][8];
#pragma unroll
        for (int ks = 0; ks < DK; ++ks)
#pragma unroll
            for (int i = 0; i < 8; ++i) x[ks][i] = (float)raw[ks][i];
        if (normed) {
            float ss = 0.f;
#pragma unroll
            for (int ks = 0; ks < DK; ++ks)
#pragma unroll
                for (int i = 0; i < 8; ++i) ss += x[ks][i] * x[ks][i];
            ss = column_sum(ss);
            const float inv = 1.0f / sqrtf(ss / (float)D + f.eps);
            auto weigh = [&](auto is_f32) {
#pragma unroll
                for (int ks = 0; ks < DK; ++ks)
#pragma unroll
                    for (int i = 0; i < 8; ++i) x[ks][i] = x[ks][i] * inv * weights8_as_f32(w[ks], i, decltype(is_f32)::value);
            };
            if (WEIGHTS < 0 ? f.weight_dtype == LLE_F32 : WEIGHTS == LLE_F32)  // (the same for the whole launch: a branch instead of 32 selects)
                weigh(std::integral_constant<bool, true>{});
            else
                weigh(std::integral_constant<bool, false>{});
        }
#pragma unroll
        for (int ks = 0; ks < DK / 2; ++ks) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float4 t = tab[ks][i];
                const float a0 = x[ks][2 * i], b0 = x[ks + DK / 2][2 * i];
                const float a1 = x[ks][2 * i + 1], b1 = x[ks + DK / 2][2 * i + 1];
                x[ks][2 * i] = a0 * t.x - b0 * t.y;
                x[ks + DK / 2][2 * i] = b0 * t.x + a0 * t.y;
                x[ks][2 * i + 1] = a1 * t.z - b1 * t.w;
                x[ks + DK / 2][2 * i + 1] = b1 * t.z + a1 * t.w;
            }
        }
#pragma unroll
        for (int ks = 0; ks < DK; ++ks)
#pragma unroll
            for (int i = 0; i < 8; ++i) qv[ks][i] = (bf16_t)x[ks][i];
    }
};

// One wavefront: K (norm, weight, rotation) and V of token `tok`, kv head `kvh`, into the pages.
// Lane l takes elements l, l + 64, ... < D / 2 and their partners D / 2 further on.  All loads
// are asked for before anything waits for one of them.
template <int DK>
__device__ __forceinline__ void fused_kv_write(const FusedQKV& f, int64_t tok, int kvh, int nq, int nkv,
                                               bf16_t* kv_layer, int P, int64_t page_stride) {
    constexpr int D = DK * 32, HALF = D / 2, PER = (HALF + LLE_WAVE - 1) / LLE_WAVE;
    const int lane = threadIdx.x % LLE_WAVE;
    const int slot = f.slots[tok];
    const bf16_t* ksrc = f.qkv + (tok * (nq + 2 * nkv) + nq + kvh) * D;
    const bf16_t* vsrc = ksrc + (int64_t)nkv * D;
    float lo[PER], hi[PER];
    uint32_t wlo[PER], whi[PER];
    bf16_t vlo[PER], vhi[PER];
    float2 tab[PER];
#pragma unroll
    for (int j = 0; j < PER; ++j) {
        const int e = min(lane + LLE_WAVE * j, HALF - 1);  // lanes past the half read its last element and drop it
        lo[j] = (float)ksrc[e];
        hi[j] = (float)ksrc[e + HALF];
        vlo[j] = vsrc[e];
        vhi[j] = vsrc[e + HALF];
        tab[j] = *(const float2*)(f.cos_sin + (tok * HALF + e) * 2);
        wlo[j] = whi[j] = 0x3f80u;  // 1 as bfloat16
    }
    const bool is_f32 = f.k_weight && f.weight_dtype == LLE_F32;
    if (f.k_weight) {
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            const int e = min(lane + LLE_WAVE * j, HALF - 1);
            wlo[j] = load_raw_weight(f.k_weight, e, f.weight_dtype);
            whi[j] = load_raw_weight(f.k_weight, e + HALF, f.weight_dtype);
        }
    }
    if (slot < 0) return;
    const int page = PageSize(P).of(slot), off = slot - page * P;
    bf16_t* page_base = kv_layer + (int64_t)page * page_stride;
    bf16_t* kdst = page_base + ((int64_t)kvh * P + off) * D;
    bf16_t* vdst = page_base + ((int64_t)nkv + kvh) * P * D + off;  // element e at vdst[e * P]
    float inv = 1.f;
    if (f.k_weight) {
        float ss = 0.f;
#pragma unroll
        for (int j = 0; j < PER; ++j)
            if (lane + LLE_WAVE * j < HALF) ss += lo[j] * lo[j] + hi[j] * hi[j];
        ss = wave_sum(ss);
        inv = 1.0f / sqrtf(ss / (float)D + f.eps);
    }
#pragma unroll
    for (int j = 0; j < PER; ++j) {
        const int e = lane + LLE_WAVE * j;
        if (e < HALF) {
            const float a = lo[j] * inv * weight_as_f32(wlo[j], is_f32), b = hi[j] * inv * weight_as_f32(whi[j], is_f32);
            kdst[e] = (bf16_t)(a * tab[j].x - b * tab[j].y);
            kdst[e + HALF] = (bf16_t)(b * tab[j].x + a * tab[j].y);
            vdst[(int64_t)e * P] = vlo[j];
            vdst[(int64_t)(e + HALF) * P] = vhi[j];
        }
    }
}

// Requests whose rows (q_len * group) fit one 16-row tile: decoded tokens and very
// short portions.  grid = (requests, kv heads, splits).
#ifndef DEC_WAVES
#define DEC_WAVES 4
#endif
template <int DK, bool FUSED, bool KEEP, bool CAP>
__global__ __launch_bounds__(DEC_WAVES* LLE_WAVE) void mfma_decode_kernel(
    const bf16_t* __restrict__ q, bf16_t* kv_layer, const int32_t* __restrict__ block_tables,
    const int32_t* __restrict__ seq_slots, const int32_t* __restrict__ cu_tokens,
    const int32_t* __restrict__ kv_lens, bf16_t* __restrict__ out, float* __restrict__ ws_o,
    float* __restrict__ ws_ml, int ws_stride, int nq, int nkv, int P, int64_t page_stride, int max_pages,
    int window, float scale_log2, FusedQKV fused, const float* __restrict__ sinks, int keep_first, float cap_log2) {
    static_assert(!(FUSED && (KEEP || CAP)), "kept first keys, capped scores: the launch that reads ready-made queries");
    static_assert(!(KEEP && CAP), "kept first keys or capped scores");
    constexpr int D = DK * 32;
    extern __shared__ float smem[];  // [waves][16][D] acc, then [waves][16] m, [waves][16] l
    float* s_o = smem;
    float* s_m = smem + DEC_WAVES * 16 * D;
    float* s_l = s_m + DEC_WAVES * 16;

    // A launch of this kernel is short, and what it waits for before its first key counts.  All
    // arguments are read here in one go, and so is all that is known of the request: read where
    // they are first used, each group would cost a round trip to memory of its own.
    // (The four tables that are read with scalar loads stay out of the statement: a pointer that
    // it has seen counts as written to, and loads through it would become vector loads.)
    asm volatile("" ::"s"(q), "s"(kv_layer), "s"(out), "s"(ws_o), "s"(ws_ml), "s"(ws_stride), "s"(nq), "s"(nkv), "s"(P),
                 "s"(page_stride), "s"(max_pages), "s"(window), "s"(scale_log2), "s"(fused.qkv), "s"(fused.slots),
                 "s"(fused.q_weight), "s"(fused.k_weight), "s"(fused.weight_dtype), "s"(fused.cos_sin),
                 "s"(fused.eps), "s"(fused.write_kv));
    int s = blockIdx.x, kvh = blockIdx.y;
    const int split = blockIdx.z, nsplit = gridDim.z;
    const int G = nq / nkv;
    if (FUSED && fused.order) {
        // More workgroups than CUs, which take one each and the next as they finish: with the longest requests first the
        // last ones to start are short (all heads of a request before the next request).  Consecutive workgroups go to
        // different dies: the heads turn from request to request, so that a die does not read the same head of every
        // page, whose places repeat every 32 KB.  (64, 128 requests of 4096 keys, 8 key heads: 191, 351 us as they come; 191,
        // 411 longest first, 180, 351 with turned heads.  32 of 16 key heads: 186, 232, 178.)
        const int id = blockIdx.y * gridDim.x + blockIdx.x, rank = id / nkv;
        s = fused.order[rank];
        kvh = (id + rank * min(nkv, 8) / 8) % nkv;
    }
    const int q_start = cu_tokens[s], q_end = cu_tokens[s + 1], kv_len = kv_lens[s], seq_slot = seq_slots[s];
    asm volatile("" ::"s"(q_start), "s"(q_end), "s"(kv_len), "s"(seq_slot));
    const int q_len = q_end - q_start;
    const int nrows = q_len * G;
    if (nrows > 16 || nrows <= 0) return;  // the prefill kernel's, or nothing to do
    const int past = kv_len - q_len;
    const int wave = threadIdx.x / LLE_WAVE, lane = threadIdx.x % LLE_WAVE;
    const int c = lane / 16, r16 = lane % 16;
    const int32_t* table = block_tables + (int64_t)seq_slot * max_pages;

    // FUSED: q is made here from the projection; the row's pointer only says that the row exists
    RowInfo row[1] = {make_row(FUSED ? fused.qkv : q, r16, nrows, G, q_start, past, nq, kvh, D, window)};
    const int lo_min = window > 0 ? max(0, past - window + 1) : 0;
    const int hi = kv_len - 1;
    const int first = lo_min / KSTEP, last = hi / KSTEP;
    const int per_split = nsplit == 1 ? last - first + 1 : (last - first + 1 + nsplit - 1) / nsplit;
    const int sb = first + split * per_split;
    const int se = min(last + 1, sb + per_split);
    // keys of later splits are not this workgroup's
    row[0].pos = min(row[0].pos, se * KSTEP - 1);
    // attend_rows asks for operands two steps ahead: past this split's last key those loads go to the
    // split's own last page (which the caches hold) instead of the next split's pages, which would
    // travel from memory twice, once for each of the two workgroups
    const int hi_loads = max(lo_min, min(hi, se * KSTEP - 1));

    RowState<DK, 1> st;
    if constexpr (!KEEP) {  // the request's tokens see from its last one's first key on, and up to its first one's own
        st.open_lo[0] = window > 0 ? max(0, hi - window + 1) : 0;
        st.open_hi[0] = min(past, se * KSTEP - 1);
    }
    if constexpr (FUSED) {
        // The raw q row, its rotation table and the norm weights are asked for while the table
        // lookup is on its way.  A new token's K and V go into the pages by the hand of the
        // wavefront that multiplies the token's step (step sb + wave, + DEC_WAVES, ...): it
        // stores them before it asks for any key, no other wavefront of this launch needs them,
        // and so no barrier stands between the write and the keys.
        FusedQRow<DK> qrow;
        typename FusedQRow<DK>::Table tab;
        const int rr = r16 < nrows ? r16 : 0;
        const int t_row = nrows == G ? 0 : rr / G;
        const int64_t tok = (int64_t)q_start + t_row;
        attend_rows<DK, 1, false, true, true, false, false>(
            st, row, kv_layer, table, kvh, nkv, P, page_stride, sb + wave, se, DEC_WAVES, lo_min, hi_loads, scale_log2,
            [&]() {
                qrow.load(fused.qkv + (tok * (nq + 2 * nkv) + kvh * G + rr - t_row * G) * D, fused.q_weight, fused.weight_dtype);
                FusedQRow<DK>::load_table(tab, fused, tok);
                if (fused.write_kv) {
                    for (int t = 0; t < q_len; ++t) {
                        const int step_of = (past + t) / KSTEP;
                        if (step_of >= sb && step_of < se && (step_of - sb) % DEC_WAVES == wave)
                            fused_kv_write<DK>(fused, (int64_t)q_start + t, kvh, nq, nkv, kv_layer, P, page_stride);
                    }
                    // The keys are read through the same pointer (no `restrict` on it: the pages are
                    // written and read in this kernel), after this point in program order; the fence
                    // keeps the compiler from moving those loads above the stores.
                    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
                    asm volatile("" ::: "memory");
                }
            },
            [&]() { qrow.finish(st.qv[0], tab, fused, fused.q_weight != nullptr); });
    } else if constexpr (KEEP) {
        // the kept first keys are the first split's work (few steps)
        init_rows<DK, 1, true>(st, row);
        const int kept = min(keep_first, max(0, hi - window + 1));  // of the row that sees the most of them
        if (split == 0 && kept > 0) {
            const RowInfo main_row = row[0];
            if (row[0].q) row[0].pos = min(keep_first, row[0].lo) - 1;
            row[0].lo = 0;
            attend_rows<DK, 1, true, false, false>(
                st, row, kv_layer, table, kvh, nkv, P, page_stride, wave, (kept + KSTEP - 1) / KSTEP, DEC_WAVES, 0, kept - 1,
                scale_log2, []() {}, []() {});
            row[0] = main_row;
        }
        attend_rows<DK, 1, true, false, true>(
            st, row, kv_layer, table, kvh, nkv, P, page_stride, sb + wave, se, DEC_WAVES, lo_min, hi_loads, scale_log2,
            []() {}, []() {});
    } else {
        attend_rows<DK, 1, true, true, true, CAP, false>(
            st, row, kv_layer, table, kvh, nkv, P, page_stride, sb + wave, se, DEC_WAVES, lo_min, hi_loads, scale_log2,
            []() {}, []() {}, cap_log2);
    }

    // merge the wavefronts (rows that do not exist are not worth the LDS traffic)
    if (r16 < nrows) {
#pragma unroll
        for (int n = 0; n < 2 * DK; ++n) *(f32x4*)(s_o + (wave * 16 + r16) * D + 16 * n + 4 * c) = st.o[0][n];
    }
    if (c == 0) {
        s_m[wave * 16 + r16] = st.m[0];
        s_l[wave * 16 + r16] = st.l[0];
    }
    __syncthreads();
    for (int idx = threadIdx.x; idx < nrows * D; idx += blockDim.x) {
        const int r = idx / D, e = idx - r * D;
        float big = s_m[r];
#pragma unroll
        for (int w = 1; w < DEC_WAVES; ++w) big = fmaxf(big, s_m[w * 16 + r]);
        float num = 0.f, den = 0.f;
#pragma unroll
        for (int w = 0; w < DEC_WAVES; ++w) {
            const float f = exp2f(s_m[w * 16 + r] - big);
            num += s_o[(w * 16 + r) * D + e] * f;
            den += s_l[w * 16 + r] * f;
        }
        const int t = nrows == G ? 0 : r / G, g = r - t * G;
        const int64_t head_row = (int64_t)(q_start + t) * nq + kvh * G + g;
        if (nsplit == 1) {
            if (sinks) den += exp2f(sinks[kvh * G + g] * 1.44269504088896340736f - big);  // (a sink: a place in the sum without a value)
            out[head_row * D + e] = (bf16_t)(num / den);
        } else {
            ws_o[(head_row * ws_stride + split) * D + e] = num;
            if (e == 0) {
                ws_ml[(head_row * ws_stride + split) * 2] = big;
                ws_ml[(head_row * ws_stride + split) * 2 + 1] = den;
            }
        }
    }
}

// One new token a request, at most SHORT_WAVES * 32 keys: grid (requests, kv heads), a wavefront for every 32 keys and one for the
// new token.  A launch of this size is bound by how many instructions stand in a row (a wavefront alone issues one in four to
// eight cycles) and by trips to memory that wait for each other, not by bytes: no loop over keys, no running maximum, no carried
// page numbers (a wavefront's keys lie at the same positions of every request), and the new token's key and value never pass
// through the page: their wavefront scores and stores them while the others wait for theirs.  The wavefronts meet once, in LDS;
// those without keys leave zeros there.
// 0.6B sizes (16 q heads, 8 kv heads of 128) at 97 keys, 1 / 8 / 32 requests: 7.9 / 8.1 / 9.7 us in mfma_decode_kernel, whose
// loop holds two steps and whose new token goes through the page, 6.1 / 6.5 / 8.0 here.
#define SHORT_WAVES 8
// a score in the base-2 domain (CAP as in tile_step)
template <bool CAP>
__device__ __forceinline__ float short_score(float s, float scale_log2, float cap_log2) {
    if constexpr (CAP) return fmaf(-2.f * cap_log2, __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(s * scale_log2)), cap_log2);
    return s * scale_log2;
}
// PAIRS, CAP: what FusedQKV says.  Rorevik's attention (16 q heads, 4 kv heads of 128, capped scores) at 8 requests of 100 keys:
// 11.9 us in two launches (rotation and cache write 6.7, attention 5.2), 4.6 here.
template <int DK, int WEIGHTS, bool PAIRS, bool CAP>
__global__ __launch_bounds__((SHORT_WAVES + 1) * LLE_WAVE) void short_decode_kernel(
    const int32_t* __restrict__ cu_tokens, const int32_t* __restrict__ kv_lens, const int32_t* __restrict__ seq_slots,
    const int32_t* __restrict__ block_tables, int max_pages, int P, int window, int G, int nkv, bf16_t* kv_layer,
    bf16_t* __restrict__ out, int64_t page_stride, float scale_log2, FusedQKV f) {
    // The first sixteen words of the arguments come with the launch: the tables that everything waits for are among them, and what is
    // known of the request is asked for before the other arguments.  Each of these statements has one trip to memory behind it:
    // read where they are first used, the same loads are five in a row.  (Pointers that are read by scalar loads stay out of them.)
    const int s = blockIdx.x, kvh = blockIdx.y;
    const int tok = cu_tokens[s], tok_end = cu_tokens[s + 1], kv_len = kv_lens[s], seq_slot = seq_slots[s];
    asm volatile("" ::"s"(tok), "s"(tok_end), "s"(kv_len), "s"(seq_slot), "s"(nkv), "s"(kv_layer), "s"(out), "s"(page_stride),
                 "s"(scale_log2), "s"(f.qkv), "s"(f.q_weight), "s"(f.k_weight), "s"(f.cos_sin), "s"(f.eps), "s"(f.write_kv));
    constexpr int D = DK * 32, WAVES = SHORT_WAVES + 1;
    extern __shared__ float smem[];  // [waves][G][D] acc, then [waves][16] m, [waves][16] l
    float* s_m = smem + WAVES * G * D;
    float* s_l = s_m + WAVES * 16;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / LLE_WAVE), lane = threadIdx.x % LLE_WAVE;
    const int c = lane / 16, r16 = lane % 16;
    if (tok_end - tok != 1) return;  // (a request without a token has nothing to do)
    const int last = kv_len - 1, lo = window > 0 ? max(0, kv_len - window) : 0;
    const int j0 = wave * KSTEP;  // the wavefront's first key
    // both halves' pages (a half outside what is seen reads the other half's page; a wavefront without keys the last key's)
    const PageSize pages(P);
    const int j0_kept = min(j0, last), j1 = j0_kept + 16 <= last ? j0_kept + 16 : j0_kept, j0_seen = j0_kept + 16 > lo ? j0_kept : j1;
    const int p0 = pages.of(j0_seen), p1 = pages.of(j1);
    const int32_t* table = block_tables + (int64_t)seq_slot * max_pages;
    const int page0 = table[p0], page1 = table[p1], slot = f.slots[tok];
    const bool fresh = f.write_kv && slot >= 0;  // (else the new token's place holds what the page does)
    const bf16_t* qkv = f.qkv + (int64_t)tok * (PAIRS ? f.cols : nkv * (G + 2) * D);
    const bf16_t* q_head = qkv + (int64_t)(kvh * G + min(r16, G - 1)) * D;  // (rows past the group's: dropped at the end)
    f32x4 o[2 * DK];
    float top = NEG_BIG, l = 0.f;
    if (wave < SHORT_WAVES && j0 <= last && j0 + KSTEP > lo) {
        FusedQRow<DK, WEIGHTS> qrow;
        typename FusedQRow<DK, WEIGHTS>::Table tab;
        qrow.load(q_head, PAIRS ? nullptr : f.q_weight, f.weight_dtype);
        if constexpr (PAIRS) qrow.load_pair_table(tab, f, tok);
        else qrow.load_table(tab, f, tok);
        const bool k_second = r16 / 8 != 0, v_second = c / 2 != 0;
        const int64_t base0 = (int64_t)page0 * page_stride, base1 = (int64_t)page1 * page_stride;
        const int off0 = j0_seen - p0 * P, off1 = j1 - p1 * P;
        const bf16_t* kp = kv_layer + (k_second ? base1 : base0) + ((int64_t)kvh * P + (k_second ? off1 : off0)) * D + 8 * c;
        const bf16_t* vp = kv_layer + (v_second ? base1 : base0) + ((int64_t)(nkv + kvh) * D + r16) * P +
                           (v_second ? off1 : off0) + 8 * (c % 2);
        StepOperands<DK> op;  // (laid out as KEY_OF_ROW says)
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
            for (int ks = 0; ks < DK; ++ks) op.k[x][ks] = *(const bf16x8*)(kp + (KEY_OF_ROW(r16, x) % 16) * D + 32 * ks);
#pragma unroll
        for (int n = 0; n < 2 * DK; ++n) op.v[n] = *(const bf16x8*)(vp + (int64_t)16 * n * P);
        bf16x8 qv[DK];
        if constexpr (PAIRS) qrow.finish_pairs(qv, tab, f);
        else qrow.finish(qv, tab, f, f.q_weight != nullptr);
        f32x4 sc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
            for (int ks = 0; ks < DK; ++ks) sc[x] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(op.k[x][ks], qv[ks], sc[x], 0, 0, 0);
        const int pos = fresh ? last - 1 : last;  // the last key that comes from the pages
        float x[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) x[i] = short_score<CAP>(sc[i / 4][i % 4], scale_log2, f.cap_log2);
        if (j0 < lo || j0 + KSTEP - 1 > pos) {  // (the same for the whole wavefront)
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int j = j0 + 8 * c + i;
                if (j < lo || j > pos) x[i] = NEG_BIG;
            }
            // (the new token's place among them, which its wavefront may be writing just now)
            drop_values(op.v, j0 + 8 * c, lo, pos);
        }
        top = column_max(max_of_8(x));
        const float base = top <= NEG_BIG ? 0.f : top;  // (no key is seen where the new token is the wavefront's first one)
        bf16x8 pb;
        float sum[2] = {0.f, 0.f};
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float p = __builtin_amdgcn_exp2f(x[i] - base);
            sum[i % 2] += p;
            pb[i] = (bf16_t)p;
        }
#pragma unroll
        for (int n = 0; n < 2 * DK; ++n)
            o[n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(op.v[n], pb, f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
        l = column_sum(sum[0] + sum[1]);
    } else if (wave == SHORT_WAVES && fresh) {
        const bf16_t* k_head = qkv + (int64_t)(nkv * G + kvh) * D;
        const bf16_t* v_head = k_head + (int64_t)nkv * D;
        FusedQRow<DK, WEIGHTS> qrow, krow;
        typename FusedQRow<DK, WEIGHTS>::Table tab;
        krow.load(k_head, PAIRS ? nullptr : f.k_weight, f.weight_dtype);
        if constexpr (PAIRS) krow.load_pair_table(tab, f, tok);
        else krow.load_table(tab, f, tok);
        qrow.load(q_head, PAIRS ? nullptr : f.q_weight, f.weight_dtype);
        bf16x4 v[2 * DK];
#pragma unroll
        for (int n = 0; n < 2 * DK; ++n) v[n] = *(const bf16x4*)(v_head + 16 * n + 4 * c);
        bf16x8 kv[DK], qv[DK];
        if constexpr (PAIRS) krow.finish_pairs(kv, tab, f);
        else krow.finish(kv, tab, f, f.k_weight != nullptr);
        const int page = pages.of(slot), off = slot - page * P;
        bf16_t* base = kv_layer + (int64_t)page * page_stride;
        if (r16 == 0) {
            bf16_t* kdst = base + ((int64_t)kvh * P + off) * D + 8 * c;
            bf16_t* vdst = base + ((int64_t)(nkv + kvh) * D + 4 * c) * P + off;
#pragma unroll
            for (int ks = 0; ks < DK; ++ks) *(bf16x8*)(kdst + 32 * ks) = kv[ks];
#pragma unroll
            for (int n = 0; n < 2 * DK; ++n)
#pragma unroll
                for (int i = 0; i < 4; ++i) vdst[(int64_t)(16 * n + i) * P] = v[n][i];
        }
        if constexpr (PAIRS) qrow.finish_pairs(qv, tab, f);
        else qrow.finish(qv, tab, f, f.q_weight != nullptr);
        float dot[2] = {0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < DK; ++ks)
#pragma unroll
            for (int i = 0; i < 8; ++i) dot[i % 2] = fmaf((float)kv[ks][i], (float)qv[ks][i], dot[i % 2]);
        top = short_score<CAP>(column_sum(dot[0] + dot[1]), scale_log2, f.cap_log2);
        l = 1.f;
#pragma unroll
        for (int n = 0; n < 2 * DK; ++n)
#pragma unroll
            for (int i = 0; i < 4; ++i) o[n][i] = (float)v[n][i];
    } else {
#pragma unroll
        for (int n = 0; n < 2 * DK; ++n) o[n] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    if (r16 < G) {
#pragma unroll
        for (int n = 0; n < 2 * DK; ++n) *(f32x4*)(smem + (wave * G + r16) * D + 16 * n + 4 * c) = o[n];
    }
    if (c == 0) {
        s_m[wave * 16 + r16] = top;
        s_l[wave * 16 + r16] = l;
    }
    __syncthreads();
    for (int idx = threadIdx.x; idx < G * D; idx += WAVES * LLE_WAVE) {
        const int r = idx / D;
        float m[WAVES], big = NEG_BIG;
#pragma unroll
        for (int w = 0; w < WAVES; ++w) {
            m[w] = s_m[w * 16 + r];
            big = fmaxf(big, m[w]);
        }
        float num = 0.f, den = 0.f;
#pragma unroll
        for (int w = 0; w < WAVES; ++w) {
            const float e = __builtin_amdgcn_exp2f(m[w] - big);
            num = fmaf(smem[w * G * D + idx], e, num);
            den = fmaf(s_l[w * 16 + r], e, den);
        }
        out[((int64_t)tok * (nkv * G) + kvh * G) * D + idx] = (bf16_t)(num / den);
    }
}

// order[0 .. S - 1]: the requests by falling length, equal ones as they come.  One workgroup, S <= 1024: a request's place is
// the number of those before it.
__global__ __launch_bounds__(1024) void decode_order_kernel(const int32_t* __restrict__ kv_lens, int32_t* __restrict__ order, int S) {
    __shared__ int lens[1024];
    const int i = threadIdx.x;
    const int own = i < S ? kv_lens[i] : 0;
    lens[i] = own;
    __syncthreads();
    if (i >= S) return;
    int place = 0;
    for (int j = 0; j < S; ++j) place += lens[j] > own || (lens[j] == own && j < i);
    order[place] = i;
}

extern "C" int lle_decode_order(const void* kv_lens, void* order, int S, hipStream_t stream) {
    if (S <= 0) return 0;
    if (S > 1024) return (int)hipErrorInvalidValue;
    decode_order_kernel<<<1, (S + LLE_WAVE - 1) / LLE_WAVE * LLE_WAVE, 0, stream>>>((const int32_t*)kv_lens, (int32_t*)order, S);
    return (int)hipGetLastError();
}

// Merges the key splits.  grid = (tokens, q heads), one wavefront each; lane k holds (m, l) of
// split k (at most 64 splits).  A token of a request with at most 16 rows was split
// `nsplit_decode` ways by the decode kernel, any other `nsplit_prefill` ways by the prefill
// kernel; a token whose kernel did not split was written by that kernel itself.
__global__ __launch_bounds__(LLE_WAVE) void mfma_combine_kernel(const float* __restrict__ ws_o,
                                                                const float* __restrict__ ws_ml, int ws_stride,
                                                                const int32_t* __restrict__ cu_tokens,
                                                                const int32_t* __restrict__ token_seq,
                                                                bf16_t* __restrict__ out, int nq, int nkv, int D,
                                                                int nsplit_decode, int nsplit_prefill,
                                                                const float* __restrict__ sinks) {
    const int64_t tok = blockIdx.x;
    const int h = blockIdx.y;
    int nsplit = nsplit_decode;
    if (nsplit_decode != nsplit_prefill) {
        const int s = token_seq ? token_seq[tok] : (int)tok;
        if ((cu_tokens[s + 1] - cu_tokens[s]) * (nq / nkv) > 16) nsplit = nsplit_prefill;
    }
    if (nsplit <= 1) return;
    const int lane = threadIdx.x;
    const int64_t head_row = tok * nq + h;
    // (m, l) of the lane's split and the first eight splits' partial sums of the lane's first two
    // elements are asked for together: the launch is as short as its chain of loads.
    const float* o = ws_o + head_row * ws_stride * D;
    const float2 ml = *(const float2*)(ws_ml + (head_row * ws_stride + min(lane, nsplit - 1)) * 2);
    const int e_first = min(2 * lane, D - 2);
    float2 first[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) first[j] = *(const float2*)(o + (int64_t)min(j, nsplit - 1) * D + e_first);
    const float m = lane < nsplit ? ml.x : NEG_BIG, l = lane < nsplit ? ml.y : 0.f;
    const float big = wave_max(m);
    const float f = exp2f(m - big);  // 0 for lanes without a split (l = 0 there anyway)
    float den = wave_sum(l * f);
    if (sinks) den += exp2f(sinks[h] * 1.44269504088896340736f - big);  // (a sink: a place in the sum without a value)
    // every lane needs every split's factor, also those of lanes that have no element below
    __shared__ float s_f[LLE_WAVE];
    s_f[lane] = f;
    __syncthreads();
    // A lane takes two neighbouring elements; the partial sums of eight splits are loaded
    // together (one load after the other would pay the memory's latency once per split).
    for (int e = 2 * lane; e < D; e += 2 * LLE_WAVE) {
        float2 num = {0.f, 0.f};
        for (int k0 = 0; k0 < nsplit; k0 += 8) {
            float2 part[8];
            if (k0 == 0 && e == e_first) {
#pragma unroll
                for (int j = 0; j < 8; ++j) part[j] = first[j];
            } else {
#pragma unroll
                for (int j = 0; j < 8; ++j) part[j] = *(const float2*)(o + (int64_t)min(k0 + j, nsplit - 1) * D + e);
            }
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const float fk = k0 + j < nsplit ? s_f[k0 + j] : 0.f;
                num.x += part[j].x * fk;
                num.y += part[j].y * fk;
            }
        }
        out[head_row * D + e] = (bf16_t)(num.x / den);
        out[head_row * D + e + 1] = (bf16_t)(num.y / den);
    }
}

// Requests with more than 16 rows.  grid = (kv heads, row blocks x key splits, requests); a
// workgroup takes a block of rows (token, head of the group) and walks the keys they see in steps
// of 32.  A short portion after a long past has few row blocks: its keys are then split over
// `nsplit` workgroups, which leave (m, l, acc) for the combine kernel.  The 32-key tiles of K and
// V^T are copied from the pages into LDS once per workgroup (all threads; two tiles are on their
// way while one is multiplied) and every wavefront reads its matrix-core operands from there:
// the rows of a workgroup share one pass over the keys.
//   LDS K tile:   [32 keys][D]    LDS V^T tile: [D][32 keys]
// both without padding, the 16-byte pieces of a row XOR-swizzled (K_SWIZZLE, V_SWIZZLE).
// Heads of 128 elements skip the registers: global_load_lds_dwordx4 writes the tiles into LDS
// directly (three buffers; see the DMA branch of the kernel).
// The shapes of a workgroup (PRE_WAVES wavefronts of PRE_RT tiles of 16 rows each):
//   4 x 1: 64 rows.  Twice the workgroups of half the height: for launches so small that these
//          all fit the chip at once.
//   4 x 2: 128 rows; every operand read from LDS serves both tiles of a wavefront.  Two
//          workgroups a CU in 256 registers a lane (heads up to 128; above, 4 x 1 only).
//   8 x 1: 128 rows, heads of 128 only.  Two workgroups a CU are four wavefronts a SIMD, in 128
//          registers each.  A wavefront issues about one instruction in eight cycles whatever
//          its kind, and a matrix instruction holds it for sixteen; the wavefronts of a SIMD run
//          side by side until they meet at an issue port, so four of them get more out of it
//          than two (measured: 118 against 128 us for 2048 rows over 4096 keys), although each
//          tile is then read from LDS by twice as many wavefronts.
#ifndef PRE_RT_MAX
#define PRE_RT_MAX 2
#endif
#define PRE_RT_OF(DK) ((DK) <= 4 ? PRE_RT_MAX : 1)
template <int DK, int PRE_RT, int PRE_WAVES, bool KEEP, bool CAP>
// (heads over 192 elements need more than the 256 registers a lane that two workgroups a CU leave)
__global__ __launch_bounds__(PRE_WAVES* LLE_WAVE, DK <= 6 ? 2 : 1) void mfma_prefill_kernel(
    const bf16_t* __restrict__ q, const bf16_t* __restrict__ kv_layer, const int32_t* __restrict__ block_tables,
    const int32_t* __restrict__ seq_slots, const int32_t* __restrict__ cu_tokens,
    const int32_t* __restrict__ kv_lens, bf16_t* __restrict__ out, float* __restrict__ ws_o,
    float* __restrict__ ws_ml, int ws_stride, int nsplit, int nq, int nkv, int P, int64_t page_stride, int max_pages,
    int window, float scale_log2, int complement_order, const float* __restrict__ sinks, int keep_first, float cap_log2) {
    constexpr int D = DK * 32;
    static_assert(PRE_RT <= PRE_RT_OF(DK), "the accumulators of two row tiles fit the registers up to heads of 128");
    constexpr int PRE_ROWS = PRE_WAVES * 16 * PRE_RT;
    constexpr bool DMA = DK == 4 && (PRE_WAVES == 4 || PRE_WAVES == 8);  // tiles straight into LDS (measured 4-5 % faster)
    static_assert(PRE_WAVES == 4 || (DK == 4 && PRE_RT == 1), "eight wavefronts: heads of 128, one row tile each");
    constexpr int TILE = 2 * KSTEP * D;  // elements of a tile: K [32 keys][D], then V^T [D][32 keys]
    __shared__ __attribute__((aligned(16))) bf16_t lds[(DMA ? 3 : 2) * TILE];

    // the kv head varies fastest: workgroups go to the eight dies in turn, each die has an L2 of
    // its own, and this way a die sees the K/V of few heads, which the row blocks of a head share
    const int s = blockIdx.z, kvh = blockIdx.x;
    const int G = nq / nkv;
    const int q_start = cu_tokens[s];
    const int q_len = cu_tokens[s + 1] - q_start;
    const int nrows = q_len * G;
    if (nrows <= 16) return;  // the decode kernel's
    // The last rows see the most keys: they are started first.  When the whole launch is
    // resident at once (two workgroups a CU) the order is: the heavy half of the row blocks,
    // heaviest first, then the light half, lightest first, so that the two workgroups that
    // come to share a CU (launch positions j and j + half) add up to about the same work.
    const int row_blocks = gridDim.y / nsplit;
    const int split = blockIdx.y / row_blocks;
    const int yb = blockIdx.y % row_blocks, heavy_blocks = (row_blocks + 1) / 2;
    const int block_row0 =
        (complement_order && yb >= heavy_blocks ? yb - heavy_blocks : row_blocks - 1 - yb) * PRE_ROWS;
    if (block_row0 >= nrows) return;
    const int wave = threadIdx.x / LLE_WAVE, lane = threadIdx.x % LLE_WAVE;
    const int c = lane / 16, r16 = lane % 16;
    const int kv_len = kv_lens[s];
    const int past = kv_len - q_len;
    const int32_t* table = block_tables + (int64_t)seq_slots[s] * max_pages;

    // the workgroup's key range, and this wavefront's own
    const int block_last_row = min(nrows, block_row0 + PRE_ROWS) - 1;
    int hi = past + block_last_row / G;
    const int block_first_pos = past + block_row0 / G;
    int lo_min = window > 0 ? max(0, block_first_pos - window + 1) : 0;
    int first_step = lo_min / KSTEP, end_step = hi / KSTEP + 1;
    if (nsplit > 1) {  // this workgroup's share of the steps (it may be empty)
        const int per_split = (end_step - first_step + nsplit - 1) / nsplit;
        first_step = first_step + split * per_split;
        end_step = min(end_step, first_step + per_split);
    }

    const int row0 = block_row0 + wave * (16 * PRE_RT);
    RowInfo row[PRE_RT];
#pragma unroll
    for (int t = 0; t < PRE_RT; ++t) row[t] = make_row(q, row0 + 16 * t + r16, nrows, G, q_start, past, nq, kvh, D, window);
    int my_first = end_step, my_end = first_step;  // a wavefront without rows multiplies nothing
    if (row0 < nrows) {
        const int my_last_row = min(nrows, row0 + 16 * PRE_RT) - 1;
        const int my_lo = window > 0 ? max(0, past + row0 / G - window + 1) : 0;
        my_first = my_lo / KSTEP;
        my_end = min(end_step, (past + my_last_row / G) / KSTEP + 1);
    }
    // (the same in every lane of a wavefront: in scalar registers the tests on them are scalar branches)
    my_first = __builtin_amdgcn_readfirstlane(my_first);
    my_end = __builtin_amdgcn_readfirstlane(my_end);
    RowState<DK, PRE_RT> st;
    init_rows<DK, PRE_RT>(st, row);
    // what this lane reads from a tile in LDS: its two keys of a step and their swizzles
    const int kx[2] = {KEY_OF_ROW(r16, 0), KEY_OF_ROW(r16, 1)};
    const int ksw[2] = {K_SWIZZLE(kx[0], DK), K_SWIZZLE(kx[1], DK)};
    const int vsw = V_SWIZZLE(r16);

    const int64_t k_head = (int64_t)kvh * P * D;
    const int64_t v_head = ((int64_t)nkv + kvh) * P * D;
    // a tile holds 4 D 16-byte pieces of K and as many of V^T; this thread copies NP of each
    constexpr int PIECES = 4 * D;
    constexpr int NP = (PIECES + PRE_WAVES * LLE_WAVE - 1) / (PRE_WAVES * LLE_WAVE);
    // then the copies stand under no condition (see one_step on what a condition costs)
    constexpr bool EVERY_THREAD_COPIES = PIECES % (PRE_WAVES * LLE_WAVE) == 0;
    // two tiles are on their way from memory at any time (register sets 0 and 1); a tile is
    // written to LDS one step after its loads were issued and multiplied one step later still
    bf16x8 stage_k[2][NP], stage_v[2][NP];
    // The pages of the two 16-key halves of a step are looked up one fetch ahead, so that the
    // table's latency is not in the way of the loads that need it.  Fetches come in step order:
    // page and offset of the next half are carried along instead of divided out (the page size
    // is no constant).  A half wholly outside [lo_min, hi] may lie in a page that is not there:
    // the page index is clamped to those of keys that are.
    int page_lo = lo_min / P, page_hi = hi / P;
    int look_page = __builtin_amdgcn_readfirstlane((first_step * KSTEP) / P);
    int look_off = __builtin_amdgcn_readfirstlane((first_step * KSTEP) % P);
    int page_id[2], page_off[2];
    auto lookup = [&]() {
#pragma unroll
        for (int x = 0; x < 2; ++x) {
            page_id[x] = table[__builtin_amdgcn_readfirstlane(min(max(look_page, page_lo), page_hi))];
            page_off[x] = look_off;
            look_off += 16;  // pages hold a multiple of 16 keys
            if (look_off == P) {
                look_off = 0;
                ++look_page;
            }
        }
    };
    if constexpr (!KEEP) lookup();
    // Piece `piece` of a tile: the wavefront-sized run it lies in belongs to ONE 16-key half
    // (half = run / DK), so the half's page is the same for the whole wavefront and its address
    // stays in scalar registers; what differs between the threads is fixed for the kernel.
    //   K: the half's keys row by row, 16 bytes of a row per piece;
    //   V^T: the half's value elements one by one, each 16 keys = two pieces.
    int k_thread[NP], v_thread[NP];  // element offsets from the half's first key, in the page
    int k_lds[NP], v_lds[NP];        // element offsets in a tile in LDS
#pragma unroll
    for (int i = 0; i < NP; ++i) {
        const int q = (threadIdx.x + PRE_WAVES * LLE_WAVE * i) % (2 * D);  // piece within its half
        const int half = (threadIdx.x + PRE_WAVES * LLE_WAVE * i) / (2 * D);
        k_thread[i] = (q / (D / 8)) * D + (q % (D / 8)) * 8;
        v_thread[i] = (q / 2) * P + (q % 2) * 8;
        const int key = 16 * half + q / (D / 8);
        k_lds[i] = key * D + (((q % (D / 8)) ^ K_SWIZZLE(key, DK)) * 8);
        v_lds[i] = KSTEP * D + (q / 2) * KSTEP + (((2 * half + q % 2) ^ V_SWIZZLE(q / 2)) * 8);
    }
    auto fetch = [&](auto set_c) {
        constexpr int set = decltype(set_c)::value;
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            const int piece = threadIdx.x + PRE_WAVES * LLE_WAVE * i;
            if (EVERY_THREAD_COPIES || piece < PIECES) {
                const int half = __builtin_amdgcn_readfirstlane(piece / (2 * D));
                const bf16_t* page = kv_layer + (int64_t)(half ? page_id[1] : page_id[0]) * page_stride;
                const int off = half ? page_off[1] : page_off[0];
                stage_k[set][i] = *(const bf16x8*)(page + k_head + (int64_t)off * D + k_thread[i]);
                stage_v[set][i] = *(const bf16x8*)(page + v_head + off + v_thread[i]);
            }
        }
        lookup();
    };
    auto stash = [&](int buf, auto set_c) {
        constexpr int set = decltype(set_c)::value;
        bf16_t* tile = lds + buf * TILE;
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            const int piece = threadIdx.x + PRE_WAVES * LLE_WAVE * i;
            if (EVERY_THREAD_COPIES || piece < PIECES) {
                *(bf16x8*)(tile + k_lds[i]) = stage_k[set][i];
                *(bf16x8*)(tile + v_lds[i]) = stage_v[set][i];
            }
        }
    };
    // one step: tile `step` is in LDS buffer `buf`; tile step + 1 sits in register set `set`
    // (loads issued a step ago) and goes to the other buffer; tile step + 2 is requested now
    // into the other register set
    // Fetch and stash run in every step, also past the last tile (the lookup clamps to a page
    // that is there; what is stashed then is never read): a load under a condition makes the
    // compiler wait, where the paths meet again, for the loads that were issued last.
    auto one_step = [&](int step, int buf, auto set_c) {
        constexpr int set = decltype(set_c)::value;
        fetch(std::integral_constant<int, 1 - set>{});  // tile step + 2
        if (step >= my_first && step < my_end) {
            const bf16_t* kt = lds + buf * TILE;
            const bf16_t* vt = kt + KSTEP * D;
            tile_step<DK, PRE_RT, CAP>(
                st, row,
                [&](int x, int ks) { return *(const bf16x8*)(kt + kx[x] * D + (((4 * ks + c) ^ ksw[x]) * 8)); },
                [&](int n) { return *(const bf16x8*)(vt + (16 * n + r16) * KSTEP + ((c ^ vsw) * 8)); },
                step * KSTEP, lo_min, hi, scale_log2, cap_log2);
        }
        stash(buf ^ 1, set_c);
        __syncthreads();
    };

    // With kept first keys the walk has two ranges: those keys (the first split's work), then the window's.
    // What the loops above and below know of a range is set anew for each; the rows' sums run on.
    [[maybe_unused]] const int w_hi = hi, w_lo_min = lo_min, w_first = first_step, w_end = end_step, w_my_first = my_first,
                               w_my_end = my_end;
    auto set_range = [&](int range) {
        const int kept = min(keep_first, max(0, w_hi - window + 1));  // of the row that sees the most of them
#pragma unroll
        for (int t = 0; t < PRE_RT; ++t) {
            row[t] = make_row(q, row0 + 16 * t + r16, nrows, G, q_start, past, nq, kvh, D, window);
            if (range == 0) {
                if (row[t].q) row[t].pos = min(keep_first, row[t].lo) - 1;
                row[t].lo = 0;
            }
        }
        hi = range == 0 ? max(0, kept - 1) : w_hi;
        lo_min = range == 0 ? 0 : w_lo_min;
        first_step = range == 0 ? 0 : w_first;
        end_step = range == 0 ? (split == 0 ? (kept + KSTEP - 1) / KSTEP : 0) : w_end;
        my_first = __builtin_amdgcn_readfirstlane(range == 0 ? 0 : w_my_first);
        my_end = __builtin_amdgcn_readfirstlane(range == 0 ? (row0 < nrows ? end_step : 0) : w_my_end);
        page_lo = lo_min / P;
        page_hi = hi / P;
        look_page = __builtin_amdgcn_readfirstlane((first_step * KSTEP) / P);
        look_off = __builtin_amdgcn_readfirstlane((first_step * KSTEP) % P);
        set_open_range<DK, PRE_RT>(st, row);
        lookup();
    };

    for (int range = KEEP ? 0 : 1; range < 2; ++range) {
    if constexpr (KEEP) {
        set_range(range);
        if (first_step >= end_step) continue;  // (the same for the whole workgroup: nothing of this range is its work)
    }
    if constexpr (DMA) {
        // Tiles go from the pages straight into LDS (no registers, no stores by the wavefronts):
        // a wavefront's load writes 1 KB of LDS in lane order (M0 holds where), so the swizzle is
        // in which piece each lane fetches: the logical piece that belongs at its place (physical
        // piece ^ swizzle).  The loads are written in assembly so that the waits are ours: the
        // compiler, seeing such a load, waits for ALL outstanding loads before every barrier.
        // vmcnt counts them in issue order, so "at most the 4 newest outstanding" means that
        // every tile requested before the last one has landed, whatever else was issued.
        // Three buffers: tile N is multiplied, N + 1 has landed or lands, N + 2 is requested.
        const unsigned lds_base = (unsigned)(size_t)(__attribute__((address_space(3))) void*)lds;
        const int tid = threadIdx.x;
        // A load's address is a base that is the same for the whole wavefront (scalar registers:
        // the page of one 16-key half) plus a byte offset per lane that never changes:
        //   K:   half i of the step, key q / 16 of it, physical piece q % 16        (q = thread + 256 i)
        //   V^T: half i of the step, element thread / 2, keys 8 (thread % 2) .. + 7 of the half
        // so V^T lies in LDS as [half][D][16 keys]: rows of 32 bytes, which the sixteen lanes that
        // a 16-byte read serves in a cycle (c0 and c0 + 1 of one half, eight different elements
        // mod 8 each) spread over the sixteen columns of the banks without a swizzle.
        constexpr int LOADS = 512 / (PRE_WAVES * LLE_WAVE);  // of K and of V^T, per thread and tile
        unsigned kd_lane[LOADS], vd_lane[LOADS];
#pragma unroll
        for (int i = 0; i < LOADS; ++i) {
            const int q = tid + PRE_WAVES * LLE_WAVE * i;  // the half is q / 256: the same for a wavefront's load
            const int key = q / 16, pk = q % 16;
            kd_lane[i] = 2u * (unsigned)((key % 16) * D + ((pk ^ K_SWIZZLE(key, DK)) * 8));
            vd_lane[i] = 2u * (unsigned)(((q % 256) / 2) * P + (q % 2) * 8);
        }
        // With one load of K and one of V^T per wavefront and tile a wavefront needs the page of
        // its own half only, and follows that alone: half the scalar arithmetic a step.
        int own_page = 0, own_off = 0, own_id = 0;
        const int own_adv_pages = KSTEP / P, own_adv_off = KSTEP % P;
        auto own_lookup = [&]() { own_id = table[__builtin_amdgcn_readfirstlane(min(max(own_page, page_lo), page_hi))]; };
        if constexpr (LOADS == 1) {
            const int key0 = first_step * KSTEP + 16 * (wave / 4);
            own_page = __builtin_amdgcn_readfirstlane(key0 / P);
            own_off = __builtin_amdgcn_readfirstlane(key0 % P);
            own_lookup();
        }
        auto dma = [&](int buf) {
#pragma unroll
            for (int i = 0; i < LOADS; ++i) {
                const int first_piece = __builtin_amdgcn_readfirstlane(wave * LLE_WAVE + PRE_WAVES * LLE_WAVE * i);
                const int half = first_piece / 256;
                // (a page's offset as an unsigned 32 x 32 -> 64 bit product: two scalar instructions)
                const int id = LOADS == 1 ? own_id : (half ? page_id[1] : page_id[0]);
                const bf16_t* page = kv_layer + (uint64_t)(uint32_t)id * (uint64_t)(uint32_t)page_stride;
                const int off = LOADS == 1 ? own_off : (half ? page_off[1] : page_off[0]);
                const bf16_t* kb = page + k_head + (int64_t)off * D;
                const bf16_t* vb = page + v_head + off;
                const unsigned kdst = lds_base + 2 * (buf * TILE + first_piece * 8);
                const unsigned vdst = kdst + 2 * KSTEP * D;
                load_into_lds(kdst, kd_lane[i], kb);
                load_into_lds(vdst, vd_lane[i], vb);
            }
            if constexpr (LOADS == 1) {
                own_page += own_adv_pages;
                own_off += own_adv_off;
                if (own_off >= P) {
                    own_off -= P;
                    ++own_page;
                }
                own_lookup();
            } else {
                lookup();
            }
        };
        const int v_read = (c / 2) * (D * 16) + r16 * 16 + (c % 2) * 8;  // this lane's place in V^T for n = 0
        auto dma_step = [&](int step, int buf, int next_buf) {
            // the key operands are asked for first: the scalar arithmetic of the loads' addresses
            // then covers their way from LDS
            const bf16_t* kt = lds + buf * TILE;
            const bf16_t* vt = kt + KSTEP * D;
            bf16x8 kreg[2][DK];
#pragma unroll
            for (int x = 0; x < 2; ++x)
#pragma unroll
                for (int ks = 0; ks < DK; ++ks)
                    kreg[x][ks] = *(const bf16x8*)(kt + kx[x] * D + (((4 * ks + c) ^ ksw[x]) * 8));
            dma(next_buf);  // tile step + 2
            if (step >= my_first && step < my_end) {
                tile_step<DK, PRE_RT, CAP>(
                    st, row, [&](int x, int ks) { return kreg[x][ks]; },
                    [&](int n) { return *(const bf16x8*)(vt + v_read + n * 256); }, step * KSTEP, lo_min, hi,
                    scale_log2, cap_log2);
            }
            // the loads just issued may stay in flight; the tile before them has landed, and this one has been read (its
            // buffer is the next one to be filled)
            if constexpr (LOADS == 2)
                asm volatile("s_waitcnt vmcnt(4) lgkmcnt(0)" ::: "memory");
            else
                asm volatile("s_waitcnt vmcnt(2) lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_s_barrier();
        };
        dma(0);  // tile first_step
        dma(1);  // tile first_step + 1
        if constexpr (LOADS == 2)
            asm volatile("s_waitcnt vmcnt(4) lgkmcnt(0)" ::: "memory");
        else
            asm volatile("s_waitcnt vmcnt(2) lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        for (int step = first_step; step < end_step; step += 3) {
            dma_step(step, 0, 2);
            dma_step(step + 1, 1, 0);
            dma_step(step + 2, 2, 1);
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // nothing may land after the workgroup has gone
    } else {
        fetch(std::integral_constant<int, 0>{});  // tile first_step
        fetch(std::integral_constant<int, 1>{});  // tile first_step + 1
        stash(0, std::integral_constant<int, 0>{});
        __syncthreads();
        for (int step = first_step; step < end_step; step += 2) {
            one_step(step, 0, std::integral_constant<int, 1>{});
            one_step(step + 1, 1, std::integral_constant<int, 0>{});  // multiplies nothing past my_end
        }
    }
    }
    finish_rows<DK, PRE_RT>(st);
#pragma unroll
    for (int t = 0; t < PRE_RT; ++t) {
        const int r = row0 + 16 * t + r16;
        if (r >= nrows) continue;
        const int tk = r / G, g = r - tk * G;
        const int64_t head_row = (int64_t)(q_start + tk) * nq + kvh * G + g;
        if (nsplit > 1) {
            float* po = ws_o + (head_row * ws_stride + split) * D;
#pragma unroll
            for (int n = 0; n < 2 * DK; ++n) *(f32x4*)(po + 16 * n + 4 * c) = st.o[t][n];
            if (c == 0) {
                ws_ml[(head_row * ws_stride + split) * 2] = st.m[t];
                ws_ml[(head_row * ws_stride + split) * 2 + 1] = st.l[t];
            }
            continue;
        }
        bf16_t* dst = out + head_row * D;
        // (a sink: a place in the sum without a value)
        const float inv = 1.0f / (sinks ? st.l[t] + exp2f(sinks[kvh * G + g] * 1.44269504088896340736f - st.m[t]) : st.l[t]);
#pragma unroll
        for (int n = 0; n < 2 * DK; ++n) {
            bf16x4 v;
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] = (bf16_t)(st.o[t][n][i] * inv);
            *(bf16x4*)(dst + 16 * n + 4 * c) = v;
        }
    }
}

// ---------------------------------------------------------------------------------
// float32 on the matrix cores: v_mfma_f32_16x16x4_f32 multiplies and adds float32 (no
// reduced-precision mode), so this is still the true 32-bit path.  One kernel for every kind
// of request, head sizes in steps of 16 up to 256, pages that hold a multiple of 16 keys:
//   * a request with at most 16 rows (token, head of the group): one tile of rows, the four
//     wavefronts take every fourth 16-key step and are merged through LDS (decoding);
//   * any other: a workgroup takes 64 rows, each wavefront a tile of 16 of them and all keys
//     that its rows see; or (TILES == 2, heads of 64 and 128) 128 rows, two tiles a wavefront.
//     (Many rows of heads of 128: split_f32_attention_kernel.)
// What bounds it: the matrix instruction (32 cycles for 1024 products) where the loads keep up.
// Every wavefront loads K and V for itself, 16 KB a step of 16 keys of 128 elements, and one tile
// multiplies them in 2048 cycles; two tiles halve the bytes and leave two independent chains of
// scores.  The registers hold one step's K and one step's V, each asked for again as soon as its
// product is through, so that two (two tiles) or three workgroups fit a CU; two steps' worth of them,
// as it was, left one.  A 2048-token prompt of 32 / 8 heads of 128: 730 -> 372 us a layer (34 GFLOP:
// 92 of the 154 TFLOP/s a large float32 product reaches), one of 4096 tokens 2455 -> 1386, 32
// prompts of 64 tokens (16 / 8 heads) 31 -> 23; 64 requests decoding at 900 keys 102 -> 92.
// grid = (kv heads, row blocks x key splits, requests); with key splits the partial (m, l, acc)
// go to the workspaces and the combine kernel merges them.
// Operands (lane = (c, r), c = lane / 16, r = lane % 16): a lane loads 16 bytes, four
// consecutive elements, and its element e is the contraction slot c of instruction e:
//   S^T = K Q^T:    A = K[key r][16 q + 4 c + e],  B = Q[row r][16 q + 4 c + e]
//   O^T += V^T P^T: A = V^T[element 16 n + r][key 4 c + e],  B = P[key 4 c + e][row r]
// and the result tile S^T leaves lane (c, r) with keys 4 c .. 4 c + 3 of row r: exactly the B
// operand of the second product, so P never leaves its registers.
// ---------------------------------------------------------------------------------
#define F32_WAVES 4
#define F32_KEYS 16
// split, yb: which of the key splits, which of the request's row blocks.  given_end >= 0: the rows of a request with more than 16 take the 16-key
// steps given_begin .. given_end - 1 in the place of the split's; `skip`, of each lane: its row of tile t stays as it is in `out` and the
// workspaces.
template <int DQ, int TILES, bool KEEP, bool CAP>
__device__ __forceinline__ void f32_attention_rows(
    const float* __restrict__ q, const float* __restrict__ kv_layer, const int32_t* __restrict__ block_tables,
    const int32_t* __restrict__ seq_slots, const int32_t* __restrict__ cu_tokens,
    const int32_t* __restrict__ kv_lens, float* __restrict__ out, float* __restrict__ ws_o,
    float* __restrict__ ws_ml, int nsplit, int parts, int nq, int nkv, int P, int64_t page_stride, int max_pages, int window,
    int keep_first, float scale_log2, const float* __restrict__ sinks, float cap_log2, int paired, float* smem, int split, int yb, int given_begin,
    int given_end, uint32_t skip) {
    static_assert(TILES == 1 || !KEEP, "kept first keys: one tile");
    constexpr int D = 16 * DQ, ROWS = 16 * TILES;
    float* s_o = smem;  // [waves][16][D] acc, then [waves][16] m, [waves][16] l
    float* s_m = smem + F32_WAVES * 16 * D;
    float* s_l = s_m + F32_WAVES * 16;
    const int s = blockIdx.z, kvh = blockIdx.x;
    const int G = nq / nkv;
    const int q_start = cu_tokens[s];
    const int q_len = cu_tokens[s + 1] - q_start;
    const int nrows = q_len * G;
    if (nrows <= 0) return;
    const int kv_len = kv_lens[s];
    const int past = kv_len - q_len;
    const bool few = nrows <= 16;  // the same for the whole workgroup
    const int wave = threadIdx.x / LLE_WAVE, lane = threadIdx.x % LLE_WAVE;
    const int c = lane / 16, r16 = lane % 16;
    const int own = few ? 1 : (nrows + ROWS * F32_WAVES - 1) / (ROWS * F32_WAVES);  // the request's blocks
    if (yb >= own) return;
    // the last rows, which see the most keys, first; or (`paired`) the later half of the blocks from
    // the longest on, then the earlier half from the shortest on
    yb = paired && 2 * yb >= own ? yb - (own + 1) / 2 : own - 1 - yb;
    const int row0 = few ? 0 : yb * (ROWS * F32_WAVES) + wave * ROWS;
    const bool wave_has_rows = row0 < nrows;
    const int32_t* table = block_tables + (int64_t)seq_slots[s] * max_pages;

    // the lane's row of each tile
    bool exists[TILES];
    int pos[TILES], lo[TILES], g[TILES];
    int64_t head_row[TILES];
    f32x4 qf[TILES][DQ];
#pragma unroll
    for (int t = 0; t < TILES; ++t) {
        const int row = row0 + 16 * t + r16;
        exists[t] = row < nrows;
        const int tok = exists[t] ? row / G : 0;
        g[t] = exists[t] ? row - tok * G : 0;
        head_row[t] = (int64_t)(q_start + tok) * nq + kvh * G + g[t];
        pos[t] = exists[t] ? past + tok : -1;
        lo[t] = (exists[t] && window > 0) ? max(0, pos[t] - window + 1) : 0;
#pragma unroll
        for (int i = 0; i < DQ; ++i)
            qf[t][i] = exists[t] ? *(const f32x4*)(q + head_row[t] * D + 16 * i + 4 * c) : f32x4{0.f, 0.f, 0.f, 0.f};
    }

    // the keys that each tile's rows see, in steps of 16, and the wavefront's share of them
    int step_begin = 0, step_end = 0, step_stride = 1;
    int first[TILES], end[TILES];
    [[maybe_unused]] int kept = 0, kept_end = 0;  // the kept first keys and their steps, which are the first split's work
    int seen_lo = 0, seen_hi = -1;  // the keys that any of its rows sees
#pragma unroll
    for (int t = 0; t < TILES; ++t) {
        const int r0 = row0 + 16 * t;
        first[t] = end[t] = 0;
        if (r0 >= nrows) continue;
        const int hi = past + (min(nrows, r0 + 16) - 1) / G;
        const int lo_tile = window > 0 ? max(0, past + r0 / G - window + 1) : 0;
        first[t] = lo_tile / F32_KEYS;
        end[t] = hi / F32_KEYS + 1;
        step_end = end[t];  // (a later tile's rows see no less far)
        seen_hi = hi;
        if (t == 0) seen_lo = lo_tile;
        if (KEEP && split == 0) {
            kept = min(keep_first, max(0, hi - window + 1));
            kept_end = (kept + F32_KEYS - 1) / F32_KEYS;
        }
    }
    seen_lo = __builtin_amdgcn_readfirstlane(seen_lo);
    seen_hi = __builtin_amdgcn_readfirstlane(seen_hi);
    if (wave_has_rows) {
        const int per_split = (step_end - first[0] + nsplit - 1) / nsplit;
        step_begin = first[0] + split * per_split;
        step_end = min(step_end, step_begin + per_split);
        if (few) {
            step_begin += wave;
            step_stride = F32_WAVES;
        } else if (given_end >= 0) {
            step_begin = max(first[0], given_begin);
            step_end = min(TILES == 2 && end[TILES - 1] > 0 ? end[TILES - 1] : end[0], given_end);
        }
    }
    f32x4 o[TILES][DQ];
    float m[TILES], l[TILES];
#pragma unroll
    for (int t = 0; t < TILES; ++t) {
#pragma unroll
        for (int n = 0; n < DQ; ++n) o[t][n] = f32x4{0.f, 0.f, 0.f, 0.f};
        m[t] = NEG_BIG;
        l[t] = 0.f;
    }
    const int64_t k_lane = ((int64_t)kvh * P + r16) * D + 4 * c;
    const int64_t v_lane = ((int64_t)nkv + kvh) * P * D + (int64_t)r16 * P + 4 * c;
    f32x4 kf[DQ], vf[DQ];
    auto place = [&](int step) {
        const int j0 = step * F32_KEYS;
        const int lp = j0 / P;  // 16 keys of a step lie in one page
        return kv_layer + (int64_t)table[__builtin_amdgcn_readfirstlane(lp)] * page_stride;
    };
    auto load_k = [&](int step) {
        const float* at = place(step) + k_lane + (int64_t)(step * F32_KEYS % P) * D;
#pragma unroll
        for (int i = 0; i < DQ; ++i) kf[i] = *(const f32x4*)(at + 16 * i);
    };
    auto load_v = [&](int step) {
        const float* at = place(step) + v_lane + step * F32_KEYS % P;
#pragma unroll
        for (int n = 0; n < DQ; ++n) vf[n] = *(const f32x4*)(at + (int64_t)16 * n * P);
    };
    auto scores = [&](auto from, auto to, f32x4* sc) {
        constexpr int T0 = decltype(from)::value, T1 = decltype(to)::value;
#pragma unroll
        for (int t = T0; t < T1; ++t) sc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < DQ; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int t = T0; t < T1; ++t)
                    sc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[i][e], qf[t][i][e], sc[t], 0, 0, 0);
    };
    // scores of a step to probabilities: the row's maximum and sum, and the factor its sums get
    auto weigh = [&](int t, int step, const f32x4 sc, f32x4& p, float& alpha) {
        const int j0 = step * F32_KEYS;
        float x[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int j = j0 + 4 * c + e;
            const float score = CAP ? cap_log2 * tanhf(sc[e] * scale_log2) : sc[e] * scale_log2;  // (CAP: scale / cap)
            x[e] = (j < lo[t] || j > pos[t]) ? NEG_BIG : score;
        }
        float top = fmaxf(fmaxf(x[0], x[1]), fmaxf(x[2], x[3]));
        top = column_max(top);
        const float new_m = fmaxf(m[t], top);
        // while the row has seen no key new_m is NEG_BIG as its masked scores are, and
        // exp2(0) = 1 would count them: shift such rows so that they give 0
        const float base = new_m <= NEG_BIG ? 0.f : new_m;
        alpha = exp2f(m[t] - base);
        m[t] = new_m;
        float psum = 0.f;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            p[e] = exp2f(x[e] - base);
            psum += p[e];
        }
        l[t] = l[t] * alpha + psum;
    };
    auto values = [&](auto from, auto to, int step, const f32x4* p, const float* alpha) {
        constexpr int T0 = decltype(from)::value, T1 = decltype(to)::value;
        if (step * F32_KEYS < seen_lo || step * F32_KEYS + F32_KEYS - 1 > seen_hi) {  // as drop_values
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int j = step * F32_KEYS + 4 * c + e;
                const bool out_of = j < seen_lo || j > seen_hi;
#pragma unroll
                for (int n = 0; n < DQ; ++n) vf[n][e] = out_of ? 0.f : vf[n][e];
            }
        }
#pragma unroll
        for (int n = 0; n < DQ; ++n) {
#pragma unroll
            for (int t = T0; t < T1; ++t) o[t][n] *= alpha[t];
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int t = T0; t < T1; ++t)
                    o[t][n] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[n][e], p[t][e], o[t][n], 0, 0, 0);
        }
    };
    using None = std::integral_constant<int, 0>;
    using One = std::integral_constant<int, 1>;
    using All = std::integral_constant<int, TILES>;
    [[maybe_unused]] const int w_pos = pos[0], w_lo = lo[0], w_begin = step_begin, w_end = step_end, w_seen_lo = seen_lo, w_seen_hi = seen_hi;
    for (int range = KEEP && kept_end > 0 ? 0 : 1; range < 2; ++range) {
    if constexpr (KEEP) {
        pos[0] = range == 0 ? (exists[0] ? min(keep_first, w_lo) - 1 : -1) : w_pos;
        lo[0] = range == 0 ? 0 : w_lo;
        step_begin = range == 0 ? (few ? wave : 0) : w_begin;
        step_end = range == 0 ? kept_end : w_end;
        seen_lo = range == 0 ? 0 : w_seen_lo;
        seen_hi = __builtin_amdgcn_readfirstlane(range == 0 ? kept - 1 : w_seen_hi);
    }
    if (step_begin >= step_end) continue;
    // K of the next step is asked for before the values of this one are multiplied, V of it before
    // its scores are: the loads fly under the other product and take no registers of their own
    load_k(step_begin);
    load_v(step_begin);
    for (int step = step_begin; step < step_end; step += step_stride) {
        const int next = step + step_stride;
        f32x4 sc[TILES], p[TILES];
        float alpha[TILES];
        // a tile takes part in the steps that its own rows see and in no other: the sums are those
        // of tiles that work alone
        const bool first_in = TILES == 1 || step < end[0];
        const bool second_in = TILES == 2 && step >= first[TILES - 1] && step < end[TILES - 1];
        if (TILES == 1 || (first_in && second_in)) {
            scores(None{}, All{}, sc);
            if (next < step_end) load_k(next);
#pragma unroll
            for (int t = 0; t < TILES; ++t) weigh(t, step, sc[t], p[t], alpha[t]);
            values(None{}, All{}, step, p, alpha);
        } else {
            if (first_in) scores(None{}, One{}, sc);
            else if (second_in) scores(One{}, All{}, sc);
            if (next < step_end) load_k(next);
            if (first_in) {
                weigh(0, step, sc[0], p[0], alpha[0]);
                values(None{}, One{}, step, p, alpha);
            } else if (second_in) {
                weigh(TILES - 1, step, sc[TILES - 1], p[TILES - 1], alpha[TILES - 1]);
                values(One{}, All{}, step, p, alpha);
            }
        }
        if (next < step_end) load_v(next);
    }
    }
#pragma unroll
    for (int t = 0; t < TILES; ++t) {
        l[t] = column_sum(l[t]);
    }

    if (!few) {  // every wavefront writes the rows of its own tiles
#pragma unroll
        for (int t = 0; t < TILES; ++t) {
            if (!exists[t] || (skip >> t & 1)) continue;
            if (parts > 1) {
                float* po = ws_o + (head_row[t] * nsplit + split) * D;
#pragma unroll
                for (int n = 0; n < DQ; ++n) *(f32x4*)(po + 16 * n + 4 * c) = o[t][n];
                if (c == 0) {
                    ws_ml[(head_row[t] * nsplit + split) * 2] = m[t];
                    ws_ml[(head_row[t] * nsplit + split) * 2 + 1] = l[t];
                }
                continue;
            }
            // (a sink: a place in the sum without a value)
            const float sum = sinks ? l[t] + exp2f(sinks[kvh * G + g[t]] * 1.44269504088896340736f - m[t]) : l[t];
            const float inv = 1.0f / sum;
#pragma unroll
            for (int n = 0; n < DQ; ++n) *(f32x4*)(out + head_row[t] * D + 16 * n + 4 * c) = o[t][n] * inv;
        }
        return;
    }
    // few rows: the four wavefronts hold parts of the same rows
    if (exists[0]) {
#pragma unroll
        for (int n = 0; n < DQ; ++n) *(f32x4*)(s_o + (wave * 16 + r16) * D + 16 * n + 4 * c) = o[0][n];
    }
    if (c == 0) {
        s_m[wave * 16 + r16] = m[0];
        s_l[wave * 16 + r16] = l[0];
    }
    __syncthreads();
    for (int idx = threadIdx.x; idx < nrows * D; idx += blockDim.x) {
        const int r = idx / D, e = idx - r * D;
        float big = s_m[r];
#pragma unroll
        for (int w = 1; w < F32_WAVES; ++w) big = fmaxf(big, s_m[w * 16 + r]);
        float num = 0.f, den = 0.f;
#pragma unroll
        for (int w = 0; w < F32_WAVES; ++w) {
            const float f = exp2f(s_m[w * 16 + r] - big);  // a wavefront without keys has l = 0, acc = 0
            num += s_o[(w * 16 + r) * D + e] * f;
            den += s_l[w * 16 + r] * f;
        }
        const int t = r / G, gg = r - t * G;
        const int64_t hr = (int64_t)(q_start + t) * nq + kvh * G + gg;
        if (nsplit == 1) {
            if (sinks) den += exp2f(sinks[kvh * G + gg] * 1.44269504088896340736f - big);
            out[hr * D + e] = num / den;
        } else {
            ws_o[(hr * nsplit + split) * D + e] = num;
            if (e == 0) {
                ws_ml[(hr * nsplit + split) * 2] = big;
                ws_ml[(hr * nsplit + split) * 2 + 1] = den;
            }
        }
    }
}

template <int DQ, int TILES, bool KEEP, bool CAP>
__global__ __launch_bounds__(F32_WAVES* LLE_WAVE, DQ > 12 ? 1 : DQ >= 8 || TILES == 2 ? 2 : 3) void mfma_f32_attention_kernel(
    const float* __restrict__ q, const float* __restrict__ kv_layer, const int32_t* __restrict__ block_tables,
    const int32_t* __restrict__ seq_slots, const int32_t* __restrict__ cu_tokens,
    const int32_t* __restrict__ kv_lens, float* __restrict__ out, float* __restrict__ ws_o,
    float* __restrict__ ws_ml, int nsplit, int nq, int nkv, int P, int64_t page_stride, int max_pages, int window,
    int keep_first, float scale_log2, const float* __restrict__ sinks, float cap_log2, int paired) {
    extern __shared__ float smem[];
    const int row_blocks = gridDim.y / nsplit;
    f32_attention_rows<DQ, TILES, KEEP, CAP>(q, kv_layer, block_tables, seq_slots, cu_tokens, kv_lens, out, ws_o, ws_ml, nsplit, nsplit, nq, nkv, P, page_stride, max_pages, window,
                                             keep_first, scale_log2, sinks, cap_log2, paired, smem, blockIdx.y / row_blocks, blockIdx.y % row_blocks, 0, -1, 0);
}

// ---------------------------------------------------------------------------------
// float32 attention of many rows on the bfloat16 matrix cores: q, K, V and the probabilities as three bfloat16 parts each, which hold all bits of what
// is not too small (parts.h), both products in six of the nine of the bfloat16 instruction (gemm_f32.hip says what that keeps), scores, maxima and sums in
// float32.  The float32 instruction bounds mfma_f32_attention_kernel (8192 cycles for 32 rows and 32 keys of 128 elements, 3072 here).
// A workgroup takes 128 rows of a request, a wavefront 32, whose first two parts of q stay in its registers and the third in its own piece of LDS.
// 32 keys a step: K and V^T are loaded once a workgroup, split once and laid out in LDS as three planes each in the layouts of
// mfma_prefill_kernel; K of the next step is on its way while this one's scores are made, V of it under the product with the values.  80 KB
// and 256 registers a lane: two workgroups a CU.  Requests of at most 16 rows are f32_attention_rows', and rows that come out not finite (an infinity
// has no parts) or whose parts may have run out of exponent (the last one ends at 2^-133): elements of q below SA_SMALL, or above SA_LARGE, where keys
// below SA_SMALL matter, and results below SA_SMALL, whose values are as small.  (Left: probabilities below SA_SMALL, which only values 2^80 times the rest
// bring back.)  V of 1e-36: error 2.7e-5 without, 4.1e-7 so.
// What bounds it: matrix cores busy 0.53 of the time and the other vector instructions, half of them splitting, most of the rest (4096 tokens; they
// hardly run beside each other, whatever the priorities: matrix instructions first made it 720 us); below two workgroups a CU a wavefront's
// own chain, 3.7 us a step.  32 / 8 heads of 128, the other kernel -> this one: a prompt of 512 / 1024 / 2048 / 4096 tokens 55 -> 40, 116 -> 78,
// 385 -> 246, 1375 -> 700 us; 300 tokens behind 4000 231 -> 131, 1000 behind 5000 914 -> 477, 512 behind 2048 beside 20 decoded tokens
// 468 -> 183.  Error against 64 bits (1024 tokens) 3.9e-7 -> 2.7e-7: fewer roundings of a sum.
// Tried: two sums in turn in place of four (2048 tokens + 15 us), all of q in registers (nothing can be asked of LDS ahead; + 4 %), whole
// blocks that fill the chip in parts (2048 tokens 252 to 265).
// ---------------------------------------------------------------------------------
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
#define SA_KEYS 32
#define SA_PLANE 8192  // bytes of a part of a step's K or V
#define SA_LDS (10 * SA_PLANE)  // three of each, and the third parts of q
#define SA_SMALL 0x1p-105f
#define SA_LARGE 0x1p100f
__global__ __launch_bounds__(F32_WAVES* LLE_WAVE, 2) void split_f32_attention_kernel(
    const float* __restrict__ q, const float* __restrict__ kv_layer, const int32_t* __restrict__ block_tables,
    const int32_t* __restrict__ seq_slots, const int32_t* __restrict__ cu_tokens,
    const int32_t* __restrict__ kv_lens, float* __restrict__ out, float* __restrict__ ws_o,
    float* __restrict__ ws_ml, int nsplit, int nq, int nkv, int P, int64_t page_stride, int max_pages, int window,
    float scale_log2, const float* __restrict__ sinks, int part_steps) {
    constexpr int D = 128, KS = D / 32, N = D / 16, TILES = 2, ROWS = 32 * F32_WAVES;
    extern __shared__ __attribute__((aligned(16))) float smem[];
    unsigned char* lds = (unsigned char*)smem;
    const int s = blockIdx.z, kvh = blockIdx.x, G = nq / nkv;
    const int q_start = cu_tokens[s], q_len = cu_tokens[s + 1] - q_start, nrows = q_len * G;
    if (nrows <= 0) return;
    const bool few = nrows <= 16;
    int split = blockIdx.y, place = blockIdx.y, parts = nsplit;  // (of few rows: a part each)
    if (few && split >= nsplit) return;
    int given_begin = 0, given_end = -1;
    uint32_t skip = 0;
    if (!few) {
        const int own = (nrows + ROWS - 1) / ROWS;
        const int past = kv_lens[s] - q_len;
        const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / LLE_WAVE), lane = threadIdx.x % LLE_WAVE, c = lane / 16, r16 = lane % 16;
        // the keys that a block of rows sees: place 0 is the last block, whose rows see the most
        auto keys_of = [&](int at_place, int& lo, int& hi) {
            const int r0 = (own - 1 - at_place) * ROWS;
            hi = past + (min(nrows, r0 + ROWS) - 1) / G, lo = window > 0 ? max(0, past + r0 / G - window + 1) : 0;
            return hi / SA_KEYS + 1 - lo / SA_KEYS;  // steps
        };
        int hi, lo;
        if (nsplit == 1) {
            if (place >= own) return;
            parts = 1;
            split = 0;
        } else {
            // Which block's part this workgroup is: of the blocks with as many parts as there can be the one with the longest, of those with a part less
            // the one with the longest, and so on, then the second of each kind (rows of one prompt: as many blocks of each), so that the parts
            // come by falling length, and a workgroup without work behind all others: the dies deal workgroups out to their engines in turn,
            // and with an idle one after every other half of the engines had nothing to do (4096 tokens of 32 / 8 heads 720 -> 1830 us).
            const int kind = (own + nsplit - 1) / nsplit;
            int before = 0, found = -1;
            for (int i0 = 0; i0 < kind * nsplit && found < 0; i0 += LLE_WAVE) {
                const int i = i0 + lane, p = i % nsplit * kind + i / nsplit;
                const bool there = i < kind * nsplit && p < own;
                const int n = there ? min(nsplit, (keys_of(p, lo, hi) + part_steps - 1) / part_steps) : 0;
                int sum = n;
#pragma unroll
                for (int d = 1; d < LLE_WAVE; d *= 2) {
                    const int up = __shfl_up(sum, d);
                    if (lane >= d) sum += up;
                }
                const uint64_t past_it = __ballot(before + sum > (int)blockIdx.y);
                if (past_it) {
                    const int at = __builtin_ctzll(past_it);
                    found = __builtin_amdgcn_readlane(p, at), parts = __builtin_amdgcn_readlane(n, at);
                    split = (int)blockIdx.y - before - (__builtin_amdgcn_readlane(sum, at) - parts);
                }
                before += __builtin_amdgcn_readlane(sum, LLE_WAVE - 1);
            }
            if (found < 0) return;
            place = found;
        }
        const int steps = keys_of(place, lo, hi);
        const int block0 = (own - 1 - place) * ROWS, row0 = block0 + 32 * wave;
        const int32_t* table = block_tables + (int64_t)seq_slots[s] * max_pages;
        // A block of few steps is in fewer parts than there can be: its first part says so of the others, and a part that is all writes the result.
        if (split == 0 && parts < nsplit) {
            for (int i = threadIdx.x; i < ROWS * nsplit; i += F32_WAVES * LLE_WAVE) {
                const int row = block0 + i / nsplit, k = i % nsplit;
                if (row >= nrows || (k < parts && parts > 1)) continue;
                float* ml = ws_ml + (((int64_t)(q_start + row / G) * nq + kvh * G + row % G) * nsplit + k) * 2;
                ml[0] = NEG_BIG;
                ml[1] = k < parts ? -1.f : 0.f;  // (below zero: the row is in `out`)
            }
        }
        const int first = lo / SA_KEYS;
        const int per_part = (steps + parts - 1) / parts, begin = first + split * per_part, end = min(first + steps, begin + per_part);
        given_begin = 2 * begin, given_end = max(0, 2 * end);
        // those that the wavefront's rows see, and those that all of them see
        const bool has_rows = row0 < nrows;
        const int w_hi = has_rows ? past + (min(nrows, row0 + 32) - 1) / G : -1, w_lo = window > 0 ? max(0, past + row0 / G - window + 1) : 0;
        const int all_hi = past + row0 / G, all_lo = window > 0 ? max(0, w_hi - window + 1) : 0;
        bool exists[TILES];
        int pos[TILES], low[TILES];
        int64_t head_row[TILES];
        u32x4 qp[TILES][KS][2];
        // (the bits of a size are in its order; 0 comes out as the largest)
        auto size_less_one = [](float x) { return __builtin_bit_cast(uint32_t, fabsf(x)) - 1u; };
        unsigned char* third = lds + 6 * SA_PLANE + (wave * LLE_WAVE + lane) * 16;  // each lane's own, [tile][32 elements of q]
#pragma unroll
        for (int t = 0; t < TILES; ++t) {
            const int row = row0 + 16 * t + r16;
            exists[t] = row < nrows;
            const int tok = exists[t] ? row / G : 0, g = exists[t] ? row - tok * G : 0;
            head_row[t] = (int64_t)(q_start + tok) * nq + kvh * G + g;
            pos[t] = exists[t] ? past + tok : -1;
            low[t] = exists[t] && window > 0 ? max(0, pos[t] - window + 1) : 0;
            uint32_t least = ~0u, most = 0;
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) {
                const float* at = q + head_row[t] * D + 32 * ks + 8 * c;
                const f32x4 a = *(const f32x4*)at, b = *(const f32x4*)(at + 4);
                u32x4 last;
#pragma unroll
                for (int h = 0; h < 4; ++h) {
                    uint32_t p1, p2, p3;
                    split2(h < 2 ? a[2 * h] : b[2 * h - 4], h < 2 ? a[2 * h + 1] : b[2 * h - 3], p1, p2, p3);
                    qp[t][ks][0][h] = p1, qp[t][ks][1][h] = p2, last[h] = p3;
                    least = min(least, min(size_less_one(a[h]), size_less_one(b[h]))), most = max(most, max(size_less_one(a[h]) + 1, size_less_one(b[h]) + 1));
                }
                *(u32x4*)(third + (t * KS + ks) * (F32_WAVES * LLE_WAVE * 16)) = last;
            }
            if (least < size_less_one(SA_SMALL) || most > size_less_one(SA_LARGE)) qp[t][0][0][0] = 0x7fc07fc0u;  // (NaN: the row comes out not finite)
        }
        // the copies: of K a thread takes pieces of eight elements of one key, of V^T pieces of eight keys of one element
        const PageSize pages(P);
        const int kr = threadIdx.x / 8, kp = threadIdx.x % 8, ve = threadIdx.x / 4, vp = threadIdx.x % 4;
        auto place_of = [&](int step, int half, int& off) {  // (of a half that no row sees, whose page may be gone: the other half's)
            int j = step * SA_KEYS + 16 * half;
            j = j > hi ? j - 16 : j + 15 < lo ? j + 16 : j;
            const int p = pages.of(j);
            off = j - p * P;
            return kv_layer + (int64_t)table[p] * page_stride;
        };
        f32x4 kreg[2][2], vreg[2][2];
        auto load_k = [&](int step) {
            int off;
            const float* at = place_of(step, wave / 2, off);
            at += ((int64_t)kvh * P + off + kr % 16) * D + 8 * kp;
#pragma unroll
            for (int i = 0; i < 2; ++i) kreg[i][0] = *(const f32x4*)(at + 64 * i), kreg[i][1] = *(const f32x4*)(at + 64 * i + 4);
        };
        auto load_v = [&](int step) {
            int off0, off1;
            const float *at0 = place_of(step, 0, off0), *at1 = place_of(step, 1, off1);
            const float* at = (vp < 2 ? at0 + off0 : at1 + off1) + (((int64_t)nkv + kvh) * D + ve) * P + 8 * (vp % 2);
#pragma unroll
            for (int i = 0; i < 2; ++i) vreg[i][0] = *(const f32x4*)(at + (int64_t)64 * i * P), vreg[i][1] = *(const f32x4*)(at + (int64_t)64 * i * P + 4);
        };
        auto put = [&](unsigned char* at, const f32x4 (&v)[2]) {
            u32x4 part[3];
#pragma unroll
            for (int h = 0; h < 4; ++h) {
                uint32_t p1, p2, p3;
                split2(v[h / 2][2 * (h % 2)], v[h / 2][2 * (h % 2) + 1], p1, p2, p3);
                part[0][h] = p1, part[1][h] = p2, part[2][h] = p3;
            }
#pragma unroll
            for (int p = 0; p < 3; ++p) *(u32x4*)(at + p * SA_PLANE) = part[p];
        };
        auto store_k = [&]() {
#pragma unroll
            for (int i = 0; i < 2; ++i) put(lds + kr * 256 + ((kp + 8 * i) ^ K_SWIZZLE(kr, 4)) * 16, kreg[i]);
        };
        auto store_v = [&](int step) {
            const int j0 = step * SA_KEYS + 8 * vp;
            if (step * SA_KEYS < lo || step * SA_KEYS + SA_KEYS - 1 > hi) {  // as drop_values
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int e = 0; e < 8; ++e) vreg[i][e / 4][e % 4] = j0 + e < lo || j0 + e > hi ? 0.f : vreg[i][e / 4][e % 4];
            }
#pragma unroll
            for (int i = 0; i < 2; ++i) put(lds + 3 * SA_PLANE + (ve + 64 * i) * 64 + (vp ^ V_SWIZZLE(ve)) * 16, vreg[i]);
        };
        auto meet = [&]() {  // what every wavefront has put into LDS is there, and what it has asked of it has come
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
        };
        f32x4 o[TILES][N];
        float m[TILES], l[TILES];
#pragma unroll
        for (int t = 0; t < TILES; ++t) {
#pragma unroll
            for (int n = 0; n < N; ++n) o[t][n] = f32x4{0.f, 0.f, 0.f, 0.f};
            m[t] = NEG_BIG;
            l[t] = 0.f;
        }
        constexpr int pa[6] = {2, 1, 0, 1, 0, 0}, pb[6] = {0, 1, 2, 0, 1, 0};  // the smallest products first
        const int key[2] = {KEY_OF_ROW(r16, 0), KEY_OF_ROW(r16, 1)};
        const int ksw[2] = {K_SWIZZLE(key[0], 4), K_SWIZZLE(key[1], 4)};
        const unsigned char* v_at = lds + 3 * SA_PLANE + r16 * 64 + (c ^ V_SWIZZLE(r16)) * 16;
        if (begin < end) {
            load_k(begin);
            load_v(begin);
            store_k();
        }
        for (int step = begin; step < end; ++step) {
            const bool active = step * SA_KEYS <= w_hi && step * SA_KEYS + SA_KEYS > w_lo;
            meet();  // K of this step is there, V of the one before has been read
            store_v(step);
            if (step + 1 < end) load_k(step + 1);
            u32x4 pp[TILES][3];
            float alpha[TILES];
            if (active) {
                f32x4 sc[TILES][2];
#pragma unroll
                for (int t = 0; t < TILES; ++t) sc[t][0] = sc[t][1] = f32x4{0.f, 0.f, 0.f, 0.f};
                bf16x8 a[2][2][3], q3[2][TILES];
                auto read_k = [&](int ks, auto set) {
                    constexpr int b = decltype(set)::value;
#pragma unroll
                    for (int x = 0; x < 2; ++x)
#pragma unroll
                        for (int p = 0; p < 3; ++p) a[b][x][p] = *(const bf16x8*)(lds + p * SA_PLANE + key[x] * 256 + ((4 * ks + c) ^ ksw[x]) * 16);
#pragma unroll
                    for (int t = 0; t < TILES; ++t) q3[b][t] = *(const bf16x8*)(third + (t * KS + ks) * (F32_WAVES * LLE_WAVE * 16));
                };
                auto score_k = [&](int ks, auto set) {
                    constexpr int b = decltype(set)::value;
#pragma unroll
                    for (int i = 0; i < 6; ++i)  // (four sums in turn: one after the other they wait for each other)
#pragma unroll
                        for (int x = 0; x < 2; ++x)
#pragma unroll
                            for (int t = 0; t < TILES; ++t)
                                sc[t][x] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[b][x][pa[i]], pb[i] == 2 ? q3[b][t] : __builtin_bit_cast(bf16x8, qp[t][ks][pb[i] == 2 ? 0 : pb[i]]), sc[t][x], 0, 0, 0);
                };
                using Set0 = std::integral_constant<int, 0>;
                using Set1 = std::integral_constant<int, 1>;
                read_k(0, Set0{});
                read_k(1, Set1{});
                score_k(0, Set0{});
                __builtin_amdgcn_sched_barrier(0);
                read_k(2, Set0{});
                score_k(1, Set1{});
                __builtin_amdgcn_sched_barrier(0);
                read_k(3, Set1{});
                score_k(2, Set0{});
                __builtin_amdgcn_sched_barrier(0);
                score_k(3, Set1{});
                const bool masked = step * SA_KEYS + SA_KEYS - 1 > all_hi || step * SA_KEYS < all_lo;  // (the same for the whole wavefront)
#pragma unroll
                for (int t = 0; t < TILES; ++t) {
                    float x[8];  // of keys 8 c + i
#pragma unroll
                    for (int i = 0; i < 8; ++i) x[i] = sc[t][i / 4][i % 4] * scale_log2;
                    if (masked) {
#pragma unroll
                        for (int i = 0; i < 8; ++i) {
                            const int j = step * SA_KEYS + 8 * c + i;
                            x[i] = j < low[t] || j > pos[t] ? NEG_BIG : x[i];
                        }
                    }
                    float top = x[0];
#pragma unroll
                    for (int i = 1; i < 8; ++i) top = fmaxf(top, x[i]);
                    const float new_m = fmaxf(m[t], column_max(top));
                    const float base = new_m <= NEG_BIG ? 0.f : new_m;  // (a row that has seen no key: as in f32_attention_rows)
                    alpha[t] = exp2f(m[t] - base);
                    m[t] = new_m;
                    float sum[2] = {0.f, 0.f};
#pragma unroll
                    for (int h = 0; h < 4; ++h) {
                        const float a = __builtin_amdgcn_exp2f(x[2 * h] - base), b = __builtin_amdgcn_exp2f(x[2 * h + 1] - base);
                        sum[0] += a, sum[1] += b;
                        uint32_t p1, p2, p3;
                        split2(a, b, p1, p2, p3);
                        pp[t][0][h] = p1, pp[t][1][h] = p2, pp[t][2][h] = p3;
                    }
                    l[t] = l[t] * alpha[t] + (sum[0] + sum[1]);
                }
            }
            meet();  // V of this step is there, K has been read
            if (step + 1 < end) {
                store_k();
                load_v(step + 1);
            }
            if (active) {
                if (!__all(alpha[0] == 1.f && alpha[1] == 1.f)) {
#pragma unroll
                    for (int t = 0; t < TILES; ++t)
#pragma unroll
                        for (int n = 0; n < N; ++n) o[t][n] *= alpha[t];
                }
                bf16x8 a[2][2][3];
                auto read_v = [&](int n, auto set) {
                    constexpr int b = decltype(set)::value;
#pragma unroll
                    for (int x = 0; x < 2; ++x)
#pragma unroll
                        for (int p = 0; p < 3; ++p) a[b][x][p] = *(const bf16x8*)(v_at + p * SA_PLANE + (n + x) * 1024);
                };
                auto add_v = [&](auto at, auto set) {
                    constexpr int n = decltype(at)::value, b = decltype(set)::value;
#pragma unroll
                    for (int i = 0; i < 6; ++i)
#pragma unroll
                        for (int x = 0; x < 2; ++x)
#pragma unroll
                            for (int t = 0; t < TILES; ++t)
                                o[t][n + x] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[b][x][pa[i]], __builtin_bit_cast(bf16x8, pp[t][pb[i]]), o[t][n + x], 0, 0, 0);
                };
                using Set0 = std::integral_constant<int, 0>;
                using Set1 = std::integral_constant<int, 1>;
                read_v(0, Set0{});
                read_v(2, Set1{});
                add_v(std::integral_constant<int, 0>{}, Set0{});
                __builtin_amdgcn_sched_barrier(0);
                read_v(4, Set0{});
                add_v(std::integral_constant<int, 2>{}, Set1{});
                __builtin_amdgcn_sched_barrier(0);
                read_v(6, Set1{});
                add_v(std::integral_constant<int, 4>{}, Set0{});
                __builtin_amdgcn_sched_barrier(0);
                add_v(std::integral_constant<int, 6>{}, Set1{});
            }
        }
        bool again = false;  // a row of the wavefront is not finite, or too small for parts
#pragma unroll
        for (int t = 0; t < TILES; ++t) {
            l[t] = column_sum(l[t]);
            float sizes = fabsf(l[t]);
            uint32_t least = ~0u;
#pragma unroll
            for (int n = 0; n < N; ++n)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    sizes = fmaxf(sizes, o[t][n][e] == o[t][n][e] ? fabsf(o[t][n][e]) : INFINITY);
                    least = min(least, size_less_one(o[t][n][e]));
                }
            const bool held = sizes < INFINITY && l[t] == l[t] && least >= size_less_one(l[t] * SA_SMALL);
            const uint64_t odd = __ballot(exists[t] && !held);  // (a row is four lanes)
            const bool row_odd = (odd >> r16 | odd >> (r16 + 16) | odd >> (r16 + 32) | odd >> (r16 + 48)) & 1;
            again = again || odd != 0;
            if (!exists[t] || row_odd) continue;
            skip |= 1u << t;
            if (parts > 1) {
                float* po = ws_o + (head_row[t] * nsplit + split) * D;
#pragma unroll
                for (int n = 0; n < N; ++n) *(f32x4*)(po + 16 * n + 4 * c) = o[t][n];
                if (c == 0) {
                    ws_ml[(head_row[t] * nsplit + split) * 2] = m[t];
                    ws_ml[(head_row[t] * nsplit + split) * 2 + 1] = l[t];
                }
                continue;
            }
            // (a sink: a place in the sum without a value)
            const float sum = sinks ? l[t] + exp2f(sinks[head_row[t] % nq] * 1.44269504088896340736f - m[t]) : l[t];
            const float inv = 1.0f / sum;
#pragma unroll
            for (int n = 0; n < N; ++n) *(f32x4*)(out + head_row[t] * D + 16 * n + 4 * c) = o[t][n] * inv;
        }
        if (!again) return;
    }
    f32_attention_rows<8, 2, false, false>(q, kv_layer, block_tables, seq_slots, cu_tokens, kv_lens, out, ws_o, ws_ml, nsplit, parts, nq, nkv, P, page_stride,
                                           max_pages, window, 0, scale_log2, sinks, 0.f, 0, smem, split, few ? 0 : place, given_begin, given_end, skip);
}

// A q or k head of a raw float32 projection in mfma_f32_attention_kernel's layout: lane (c, r) holds elements 16 i + 4 c .. + 3,
// element e and its partner of the rotation, D / 2 further on, in one lane.  load asks for everything, finish works on it.
template <int DQ, int WEIGHTS>
struct F32Head {
    f32x4 x[DQ], w[DQ];
    typedef f32x4 Table[DQ / 2][2];  // cos, sin of two elements each
    __device__ __forceinline__ void load(const float* src, const void* weight, int c) {
#pragma unroll
        for (int i = 0; i < DQ; ++i) x[i] = *(const f32x4*)(src + 16 * i + 4 * c);
        if (!weight) return;  // (the same for the whole launch)
#pragma unroll
        for (int i = 0; i < DQ; ++i) {
            if constexpr (WEIGHTS == LLE_F32) {
                w[i] = *(const f32x4*)((const float*)weight + 16 * i + 4 * c);
            } else {
                const bf16x4 b = *(const bf16x4*)((const bf16_t*)weight + 16 * i + 4 * c);
                w[i] = f32x4{(float)b[0], (float)b[1], (float)b[2], (float)b[3]};
            }
        }
    }
    static __device__ __forceinline__ void load_table(Table& tab, const float* cos_sin, int tok, int c) {
#pragma unroll
        for (int i = 0; i < DQ / 2; ++i) {
            const f32x4* t = (const f32x4*)(cos_sin + ((int64_t)tok * (8 * DQ) + 16 * i + 4 * c) * 2);
            tab[i][0] = t[0];
            tab[i][1] = t[1];
        }
    }
    __device__ __forceinline__ void norm(float eps) {
        f32x4 ss = x[0] * x[0];
#pragma unroll
        for (int i = 1; i < DQ; ++i) ss += x[i] * x[i];
        const float inv = 1.0f / sqrtf(column_sum((ss[0] + ss[1]) + (ss[2] + ss[3])) / (float)(16 * DQ) + eps);
#pragma unroll
        for (int i = 0; i < DQ; ++i) x[i] = x[i] * inv * w[i];
    }
    __device__ __forceinline__ void turn(const Table& tab) {
#pragma unroll
        for (int i = 0; i < DQ / 2; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float cs = tab[i][e / 2][e % 2 * 2], sn = tab[i][e / 2][e % 2 * 2 + 1], a = x[i][e], b = x[i + DQ / 2][e];
                x[i][e] = a * cs - b * sn;
                x[i + DQ / 2][e] = b * cs + a * sn;
            }
    }
};

// short_decode_kernel in float32: one new token a request, at most SHORT_F32_KEYS keys, a wavefront for every 16 of them (past 176:
// a second 16) and one for the new token; products on the float32 matrix instruction as in mfma_f32_attention_kernel (1024 cycles for the scores of
// 16 keys of 128, as many for the values: V flies under the scores).  Twelve wavefronts leave a lane the 168 registers that a
// head, its weights, its rotation and K need side by side.  0.6B sizes (16 q heads, 8 kv heads of 128) at 97 keys, 32 requests:
// 12.0 us in two launches (rotation and cache write, attention), 9.1 here; at 200 keys 19.2 and 15.7.  1 / 8 requests 9.0 / 10.0 and
// 7.0 / 7.7, at 256 keys 8 requests 11.4 and 12.5 (the two launches' key splits reach CUs that this one leaves idle).  Which of
// them takes a step is can_fuse_rope_attention's to say, from the bound on the keys that it is given: a step that runs as a graph
// has a bound of 256 at least, so there 1 to 11 requests of 8 kv heads are the two launches' whatever their length.  Tried and
// not kept: the second step's K asked for before the first's values.
#define SHORT_F32_WAVES 11
#define SHORT_F32_KEYS 256
static_assert(SHORT_F32_KEYS <= 2 * SHORT_F32_WAVES * F32_KEYS, "two steps a wavefront");
template <int DQ, int WEIGHTS>
__global__ __launch_bounds__((SHORT_F32_WAVES + 1) * LLE_WAVE) void short_decode_f32_kernel(
    const int32_t* __restrict__ cu_tokens, const int32_t* __restrict__ kv_lens, const int32_t* __restrict__ seq_slots,
    const int32_t* __restrict__ block_tables, int max_pages, int P, int window, int G, int nkv, float* kv_layer,
    float* __restrict__ out, int64_t page_stride, float scale_log2, FusedQKV f) {
    const int s = blockIdx.x, kvh = blockIdx.y;
    const int tok = cu_tokens[s], tok_end = cu_tokens[s + 1], kv_len = kv_lens[s], seq_slot = seq_slots[s];
    asm volatile("" ::"s"(tok), "s"(tok_end), "s"(kv_len), "s"(seq_slot), "s"(nkv), "s"(kv_layer), "s"(out), "s"(page_stride),
                 "s"(scale_log2), "s"(f.qkv), "s"(f.q_weight), "s"(f.k_weight), "s"(f.cos_sin), "s"(f.eps), "s"(f.write_kv));
    constexpr int D = DQ * 16, WAVES = SHORT_F32_WAVES + 1;
    extern __shared__ float smem[];  // [waves][G][D] acc, then [waves][16] m, [waves][16] l
    float* s_m = smem + WAVES * G * D;
    float* s_l = s_m + WAVES * 16;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / LLE_WAVE), lane = threadIdx.x % LLE_WAVE;
    const int c = lane / 16, r16 = lane % 16;
    if (tok_end - tok != 1) return;  // (a request without a token has nothing to do)
    const int last = kv_len - 1, lo = window > 0 ? max(0, kv_len - window) : 0;
    // the wavefront's steps of 16 keys: its own number and, past SHORT_F32_WAVES steps, the one that many further on
    int j0 = wave * F32_KEYS;
    constexpr int ROUND = SHORT_F32_WAVES * F32_KEYS;
    if (j0 + F32_KEYS <= lo) j0 += ROUND;
    const PageSize pages(P);
    const int32_t* table = block_tables + (int64_t)seq_slot * max_pages;
    int at = min(j0, max(last, 0)), lp = pages.of(at);  // (16 keys of a step lie in one page)
    int page = table[lp];
    const int slot = f.slots[tok];
    const bool fresh = f.write_kv && slot >= 0;  // (else the new token's place holds what the page does)
    const float* qkv = (const float*)f.qkv + (int64_t)tok * (nkv * (G + 2) * D);
    const float* q_head = qkv + (int64_t)(kvh * G + min(r16, G - 1)) * D;  // (rows past the group's: dropped at the end)
    f32x4 o[DQ];
#pragma unroll
    for (int n = 0; n < DQ; ++n) o[n] = f32x4{0.f, 0.f, 0.f, 0.f};
    float top = NEG_BIG, l = 0.f;
    if (wave < SHORT_F32_WAVES && j0 <= last && j0 + F32_KEYS > lo) {
        F32Head<DQ, WEIGHTS> q;
        typename F32Head<DQ, WEIGHTS>::Table tab;
        q.load(q_head, f.q_weight, c);
        q.load_table(tab, f.cos_sin, tok, c);
        f32x4 k[DQ], v[DQ];
        auto load_k = [&] {
            const float* kp = kv_layer + (int64_t)page * page_stride + ((int64_t)kvh * P + (at - lp * P) + r16) * D + 4 * c;
#pragma unroll
            for (int i = 0; i < DQ; ++i) k[i] = *(const f32x4*)(kp + 16 * i);
        };
        load_k();
        if (f.q_weight) q.norm(f.eps);
        q.turn(tab);
        const int pos = fresh ? last - 1 : last;  // the last key that comes from the pages
        for (;;) {
            const float* vp = kv_layer + (int64_t)page * page_stride + ((int64_t)(nkv + kvh) * D + r16) * P + (at - lp * P) + 4 * c;
#pragma unroll
            for (int n = 0; n < DQ; ++n) v[n] = *(const f32x4*)(vp + (int64_t)16 * n * P);
            f32x4 sc = {0.f, 0.f, 0.f, 0.f}, sc2 = sc;  // (two chains)
#pragma unroll
            for (int i = 0; i < DQ; ++i)
#pragma unroll
                for (int e = 0; e < 4; e += 2) {
                    sc = __builtin_amdgcn_mfma_f32_16x16x4f32(k[i][e], q.x[i][e], sc, 0, 0, 0);
                    sc2 = __builtin_amdgcn_mfma_f32_16x16x4f32(k[i][e + 1], q.x[i][e + 1], sc2, 0, 0, 0);
                }
            sc += sc2;
            f32x4 x = sc * scale_log2;
            if (j0 < lo || j0 + F32_KEYS - 1 > pos) {  // (the same for the whole wavefront) places without a key: whatever lies there
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int key = j0 + 4 * c + e;
                    const bool out_of = key < lo || key > pos;
                    if (out_of) x[e] = NEG_BIG;
#pragma unroll
                    for (int n = 0; n < DQ; ++n) v[n][e] = out_of ? 0.f : v[n][e];
                }
            }
            const float before = top;
            top = fmaxf(top, column_max(fmaxf(fmaxf(x[0], x[1]), fmaxf(x[2], x[3]))));
            const float base = top <= NEG_BIG ? 0.f : top;  // (no key is seen where the new token is the step's first one)
            f32x4 p;
#pragma unroll
            for (int e = 0; e < 4; ++e) p[e] = exp2f(x[e] - base);
            const float sum = (p[0] + p[1]) + (p[2] + p[3]);
            if (j0 >= ROUND && before > NEG_BIG) {  // a second step
                const float alpha = exp2f(before - base);
                l = fmaf(l, alpha, sum);
#pragma unroll
                for (int n = 0; n < DQ; ++n) o[n] *= alpha;
            } else {
                l = sum;
            }
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int n = 0; n < DQ; ++n) o[n] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[n][e], p[e], o[n], 0, 0, 0);
            j0 += ROUND;
            if (j0 > last) break;
            at = j0, lp = pages.of(at), page = table[lp];
            load_k();
        }
        l = column_sum(l);
    } else if (wave == SHORT_F32_WAVES && fresh) {
        const float* k_head = qkv + (int64_t)(nkv * G + kvh) * D;
        const float* v_head = k_head + (int64_t)nkv * D;
        F32Head<DQ, WEIGHTS> k, q;
        typename F32Head<DQ, WEIGHTS>::Table tab;
        k.load(k_head, f.k_weight, c);
        k.load_table(tab, f.cos_sin, tok, c);
        if (f.k_weight) k.norm(f.eps);
        q.load(q_head, f.q_weight, c);
        k.turn(tab);
        const int own = pages.of(slot), off = slot - own * P;
        float* base = kv_layer + (int64_t)own * page_stride;
        if (r16 == 0) {
            float* kdst = base + ((int64_t)kvh * P + off) * D + 4 * c;
#pragma unroll
            for (int i = 0; i < DQ; ++i) *(f32x4*)(kdst + 16 * i) = k.x[i];
        }
        if (f.q_weight) q.norm(f.eps);
        // (v only now, where the weights' registers are free)
#pragma unroll
        for (int n = 0; n < DQ; ++n) o[n] = *(const f32x4*)(v_head + 16 * n + 4 * c);
        q.turn(tab);
        f32x4 dot = k.x[0] * q.x[0];
#pragma unroll
        for (int i = 1; i < DQ; ++i) dot += k.x[i] * q.x[i];
        top = column_sum((dot[0] + dot[1]) + (dot[2] + dot[3])) * scale_log2;
        l = 1.f;
        if (r16 == 0) {
            float* vdst = base + ((int64_t)(nkv + kvh) * D + 4 * c) * P + off;
#pragma unroll
            for (int n = 0; n < DQ; ++n)
#pragma unroll
                for (int e = 0; e < 4; ++e) vdst[(int64_t)(16 * n + e) * P] = o[n][e];
        }
    }
    if (r16 < G) {
#pragma unroll
        for (int n = 0; n < DQ; ++n) *(f32x4*)(smem + (wave * G + r16) * D + 16 * n + 4 * c) = o[n];
    }
    if (c == 0) {
        s_m[wave * 16 + r16] = top;
        s_l[wave * 16 + r16] = l;
    }
    __syncthreads();
    for (int idx = threadIdx.x; idx < G * D; idx += WAVES * LLE_WAVE) {
        const int r = idx / D;
        float m[WAVES], big = NEG_BIG;
#pragma unroll
        for (int w = 0; w < WAVES; ++w) {
            m[w] = s_m[w * 16 + r];
            big = fmaxf(big, m[w]);
        }
        float num = 0.f, den = 0.f;
#pragma unroll
        for (int w = 0; w < WAVES; ++w) {
            const float e = exp2f(m[w] - big);
            num = fmaf(smem[w * G * D + idx], e, num);
            den = fmaf(s_l[w * 16 + r], e, den);
        }
        out[((int64_t)tok * (nkv * G) + kvh * G) * D + idx] = num / den;
    }
}

// merges the key splits of mfma_f32_attention_kernel: grid = (tokens, q heads), one wavefront each
__global__ __launch_bounds__(LLE_WAVE) void f32_combine_kernel(const float* __restrict__ ws_o,
                                                               const float* __restrict__ ws_ml, int nsplit,
                                                               float* __restrict__ out, int nq, int D,
                                                               const float* __restrict__ sinks) {
    const int64_t head_row = (int64_t)blockIdx.x * nq + blockIdx.y;
    const int lane = threadIdx.x;
    __shared__ float s_f[LLE_WAVE];
    const float2 ml = *(const float2*)(ws_ml + (head_row * nsplit + min(lane, nsplit - 1)) * 2);
    const float m = lane < nsplit ? ml.x : NEG_BIG, l = lane < nsplit ? ml.y : 0.f;
    const float big = wave_max(m);
    const float f = exp2f(m - big);
    float den = wave_sum(l * f);
    if (sinks) den += exp2f(sinks[blockIdx.y] * 1.44269504088896340736f - big);
    s_f[lane] = f;
    __syncthreads();
    const float* o = ws_o + head_row * nsplit * D;
    for (int e = lane; e < D; e += LLE_WAVE) {
        float num = 0.f;
        for (int k = 0; k < nsplit; ++k) num += o[(int64_t)k * D + e] * s_f[k];
        out[head_row * D + e] = num / den;
    }
}

// The same of split_f32_attention_kernel, whose rows may have fewer parts than nsplit, or be in `out` already: rows of 128, one a wavefront, two
// neighbouring elements a lane.
__global__ __launch_bounds__(256) void split_f32_combine_kernel(const float* __restrict__ ws_o, const float* __restrict__ ws_ml, int nsplit,
                                                                float* __restrict__ out, int64_t rows, int nq, const float* __restrict__ sinks) {
    const int64_t head_row = (int64_t)blockIdx.x * 4 + threadIdx.x / LLE_WAVE;
    const int lane = threadIdx.x % LLE_WAVE;
    if (head_row >= rows) return;
    const float2 ml = *(const float2*)(ws_ml + (head_row * nsplit + min(lane, nsplit - 1)) * 2);
    const float m = lane < nsplit ? ml.x : NEG_BIG, l = lane < nsplit ? ml.y : 0.f;
    const uint64_t some = __ballot(l != 0.f);  // (behind the last of them there may be nothing written)
    if (__ballot(l < 0.f) & 1) return;
    // (none: every score is -inf or as good as, and the row 0 / 0 as in f32_combine_kernel, or 0 beside a sink)
    const int held = some ? 64 - __builtin_clzll(some) : 0;
    const float big = wave_max(m);
    const float f = exp2f(m - big);
    float den = wave_sum(l * f);
    if (sinks) den += exp2f(sinks[head_row % nq] * 1.44269504088896340736f - big);
    const float* o = ws_o + head_row * nsplit * 128 + 2 * lane;
    float2 num = {0.f, 0.f};
    for (int k0 = 0; k0 < held; k0 += 4) {
        float2 part[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) part[j] = *(const float2*)(o + (int64_t)min(k0 + j, held - 1) * 128);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float fk = __shfl(f, k0 + j);
            if (k0 + j < held) num.x += part[j].x * fk, num.y += part[j].y * fk;
        }
    }
    *(float2*)(out + head_row * 128 + 2 * lane) = float2{num.x / den, num.y / den};
}

// float32, head_dim a multiple of 16 (<= 256), page size a multiple of 16.  `row_blocks`: the
// most 64-row blocks that a request of this batch has (1 when every request has at most 16
// rows); with nsplit > 1 the workspaces ws_o [N * nq * nsplit * d] and ws_ml [N * nq * nsplit * 2]
// floats are needed (nsplit <= 64).  tiles 3: split_f32_attention_kernel, heads of 128; `row_blocks` then the workgroups for the parts of a request's
// blocks, `paired` the most steps of 32 keys of a part, nsplit the most parts of a block.
extern "C" int lle_paged_attention_mfma_f32(const void* q, const void* kv_layer, const void* block_tables,
                                            const void* seq_slots, const void* cu_tokens, const void* kv_lens,
                                            void* out, void* ws_o, void* ws_ml, int N, int S, int nq, int nkv, int d,
                                            int page_size, int64_t page_stride, int max_pages, int window,
                                            int keep_first, float scale, int row_blocks, int tiles, int paired, int nsplit,
                                            const void* sinks, float softcap, hipStream_t stream) {
    if (N <= 0) return 0;
    if (tiles < 1 || tiles > 3 || (tiles > 1 && ((d != 64 && d != 128) || keep_first > 0 || softcap > 0.f)) || (tiles == 3 && (d != 128 || paired < 1)))
        return (int)hipErrorInvalidValue;
    if (d % 16 != 0 || d > 256 || d <= 0 || page_size % 16 != 0 || nq % nkv != 0) return (int)hipErrorInvalidValue;
    const int64_t grid_y = tiles == 3 ? row_blocks : (int64_t)row_blocks * nsplit;
    if (S > 65535 || nkv <= 0 || row_blocks < 1 || nsplit < 1 || nsplit > 64 || grid_y > 65535) return (int)hipErrorInvalidValue;
    if (nsplit > 1 && (!ws_o || !ws_ml)) return (int)hipErrorInvalidValue;
    if (keep_first < 0 || (keep_first > 0 && window <= 0)) return (int)hipErrorInvalidValue;
    if (softcap < 0.f || (softcap > 0.f && keep_first > 0)) return (int)hipErrorInvalidValue;
    // with a cap: the factor that tanh's argument gets, and the cap in the base-2 domain
    const float scale_log2 = softcap > 0.f ? scale / softcap : scale * 1.44269504088896340736f;
    const float cap_log2 = softcap * 1.44269504088896340736f;
    const dim3 grid(nkv, (int)grid_y, S);
    const size_t smem = tiles == 3 ? SA_LDS : (size_t)(F32_WAVES * 16 * d + 2 * F32_WAVES * 16) * sizeof(float);
    auto launch = [&](auto kernel) {
        if (smem > 64 * 1024) {
            const hipError_t e = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
            if (e != hipSuccess) return e;
        }
        kernel<<<grid, F32_WAVES * LLE_WAVE, smem, stream>>>(
            (const float*)q, (const float*)kv_layer, (const int32_t*)block_tables, (const int32_t*)seq_slots,
            (const int32_t*)cu_tokens, (const int32_t*)kv_lens, (float*)out, (float*)ws_o, (float*)ws_ml, nsplit, nq, nkv,
            page_size, page_stride, max_pages, window, keep_first, scale_log2, (const float*)sinks, cap_log2, paired);
        return hipGetLastError();
    };
    hipError_t launched = hipSuccess;
#define LLE_F32_CASE(DQV)                                                                     \
    case DQV:                                                                                 \
        if constexpr (DQV == 4 || DQV == 8) {                                                 \
            if (tiles == 2) {                                                                 \
                launched = launch(mfma_f32_attention_kernel<DQV, 2, false, false>);           \
                break;                                                                        \
            }                                                                                 \
        }                                                                                     \
        launched = keep_first > 0 ? launch(mfma_f32_attention_kernel<DQV, 1, true, false>)    \
                   : softcap > 0.f ? launch(mfma_f32_attention_kernel<DQV, 1, false, true>)   \
                                   : launch(mfma_f32_attention_kernel<DQV, 1, false, false>); \
        break;
    if (tiles == 3) {
        static std::atomic<uint64_t> granted{0};
        const hipError_t e = lle_grant_lds((const void*)split_f32_attention_kernel, SA_LDS, granted);
        if (e != hipSuccess) return (int)e;
        split_f32_attention_kernel<<<grid, F32_WAVES * LLE_WAVE, smem, stream>>>(
            (const float*)q, (const float*)kv_layer, (const int32_t*)block_tables, (const int32_t*)seq_slots, (const int32_t*)cu_tokens,
            (const int32_t*)kv_lens, (float*)out, (float*)ws_o, (float*)ws_ml, nsplit, nq, nkv, page_size, page_stride, max_pages, window,
            scale_log2, (const float*)sinks, paired);
        launched = hipGetLastError();
    } else switch (d / 16) {
        LLE_F32_CASE(1) LLE_F32_CASE(2) LLE_F32_CASE(3) LLE_F32_CASE(4) LLE_F32_CASE(5) LLE_F32_CASE(6)
        LLE_F32_CASE(7) LLE_F32_CASE(8) LLE_F32_CASE(9) LLE_F32_CASE(10) LLE_F32_CASE(11) LLE_F32_CASE(12)
        LLE_F32_CASE(13) LLE_F32_CASE(14) LLE_F32_CASE(15) LLE_F32_CASE(16)
    }
#undef LLE_F32_CASE
    if (launched != hipSuccess) return (int)launched;
    const int64_t out_rows = (int64_t)N * nq;
    if (nsplit > 1 && tiles == 3)
        split_f32_combine_kernel<<<(int)((out_rows + 3) / 4), 256, 0, stream>>>((const float*)ws_o, (const float*)ws_ml, nsplit, (float*)out, out_rows,
                                                                                nq, (const float*)sinks);
    else if (nsplit > 1)
        f32_combine_kernel<<<dim3(N, nq), LLE_WAVE, 0, stream>>>((const float*)ws_o, (const float*)ws_ml, nsplit,
                                                                 (float*)out, nq, d, (const float*)sinks);
    return (int)hipGetLastError();
}

// CUs of the current device (asked once per device)
static int compute_units() {
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

template <int DK, bool FUSED, bool KEEP, bool CAP = false>
static int launch_decode(const bf16_t* q, bf16_t* kv_layer, const int32_t* block_tables, const int32_t* seq_slots,
                         const int32_t* cu_tokens, const int32_t* kv_lens, bf16_t* out, float* ws_o, float* ws_ml,
                         int ws_stride, int S, int nq, int nkv, int P, int64_t page_stride, int max_pages, int window,
                         float scale_log2, int nsplit, const FusedQKV& fused, const float* sinks, int keep_first,
                         float cap_log2, hipStream_t stream) {
    constexpr int D = DK * 32;
    const size_t smem = (size_t)(DEC_WAVES * 16 * D + 2 * DEC_WAVES * 16) * sizeof(float);
    if (smem > 64 * 1024) {
        hipError_t e = hipFuncSetAttribute((const void*)mfma_decode_kernel<DK, FUSED, KEEP, CAP>,
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
        if (e != hipSuccess) return (int)e;
    }
    mfma_decode_kernel<DK, FUSED, KEEP, CAP><<<dim3(S, nkv, nsplit), DEC_WAVES * LLE_WAVE, smem, stream>>>(
        q, kv_layer, block_tables, seq_slots, cu_tokens, kv_lens, out, ws_o, ws_ml, ws_stride, nq, nkv, P,
        page_stride, max_pages, window, scale_log2, fused, sinks, keep_first, cap_log2);
    return 0;
}

template <int DK, int WEIGHTS, bool PAIRS = false, bool CAP = false>
static int launch_short_decode(const FusedQKV& f, bf16_t* kv_layer, const int32_t* block_tables, const int32_t* seq_slots,
                               const int32_t* cu_tokens, const int32_t* kv_lens, bf16_t* out, int S, int nq, int nkv, int P,
                               int64_t page_stride, int max_pages, int window, float scale_log2, hipStream_t stream) {
    const int G = nq / nkv;
    const size_t smem = (size_t)(SHORT_WAVES + 1) * (G * DK * 32 + 2 * 16) * sizeof(float);
    short_decode_kernel<DK, WEIGHTS, PAIRS, CAP><<<dim3(S, nkv), (SHORT_WAVES + 1) * LLE_WAVE, smem, stream>>>(
        cu_tokens, kv_lens, seq_slots, block_tables, max_pages, P, window, G, nkv, kv_layer, out, page_stride, scale_log2, f);
    LLE_RETURN_LAUNCH_STATUS();
}

// A second stream of this library's own (per device, made at first use, default priority) and the
// two events that fork it from and join it to the caller's stream: in a batch that holds prompt
// portions beside decoded tokens the two attention kernels work on different requests, one bound by
// memory and one by the matrix cores, and share the chip instead of taking turns.
struct SideLane {
    hipStream_t stream;
    hipEvent_t fork, join;
};
static SideLane* side_lane() {
    static SideLane lanes[64];
    static int state[64] = {0};  // 0: not made, 1: there, -1: could not be made
    static std::mutex lock;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return nullptr;
    std::lock_guard<std::mutex> guard(lock);
    if (state[dev] == 0) {
        SideLane& l = lanes[dev];
        const bool ok = hipStreamCreateWithFlags(&l.stream, hipStreamNonBlocking) == hipSuccess &&
                        hipEventCreateWithFlags(&l.fork, hipEventDisableTiming) == hipSuccess &&
                        hipEventCreateWithFlags(&l.join, hipEventDisableTiming) == hipSuccess;
        state[dev] = ok ? 1 : -1;
    }
    return state[dev] == 1 ? &lanes[dev] : nullptr;
}

template <int DK>
static int launch_mfma(const bf16_t* q, bf16_t* kv_layer, const int32_t* block_tables,
                       const int32_t* seq_slots, const int32_t* cu_tokens, const int32_t* kv_lens,
                       const int32_t* token_seq, bf16_t* out, float* ws_o, float* ws_ml, int N, int S, int nq,
                       int nkv, int P, int64_t page_stride, int max_pages, int window, float scale_log2,
                       int run_decode, int nsplit_decode, int run_prefill, int nsplit_prefill, int max_q_len,
                       int prefill_form, const FusedQKV& fused, const float* sinks, int keep_first, float cap_log2,
                       hipStream_t stream) {
    constexpr int D = DK * 32;
    const int G = nq / nkv;
    if (!run_decode) nsplit_decode = 1;
    if (!run_prefill) nsplit_prefill = 1;
    const int ws_stride = nsplit_decode > nsplit_prefill ? nsplit_decode : nsplit_prefill;
    if (fused.qkv && (run_prefill || !run_decode || DK % 2 != 0 || keep_first || cap_log2 > 0.f)) return (int)hipErrorInvalidValue;
    // both kinds in one batch: the decode kernel goes to the side stream, forked from and joined to `stream`
    SideLane* lane = (run_decode && run_prefill) ? side_lane() : nullptr;
    hipStream_t prefill_stream = stream;
    if (lane) {
        if (hipEventRecord(lane->fork, stream) != hipSuccess || hipStreamWaitEvent(lane->stream, lane->fork, 0) != hipSuccess)
            lane = nullptr;
    }
    if (lane) stream = lane->stream;  // for the decode kernel below
    if (run_decode) {
        int e;
        if (keep_first > 0) {
            e = launch_decode<DK, false, true>(q, kv_layer, block_tables, seq_slots, cu_tokens, kv_lens, out, ws_o, ws_ml,
                                               ws_stride, S, nq, nkv, P, page_stride, max_pages, window, scale_log2,
                                               nsplit_decode, fused, sinks, keep_first, 0.f, stream);
        } else if (cap_log2 > 0.f) {
            e = launch_decode<DK, false, false, true>(q, kv_layer, block_tables, seq_slots, cu_tokens, kv_lens, out, ws_o, ws_ml,
                                                      ws_stride, S, nq, nkv, P, page_stride, max_pages, window, scale_log2,
                                                      nsplit_decode, fused, sinks, 0, cap_log2, stream);
        } else if constexpr (DK % 2 == 0) {
            e = fused.qkv ? launch_decode<DK, true, false>(q, kv_layer, block_tables, seq_slots, cu_tokens, kv_lens, out, ws_o,
                                                    ws_ml, ws_stride, S, nq, nkv, P, page_stride, max_pages, window,
                                                    scale_log2, nsplit_decode, fused, sinks, 0, 0.f, stream)
                          : launch_decode<DK, false, false>(q, kv_layer, block_tables, seq_slots, cu_tokens, kv_lens, out,
                                                     ws_o, ws_ml, ws_stride, S, nq, nkv, P, page_stride, max_pages,
                                                     window, scale_log2, nsplit_decode, fused, sinks, 0, 0.f, stream);
        } else {
            e = launch_decode<DK, false, false>(q, kv_layer, block_tables, seq_slots, cu_tokens, kv_lens, out, ws_o, ws_ml,
                                         ws_stride, S, nq, nkv, P, page_stride, max_pages, window, scale_log2,
                                         nsplit_decode, fused, sinks, 0, 0.f, stream);
        }
        if (e != 0) {
            if (lane) (void)hipStreamSynchronize(lane->stream);
            return e;
        }
    }
    // After the fork an error may not leave the side stream running behind the caller's back: the
    // caller frees `out` and the workspaces on its own stream, and the decode kernel still writes them.
    if (lane) {
        if (hipEventRecord(lane->join, lane->stream) != hipSuccess) {
            const int e = (int)hipGetLastError();
            (void)hipStreamSynchronize(lane->stream);
            return e;
        }
        stream = prefill_stream;
    }
    if (run_prefill) {
        const int rows = max_q_len * G;
        auto launch = [&](auto rt, auto waves) {
            constexpr int RT = decltype(rt)::value, WAVES = decltype(waves)::value;
            constexpr int PRE_ROWS = WAVES * 16 * RT;
            const int blocks = (rows + PRE_ROWS - 1) / PRE_ROWS;
            const int64_t workgroups = (int64_t)nkv * blocks * nsplit_prefill * S;
            auto go = [&](auto kernel) {
                kernel<<<dim3(nkv, blocks * nsplit_prefill, S), WAVES * LLE_WAVE, 0, stream>>>(
                    q, kv_layer, block_tables, seq_slots, cu_tokens, kv_lens, out, ws_o, ws_ml, ws_stride, nsplit_prefill,
                    nq, nkv, P, page_stride, max_pages, window, scale_log2, workgroups <= 2 * compute_units() ? 1 : 0, sinks,
                    keep_first, cap_log2);
            };
            if (keep_first > 0) go(mfma_prefill_kernel<DK, RT, WAVES, true, false>);
            else if (cap_log2 > 0.f) go(mfma_prefill_kernel<DK, RT, WAVES, false, true>);
            else go(mfma_prefill_kernel<DK, RT, WAVES, false, false>);
        };
        using Four = std::integral_constant<int, 4>;
        if (DK == 4 && prefill_form == 3) {
            if constexpr (DK == 4) launch(std::integral_constant<int, 1>{}, std::integral_constant<int, 8>{});
        } else if (PRE_RT_OF(DK) == 1 || prefill_form == 1) {
            launch(std::integral_constant<int, 1>{}, Four{});
        } else {
            launch(std::integral_constant<int, PRE_RT_OF(DK)>{}, Four{});
        }
    }
    if (lane && hipStreamWaitEvent(stream, lane->join, 0) != hipSuccess) {
        const int e = (int)hipGetLastError();
        (void)hipStreamSynchronize(lane->stream);
        return e;
    }
    if (ws_stride > 1)  // a batch of one kind needs no look at the tokens' requests
        mfma_combine_kernel<<<dim3(N, nq), LLE_WAVE, 0, stream>>>(
            ws_o, ws_ml, ws_stride, cu_tokens, token_seq, out, nq, nkv, D, run_decode ? nsplit_decode : nsplit_prefill,
            run_prefill ? nsplit_prefill : nsplit_decode, sinks);
    return (int)hipGetLastError();
}

// bfloat16, head_dim a multiple of 32 (<= 256), page size a multiple of 16.
// run_decode / run_prefill say which kinds of request the batch holds (requests
// with q_len * group <= 16 rows are the decode kernel's); with ns = max(nsplit_decode,
// nsplit_prefill) > 1 the workspaces ws_o [N * nq * ns * d] and ws_ml [N * nq * ns * 2]
// floats are needed (ns <= 64).
static int paged_attention_mfma(const void* q, void* kv_layer, const void* block_tables, const void* seq_slots,
                                const void* cu_tokens, const void* kv_lens, const void* token_seq, void* out,
                                void* ws_o, void* ws_ml, int N, int S, int nq, int nkv, int d, int page_size,
                                int64_t page_stride, int max_pages, int window, float scale, int run_decode,
                                int nsplit_decode, int run_prefill, int nsplit_prefill, int max_q_len,
                                int prefill_form, const FusedQKV& fused, const float* sinks, int keep_first,
                                float softcap, hipStream_t stream) {
    if (N <= 0) return 0;
    if (keep_first < 0 || (keep_first > 0 && window <= 0)) return (int)hipErrorInvalidValue;
    if (d % 32 != 0 || d > 256 || page_size % 16 != 0 || nq % nkv != 0) return (int)hipErrorInvalidValue;
    if (S > 65535 || nkv > 65535 || page_stride < 0 || page_stride >= ((int64_t)1 << 32)) return (int)hipErrorInvalidValue;
    if (nsplit_decode < 1 || nsplit_decode > 64 || nsplit_prefill < 1 || nsplit_prefill > 64)
        return (int)hipErrorInvalidValue;
    if (softcap < 0.f || (softcap > 0.f && keep_first > 0)) return (int)hipErrorInvalidValue;
    const float cap_log2 = softcap * 1.44269504088896340736f;
    const float scale_log2 = softcap > 0.f ? 2.f * scale / softcap * 1.44269504088896340736f : scale * 1.44269504088896340736f;
#define LLE_ATT_CASE(DKV)                                                                                          \
    case DKV:                                                                                                      \
        return launch_mfma<DKV>((const bf16_t*)q, (bf16_t*)kv_layer, (const int32_t*)block_tables,                  \
                                (const int32_t*)seq_slots, (const int32_t*)cu_tokens, (const int32_t*)kv_lens,      \
                                (const int32_t*)token_seq, (bf16_t*)out, (float*)ws_o, (float*)ws_ml, N, S, nq, nkv, \
                                page_size, page_stride, max_pages, window, scale_log2, run_decode, nsplit_decode,   \
                                run_prefill, nsplit_prefill, max_q_len, prefill_form, fused, sinks, keep_first, cap_log2,     \
                                stream);
    switch (d / 32) {
        LLE_ATT_CASE(1)
        LLE_ATT_CASE(2)
        LLE_ATT_CASE(3)
        LLE_ATT_CASE(4)
        LLE_ATT_CASE(5)
        LLE_ATT_CASE(6)
        LLE_ATT_CASE(7)
        LLE_ATT_CASE(8)
    }
#undef LLE_ATT_CASE
    return (int)hipErrorInvalidValue;
}

extern "C" int lle_paged_attention_mfma(const void* q, const void* kv_layer, const void* block_tables,
                                        const void* seq_slots, const void* cu_tokens, const void* kv_lens,
                                        const void* token_seq, void* out, void* ws_o, void* ws_ml, int N, int S,
                                        int nq, int nkv, int d, int page_size, int64_t page_stride, int max_pages,
                                        int window, float scale, int run_decode, int nsplit_decode, int run_prefill,
                                        int nsplit_prefill, int max_q_len, int prefill_form, const void* sinks,
                                        int keep_first, float softcap, hipStream_t stream) {
    const FusedQKV none = {};
    return paged_attention_mfma(q, (void*)kv_layer, block_tables, seq_slots, cu_tokens, kv_lens, token_seq, out, ws_o,
                                ws_ml, N, S, nq, nkv, d, page_size, page_stride, max_pages, window, scale, run_decode,
                                nsplit_decode, run_prefill, nsplit_prefill, max_q_len, prefill_form, none,
                                (const float*)sinks, keep_first, softcap, stream);
}

// The most keys of a request, and the LDS, of short_decode_kernel.
extern "C" int lle_short_decode_max_keys(void) { return SHORT_WAVES * KSTEP; }
static bool short_decode_fits(int S, int nq, int nkv, int d, int page_size, int max_kv_len) {
    return S > 0 && S <= 65535 && nkv > 0 && nkv <= 65535 && nq > 0 && nq % nkv == 0 && nq / nkv <= 16 && (d == 64 || d == 128) && page_size > 0 &&
           page_size % 16 == 0 && max_kv_len > 0 && max_kv_len <= SHORT_WAVES * KSTEP &&
           (size_t)(SHORT_WAVES + 1) * (nq / nkv * d + 2 * 16) * sizeof(float) <= 64 * 1024;
}

// Whether it takes a step of S requests in place of mfma_decode_kernel, of which twice as many workgroups fit a CU where heads
// are of 64: only while all of its own are at work at once.  Heads of 64 in groups of 1 to 8 at 512 workgroups and 24 / 97 / 160
// / 256 keys: 8.8 / 9.7 / 9.6 / 10.3 -> 7.1 / 7.9 / 8.8 / 10.1 us, at 768 10.1 / 12.3 / 12.5 / 14.4 -> 9.6 / 10.8 / 12.3 / 16.1, at 2048
// 21 / 27 / 28 / 29 -> 22 / 27 / 31 / 35; groups of 16 at 256: 8.3 / 8.5 / 8.5 / 8.5 -> 5.3 / 5.8 / 6.2 / 6.9, at 320 10.6 -> 11.6
// with 256 keys.  (Heads of 128: 0.95 of the time at 2048 workgroups of 256 keys, less at fewer.)
static bool short_decode_pays(int S, int G, int nkv, int d) { return d != 64 || (int64_t)S * nkv <= (G > 8 ? 256 : 512); }

// One token a request (S of them): the rotation of q and k in neighbouring pairs, the write of K and V and the attention of
// lle_pair_rope_write and lle_paged_attention_mfma in one launch, for heads of 64 or 128 of q, k and v alike without biases.  A row of u
// has `cols` columns, a multiple of 8: q, k, v, then others.  rot: a multiple of 8 (0: nothing turns); softcap <= 0: none.
extern "C" int lle_pair_rope_attention_decode(const void* u, int cols, const void* slots, const void* cos_sin, int rot, int write_kv,
                                              void* kv_layer, const void* block_tables, const void* seq_slots, const void* cu_tokens,
                                              const void* kv_lens, void* out, int S, int nq, int nkv, int d, int page_size,
                                              int64_t page_stride, int max_pages, int window, float scale, float softcap, int max_kv_len,
                                              hipStream_t stream) {
    if (!short_decode_fits(S, nq, nkv, d, page_size, max_kv_len) || cols % 8 != 0 || cols < (nq + 2 * nkv) * d || rot < 0 || rot % 8 != 0 ||
        rot > d || (rot > 0 && !cos_sin) || !u || !slots || ((uintptr_t)u & 15))
        return (int)hipErrorInvalidValue;
    FusedQKV f = {};
    f.qkv = (const bf16_t*)u;
    f.slots = (const int32_t*)slots;
    f.cos_sin = (const float*)cos_sin;
    f.write_kv = write_kv;
    f.cols = cols;
    f.rot = rot;
    constexpr float LOG2E = 1.44269504088896340736f;
    const bool cap = softcap > 0.f;
    f.cap_log2 = cap ? softcap * LOG2E : 0.f;
    const float scale_log2 = cap ? 2.f * LOG2E * scale / softcap : scale * LOG2E;
    return (d == 64 ? (cap ? launch_short_decode<2, LLE_BF16, true, true> : launch_short_decode<2, LLE_BF16, true, false>)
                    : (cap ? launch_short_decode<4, LLE_BF16, true, true> : launch_short_decode<4, LLE_BF16, true, false>))(
        f, (bf16_t*)kv_layer, (const int32_t*)block_tables, (const int32_t*)seq_slots, (const int32_t*)cu_tokens, (const int32_t*)kv_lens,
        (bf16_t*)out, S, nq, nkv, page_size, page_stride, max_pages, window, scale_log2, stream);
}

// The most keys of a request of short_decode_f32_kernel.
extern "C" int lle_short_decode_max_keys_f32(void) { return SHORT_F32_KEYS; }

// One token a request (S of them), float32 throughout (norm weights: weight_dtype, or none): q/k norm, rotation over the whole
// head, the write of K and V and the attention in one launch, for heads of 64 or 128 and at most SHORT_F32_KEYS keys.  Else as
// lle_qk_norm_rope_attention_decode below.
extern "C" int lle_qk_norm_rope_attention_decode_f32(const void* qkv, const void* slots, const void* q_weight, const void* k_weight,
                                                     int weight_dtype, const void* cos_sin, float eps, int write_kv, void* kv_layer,
                                                     const void* block_tables, const void* seq_slots, const void* cu_tokens,
                                                     const void* kv_lens, void* out, int S, int nq, int nkv, int d, int page_size,
                                                     int64_t page_stride, int max_pages, int window, float scale, int max_kv_len,
                                                     hipStream_t stream) {
    if (S <= 0) return 0;
    if (!qkv || !cos_sin || !slots || (q_weight == nullptr) != (k_weight == nullptr) || S > 65535 || nkv <= 0 || nkv > 65535 || nq <= 0 ||
        nq % nkv != 0 || nq / nkv > 16 || (d != 64 && d != 128) || page_size <= 0 || page_size % 16 != 0 || max_kv_len <= 0 ||
        max_kv_len > SHORT_F32_KEYS || (((uintptr_t)qkv | (uintptr_t)cos_sin | (uintptr_t)kv_layer) & 15) || page_stride % 4 != 0)
        return (int)hipErrorInvalidValue;
    const size_t smem = (size_t)(SHORT_F32_WAVES + 1) * (nq / nkv * d + 2 * 16) * sizeof(float);
    if (smem > 64 * 1024) return (int)hipErrorInvalidValue;
    FusedQKV f = {};
    f.qkv = (const bf16_t*)qkv;
    f.slots = (const int32_t*)slots;
    f.q_weight = q_weight;
    f.k_weight = k_weight;
    f.cos_sin = (const float*)cos_sin;
    f.eps = eps;
    f.write_kv = write_kv;
    const bool f32 = weight_dtype == LLE_F32;
    auto kernel = d == 64 ? (f32 ? short_decode_f32_kernel<4, LLE_F32> : short_decode_f32_kernel<4, LLE_BF16>)
                          : (f32 ? short_decode_f32_kernel<8, LLE_F32> : short_decode_f32_kernel<8, LLE_BF16>);
    kernel<<<dim3(S, nkv), (SHORT_F32_WAVES + 1) * LLE_WAVE, smem, stream>>>(
        (const int32_t*)cu_tokens, (const int32_t*)kv_lens, (const int32_t*)seq_slots, (const int32_t*)block_tables, max_pages, page_size,
        window, nq / nkv, nkv, (float*)kv_layer, (float*)out, page_stride, scale * 1.44269504088896340736f, f);
    LLE_RETURN_LAUNCH_STATUS();
}

// Decode steps only (every request has at most 16 / group tokens), head_dim a multiple of 64, a
// rotation over the whole head: the q/k norm, the rotation and the write of the new K and V
// (write_kv != 0; slots [N], < 0: not written) happen inside the attention launch.  qkv is
// [N, (nq + 2 nkv) * d] as the projection left it; q_weight / k_weight [d] or null; cos_sin
// [N, d / 2, 2] float32.  token_seq null: one token a request.  Then, with no more than SHORT_WAVES * 32 keys a request (`max_kv_len` > 0 is a
// bound), heads of 64 or 128 and partial results that 64 KB of LDS hold (groups of up to 13 at 128): short_decode_kernel, where
// short_decode_pays.
// (`order` serves more keys.)
extern "C" int lle_qk_norm_rope_attention_decode(const void* qkv, const void* slots, const void* q_weight,
                                                 const void* k_weight, int weight_dtype, const void* cos_sin,
                                                 float eps, int write_kv, void* kv_layer, const void* block_tables,
                                                 const void* seq_slots, const void* cu_tokens, const void* kv_lens,
                                                 const void* token_seq, void* out, void* ws_o, void* ws_ml, int N,
                                                 int S, int nq, int nkv, int d, int page_size, int64_t page_stride,
                                                 int max_pages, int window, float scale, int nsplit_decode,
                                                 const void* order, int max_kv_len, hipStream_t stream) {
    if (!qkv || !cos_sin || !slots || d % 64 != 0) return (int)hipErrorInvalidValue;
    if ((q_weight == nullptr) != (k_weight == nullptr)) return (int)hipErrorInvalidValue;
    FusedQKV fused = {};
    fused.qkv = (const bf16_t*)qkv;
    fused.slots = (const int32_t*)slots;
    fused.q_weight = q_weight;
    fused.k_weight = k_weight;
    fused.weight_dtype = weight_dtype;
    fused.cos_sin = (const float*)cos_sin;
    fused.eps = eps;
    fused.write_kv = write_kv;
    fused.order = (const int32_t*)order;
    if (!token_seq && N == S && nsplit_decode == 1 && !order && short_decode_fits(S, nq, nkv, d, page_size, max_kv_len) &&
        short_decode_pays(S, nq / nkv, nkv, d)) {
        const float scale_log2 = scale * 1.44269504088896340736f;
        const bool f32 = weight_dtype == LLE_F32;
        return (d == 64 ? (f32 ? launch_short_decode<2, LLE_F32> : launch_short_decode<2, LLE_BF16>)
                        : (f32 ? launch_short_decode<4, LLE_F32> : launch_short_decode<4, LLE_BF16>))(
            fused, (bf16_t*)kv_layer, (const int32_t*)block_tables, (const int32_t*)seq_slots, (const int32_t*)cu_tokens,
                (const int32_t*)kv_lens, (bf16_t*)out, S, nq, nkv, page_size, page_stride, max_pages, window, scale_log2, stream);
    }
    return paged_attention_mfma(nullptr, kv_layer, block_tables, seq_slots, cu_tokens, kv_lens, token_seq, out, ws_o,
                                ws_ml, N, S, nq, nkv, d, page_size, page_stride, max_pages, window, scale, 1,
                                nsplit_decode, 0, 1, 1, 0, fused, nullptr, 0, 0.f, stream);
}
