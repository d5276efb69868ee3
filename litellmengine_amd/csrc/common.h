// Shared device helpers for the gfx950 kernels: element types, conversions,
// wavefront (64 lanes) and workgroup reductions.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <float.h>

typedef __bf16 bf16_t;

// dtype codes shared with the Python side (csrc/ops.py)
#define LLE_F32 0
#define LLE_BF16 1

#define LLE_WAVE 64

template <typename T> __device__ __forceinline__ float to_f32(T x);
template <> __device__ __forceinline__ float to_f32<float>(float x) { return x; }
template <> __device__ __forceinline__ float to_f32<bf16_t>(bf16_t x) { return (float)x; }

template <typename T> __device__ __forceinline__ T from_f32(float x);
template <> __device__ __forceinline__ float from_f32<float>(float x) { return x; }
template <> __device__ __forceinline__ bf16_t from_f32<bf16_t>(float x) { return (bf16_t)x; }

// a value of either float type behind a void pointer (norm weights may be
// stored in 32-bit while activations are 16-bit)
__device__ __forceinline__ float load_as_f32(const void* p, int64_t i, int dtype) {
    return dtype == LLE_F32 ? ((const float*)p)[i] : (float)((const bf16_t*)p)[i];
}

// Lanes i and i ^ 32 (or i ^ 16) combined by `op`, in every lane: the two operands of the swap come out as the lower and the
// upper halves (even and odd rows of 16) repeated.  All lanes of the wavefront must be active here and below.
template <typename Op>
__device__ __forceinline__ float combine_xor32(float v, Op op) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return op(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
template <typename Op>
__device__ __forceinline__ float combine_xor16(float v, Op op) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return op(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
// the lane's own value and that of the lane N further on in its row of 16 (around its end)
template <int N, typename Op>
__device__ __forceinline__ float combine_row_ror(float v, Op op) {
    return op(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x120 + N, 0xf, 0xf, true)));
}
struct AddF32 {
    __device__ __forceinline__ float operator()(float a, float b) const { return a + b; }
};
struct MaxF32 {
    __device__ __forceinline__ float operator()(float a, float b) const { return fmaxf(a, b); }
};

// All 64 lanes by the tree of i ^ 32, i ^ 16, i ^ 8, ... i ^ 1.  (Once lanes 8 apart hold the same, the lane 4 further on in the
// row holds what lane i ^ 4 does, and so on.)  Ten instructions between registers instead of six trips through LDS of nine
// each: a wavefront alone issues an instruction in four to eight cycles, so a decode step's short launches pay for every one.
template <typename Op>
__device__ __forceinline__ float combine_wave(float v, Op op) {
    v = combine_xor32(v, op);
    v = combine_xor16(v, op);
    v = combine_row_ror<8>(v, op);
    v = combine_row_ror<4>(v, op);
    v = combine_row_ror<2>(v, op);
    return combine_row_ror<1>(v, op);
}
__device__ __forceinline__ float wave_sum(float v) { return combine_wave(v, AddF32{}); }
__device__ __forceinline__ float wave_max(float v) { return combine_wave(v, MaxF32{}); }
// the lane's row of 16: i ^ 1, then i ^ 2, 4, 8.  (Once neighbours hold the same, the other pair of a quad is as good as lane
// i ^ 2; then the mirrored half row as lane i ^ 4, and the mirrored row as lane i ^ 8.)
template <int CTRL>
__device__ __forceinline__ float add_dpp(float v) {
    return v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}
__device__ __forceinline__ float row16_sum(float v) {
    v = add_dpp<0xb1>(v);   // quad_perm 1 0 3 2
    v = add_dpp<0x4e>(v);   // quad_perm 2 3 0 1
    v = add_dpp<0x141>(v);  // row_half_mirror
    return add_dpp<0x140>(v);  // row_mirror
}
// the four lanes i % 16 (a column of a matrix-core tile): i ^ 16, then i ^ 32
__device__ __forceinline__ float column_sum(float v) { return combine_xor32(combine_xor16(v, AddF32{}), AddF32{}); }
__device__ __forceinline__ float column_max(float v) { return combine_xor32(combine_xor16(v, MaxF32{}), MaxF32{}); }

// 16 bytes a lane from `base` and its byte offset straight into LDS, the lanes' one behind the other from byte `at` on (both
// the same for the wavefront).  The load takes its address in LDS from M0 and wants a wait state behind a write of it, which the
// compiler cannot put into an asm.  Nothing waits for the load here: vmcnt counts it.
__device__ __forceinline__ void load_into_lds(unsigned at, unsigned offset, const void* base) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(at), "v"(offset), "s"(base) : "memory", "m0");
}

// the same with 4 bytes a lane
__device__ __forceinline__ void load_word_into_lds(unsigned at, unsigned offset, const void* base) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" ::"s"(at), "v"(offset), "s"(base) : "memory", "m0");
}

// The values of keys outside [lo, hi] become zeros; v[n][i], of eight 16-bit numbers, belongs to key `first` + i.  Their weight is
// 0, which drops whatever lies there but an infinity or a NaN (pages are handed on as they are).
template <typename Vec, int N>
__device__ __forceinline__ void drop_values(Vec (&v)[N], int first, int lo, int hi) {
    typedef uint32_t quad __attribute__((ext_vector_type(4)));
    static_assert(sizeof(Vec) == sizeof(quad), "eight 16-bit numbers");
    quad keep;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int j = first + 2 * i;
        keep[i] = (j >= lo && j <= hi ? 0xffffu : 0u) | (j + 1 >= lo && j + 1 <= hi ? 0xffff0000u : 0u);
    }
#pragma unroll
    for (int n = 0; n < N; ++n) v[n] = __builtin_bit_cast(Vec, __builtin_bit_cast(quad, v[n]) & keep);
}

// Sum over a workgroup of up to 1024 threads; `smem` holds >= 16 floats.
// Every thread gets the result; the order of the additions is fixed.
__device__ __forceinline__ float block_sum(float v, float* smem) {
    const int lane = threadIdx.x % LLE_WAVE, wave = threadIdx.x / LLE_WAVE;
    const int nwaves = (blockDim.x + LLE_WAVE - 1) / LLE_WAVE;
    v = wave_sum(v);
    __syncthreads();
    if (lane == 0) smem[wave] = v;
    __syncthreads();
    float total = 0.f;
    for (int w = 0; w < nwaves; ++w) total += smem[w];
    return total;
}

__device__ __forceinline__ float block_max(float v, float* smem) {
    const int lane = threadIdx.x % LLE_WAVE, wave = threadIdx.x / LLE_WAVE;
    const int nwaves = (blockDim.x + LLE_WAVE - 1) / LLE_WAVE;
    v = wave_max(v);
    __syncthreads();
    if (lane == 0) smem[wave] = v;
    __syncthreads();
    float total = smem[0];
    for (int w = 1; w < nwaves; ++w) total = fmaxf(total, smem[w]);
    return total;
}

// launch check shared by the extern "C" entry points: 0 or the hipError_t
#define LLE_RETURN_LAUNCH_STATUS() return (int)hipGetLastError()

extern "C" const char* lle_error_string(int code);
#define LLE_DEFINE_ERROR_STRING() \
    extern "C" const char* lle_error_string(int code) { return hipGetErrorString((hipError_t)code); }
