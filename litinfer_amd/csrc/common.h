// Shared device helpers for the gfx950 kernels: element types, conversions,
// wave and block reductions with a fixed order.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#define LI_OK 0
#define LI_ERR_DTYPE 1
#define LI_ERR_SIZE 2
#define LI_ERR_LAUNCH 3

#define LI_F32 0
#define LI_BF16 1

#define LI_WAVE 64

struct bf16_t { uint16_t bits; };

__device__ __forceinline__ float bf16_to_float(uint16_t b) {
    return __uint_as_float(((uint32_t)b) << 16);
}

// round to nearest even; NaN stays NaN (v_cvt_pk_bf16_f32, one instruction for one or two values)
__device__ __forceinline__ uint16_t float_to_bf16(float f) {
    return __builtin_bit_cast(uint16_t, (__bf16)f);
}

typedef __bf16 li_bf16x2 __attribute__((ext_vector_type(2)));
typedef float li_f32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t pack2_bf16(float lo, float hi) {      // lo in bits 0..15
    li_f32x2 v = {lo, hi};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, li_bf16x2));
}

__device__ __forceinline__ float load_as_float(const float* p) { return *p; }
__device__ __forceinline__ float load_as_float(const bf16_t* p) { return bf16_to_float(p->bits); }
__device__ __forceinline__ void store_from_float(float* p, float v) { *p = v; }
__device__ __forceinline__ void store_from_float(bf16_t* p, float v) { p->bits = float_to_bf16(v); }

// GELU with the error function
__device__ __forceinline__ float gelu_erf(float z) { return 0.5f * z * (1.0f + erff(z * 0.70710678118654752f)); }
// ... and in its tanh form
__device__ __forceinline__ float gelu_tanh(float z) {
    return 0.5f * z * (1.0f + tanhf(0.7978845608028654f * (z + 0.044715f * z * z * z)));
}
// ... for results that are rounded to bfloat16: z / 2 (1 + tanh(u)) = z / (1 + exp(-2 u)), with the exponential and reciprocal
// instructions (one unit in the last float32 place each), a third of the instructions
__device__ __forceinline__ float gelu_tanh_bf16(float z) {
    return z * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.5957691216057308f * 1.44269504088896341f * (z + 0.044715f * z * z * z)));
}
// xIELU with two numbers worked out by the caller, sp = softplus(p) and sq = 1/2 + softplus(q):
// z > 0: sp z^2 + z / 2;  z <= 0: sq (exp(z) - 1 - z) + z / 2
__device__ __forceinline__ float xielu(float z, float sp, float sq) {
    return (z > 0.f ? sp * z * z : sq * (expm1f(z) - z)) + 0.5f * z;
}
// What a product may leave instead of its sums (li_linear_act): 1 max(z, 0)^2, 2 and 3 GELU in its tanh form and with the
// error function, 4 xIELU with the numbers a0 and a1
#define LI_ACT_RELU2 1
#define LI_ACT_GELU_TANH 2
#define LI_ACT_GELU_ERF 3
#define LI_ACT_XIELU 4
// (a product of gate and up columns, li_linear_swiglu: 2 up * GELU(gate), 5 the clamped form with the limit a0; 0 the plain one)
#define LI_ACT_CLAMPED 5
struct LiAct { int act; float a0, a1; };
__device__ __forceinline__ float activation(float z, const LiAct& e) {
    if (e.act == LI_ACT_RELU2) { const float r = fmaxf(z, 0.f); return r * r; }
    if (e.act == LI_ACT_GELU_TANH) return gelu_tanh(z);
    if (e.act == LI_ACT_GELU_ERF) return gelu_erf(z);
    return xielu(z, e.a0, e.a1);
}

// Exchanges between the lanes of a wave inside the vector ALU.  __shfl_xor goes through the LDS crossbar: sixty cycles and more a step, in a
// chain of six for a sum over a wave, behind which every other LDS access waits; a DPP move (within rows of 16 lanes) or v_permlane16/32_swap
// (between them) is an instruction of a few.  In launches whose work is one row or a few this chain is a good part of the time.
// All lanes of a row (o < 16) or of the wave have to take part.
template <int CTRL>
__device__ __forceinline__ int dpp_mov(int v) { return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xf, 0xf, true); }
// v of lane l ^ o; o a constant once the caller's loop is unrolled: 1, 2, 4, 8, 16 or 32
__device__ __forceinline__ int lane_xor(int v, const int o) {
    if (o == 1) return dpp_mov<0xB1>(v);                       // quad_perm [1,0,3,2]
    if (o == 2) return dpp_mov<0x4E>(v);                       // quad_perm [2,3,0,1]
    if (o == 4) return dpp_mov<0x141>(dpp_mov<0x1B>(v));       // quad_perm [3,2,1,0], then row_half_mirror: l ^ 3 ^ 7
    if (o == 8) return dpp_mov<0x128>(v);                      // row_ror:8
    // (the swap leaves the even rows' (the lower half's) values in every lane of one result, the others' in the other)
    const bool upper = (__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0)) & o) != 0;
    if (o == 16) { const auto r = __builtin_amdgcn_permlane16_swap(v, v, false, false); return upper ? r[0] : r[1]; }
    const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    return upper ? r[0] : r[1];
}
__device__ __forceinline__ float lane_xor(float v, const int o) { return __int_as_float(lane_xor(__float_as_int(v), o)); }
// v + lane_xor(v, o), max(v, lane_xor(v, o)): no choice between the swap's results
template <typename Op>
__device__ __forceinline__ float lane_xor_with(float v, const int o, Op op) {
    if (o < 16) return op(v, lane_xor(v, o));
    const uint32_t u = __float_as_uint(v);
    if (o == 16) { const auto r = __builtin_amdgcn_permlane16_swap(u, u, false, false); return op(__uint_as_float(r[0]), __uint_as_float(r[1])); }
    const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    return op(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float lane_xor_add(float v, const int o) { return lane_xor_with(v, o, [](float a, float b) { return a + b; }); }
__device__ __forceinline__ float lane_xor_max(float v, const int o) { return lane_xor_with(v, o, [](float a, float b) { return fmaxf(a, b); }); }

// Over the wave, in the order 32, 16, 8, 4, 2, 1.  (Once the values repeat every eight lanes, a rotation of the row by 4 brings lane l ^ 4's.)
template <typename Op>
__device__ __forceinline__ float wave_with(float v, Op op) {
    v = lane_xor_with(v, 32, op);
    v = lane_xor_with(v, 16, op);
    v = op(v, __int_as_float(dpp_mov<0x128>(__float_as_int(v))));
    v = op(v, __int_as_float(dpp_mov<0x124>(__float_as_int(v))));
    v = op(v, __int_as_float(dpp_mov<0x122>(__float_as_int(v))));
    return op(v, __int_as_float(dpp_mov<0x121>(__float_as_int(v))));
}
__device__ __forceinline__ float wave_sum(float v) { return wave_with(v, [](float a, float b) { return a + b; }); }
__device__ __forceinline__ float wave_max(float v) { return wave_with(v, [](float a, float b) { return fmaxf(a, b); }); }

// Sum over a block of NT threads (NT a multiple of 64, at most 1024); every
// thread gets the result.  The order of additions depends on NT only.
template <int NT>
__device__ __forceinline__ float block_sum(float v, float* smem /* NT/64 floats */) {
    v = wave_sum(v);
    const int lane = threadIdx.x & (LI_WAVE - 1), w = threadIdx.x / LI_WAVE;
    __syncthreads();
    if (lane == 0) smem[w] = v;
    __syncthreads();
    float t = 0.f;
#pragma unroll
    for (int i = 0; i < NT / LI_WAVE; ++i) t += smem[i];
    return t;
}

static inline int li_launch_status() {
    return hipGetLastError() == hipSuccess ? LI_OK : LI_ERR_LAUNCH;
}
