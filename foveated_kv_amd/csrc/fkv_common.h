// Shared device/host definitions for the FoveatedKV gfx950 library.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <string>

#include "../../include/fkv.h"

typedef _Float16 fkv_h2 __attribute__((ext_vector_type(2)));
typedef float fkv_f2 __attribute__((ext_vector_type(2)));

namespace fkv {

constexpr int kWave = 64;          // CDNA wavefront
constexpr int kTile = 64;          // tokens per wave iteration (one per lane)
constexpr int kWavesPerGroup = 4;  // waves per workgroup of the attention kernel

// Sets the thread-local error string returned by fkv_last_error().
int set_error(const std::string& msg);
int check_hip(hipError_t e, const char* what);

__host__ __device__ inline int64_t cdiv(int64_t a, int64_t b) { return (a + b - 1) / b; }
__host__ __device__ inline int64_t round_up(int64_t a, int64_t b) { return cdiv(a, b) * b; }

// ---------------------------------------------------------------------------
// device helpers
// ---------------------------------------------------------------------------

__device__ inline float h2f(uint16_t b) { return (float)__builtin_bit_cast(_Float16, b); }
__device__ inline uint16_t f2h(float f) { return __builtin_bit_cast(uint16_t, (_Float16)f); }
__device__ inline float bf2f(uint16_t b) { return __uint_as_float((uint32_t)b << 16); }

__device__ inline fkv_h2 as_h2(uint32_t u) { return __builtin_bit_cast(fkv_h2, u); }
__device__ inline uint32_t as_u32(fkv_h2 h) { return __builtin_bit_cast(uint32_t, h); }

// acc + a.x*b.x + a.y*b.y with fp32 accumulation (v_dot2_f32_f16).
__device__ inline float dot2(fkv_h2 a, fkv_h2 b, float acc) {
    return __builtin_amdgcn_fdot2(a, b, acc, false);
}

// Two E4M3 codes (selected 16-bit word of src) -> two fp16 values, exact for
// every normal E4M3 value (v_cvt_scalef32_pk_f16_fp8 with unit scale).
__device__ inline fkv_h2 e4m3x2_to_h2(uint32_t src, bool hi_word) {
    return hi_word ? __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(src, 1.0f, true)
                   : __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(src, 1.0f, false);
}

template <typename T>
__device__ inline T wave_xor(T v, int mask) {
    return __shfl_xor(v, mask, kWave);
}

__device__ inline float wave_max(float v) {
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v = fmaxf(v, wave_xor(v, o));
    return v;
}

__device__ inline float wave_sum(float v) {
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v += wave_xor(v, o);
    return v;
}

__device__ inline float wave_min(float v) {
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v = fminf(v, wave_xor(v, o));
    return v;
}

// 16-byte accesses that leave the caches to others (non-temporal).
typedef uint32_t fkv_u2 __attribute__((ext_vector_type(2)));
typedef uint32_t fkv_u4 __attribute__((ext_vector_type(4)));
__device__ inline uint4 load16_nt(const void* p) {
    const fkv_u4 v = __builtin_nontemporal_load((const fkv_u4*)p);
    return make_uint4(v.x, v.y, v.z, v.w);
}
template <bool NT>
__device__ inline void store16(void* p, uint4 v) {
    const fkv_u4 x = {v.x, v.y, v.z, v.w};
    if (NT) __builtin_nontemporal_store(x, (fkv_u4*)p);
    else *(fkv_u4*)p = x;
}
template <bool NT>
__device__ inline void store8(void* p, uint32_t lo, uint32_t hi) {
    const fkv_u2 x = {lo, hi};
    if (NT) __builtin_nontemporal_store(x, (fkv_u2*)p);
    else *(fkv_u2*)p = x;
}

// 8 consecutive elements, read once (non-temporal), as packed fp16 bits
// (astype(float16) semantics: RNE).  float32 elements, whose 32 bytes take two
// loads, pass the caches by only with nt32: what the first load brings the
// second one then has to fetch again from beyond them.
__device__ inline uint4 load8(const void* base, int dtype, int64_t elem, bool nt32 = true) {
    if (dtype == FKV_F16) return load16_nt((const uint16_t*)base + elem);
    auto pk = [](float a, float b) { return (uint32_t)f2h(a) | ((uint32_t)f2h(b) << 16); };
    if (dtype == FKV_BF16) {
        const uint4 w = load16_nt((const uint16_t*)base + elem);
        auto two = [&](uint32_t u) { return pk(__uint_as_float(u << 16), __uint_as_float(u & 0xFFFF0000u)); };
        return make_uint4(two(w.x), two(w.y), two(w.z), two(w.w));
    }
    const uint4* p = (const uint4*)((const float*)base + elem);
    const uint4 a = nt32 ? load16_nt(p) : p[0], b = nt32 ? load16_nt(p + 1) : p[1];
    auto two = [&](uint32_t x, uint32_t y) { return pk(__uint_as_float(x), __uint_as_float(y)); };
    return make_uint4(two(a.x, a.y), two(a.z, a.w), two(b.x, b.y), two(b.z, b.w));
}

// a / b rounded to nearest even, from y = 1.0f / b (so rounded itself):
// Markstein's correction of a * y.  One step gives the correctly rounded
// quotient where a * y is within one unit in the last place; a second one
// (STEPS = 2) holds for any rounding of a * y.  A non-finite b gives NaN
// where the division gives 0 or NaN.
template <int STEPS>
__device__ inline float div_by(float a, float b, float y) {
    float q = a * y;
#pragma unroll
    for (int i = 0; i < STEPS; i++) q = fmaf(fmaf(-b, q, a), y, q);
    return q;
}

// v of another lane by DPP (a quad_perm or row mirror control).
template <int CTRL>
__device__ inline float dpp_f32(float v) {
    const int i = __float_as_int(v);
    return __int_as_float(__builtin_amdgcn_update_dpp(i, i, CTRL, 0xF, 0xF, true));
}
constexpr int kDppXor1 = 0xB1, kDppXor2 = 0x4E;  // quad_perm 1,0,3,2 and 2,3,0,1

// Wave-wide (max, first index) reduction: larger value wins, ties go to the
// smaller index.  Lanes with no candidate hold (-inf, INT_MAX).
__device__ inline void wave_argmax(float& v, int& idx) {
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
        float ov = wave_xor(v, o);
        int oi = wave_xor(idx, o);
        if (ov > v || (ov == v && oi < idx)) {
            v = ov;
            idx = oi;
        }
    }
}

}  // namespace fkv
