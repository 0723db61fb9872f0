// TurboQuant far tier for gfx950: handle construction and the compression
// kernels.
//
// Replaces the reference's TurboFoveatedHandle (csrc/foveated_attn.cpp:
// 280-491) and its Python compression (src/foveated_kv/turbo_quantize.py:
// 25-178).  The fused attention over a TurboQuant blob is attn_kernel<D,
// NQ, 1> in fkv_attn.hip; the record layout is described in fkv_attn.h.
#include <hip/hip_runtime.h>

#include <cmath>
#include <string>

#include "fkv_attn.h"
#include "fkv_common.h"

namespace fkv {

// ---------------------------------------------------------------------------
// compression (src/foveated_kv/turbo_quantize.py:25-91, 139-178), fp32
// ---------------------------------------------------------------------------
//
//   n = |k|; y = (k / max(n, 1e-8)) Pi^T; idx = [y >= b0] + [y >= b1] + [y >= b2]
//   r = k - n * (cb[idx] Pi); gamma = |r|; sign = (r S^T >= 0)
//
// Three D x D products per token, all on the matrix cores
// (v_mfma_f32_32x32x16_f16) at fp32 precision: every fp32 operand is split
// into fp16 hi + lo after a power-of-two scale that puts its row's (token's)
// largest value near 1,024 (256), so that lo keeps its 11 bits above fp16's
// subnormals: 22 bits of an element down to 2^-13 of its row's largest, an
// absolute 2^-35 of that below.  The keys are fp16 already; products of fp16
// values are exact and summed in fp32, and the lo products run first, while
// the sums are small.  lo x lo, at most 2^-22 of the product of its elements,
// is left out of the second and third product.  Fewer bits per operand than
// the fp32 FMA chains had, but a smaller error of a product: rms, over the
// norms of the vector and the row, 8.1e-9 against the chains' 1.8e-8 at D =
// 128, 1.1e-8 against 1.8e-8 at D = 64 (both modelled on the CPU).  A token
// with a rotated coordinate within 6e-8 of its norm of a boundary (1 in
// 6,000) takes its codes from 64-bit sums: twelve standard deviations of the
// error measured with the orthonormal Pi and the boundaries of
// get_turbo_constants; no bound, and not scaled for other matrices.  Against
// 64 bits over N(0, 1) keys with outlier channels, 20 x 262,112 tokens: no
// code and 62 signs off of 6.7e8 at D = 128 (59 and 121 with fp32 FMA
// chains), none and 36 of 3.4e8 at D = 64 (18 and 48).
// The matrix is the A operand (rows = output dims) and the tokens are the B
// operand (columns), so a lane's accumulators hold its own token's output
// dims 32 rb + 8 a + 4 (lane / 32) + b; every product's K slots are numbered
// in that order too, so one product's results are the next one's B operand
// without leaving the lane's registers.

typedef _Float16 fkv_h8 __attribute__((ext_vector_type(8)));
typedef float fkv_f16v __attribute__((ext_vector_type(16)));

constexpr int kTqTok = 128;  // tokens per workgroup of the key compressor (32 per wave)
constexpr float kTqRow = 1024.0f, kTqVec = 256.0f;  // the largest value of a matrix row / of a token's operand

// The key compressor's prepared constants: per product (Pi, Pi^T, S) the lo
// and the hi operand, [part][row block][K step][lane][8 halves]; the inverse
// row scales of the first two products (the second times the centroids'
// inverse scale); the boundaries ascending; the four centroids' hi, then
// their lo halves as byte tables (code c at bytes 2 (3 - c), 2 (3 - c) + 1).
__host__ __device__ constexpr size_t tq_op_bytes(int D) { return (size_t)4 * D * D; }
__host__ __device__ constexpr size_t tq_scale_section(int D) { return 3 * tq_op_bytes(D); }
__host__ __device__ constexpr size_t tq_const_section(int D) { return tq_scale_section(D) + (size_t)8 * D; }
__host__ __device__ constexpr size_t tq_prep_bytes(int D) { return tq_const_section(D) + 32; }

// Power of two that brings |x| <= m near 1, and its inverse.
__device__ inline float pow2_scale(float m, float& inv) {
    const int e = min((int)((__float_as_uint(m) >> 23) & 0xFF), 253);
    inv = e ? __uint_as_float((uint32_t)e << 23) : 0x1p-127f;
    return m < INFINITY ? __uint_as_float((uint32_t)(254 - e) << 23) : (inv = 1.0f);
}
__device__ inline void split_half(float x, uint16_t& hi, uint16_t& lo) {
    hi = f2h(x);
    lo = f2h(x - h2f(hi));
}

// Blocks 0 .. 3 D - 1: one output row of one product (64 threads); the last
// block: the scalar constants.
__global__ __launch_bounds__(kWave) void tq_prep_kernel(const float* __restrict__ Pi, const float* __restrict__ S,
                                                        const float* __restrict__ cb, const float* __restrict__ bd,
                                                        int D, uint8_t* __restrict__ prep) {
    const int lane = threadIdx.x;
    float* const scales = (float*)(prep + tq_scale_section(D));
    float cinv;
    const float cscale =
        pow2_scale(fmaxf(fmaxf(fabsf(cb[0]), fabsf(cb[1])), fmaxf(fabsf(cb[2]), fabsf(cb[3]))), cinv);
    if (blockIdx.x == 3 * D) {
        if (lane != 0) return;
        // ascending (the code counts the boundaries at or below y); NaN, which none reaches, last
        float b[3];
        for (int i = 0; i < 3; i++) b[i] = bd[i] == bd[i] ? bd[i] : INFINITY;
        for (int i : {0, 1, 0})
            if (b[i] > b[i + 1]) {
                const float t = b[i];
                b[i] = b[i + 1];
                b[i + 1] = t;
            }
        float* const c = (float*)(prep + tq_const_section(D));
        for (int i = 0; i < 3; i++) c[i] = b[i];
        for (int i = 0; i < 4; i++)  // entry 3 - code
            split_half(cb[3 - i] * cscale * kTqVec, ((uint16_t*)(c + 4))[i], ((uint16_t*)(c + 6))[i]);
        return;
    }
    const int op = blockIdx.x / D, i = blockIdx.x % D;
    auto at = [&](int j) { return op == 1 ? Pi[(int64_t)j * D + i] : (op ? S : Pi)[(int64_t)i * D + j]; };
    float m = 0.f;
    for (int j = lane; j < D; j += kWave) m = fmaxf(m, fabsf(at(j)));
    m = wave_max(m);
    float inv;
    const float scale = pow2_scale(m, inv);
    if (op < 2 && lane == 0) scales[op * D + i] = (op == 1 ? inv * cinv / kTqVec : inv) / kTqRow;
    uint16_t* const out = (uint16_t*)(prep + op * tq_op_bytes(D));
    for (int j = lane; j < D; j += kWave) {
        uint16_t hi, lo;
        split_half(at(j) * scale * kTqRow, hi, lo);
        // K step j / 16, lane half (j % 8) / 4, slot 4 ((j % 16) / 8) + j % 4
        const int64_t o = ((int64_t)((i / 32) * (D / 16) + j / 16) * 64 + (i % 32) + 32 * ((j % 8) / 4)) * 8 +
                          4 * ((j % 16) / 8) + j % 4;
        out[o] = lo;
        out[(int64_t)D * D + o] = hi;
    }
}

template <int D>
struct TqGemm {
    static constexpr int NB = D / 32, NS = D / 16;
    const uint8_t* op;  // the product's operands in LDS
    int lane;
    fkv_f16v acc[NB];
    __device__ inline void clear() {
#pragma unroll
        for (int rb = 0; rb < NB; rb++)
#pragma unroll
            for (int i = 0; i < 16; i++) acc[rb][i] = 0.f;
    }
    // acc += A_part B.  The next step's operands are read while this step's
    // are multiplied, and the address is opaque, so that no pass keeps
    // operands in registers for a later one (32 fragments of 4 VGPRs: spills).
    __device__ inline void add(int part, const fkv_h8 (&b)[NS]) {
        int o = part * (2 * D * D) + lane * 16;
        asm volatile("" : "+v"(o));
        const fkv_h8* f = (const fkv_h8*)(op + o);
        fkv_h8 cur[NB], nxt[NB];
#pragma unroll
        for (int rb = 0; rb < NB; rb++) cur[rb] = f[rb * NS * 64];
#pragma unroll
        for (int s = 0; s < NS; s++) {
#pragma unroll
            for (int rb = 0; rb < NB; rb++)
                if (s + 1 < NS) nxt[rb] = f[(rb * NS + s + 1) * 64];
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int rb = 0; rb < NB; rb++)
                acc[rb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(cur[rb], b[s], acc[rb], 0, 0, 0);
#pragma unroll
            for (int rb = 0; rb < NB; rb++) cur[rb] = nxt[rb];
        }
    }
    // fp32-precision product with the split operand hi + lo
    __device__ inline void split(const fkv_h8 (&hi)[NS], const fkv_h8 (&lo)[NS]) {
        clear();
        add(0, hi);
        add(1, lo);
        add(1, hi);
    }
};

// Sum of eight partial sums of this lane and of lane ^ 32 (the token's other dims).
__device__ inline float tq_half_sum(const float (&p)[8]) {
    const float s = ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
    return s + __shfl_xor(s, 32);
}

// fp16 bits of the centroids of two codes (given as 3 - code in the halves of
// c01, c23) from the byte tables: two per dword.
__device__ inline void centroids4(uint32_t t01, uint32_t t23, uint32_t c01, uint32_t c23, uint32_t& o01, uint32_t& o23) {
    o01 = __builtin_amdgcn_perm(t23, t01, ((c01 << 1) | (c01 << 9)) + 0x01000100u);
    o23 = __builtin_amdgcn_perm(t23, t01, ((c23 << 1) | (c23 << 9)) + 0x01000100u);
}

// Slots 4 u .. 4 u + 3 of an operand.
__device__ inline void put4(fkv_h8& o, int u, uint32_t w01, uint32_t w23) {
    const fkv_h2 x = as_h2(w01), y = as_h2(w23);
    o[4 * u] = x[0];
    o[4 * u + 1] = x[1];
    o[4 * u + 2] = y[0];
    o[4 * u + 3] = y[1];
}

// The codes of one token in 64 bits, by the whole wave: dim i's code from
// lane i % 64, returned as masks of the codes' low and high bits per 64 dims.
// For tokens with a rotated coordinate so near a boundary that the fp32-precision
// sums may fall on the wrong side of it (one token in 6,000).
template <int D, bool WIDE>
__device__ inline void exact_codes(const void* keys, int dtype, int64_t t, const float* __restrict__ Pi, const float* bd,
                                   int lane, uint64_t (&m0)[D / 64], uint64_t (&m1)[D / 64]) {
    float k[D / 64];
    double ss = 0.0, y[D / 64];
#pragma unroll
    for (int i = 0; i < D / 64; i++) {
        k[i] = h2f(load_as_f16(keys, t * D + 64 * i + lane, dtype));
        ss += (double)k[i] * (double)k[i];
        y[i] = 0.0;
    }
    for (int o = 32; o >= 1; o >>= 1) ss += __shfl_xor(ss, o);
    const double nc = fmax(sqrt(ss), (double)1e-8f);
    // matrix elements in flight per row (a lane reads along its own rows): the
    // wave waits for D / U of these round trips, and its workgroup for it
    constexpr int U = WIDE ? 32 : 8;
#pragma unroll
    for (int jj = 0; jj < D / 64; jj++)
#pragma unroll 1
        for (int j0 = 0; j0 < 64; j0 += U) {
            float m[D / 64][U];
#pragma unroll
            for (int i = 0; i < D / 64; i++) {
                const float* p = Pi + (int64_t)(64 * i + lane) * D + 64 * jj + j0;
#pragma unroll
                for (int u = 0; u < U; u += 4) {
                    if (WIDE) {
                        const float4 v = *(const float4*)(p + u);
                        m[i][u] = v.x;
                        m[i][u + 1] = v.y;
                        m[i][u + 2] = v.z;
                        m[i][u + 3] = v.w;
                    } else {
#pragma unroll
                        for (int e = 0; e < 4; e++) m[i][u + e] = p[u + e];
                    }
                }
            }
#pragma unroll
            for (int u = 0; u < U; u++) {
                const double kj = (double)__int_as_float(__builtin_amdgcn_readlane(__float_as_int(k[jj]), j0 + u));
#pragma unroll
                for (int i = 0; i < D / 64; i++) y[i] = fma(kj, (double)m[i][u], y[i]);
            }
        }
#pragma unroll
    for (int i = 0; i < D / 64; i++) {
        const double v = y[i] / nc;
        const int c = (v >= (double)bd[0]) + (v >= (double)bd[1]) + (v >= (double)bd[2]);
        m0[i] = __ballot(c & 1);
        m1[i] = __ballot(c & 2);
    }
}

// One workgroup of four waves per 128 tokens, two workgroups per CU (64 KB of
// LDS each at D = 128): one's vector work overlaps the other's matrix work.
// Each product's operands come to LDS by LDS DMA once the previous product
// is done with them, while its results are turned into codes, residuals or
// signs.  WIDE: keys, Pi and code buffers 16-byte aligned (else element loads
// and byte stores).  Bound by issue: per 32 tokens of a wave 256 MFMAs (27 us
// over 262K tokens at D = 128) and 2,200 vector instructions (29 us), and the
// LDS reads of the operands (27 us).  4 x 8 heads x 8,191 tokens: 869 us with
// fp32 FMA chains (30 TFLOP/s), 84 us now: 78 without the test for close
// coordinates, 81 without the few 64-bit ones, whose wave its workgroup and
// at the end the launch wait for.
template <int D, bool WIDE>
__global__ __launch_bounds__(256, 2) void tq_compress_keys_kernel(const void* __restrict__ keys, int dtype, int64_t n_tok,
                                                                  const uint8_t* __restrict__ prep,
                                                                  const float* __restrict__ Pi,
                                                                  uint8_t* __restrict__ out_idx,
                                                                  uint8_t* __restrict__ out_sgn,
                                                                  uint16_t* __restrict__ out_norm,
                                                                  uint16_t* __restrict__ out_gamma) {
    constexpr int NB = D / 32, NS = D / 16;
    __shared__ __attribute__((aligned(16))) uint8_t op_s[tq_op_bytes(D)];
    __shared__ __attribute__((aligned(16))) float sc_s[2 * D];
    const int tid = threadIdx.x, lane = tid % kWave, wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int h = lane >> 5;
    const uint32_t upper = h ? ~0u : 0u;  // selects by mask (a select between array elements became an indexed access)
    const int64_t t = (int64_t)blockIdx.x * kTqTok + wave * 32 + (lane & 31);
    const bool live = t < n_tok;
    auto fetch = [&](int op) __attribute__((always_inline)) {
        constexpr int CH = (int)tq_op_bytes(D) / 1024 / 4;  // 1-KB chunks per wave
#pragma unroll
        for (int c = 0; c < CH; c++) {
            const size_t o = (size_t)(wave * CH + c) * 1024;
            __builtin_amdgcn_global_load_lds((const void*)(prep + op * tq_op_bytes(D) + o + lane * 16),
                                             (__attribute__((address_space(3))) void*)(op_s + o), 16, 0, 0);
        }
    };
    auto ready = [&]() __attribute__((always_inline)) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
    };
    fetch(0);
    for (int i = tid; i < 2 * D; i += 256) sc_s[i] = ((const float*)(prep + tq_scale_section(D)))[i];
    const float* const cst = (const float*)(prep + tq_const_section(D));
    float b0 = cst[0], b1 = cst[1], b2 = cst[2];
    const uint32_t* const tab = (const uint32_t*)cst + 4;
    const uint32_t hi01 = tab[0], hi23 = tab[1], lo01 = tab[2], lo23 = tab[3];
    // the token's keys as the B operand: slots 0..3 of step s are dims 16 s +
    // 4 h .., slots 4..7 dims 16 s + 8 + 4 h ..
    fkv_h8 kb[NS];
    if (WIDE && dtype != FKV_F32) {
        // lane half h loads dims 16 s + 8 h .. + 7; the halves then exchange
        // their outer four dims
#pragma unroll
        for (int s = 0; s < NS; s++) {
            uint4 w = make_uint4(0, 0, 0, 0);
            if (live) w = *(const uint4*)((const uint16_t*)keys + t * D + 16 * s + 8 * h);
            if (dtype == FKV_BF16) {
                auto two = [](uint32_t u) {
                    return (uint32_t)f2h(__uint_as_float(u << 16)) |
                           ((uint32_t)f2h(__uint_as_float(u & 0xFFFF0000u)) << 16);
                };
                w = make_uint4(two(w.x), two(w.y), two(w.z), two(w.w));
            }
            // given to the other half: h = 0 its dims 4..7, h = 1 its dims 8..11
            const uint32_t g0 = __shfl_xor(h ? w.x : w.z, 32), g1 = __shfl_xor(h ? w.y : w.w, 32);
            const uint4 o = h ? make_uint4(g0, g1, w.z, w.w) : make_uint4(w.x, w.y, g0, g1);
            kb[s] = __builtin_bit_cast(fkv_h8, o);
        }
    } else if (WIDE) {
#pragma unroll
        for (int s = 0; s < NS; s++) {
            float4 x = make_float4(0.f, 0.f, 0.f, 0.f), y = x;
            if (live) {
                x = *(const float4*)((const float*)keys + t * D + 16 * s + 4 * h);
                y = *(const float4*)((const float*)keys + t * D + 16 * s + 8 + 4 * h);
            }
            kb[s] = fkv_h8{(_Float16)x.x, (_Float16)x.y, (_Float16)x.z, (_Float16)x.w,
                           (_Float16)y.x, (_Float16)y.y, (_Float16)y.z, (_Float16)y.w};
        }
    } else {
#pragma unroll
        for (int s = 0; s < NS; s++)
#pragma unroll
            for (int e = 0; e < 8; e++)
                kb[s][e] = live ? __builtin_bit_cast(_Float16, load_as_f16(keys, t * D + 16 * s + 8 * (e / 4) + 4 * h + e % 4,
                                                                           dtype))
                                : (_Float16)0.f;
    }
    // eight partial sums, added pairwise: the norm's rounding moves every boundary
    float ss[8] = {};
#pragma unroll
    for (int s = 0; s < NS; s++)
#pragma unroll
        for (int e = 0; e < 8; e++) ss[e] = fmaf((float)kb[s][e], (float)kb[s][e], ss[e]);
    const float norm = sqrtf(tq_half_sum(ss));
    // Keys of a small norm times 2^14 (exact; everything below scales with
    // them): products of fp16 subnormals would be summed with fewer bits (keys
    // of standard deviation 2^-22, 400,000 tokens of 128: 85 codes off 64 bits).
    const bool tiny = norm < 0x1p-6f;
    float nrm = norm, nc = fmaxf(norm, 1e-8f);
    if (__ballot(tiny)) {
        const float up = tiny ? 0x1p14f : 1.0f;
#pragma unroll
        for (int s = 0; s < NS; s++) kb[s] *= (_Float16)up;
        nrm *= up;
        nc *= up;
    }
    // y >= b  <=>  k Pi^T >= b max(n, 1e-8)
    b0 *= nc;
    b1 *= nc;
    b2 *= nc;
    TqGemm<D> g{op_s, lane, {}};
    // ---- codes ----
    ready();
    g.clear();
    g.add(0, kb);
    g.add(1, kb);
    __syncthreads();  // every wave is done with the operands
    fetch(1);
    fkv_h8 hi[NS], lo[NS];
    uint32_t w[NB];
    float gap = INFINITY;  // the least distance of a coordinate from a boundary
#pragma unroll
    for (int rb = 0; rb < NB; rb++) {
        w[rb] = 0;
#pragma unroll
        for (int a = 0; a < 4; a++) {
            const float4 sc = *(const float4*)&sc_s[32 * rb + 8 * a + 4 * h];
            const float f[4] = {sc.x, sc.y, sc.z, sc.w};
            uint32_t c[4];
#pragma unroll
            for (int b = 0; b < 4; b++) {
                // the boundaries above the coordinate: 3 - code.  The signs of
                // the differences are exact (f is a power of two), and a zero
                // one is positive; compares would leave lane masks to spill
                const float y = g.acc[rb][4 * a + b];
                const float d0 = fmaf(y, f[b], -b0), d1 = fmaf(y, f[b], -b1), d2 = fmaf(y, f[b], -b2);
                c[b] = (__float_as_uint(d0) >> 31) + (__float_as_uint(d1) >> 31) + (__float_as_uint(d2) >> 31);
                gap = fminf(fminf(fminf(fabsf(d0), fabsf(d1)), fabsf(d2)), gap);
                w[rb] |= c[b] << (8 * a + 2 * b);
            }
            // the centroids' halves, two codes at a time
            uint32_t h01, h23, l01, l23;
            centroids4(hi01, hi23, c[0] | (c[1] << 16), c[2] | (c[3] << 16), h01, h23);
            centroids4(lo01, lo23, c[0] | (c[1] << 16), c[2] | (c[3] << 16), l01, l23);
            put4(hi[2 * rb + a / 2], a % 2, h01, h23);
            put4(lo[2 * rb + a / 2], a % 2, l01, l23);
        }
        w[rb] = ~w[rb];  // the codes
    }
    // tokens with a coordinate within twelve standard deviations of the sums'
    // error (5e-9 of the norm for an orthonormal Pi) take their codes from 64-bit sums
    const uint64_t close = __ballot(live && nrm > 0.f && nrm < INFINITY && gap < 6e-8f * nrm);
    const bool odd_norm = !(nrm < INFINITY);
    uint32_t redo = (uint32_t)close | (uint32_t)(close >> 32);
    if (redo || __ballot(odd_norm)) {
        while (redo) {
            const int tl = __builtin_ctz(redo);
            redo &= redo - 1;
            uint64_t m0[D / 64], m1[D / 64];
            exact_codes<D, WIDE>(keys, dtype, (int64_t)blockIdx.x * kTqTok + wave * 32 + tl, Pi, cst, lane, m0, m1);
            if ((lane & 31) == tl) {
#pragma unroll
                for (int rb = 0; rb < NB; rb++) {
                    w[rb] = 0;
#pragma unroll
                    for (int a = 0; a < 4; a++) {
                        // four low and four high bits interleaved
                        const int at = (32 * rb + 8 * a) % 64 + 4 * h;
                        uint32_t x = (uint32_t)(m0[rb / 2] >> at) & 15u, z = (uint32_t)(m1[rb / 2] >> at) & 15u;
                        x = (x | (x << 2)) & 0x33u;
                        x = (x | (x << 1)) & 0x55u;
                        z = (z | (z << 2)) & 0x33u;
                        z = (z | (z << 1)) & 0x55u;
                        w[rb] |= (x | (z << 1)) << (8 * a);
                    }
                }
            }
        }
#pragma unroll
        for (int rb = 0; rb < NB; rb++) {
            if (odd_norm) w[rb] = 0;  // no code of a non-finite norm
#pragma unroll
            for (int a = 0; a < 4; a++) {
                const uint32_t q = ~w[rb] >> (8 * a);
                const uint32_t c01 = (q & 3u) | ((q & 12u) << 14), c23 = ((q >> 4) & 3u) | ((q & 192u) << 10);
                uint32_t h01, h23, l01, l23;
                centroids4(hi01, hi23, c01, c23, h01, h23);
                centroids4(lo01, lo23, c01, c23, l01, l23);
                put4(hi[2 * rb + a / 2], a % 2, h01, h23);
                put4(lo[2 * rb + a / 2], a % 2, l01, l23);
            }
        }
    }
    // byte 8 rb + 2 a + h of the token's codes: dword pairs interleave the halves' bytes
    uint32_t ix[2 * NB];
#pragma unroll
    for (int rb = 0; rb < NB; rb++) {
        const uint32_t o = __shfl_xor(w[rb], 32), w0 = h ? o : w[rb], w1 = h ? w[rb] : o;
        ix[2 * rb] = __builtin_amdgcn_perm(w1, w0, 0x05010400u);
        ix[2 * rb + 1] = __builtin_amdgcn_perm(w1, w0, 0x07030602u);
    }
    if (live) {
        uint8_t* const dst = out_idx + t * (D / 4) + h * (D / 8);  // each half writes half the token's bytes
        uint32_t mine[NB];
#pragma unroll
        for (int i = 0; i < NB; i++) mine[i] = (ix[i] & ~upper) | (ix[NB + i] & upper);
        if (WIDE) {
            if constexpr (NB == 4) *(uint4*)dst = make_uint4(mine[0], mine[1], mine[2], mine[3]);
            else *(uint2*)dst = make_uint2(mine[0], mine[1]);
        } else {
#pragma unroll
            for (int i = 0; i < 4 * NB; i++) dst[i] = (uint8_t)(mine[i / 4] >> (8 * (i % 4)));
        }
    }
    // ---- residual ----
    ready();
    g.split(hi, lo);
    __syncthreads();
    fetch(2);
#pragma unroll
    for (int e = 0; e < 8; e++) ss[e] = 0.f;
#pragma unroll
    for (int rb = 0; rb < NB; rb++)
#pragma unroll
        for (int a = 0; a < 4; a++) {
            const float4 sc = *(const float4*)&sc_s[D + 32 * rb + 8 * a + 4 * h];
            const float f[4] = {sc.x, sc.y, sc.z, sc.w};
#pragma unroll
            for (int b = 0; b < 4; b++) {
                const int s = 2 * rb + a / 2, e = 4 * (a % 2) + b;
                const float r = fmaf(-nrm, g.acc[rb][4 * a + b] * f[b], (float)kb[s][e]);
                g.acc[rb][4 * a + b] = r;
                ss[e] = fmaf(r, r, ss[e]);
            }
        }
    const float gamma = sqrtf(tq_half_sum(ss));
    if (live && h == 0) {
        out_norm[t] = f2h(norm);
        out_gamma[t] = f2h(tiny ? gamma * 0x1p-14f : gamma);
    }
    // the residual scaled so that its largest value is at most 512 (only the
    // sign of its projections is kept); a non-finite one gives no sign
    const int ge = (int)((__float_as_uint(gamma) >> 23) & 0xFF);
    const float rs = gamma < INFINITY ? __uint_as_float((uint32_t)(254 - min(ge, 253)) << 23) * (ge ? kTqVec : 1.0f) : 0.f;
#pragma unroll
    for (int rb = 0; rb < NB; rb++)
#pragma unroll
        for (int i = 0; i < 16; i++) {
            uint16_t vh, vl;
            split_half(g.acc[rb][i] * rs, vh, vl);
            hi[2 * rb + i / 8][i % 8] = __builtin_bit_cast(_Float16, vh);
            lo[2 * rb + i / 8][i % 8] = __builtin_bit_cast(_Float16, vl);
        }
    // ---- signs ----
    ready();
    g.split(hi, lo);
#pragma unroll
    for (int rb = 0; rb < NB; rb++) {
        w[rb] = 0;
#pragma unroll
        for (int i = 0; i < 16; i++) w[rb] |= (g.acc[rb][i] >= 0.f ? 1u : 0u) << (8 * (i / 4) + i % 4);
        w[rb] <<= 4 * h;
        w[rb] |= __shfl_xor(w[rb], 32);
    }
    if (live) {
        uint8_t* const dst = out_sgn + t * (D / 8) + h * (D / 16);
        uint32_t mine[NB / 2];
#pragma unroll
        for (int i = 0; i < NB / 2; i++) mine[i] = (w[i] & ~upper) | (w[NB / 2 + i] & upper);
        if (WIDE) {
            if constexpr (NB == 4) *(uint2*)dst = make_uint2(mine[0], mine[1]);
            else *(uint32_t*)dst = mine[0];
        } else {
#pragma unroll
            for (int i = 0; i < 2 * NB; i++) dst[i] = (uint8_t)(mine[i / 4] >> (8 * (i % 4)));
        }
    }
}


// Four lanes per (token, 32-dim group), 8 values each: scale = max(max|v|,
// 1e-8), code = clip(rint((v / scale + 1) * 1.5), 0, 3) (round half to even,
// as mx.round).  Bound by the one read of the values: 16-byte loads
// (WIDE: values 16-byte aligned; else element loads) and contiguous 2-byte
// stores; one thread per group with element loads 64 bytes apart took 70 us
// for 4 x 8 heads x 8,191 tokens of 128, 18 us now.  The quotient needs one
// division per group: one correction step of v * (1 / scale) is the IEEE
// quotient for every pair of fp16 values |v| <= scale (all pairs checked;
// an infinite scale takes the product, 0 or NaN as the division gives).
template <bool WIDE>
__global__ __launch_bounds__(256) void tq_compress_values_kernel(const void* __restrict__ vals, int dtype,
                                                                 int64_t n_groups, uint8_t* __restrict__ out_packed,
                                                                 uint16_t* __restrict__ out_scale) {
    const int64_t n = n_groups * 4;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        uint32_t w[4];
        if (WIDE) {
            const uint4 x = load8(vals, dtype, i * 8);
            w[0] = x.x;
            w[1] = x.y;
            w[2] = x.z;
            w[3] = x.w;
        } else {
#pragma unroll
            for (int k = 0; k < 4; k++)
                w[k] = (uint32_t)load_as_f16(vals, i * 8 + 2 * k, dtype) |
                       ((uint32_t)load_as_f16(vals, i * 8 + 2 * k + 1, dtype) << 16);
        }
        float v[8], mx = 0.f;
#pragma unroll
        for (int k = 0; k < 8; k++) {
            v[k] = h2f((uint16_t)(w[k / 2] >> (16 * (k & 1))));
            mx = fmaxf(mx, fabsf(v[k]));
        }
        mx = fmaxf(mx, dpp_f32<kDppXor1>(mx));  // n is a multiple of 4: the group's lanes are here
        mx = fmaxf(mx, dpp_f32<kDppXor2>(mx));
        const float sc = fmaxf(mx, 1e-8f), rsc = 1.0f / sc;
        uint32_t c = 0;
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const float q = sc < INFINITY ? div_by<1>(v[k], sc, rsc) : v[k] * rsc;
            const float r = fminf(fmaxf(rintf((q + 1.0f) * 1.5f), 0.f), 3.f);
            c |= (uint32_t)r << (2 * k);
        }
        ((uint16_t*)out_packed)[i] = (uint16_t)c;
        if (i % 4 == 0) out_scale[i / 4] = f2h(sc);
    }
}

}  // namespace fkv

using fkv::check_hip;
using fkv::set_error;

namespace {

int turbo_create(const char* fn, fkv_attn** out, int32_t B, int32_t Hkv, int32_t D, int32_t Na, int32_t F,
                     const void* near_k, const void* near_v, int32_t near_dtype, const uint8_t* k_idx,
                     const uint8_t* k_signs, const void* k_norm, const void* k_gamma, const uint8_t* v_packed,
                     const void* v_scale, int32_t nz_dtype, const int32_t* near_valid, const float* Pi,
                     const float* S, const float* centroids, float spike_margin, void* blob, int64_t blob_bytes,
                 void* stream) {
    const std::string name(fn);
    if (!out) return set_error(name + ": out is NULL");
    *out = nullptr;
    if (B <= 0 || Hkv <= 0 || Na < 0 || F < 0)
        return set_error(name + ": bad shape B=" + std::to_string(B) + " Hkv=" + std::to_string(Hkv) +
                         " Na=" + std::to_string(Na) + " F=" + std::to_string(F));
    if (D != 64 && D != 128) return set_error(name + ": head dim must be 64 or 128, got " + std::to_string(D));
    if (near_dtype < FKV_F16 || near_dtype > FKV_F32 || nz_dtype < FKV_F16 || nz_dtype > FKV_F32)
        return set_error(name + ": unsupported dtype");
    if ((Na > 0 && (!near_k || !near_v)) ||
        (F > 0 && (!k_idx || !k_signs || !k_norm || !k_gamma || !v_packed || !v_scale)) || !near_valid || !Pi ||
        !S || !centroids)
        return set_error(name + ": NULL array");
    hipStream_t st = (hipStream_t)stream;
    fkv_attn* h = new fkv_attn();
    fkv::PackSrc src{};
    src.near_k = near_k;
    src.near_v = near_v;
    src.near_dtype = near_dtype;
    src.near_valid = near_valid;
    src.k_idx = k_idx;
    src.k_signs = k_signs;
    src.k_norm = k_norm;
    src.k_gamma = k_gamma;
    src.v_packed = v_packed;
    src.v_scale = v_scale;
    src.nz_dtype = nz_dtype;
    src.Pi = Pi;
    src.S = S;
    int rc = fkv::attn_begin(fn, h, B, Hkv, D, Na, F, 1, src, spike_margin, blob, blob_bytes, st);
    float cb[4] = {0.f, 0.f, 0.f, 0.f};
    if (!rc) rc = check_hip(hipMemcpyAsync(cb, centroids, sizeof(cb), hipMemcpyDeviceToHost, st), "hipMemcpyAsync");
    if (!rc) rc = fkv::attn_finish(fn, h, st);
    if (!rc) {
        h->tq.rot = (const uint16_t*)(h->blob + fkv::tq_rot_section(h->L));
        // centroid(c) = alpha + beta*sh + gamma*sl + delta*sh*sl, sh/sl = +-1 bits of c
        const double c0 = cb[0], c1 = cb[1], c2 = cb[2], c3 = cb[3];
        h->tq.alpha = (float)((c0 + c1 + c2 + c3) / 4);
        h->tq.beta = (float)((c2 + c3 - c0 - c1) / 4);
        h->tq.gamma = (float)((c1 + c3 - c0 - c2) / 4);
        h->tq.delta = (float)((c0 + c3 - c1 - c2) / 4);
        // value levels {-1, -0.333333, 0.333333, 1} (csrc/kernels/foveated_attn.metal:529)
        const double l0 = -1.0, l1 = (double)-0.333333f, l2 = (double)0.333333f, l3 = 1.0;
        h->tq.lvh = (float)((l2 + l3 - l0 - l1) / 4);
        h->tq.lvl = (float)((l1 + l3 - l0 - l2) / 4);
        // the kernel expands the high-bit value plane to +-2 against
        // weights scaled by lvl (one weight for both planes)
        if (std::fabs(h->tq.lvh - 2.0 * h->tq.lvl) > 2e-6 * h->tq.lvh)
            rc = fkv::set_error(name + ": value levels with lvh != 2 lvl (internal error)");
    }
    if (rc) {
        fkv_attn_destroy(h);
        return rc;
    }
    *out = h;
    return FKV_OK;
}

}  // namespace

extern "C" {

int fkv_turbo_create(fkv_attn** out, int32_t B, int32_t Hkv, int32_t D, int32_t Na, int32_t F,
                     const void* near_k, const void* near_v, int32_t near_dtype, const uint8_t* k_idx,
                     const uint8_t* k_signs, const void* k_norm, const void* k_gamma, const uint8_t* v_packed,
                     const void* v_scale, int32_t nz_dtype, const int32_t* near_valid, const float* Pi,
                     const float* S, const float* centroids, float spike_margin, void* stream) {
    return turbo_create("fkv_turbo_create", out, B, Hkv, D, Na, F, near_k, near_v, near_dtype, k_idx, k_signs, k_norm,
                        k_gamma, v_packed, v_scale, nz_dtype, near_valid, Pi, S, centroids, spike_margin, nullptr, 0,
                        stream);
}

int fkv_turbo_create_at(fkv_attn** out, int32_t B, int32_t Hkv, int32_t D, int32_t Na, int32_t F,
                        const void* near_k, const void* near_v, int32_t near_dtype, const uint8_t* k_idx,
                        const uint8_t* k_signs, const void* k_norm, const void* k_gamma, const uint8_t* v_packed,
                        const void* v_scale, int32_t nz_dtype, const int32_t* near_valid, const float* Pi,
                        const float* S, const float* centroids, float spike_margin, void* blob, int64_t blob_bytes,
                        void* stream) {
    if (!blob) return set_error("fkv_turbo_create_at: NULL blob");
    return turbo_create("fkv_turbo_create_at", out, B, Hkv, D, Na, F, near_k, near_v, near_dtype, k_idx, k_signs,
                        k_norm, k_gamma, v_packed, v_scale, nz_dtype, near_valid, Pi, S, centroids, spike_margin, blob,
                        blob_bytes, stream);
}

int fkv_turbo_compress_keys(const void* keys, int32_t dtype, int64_t n_tokens, int32_t D, const float* Pi,
                            const float* S, const float* centroids, const float* boundaries, uint8_t* out_idx,
                            uint8_t* out_signs, void* out_norm, void* out_gamma, void* stream) {
    if (D != 64 && D != 128) return set_error("fkv_turbo_compress_keys: head dim must be 64 or 128");
    if (dtype < FKV_F16 || dtype > FKV_F32) return set_error("fkv_turbo_compress_keys: unsupported dtype");
    if (n_tokens < 0) return set_error("fkv_turbo_compress_keys: negative token count");
    if (n_tokens == 0) return FKV_OK;
    if (!keys || !Pi || !S || !centroids || !boundaries || !out_idx || !out_signs || !out_norm || !out_gamma)
        return set_error("fkv_turbo_compress_keys: NULL argument");
    hipStream_t st = (hipStream_t)stream;
    // the constants' workspace is allocated and freed by each call, which a
    // captured graph could not replay
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    if (int rc = check_hip(hipStreamIsCapturing(st, &cs), "hipStreamIsCapturing")) return rc;
    if (cs != hipStreamCaptureStatusNone) return set_error("fkv_turbo_compress_keys: not under graph capture");
    uint8_t* prep = nullptr;
    int rc = check_hip(hipMallocAsync((void**)&prep, fkv::tq_prep_bytes(D), st), "hipMallocAsync");
    if (rc) return rc;
    hipLaunchKernelGGL(fkv::tq_prep_kernel, dim3((unsigned)(3 * D + 1)), dim3(fkv::kWave), 0, st, Pi, S, centroids,
                       boundaries, D, prep);
    // vector loads and stores where the caller's arrays are 16-byte aligned
    // (a token's rows then are too)
    const bool wide = (((uintptr_t)keys | (uintptr_t)Pi | (uintptr_t)out_idx | (uintptr_t)out_signs) & 15) == 0;
    auto* kern = D == 128 ? (wide ? fkv::tq_compress_keys_kernel<128, true> : fkv::tq_compress_keys_kernel<128, false>)
                          : (wide ? fkv::tq_compress_keys_kernel<64, true> : fkv::tq_compress_keys_kernel<64, false>);
    hipLaunchKernelGGL(kern, dim3((unsigned)fkv::cdiv(n_tokens, fkv::kTqTok)), dim3(256), 0, st, keys, dtype, n_tokens,
                       prep, Pi, out_idx, out_signs, (uint16_t*)out_norm, (uint16_t*)out_gamma);
    rc = check_hip(hipGetLastError(), "tq_compress_keys_kernel launch");
    (void)hipFreeAsync(prep, st);
    return rc;
}

int fkv_turbo_compress_values(const void* values, int32_t dtype, int64_t n_tokens, int32_t D, uint8_t* out_packed,
                              void* out_scale, void* stream) {
    if (D <= 0 || D % 32 != 0) return set_error("fkv_turbo_compress_values: head dim must be a multiple of 32");
    if (dtype < FKV_F16 || dtype > FKV_F32) return set_error("fkv_turbo_compress_values: unsupported dtype");
    if (n_tokens < 0) return set_error("fkv_turbo_compress_values: negative token count");
    if (n_tokens == 0) return FKV_OK;
    if (!values || !out_packed || !out_scale) return set_error("fkv_turbo_compress_values: NULL argument");
    const int64_t ng = n_tokens * (D / 32);
    auto* kern = ((uintptr_t)values & 15) == 0 ? fkv::tq_compress_values_kernel<true>
                                               : fkv::tq_compress_values_kernel<false>;
    hipLaunchKernelGGL(kern, dim3(fkv::grid_for(4 * ng, 256)), dim3(256), 0, (hipStream_t)stream, values, dtype, ng,
                       out_packed, (uint16_t*)out_scale);
    return check_hip(hipGetLastError(), "tq_compress_values_kernel launch");
}

}  // extern "C"
