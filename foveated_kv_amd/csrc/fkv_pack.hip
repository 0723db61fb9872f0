// Blob packing for gfx950: a layer's tiers, as the compress kernels write
// them, into the attention kernel's operand layouts (fkv_attn.h).  Runs once
// per handle (csrc/foveated_attn.cpp:83-128, 297-345 of the reference).
//
// Two launches per handle: pack_header_kernel (near_valid, key scales, the
// bad-code flag, TurboQuant's rotation operands) and pack_blob_kernel, one
// workgroup per 64-token tile of the near or the far tier.  Every byte of
// every tile is written, padding tokens as zeros, so the blob needs no
// clearing.  Bound by memory: all operand layouts are transpositions inside
// a tile, done on 16-byte units or in registers, with wide loads and stores
// on both sides (element loads, one thread per 16 elements, took 129 us for
// 4 x 8 heads x 8,192 tokens at D = 128 and a clear of the blob 12 us more;
// 33 us now, 159 MB in and out).  WIDE: every source array 16-byte aligned; else the same
// units are put together from element loads.
#include <hip/hip_runtime.h>

#include "fkv_attn.h"
#include "fkv_common.h"

namespace fkv {

namespace {

constexpr int kPackThreads = 256;

__global__ void pack_header_kernel(PackSrc s, BlobLayout L, uint8_t* __restrict__ blob) {
    const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i < L.Hkv) {
        const int v = s.near_valid[i];
        ((uint32_t*)(blob + L.near_valid))[i] = (uint32_t)(v < 0 ? 0 : (v > L.Na ? L.Na : v));
    }
    if (i == L.Hkv) ((uint32_t*)(blob + L.near_valid))[i] = 0;  // bad far codes found
    if (i < (int64_t)L.B * L.Hkv) ((float*)(blob + L.kscale))[i] = 1.0f;
    const int64_t DD = (int64_t)L.D * L.D;
    if (L.fmt == 1 && i < 2 * DD) {
        // Pi and S -> the query rotation's fp16 operands
        const int mat = (int)(i / DD), r = (int)(i / L.D % L.D), c = (int)(i % L.D);
        ((uint16_t*)(blob + tq_rot_section(L)))[tq_rot_index(L.D, mat, r, c)] = f2h((mat ? s.S : s.Pi)[(int64_t)r * L.D + c]);
    }
}

// 16 bytes from any address / from a 16-byte aligned one.
template <bool WIDE>
__device__ inline uint4 load16(const uint8_t* p) {
    if (WIDE) return *(const uint4*)p;
    uint32_t w[4] = {0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < 16; i++) w[i / 4] |= (uint32_t)p[i] << (8 * (i % 4));
    return make_uint4(w[0], w[1], w[2], w[3]);
}
template <bool WIDE>
__device__ inline uint32_t load4(const uint8_t* p) {
    if (WIDE) return *(const uint32_t*)p;
    return p[0] | ((uint32_t)p[1] << 8) | ((uint32_t)p[2] << 16) | ((uint32_t)p[3] << 24);
}
// Elements e, e + 1 / e .. e + 7 as packed fp16.
template <bool WIDE>
__device__ inline uint32_t load_h2(const void* p, int dtype, int64_t e) {
    if (WIDE && dtype == FKV_F16) return *(const uint32_t*)((const uint16_t*)p + e);
    if (WIDE && dtype == FKV_F32) {
        const float2 x = *(const float2*)((const float*)p + e);
        return (uint32_t)f2h(x.x) | ((uint32_t)f2h(x.y) << 16);
    }
    return (uint32_t)load_as_f16(p, e, dtype) | ((uint32_t)load_as_f16(p, e + 1, dtype) << 16);
}
template <bool WIDE>
__device__ inline uint4 load_h8(const void* p, int dtype, int64_t e) {
    if (WIDE) return load8(p, dtype, e);
    return make_uint4(load_h2<false>(p, dtype, e), load_h2<false>(p, dtype, e + 2), load_h2<false>(p, dtype, e + 4),
                      load_h2<false>(p, dtype, e + 6));
}

// Near tile: K 16-byte units (8 dims of a token) from token-major to
// chunk-major; V units of 8 tokens x 2 dims transposed in registers.
template <int D, bool WIDE>
__device__ inline void pack_near_tile(const PackSrc& s, const BlobLayout& L, uint8_t* blob, int64_t bkv, int tile) {
    constexpr int KU = D / 8 * 64 / kPackThreads, VU = D / 2 * 8 / kPackThreads;  // units per thread
    const int tid = threadIdx.x;
    const int t0 = tile * kTile;
    const int64_t src = (bkv * L.Na + t0) * D;
    const int64_t dst = (bkv * L.Na_pad + t0) * D * 2;  // bytes
    const uint4 zero = make_uint4(0, 0, 0, 0);
    uint4 kw[KU];
#pragma unroll
    for (int u = 0; u < KU; u++) {
        const int i = u * kPackThreads + tid, c = i / 64, t = i % 64;  // lanes = tokens: contiguous stores
        kw[u] = t0 + t < L.Na ? load_h8<WIDE>(s.near_k, s.near_dtype, src + (int64_t)t * D + 8 * c) : zero;
    }
    uint32_t vw[VU][8];
#pragma unroll
    for (int u = 0; u < VU; u++) {
        const int i = u * kPackThreads + tid, g = i / (D / 2), d = 2 * (i % (D / 2));  // tokens 8 g .., dims d, d + 1
#pragma unroll
        for (int e = 0; e < 8; e++)
            vw[u][e] = t0 + 8 * g + e < L.Na ? load_h2<WIDE>(s.near_v, s.near_dtype, src + (int64_t)(8 * g + e) * D + d)
                                             : 0u;
    }
#pragma unroll
    for (int u = 0; u < KU; u++) *(uint4*)(blob + L.near_k + dst + (int64_t)(u * kPackThreads + tid) * 16) = kw[u];
#pragma unroll
    for (int u = 0; u < VU; u++) {
        const int i = u * kPackThreads + tid, g = i / (D / 2), d = 2 * (i % (D / 2));
        uint32_t lo[4], hi[4];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            lo[e] = __builtin_amdgcn_perm(vw[u][2 * e + 1], vw[u][2 * e], 0x05040100u);
            hi[e] = __builtin_amdgcn_perm(vw[u][2 * e + 1], vw[u][2 * e], 0x07060302u);
        }
        uint4* o = (uint4*)(blob + L.near_v + dst + near_v_index(8 * g, d, D) * 2);
        o[0] = make_uint4(lo[0], lo[1], lo[2], lo[3]);
        o[1] = make_uint4(hi[0], hi[1], hi[2], hi[3]);  // dim d + 1: the next 16 bytes
    }
}

// Eight dwords of eight nibbles: out[j] = nibble j of every in[m] at nibble m.
__device__ inline void transpose_nibbles(uint32_t (&x)[8]) {
#pragma unroll
    for (int i = 0; i < 8; i += 2) {
        const uint32_t a = x[i], b = x[i + 1];
        x[i] = (a & 0x0F0F0F0Fu) | ((b & 0x0F0F0F0Fu) << 4);
        x[i + 1] = ((a >> 4) & 0x0F0F0F0Fu) | (b & 0xF0F0F0F0u);
    }
#pragma unroll
    for (int i = 0; i < 8; i++)
        if (!(i & 2)) {
            const uint32_t a = x[i], b = x[i + 2];
            x[i] = __builtin_amdgcn_perm(b, a, 0x06020400u);
            x[i + 2] = __builtin_amdgcn_perm(b, a, 0x07030501u);
        }
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const uint32_t a = x[i], b = x[i + 4];
        x[i] = __builtin_amdgcn_perm(b, a, 0x05040100u);
        x[i + 4] = __builtin_amdgcn_perm(b, a, 0x07060302u);
    }
}

// fp8 K / INT4 V far record (fmt 0: per-token, fmt 2: group-32 values).
// K: 16-byte units (16 codes of a token) from token-major to chunk-major;
// exponent-0 codes become signed zeros (the reference LUT ignores their
// mantissa), the NaN codes 0x7F / 0xFF are reported.  V: a unit is 8 tokens
// x 8 dims of nibbles, transposed in registers and put in place in LDS.
template <int D, int FMT, bool WIDE>
__device__ inline void pack_far_tile(const PackSrc& s, const BlobLayout& L, uint8_t* blob, int64_t bkv, int tile) {
    constexpr int KU = D / 16 * 64 / kPackThreads;
    constexpr int VN = D / 8 * 8;  // V units (at most kPackThreads)
    __shared__ __attribute__((aligned(16))) uint32_t v_s[8 * D];
    const int tid = threadIdx.x;
    const int t0 = tile * kTile;
    uint8_t* const rec = blob + L.far + far_rec_index(L, bkv, tile) * (int64_t)L.far_rec;
    uint4 kw[KU];
#pragma unroll
    for (int u = 0; u < KU; u++) {
        const int i = u * kPackThreads + tid, c = i / 64, t = t0 + i % 64;
        kw[u] = t < L.F ? load16<WIDE>(s.far_k + (bkv * L.F + t) * D + 16 * c) : make_uint4(0, 0, 0, 0);
    }
    // tokens of a unit in the nibble order of a dword: 0 2 4 6 1 3 5 7
    constexpr int order[8] = {0, 2, 4, 6, 1, 3, 5, 7};
    const int g = tid / (D / 8), dg = tid % (D / 8);  // tokens 8 g .., dims 8 dg ..
    uint32_t x[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    if (tid < VN) {
#pragma unroll
        for (int m = 0; m < 8; m++) {
            const int t = t0 + 8 * g + order[m];
            if (t < L.F) x[m] = load4<WIDE>(s.far_v + (bkv * L.F + t) * (D / 2) + 4 * dg);
        }
    }
    constexpr int NG = FMT == 2 ? D / 32 : 1;  // scale / zero pairs of a token
    uint32_t sz = 0;
    if (tid < 64 * NG && t0 + tid / NG < L.F) {
        const int64_t k = (bkv * L.F + t0) * NG + tid;
        sz = (uint32_t)load_as_f16(s.far_v_scale, k, s.sz_dtype) | ((uint32_t)load_as_f16(s.far_v_zero, k, s.sz_dtype) << 16);
    }
    bool bad = false;
#pragma unroll
    for (int u = 0; u < KU; u++) {
        uint32_t w[4] = {kw[u].x, kw[u].y, kw[u].z, kw[u].w};
#pragma unroll
        for (int i = 0; i < 4; i++) {
            bad |= (((w[i] & 0x7F7F7F7Fu) + 0x01010101u) & 0x80808080u) != 0;
            const uint32_t nz = ((w[i] & 0x78787878u) + 0x78787878u) & 0x80808080u;  // exponent not 0
            w[i] &= (nz - (nz >> 7)) | 0x80808080u;
        }
        *(uint4*)(rec + (int64_t)(u * kPackThreads + tid) * 16) = make_uint4(w[0], w[1], w[2], w[3]);
    }
    if (__ballot(bad) && (tid % kWave) == 0) atomicOr((unsigned*)(blob + L.near_valid) + L.Hkv, 1u);
    if (tid < VN) {
        transpose_nibbles(x);
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const int d = 8 * dg + j, dh = d / 64, l = d % 64;
            const int chunk = FMT == 2 ? 2 * dh + ((l >> 5) ^ (g >> 2)) : 2 * dh + (g >> 2);
            v_s[chunk * 256 + l * 4 + (g & 3)] = x[j];
        }
    }
    if (tid < 64 * NG) ((uint32_t*)(rec + (FMT == 2 ? g32_sz_section(D) : far_sz_section(D))))[tid] = sz;
    __syncthreads();
#pragma unroll
    for (int i = tid; i < 2 * D; i += kPackThreads) ((uint4*)(rec + far_v_section(D)))[i] = ((const uint4*)v_s)[i];
}

// Bits 4 i + r of a dword, i = 0..7, in the low byte.
__device__ inline uint32_t every_4th(uint32_t w, int r) {
    uint32_t x = (w >> r) & 0x11111111u;
    x = (x | (x >> 3)) & 0x03030303u;
    x = (x | (x >> 6)) & 0x000F000Fu;
    return (x | (x >> 12)) & 0xFFu;
}

// TurboQuant far record.  Key planes: one dword of a token's 32 dims per
// thread; the codes' bits are reversed as a whole and picked apart by
// residue.  Value planes: a lane holds 32 dims' codes of the token whose bit
// position is its lane, so a ballot per dim and plane is the dim's dword pair.
template <int D, bool WIDE>
__device__ inline void pack_tq_tile(const PackSrc& s, const BlobLayout& L, uint8_t* blob, int64_t bkv, int tile) {
    constexpr int NK = D / 32, NG = D / 32;
    const int tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
    const int t0 = tile * kTile;
    uint8_t* const rec = blob + L.far + far_rec_index(L, bkv, tile) * (int64_t)L.far_rec;
    // value codes: wave w < NG takes dims 32 w ..; lane l's token of its half
    // sits at bit l % 32 of the half's dword: 2 i at 15 - i, 2 i + 1 at 31 - i
    const int b = lane % 32, vt = t0 + (lane & 32) + (b < 16 ? 2 * (15 - b) : 2 * (31 - b) + 1);
    const bool vin = vt < L.F;
    uint32_t v0 = ~0u, v1 = ~0u;  // padding tokens: code 3
    if (wave < NG && vin) {
        const uint8_t* p = s.v_packed + (bkv * L.F + vt) * (D / 4) + 8 * wave;
        v0 = load4<WIDE>(p);
        v1 = load4<WIDE>(p + 4);
    }
    const int kt = tid / NK, k = tid % NK;  // token, dword
    uint32_t c0 = ~0u, c1 = ~0u, sg = ~0u, ng = 0, sc = 0;
    const bool kin = kt < 64 && t0 + kt < L.F;
    if (kin) {
        const int64_t tok = bkv * L.F + t0 + kt;
        const uint8_t* p = s.k_idx + tok * (D / 4) + 8 * k;
        c0 = load4<WIDE>(p);
        c1 = load4<WIDE>(p + 4);
        sg = load4<WIDE>(s.k_signs + tok * (D / 8) + 4 * k);
        sc = load_as_f16(s.v_scale, tok * NG + k, s.nz_dtype);
        if (k == 0)
            ng = (uint32_t)load_as_f16(s.k_norm, tok, s.nz_dtype) | ((uint32_t)load_as_f16(s.k_gamma, tok, s.nz_dtype) << 16);
    }
    if (kt < 64) {
        // complemented and reversed: bit 4 (7 - m) + 3 - q of r0 is plane q & 1 of
        // dim 2 m + (q >> 1) (dims 0..15; r1: 16..31)
        const uint32_t r0 = __brev(~c0), r1 = __brev(~c1), rs = __brev(~sg);
        auto plane = [&](int q) {  // 16 dims 2 m + (q >> 1), the first at bit 15
            return (every_4th(r0, 3 - q) << 8) | every_4th(r1, 3 - q);
        };
        auto sign = [&](int odd) {  // bits 2 m + odd, the first at bit 15
            uint32_t x = (rs >> (1 - odd)) & 0x55555555u;
            x = (x | (x >> 1)) & 0x33333333u;
            x = (x | (x >> 2)) & 0x0F0F0F0Fu;
            x = (x | (x >> 4)) & 0x00FF00FFu;
            return (x | (x >> 8)) & 0xFFFFu;
        };
        uint32_t* const kp = (uint32_t*)rec + kt * NK + k;
        kp[0] = plane(1) | (plane(3) << 16);              // high bit: dims 2 i, 2 i + 1
        kp[2 * D] = plane(0) | (plane(2) << 16);          // low bit
        kp[4 * D] = sign(0) | (sign(1) << 16);            // QJL sign
        ((uint16_t*)(rec + tq_sc_section(D)))[tq_sc_index(D, kt / 4, k % 2, kt % 4, k / 2)] = (uint16_t)sc;
        if (k == 0) ((uint32_t*)(rec + tq_ng_section(D)))[kt] = ng;
    }
    if (wave < NG) {
        uint32_t o[4] = {0, 0, 0, 0};  // lane j: dim 32 wave + j -- high bit of tokens 0..31, 32..63, low bit
#pragma unroll
        for (int j = 0; j < 32; j++) {
            const uint32_t c = (j < 16 ? v0 : v1) >> (2 * (j % 16));
            const uint64_t h = __ballot(!(c & 2)), l = __ballot(!(c & 1));
            const bool mine = lane == j;
            o[0] = mine ? (uint32_t)h : o[0];
            o[1] = mine ? (uint32_t)(h >> 32) : o[1];
            o[2] = mine ? (uint32_t)l : o[2];
            o[3] = mine ? (uint32_t)(l >> 32) : o[3];
        }
        if (lane < 32) {
            const int d = 32 * wave + lane, half = wave & 1;  // [own, other] half of the tokens
            *(uint4*)(rec + tq_vp_section(D) + (d / 64) * 1024 + (d % 64) * 16) =
                half ? make_uint4(o[1], o[0], o[3], o[2]) : make_uint4(o[0], o[1], o[2], o[3]);
        }
    }
}

template <int D, int FMT, bool WIDE>
__global__ __launch_bounds__(kPackThreads) void pack_blob_kernel(PackSrc s, BlobLayout L, uint8_t* __restrict__ blob) {
    const int bkv_n = L.B * L.Hkv;
    const int64_t near_wgs = (int64_t)(L.Na_pad / kTile) * bkv_n;
    const int64_t wg = blockIdx.x;
    if (wg < near_wgs) {
        const int tiles = L.Na_pad / kTile;
        pack_near_tile<D, WIDE>(s, L, blob, wg / tiles, (int)(wg % tiles));
        return;
    }
    const int tiles = L.F_pad / kTile;
    const int64_t f = wg - near_wgs;
    if (FMT == 1) pack_tq_tile<D, WIDE>(s, L, blob, f / tiles, (int)(f % tiles));
    else pack_far_tile<D, FMT == 1 ? 0 : FMT, WIDE>(s, L, blob, f / tiles, (int)(f % tiles));
}

using PackKernel = void (*)(PackSrc, BlobLayout, uint8_t*);
template <int D, bool WIDE>
PackKernel pick_pack(int fmt) {
    return fmt == 1 ? pack_blob_kernel<D, 1, WIDE> : fmt == 2 ? pack_blob_kernel<D, 2, WIDE> : pack_blob_kernel<D, 0, WIDE>;
}

}  // namespace

int pack_blob(const PackSrc& s, const BlobLayout& L, uint8_t* blob, hipStream_t st) {
    int64_t n = (int64_t)L.B * L.Hkv;
    if (n < L.Hkv + 1) n = L.Hkv + 1;
    if (L.fmt == 1 && n < 2 * (int64_t)L.D * L.D) n = 2 * (int64_t)L.D * L.D;
    hipLaunchKernelGGL(pack_header_kernel, dim3((unsigned)cdiv(n, 256)), dim3(256), 0, st, s, L, blob);
    const int64_t wgs = (int64_t)(L.Na_pad / kTile + L.F_pad / kTile) * L.B * L.Hkv;
    if (wgs > 0) {
        uintptr_t all = (uintptr_t)s.near_k | (uintptr_t)s.near_v | (uintptr_t)s.far_k | (uintptr_t)s.far_v |
                        (uintptr_t)s.k_idx | (uintptr_t)s.k_signs | (uintptr_t)s.v_packed;
        const bool wide = (all & 15) == 0;
        const PackKernel kern = L.D == 128 ? (wide ? pick_pack<128, true>(L.fmt) : pick_pack<128, false>(L.fmt))
                                           : (wide ? pick_pack<64, true>(L.fmt) : pick_pack<64, false>(L.fmt));
        hipLaunchKernelGGL(kern, dim3((unsigned)wgs), dim3(kPackThreads), 0, st, s, L, blob);
    }
    return check_hip(hipGetLastError(), "pack kernels");
}

}  // namespace fkv
