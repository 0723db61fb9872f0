// Fused tier compression for gfx950: one pass over a layer's K and V builds
// the fp16 near tier (with zero headroom), the E4M3 far keys, the INT4
// per-token far values (+ fp16 scale / zero) and the fp16 far-row archive.
//
// Replaces CompressHandle::compress_layer (csrc/foveated_compress.cpp:95-201)
// and its three Metal kernels compress_foveal / compress_fp8 / compress_int4
// (csrc/kernels/foveated_compress.metal:76-205), whose outputs are
// reproduced bit-exactly:
//   * E4M3: re-biased exponent tested for saturation/underflow BEFORE
//     rounding, round-to-nearest-even on the 10->3 mantissa bits, a carry
//     into exponent 15 saturates to 0x7E (:39-66);
//   * INT4: fp32 row min/max, scale = max((max-min)/15, 1e-8) in fp32 with a
//     correctly rounded divide, codes = clamp(round((v-min)/scale), 0, 15)
//     with round-half-away-from-zero, even dim in the low nibble; the stored
//     scale and zero are the fp16 roundings (:153-205).
// Each row of D elements is owned by D/8 lanes (16 bytes of fp16 each).
#include <hip/hip_runtime.h>

#include <string>
#include <type_traits>

#include "fkv_common.h"
#include "../../include/fkv.h"

namespace fkv {

struct CompressArgs {
    const void* k;
    const void* v;
    int dtype;
    int B, H, S;
    fkv_tiers tb;
    uint16_t* near_k;
    uint16_t* near_v;
    uint8_t* far_k;
    uint8_t* far_v;
    uint16_t* fvs;
    uint16_t* fvz;
    int32_t* near_valid;
    uint16_t* arc_k;
    uint16_t* arc_v;
    // per-head-scaled fp8 keys (cfg->k_scale): (B*H) fp32 scales the far
    // keys are divided by before encoding; NULL = unscaled (the reference)
    const float* kscale;
    bool nt_in;  // float32 K and V pass the caches by (load8)
};

// Packed-half integer operations (two fp16 bit patterns per dword).
typedef uint16_t fkv_us2 __attribute__((ext_vector_type(2)));
typedef short fkv_s2 __attribute__((ext_vector_type(2)));
__device__ inline fkv_us2 as_us2(uint32_t w) { return __builtin_bit_cast(fkv_us2, w); }

// The reference's encoder on eight fp16 values (four dwords of two) with the
// hardware's converter, which rounds to nearest even as well but keeps
// subnormal codes and the values 256..448: magnitudes below 2^-6 (0x2400)
// become zero first, infinities, NaN and magnitudes above 448 (0x5F00)
// become 448, and afterwards every code of exponent 15 -- whatever reached
// 256, before rounding or by it -- becomes 0x7E.  About six instructions per
// value; bit tests and selects on each value took twenty, which bound the
// long-context compress with every option (see far_row).
__device__ inline uint32_t e4m3_flush_clamp(uint32_t w) {
    const fkv_us2 m = as_us2(w & 0x7FFF7FFFu);
    const fkv_us2 one = {1, 1}, top = {0x5F00, 0x5F00}, low = {0x23FF, 0x23FF};
    const fkv_us2 keep = -__builtin_elementwise_min(__builtin_elementwise_sub_sat(m, low), one);  // 0xFFFF from 2^-6 on
    const uint32_t c = __builtin_bit_cast(uint32_t, __builtin_elementwise_min(m, top) & keep);
    return c | (w & 0x80008000u);
}
__device__ inline uint32_t encode_e4m3x4(uint32_t w0, uint32_t w1) {
    const fkv_s2 none = {0, 0};
    fkv_s2 c = __builtin_amdgcn_cvt_scalef32_pk_fp8_f16(none, as_h2(e4m3_flush_clamp(w0)), 1.0f, false);
    c = __builtin_amdgcn_cvt_scalef32_pk_fp8_f16(c, as_h2(e4m3_flush_clamp(w1)), 1.0f, true);
    const uint32_t codes = __builtin_bit_cast(uint32_t, c);
    const uint32_t t = ((codes & 0x78787878u) + 0x08080808u) & 0x80808080u;  // exponent 15
    const uint32_t mask = t - (t >> 7);                                     // 0x7F there
    return (codes & ~mask) | (mask & 0x7E7E7E7Eu);
}

// fp16(a / b), the quotient rounded to fp32 first (y = 1.0f / b).  The empty
// asm keeps the two roundings apart: the compiler would fuse the quotient's
// last fma with the conversion into one that rounds once, which gives another
// fp16 value where fp32's rounding has moved the quotient onto a tie.
__device__ inline uint16_t quotient_h(float a, float b, float y) {
    float q = div_by<1>(a, b, y);
    asm volatile("" : "+v"(q));
    return f2h(q);
}

// The fp16 value a key is encoded from with a per-head scale: fp16(key /
// scale), fp32 division rounded to nearest even.  One correction step is
// enough for every fp16 key and every scale that is an fp16 amax over 240
// (all pairs checked) but turns -0 into +0, so the sign is the key's;
// infinities and NaN, which the scale leaves out, go to the encoder as they
// are.
__device__ inline uint32_t scaled_keys(uint32_t w, float scale, float rscale) {
    const uint16_t lo = (uint16_t)w, hi = (uint16_t)(w >> 16);
    const uint16_t ql = quotient_h(h2f(lo), scale, rscale), qh = quotient_h(h2f(hi), scale, rscale);
    const uint32_t q = ((lo & 0x7C00u) == 0x7C00u ? lo : ql) | ((uint32_t)((hi & 0x7C00u) == 0x7C00u ? hi : qh) << 16);
    return (q & 0x7FFF7FFFu) | (w & 0x80008000u);
}

// Minimum and maximum over the RL lanes (4, 8 or 16, aligned) of a row by DPP: lane
// pairs, quads, then the mirrored halves of 8 and of 16 lanes.
template <int RL>
__device__ inline void row_minmax(float& mn, float& mx) {
    static_assert(RL == 4 || RL == 8 || RL == 16, "rows of 4, 8 or 16 lanes");
    mn = fminf(mn, dpp_f32<kDppXor1>(mn));
    mx = fmaxf(mx, dpp_f32<kDppXor1>(mx));
    mn = fminf(mn, dpp_f32<kDppXor2>(mn));
    mx = fmaxf(mx, dpp_f32<kDppXor2>(mx));
    if (RL >= 8) {
        mn = fminf(mn, dpp_f32<0x141>(mn));  // row_half_mirror
        mx = fmaxf(mx, dpp_f32<0x141>(mx));
    }
    if (RL >= 16) {
        mn = fminf(mn, dpp_f32<0x140>(mn));  // row_mirror
        mx = fmaxf(mx, dpp_f32<0x140>(mx));
    }
}

// One far row (fr = bh * F + f) from its fp16 K / V (8 elements per lane):
// E4M3 keys, INT4 values per token (VG = 0) or per VG-dim group, archive.
// Meant to be bound by memory; the arithmetic per value is kept to what that
// leaves room for (one division per row and lane instead of one per value,
// the converter for the keys, lane reductions by DPP instead of LDS
// permutes): the 64K x 8 head layer from bf16 with key scales and group-32
// values took 191 us without (3.4 TB/s), 124 us now (5.3 TB/s); the 8 x 8 x
// 16K fp16 layer was at the memory's rate before (219 us) and still is (218).
template <int D, int VG, bool NT>
__device__ inline void far_row(const CompressArgs& a, int bh, int64_t fr, int sub, uint4 kw, uint4 vw) {
    constexpr int LPR = D / 8;
    if (!a.far_k) {  // near tier and archive only (the archive is read next)
        store16<false>(a.arc_k + fr * D + sub * 8, kw);
        store16<false>(a.arc_v + fr * D + sub * 8, vw);
        return;
    }
    if (a.arc_k) store16<true>(a.arc_k + fr * D + sub * 8, kw);
    if (a.arc_v) store16<true>(a.arc_v + fr * D + sub * 8, vw);
    // far K: E4M3 codes
    if (a.kscale) {
        const float scale = a.kscale[bh], rscale = 1.0f / scale;
        kw = make_uint4(scaled_keys(kw.x, scale, rscale), scaled_keys(kw.y, scale, rscale),
                        scaled_keys(kw.z, scale, rscale), scaled_keys(kw.w, scale, rscale));
    }
    store8<NT>(a.far_k + fr * D + sub * 8, encode_e4m3x4(kw.x, kw.y), encode_e4m3x4(kw.z, kw.w));
    // far V: INT4 per token (VG = 0) or per 32-dim group
    constexpr int RL = VG ? VG / 8 : LPR;  // lanes of one quantisation row
    const uint32_t vs[4] = {vw.x, vw.y, vw.z, vw.w};
    float vf[8];
    float mn = INFINITY, mx = -INFINITY;
#pragma unroll
    for (int i = 0; i < 8; i++) {
        vf[i] = h2f((uint16_t)(vs[i / 2] >> (16 * (i & 1))));
        mn = fminf(mn, vf[i]);
        mx = fmaxf(mx, vf[i]);
    }
    row_minmax<RL>(mn, mx);
    const float scale = fmaxf((mx - mn) / 15.0f, 1e-8f), rscale = 1.0f / scale;
    uint32_t packed = 0;
#pragma unroll
    for (int i = 0; i < 8; i++) {
        // round half away from zero of a quotient >= 0, clamped to 15 (NaN: 0)
        const float q = div_by<2>(vf[i] - mn, scale, rscale);
        uint32_t c = (uint32_t)fminf(fmaxf(q, 0.0f), 15.0f);
        c += q - (float)c >= 0.5f ? 1u : 0u;
        packed |= min(c, 15u) << (4 * i);
    }
    uint32_t* const pv = (uint32_t*)(a.far_v + fr * (D / 2) + sub * 4);
    if (NT) __builtin_nontemporal_store(packed, pv);
    else *pv = packed;
    if (sub % RL == 0) {
        const int64_t si = VG ? fr * (D / VG) + sub / RL : fr;
        a.fvs[si] = f2h(scale);
        a.fvz[si] = f2h(mn);
    }
}

// VG = 0: one INT4 scale / zero per token (the reference); VG = 32: one per
// 32-dim group (4 lanes), the same quantiser applied to every group.
template <int D, int VG, bool NT>
__global__ __launch_bounds__(256) void compress_kernel(CompressArgs a) {
    constexpr int LPR = D / 8;       // lanes per row
    constexpr int RPB = 256 / LPR;   // rows per block
    const fkv_tiers& tb = a.tb;
    const int bh = blockIdx.y;
    const int r = blockIdx.x * RPB + threadIdx.x / LPR;
    const int sub = threadIdx.x % LPR;
    if (blockIdx.x == 0 && threadIdx.x == 0 && bh < a.H) a.near_valid[bh] = tb.r_actual;
    const int npad = tb.n_near_padded;
    const int F = tb.far_count;
    if (r >= a.S + tb.headroom) return;  // whole row group leaves together
    const uint4 zero4 = make_uint4(0, 0, 0, 0);
    if (r >= a.S) {  // headroom slot: zeros
        const int64_t o = ((int64_t)bh * npad + tb.r_actual + (r - a.S)) * D + sub * 8;
        store16<NT>(a.near_k + o, zero4);
        store16<NT>(a.near_v + o, zero4);
        return;
    }
    const int t = r;
    int slot = -1, f = -1;
    if (t < tb.n_sinks) slot = t;
    else if (t >= tb.near_mid_start && t < tb.mid_end) slot = tb.n_sinks + (t - tb.near_mid_start);
    else if (tb.window > 0 && t >= a.S - tb.window) slot = tb.n_sinks + tb.near_from_mid + (t - (a.S - tb.window));
    else if (t >= tb.mid_start && t < tb.near_mid_start) f = t - tb.mid_start;

    const int64_t src = ((int64_t)bh * a.S + t) * D + sub * 8;
    const uint4 kw = load8(a.k, a.dtype, src, a.nt_in), vw = load8(a.v, a.dtype, src, a.nt_in);
    if (slot >= 0) {
        const int64_t o = ((int64_t)bh * npad + slot) * D + sub * 8;
        store16<NT>(a.near_k + o, kw);
        store16<NT>(a.near_v + o, vw);
        return;
    }
    if (f < 0) return;  // unreachable: every position is near or far
    far_row<D, VG, NT>(a, bh, (int64_t)bh * F + f, sub, kw, vw);
}


// ---------------------------------------------------------------------------
// Per-head fp8 key scale (the benchmark's "per-head-scaled fp8 E4M3" keys;
// an extension: the reference encodes keys unscaled,
// foveated_compress.metal:39-66).  scale = amax / 240 over the finite
// values of the head's far keys (fp32 division; 1 when amax is 0), so the
// head's largest |key| encodes to 240 (0x77): the encoder above emits
// exponent 15 only as the saturation code 0x7E (448), so 240 is the top of
// its 3-bit-mantissa range, and a scale of amax / 448 would put every key
// in (240, 448] x scale on 448.
// ---------------------------------------------------------------------------

constexpr int kScaleThreads = 256;
constexpr int kScaleRows = 4;      // rows a lane group loads together
constexpr int kScaleBlocks = 2048; // workgroups the reduction aims for
constexpr int kScaleOneThreads = 1024, kScaleOneSweeps = 4;  // one workgroup per (batch, head)

// Whether one workgroup of 1,024 threads takes a (batch, head)'s far rows and
// writes the scale: up to 1,024 rows of 128 (2,048 of 64).  The second launch
// costs a small call more than the rows do: 300 tokens of 128, 1 head, a call
// 33 us with one workgroup of 256 threads, 35-36 with two launches, 32 here
// (in a graph 13.5, 7.4 and 6.3); 2,000 tokens of 64 35, 36 and 33 (28, 7.7 and
// 8.7).  At 3,000 tokens of 64 the rows of one workgroup take 10.4 in a graph
// against 7.8.
__host__ __device__ inline bool kscale_one(int F, int D) {
    return F <= kScaleOneSweeps * kScaleRows * (kScaleOneThreads / (D / 8));
}

// Workgroups per (batch, head) of the reduction: each takes at least
// kScaleRows rows per lane group, so their maxima (one fp32 each) always fit
// the head's F * D bytes of far codes, where they wait for kscale_finish.
__host__ __device__ inline int kscale_parts(int F, int D, int BH) {
    const int64_t rows = (int64_t)kScaleRows * (kScaleThreads / (D / 8));
    int64_t p = cdiv(F, rows);
    const int64_t most = cdiv(kScaleBlocks, BH);
    if (p > most) p = most;
    return p < 1 ? 1 : (int)p;
}

// The largest magnitude among elements that are finite as fp16, over packed
// or single elements: a magnitude's bits order as integers, and adding BIAS
// makes those that fp16 does not hold as finite numbers negative, which a
// signed maximum passes over.  Three instructions per dword instead of a
// conversion, a test and a maximum per element.
template <int DT>
struct FiniteMax {
    // the smallest magnitude that fp16 rounds to infinity (or holds as one)
    static constexpr uint32_t kTop = DT == FKV_F16 ? 0x7C00u : DT == FKV_BF16 ? 0x4780u : 0x477FF000u;
    static constexpr uint32_t kBias = DT == FKV_F32 ? 0x80000000u - kTop : 0x8000u - kTop;
    uint32_t m = DT == FKV_F32 ? kBias : kBias | (kBias << 16);
    __device__ inline void add(uint32_t w) {
        if constexpr (DT == FKV_F32) {
            m = (uint32_t)max((int32_t)m, (int32_t)((w & 0x7FFFFFFFu) + kBias));
        } else {
            const fkv_us2 bias = {(uint16_t)kBias, (uint16_t)kBias};
            const fkv_s2 x = __builtin_bit_cast(fkv_s2, as_us2(w & 0x7FFF7FFFu) + bias);
            m = __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(fkv_s2, m), x));
        }
    }
    // as the fp16 value it is encoded from (rounding keeps the order)
    __device__ inline float value() const {
        if constexpr (DT == FKV_F32) return h2f(f2h(__uint_as_float(m - kBias)));
        const uint32_t lo = (m & 0xFFFFu) - kBias, hi = (m >> 16) - kBias, x = lo > hi ? lo : hi;
        return DT == FKV_F16 ? h2f((uint16_t)x) : h2f(f2h(bf2f((uint16_t)x)));
    }
};

__device__ inline float kscale_of(float amax) { return amax > 0.f ? amax / 240.0f : 1.0f; }

// Bound by the one read of the far keys.  A maximum does not depend on the
// order, so the rows of a (batch, head) are dealt over as many workgroups as
// fill the chip (one workgroup per head read 121 MB of keys at 8 heads x 59K
// rows in 3,690 us: eight CUs), and each lane group has kScaleRows rows in
// flight; 41 us with a conversion and a test per element, 36 us here (8 or
// 16 rows in flight: no faster).
// Far rows are positions mid_start.. (far_idx NULL) or far_idx[bh][f];
// out-of-range indices are zero rows.
template <int D, int DT, bool ONE>
__global__ __launch_bounds__(ONE ? kScaleOneThreads : kScaleThreads) void kscale_kernel(
    CompressArgs a, const int32_t* __restrict__ far_idx, float* __restrict__ out) {
    constexpr int NT = ONE ? kScaleOneThreads : kScaleThreads;
    constexpr int LPR = D / 8, RPB = NT / LPR, NQ = DT == FKV_F32 ? 2 : 1;  // 16-byte loads per lane and row
    __shared__ float red[NT / kWave];
    const int bh = blockIdx.y, sub = threadIdx.x % LPR, parts = gridDim.x;
    const int F = a.tb.far_count;
    FiniteMax<DT> amax;
    for (int64_t f0 = (int64_t)blockIdx.x * kScaleRows * RPB + threadIdx.x / LPR; f0 < F;
         f0 += (int64_t)parts * kScaleRows * RPB) {
        int t[kScaleRows];
#pragma unroll
        for (int u = 0; u < kScaleRows; u++) {
            const int64_t f = f0 + u * RPB;
            t[u] = f >= F ? -1 : far_idx ? far_idx[(int64_t)bh * F + f] : a.tb.mid_start + (int)f;
        }
        uint4 kx[kScaleRows][NQ];
#pragma unroll
        for (int u = 0; u < kScaleRows; u++) {
            // a row outside the sequence reads row 0 and is left out below
            const bool in = t[u] >= 0 && t[u] < a.S;
            const uint4* p = (const uint4*)a.k + (((int64_t)bh * a.S + (in ? t[u] : 0)) * LPR + sub) * NQ;
#pragma unroll
            for (int q = 0; q < NQ; q++) kx[u][q] = p[q];
        }
#pragma unroll
        for (int u = 0; u < kScaleRows; u++)
            if (t[u] >= 0 && t[u] < a.S)
#pragma unroll
                for (int q = 0; q < NQ; q++) {
                    amax.add(kx[u][q].x);
                    amax.add(kx[u][q].y);
                    amax.add(kx[u][q].z);
                    amax.add(kx[u][q].w);
                }
    }
    const float m0 = wave_max(amax.value());
    if (threadIdx.x % kWave == 0) red[threadIdx.x / kWave] = m0;
    __syncthreads();
    if (threadIdx.x == 0) {
        float m = 0.f;
        for (int w = 0; w < NT / kWave; w++) m = fmaxf(m, red[w]);
        if (ONE) out[bh] = kscale_of(m);
        else out[(int64_t)bh * parts + blockIdx.x] = m;
    }
}

// One wave per (batch, head): the largest of its workgroups' maxima -> scale.
__global__ __launch_bounds__(kWave) void kscale_finish_kernel(const float* __restrict__ part_max, int parts,
                                                              float* __restrict__ out) {
    const int bh = blockIdx.x;
    float m = 0.f;
    for (int i = threadIdx.x; i < parts; i += kWave) m = fmaxf(m, part_max[(int64_t)bh * parts + i]);
    m = wave_max(m);
    if (threadIdx.x == 0) out[bh] = kscale_of(m);
}

// ---------------------------------------------------------------------------
// Importance partition: near = sinks + the near_from_mid middle tokens of
// highest importance + window, per (batch, head).
// ---------------------------------------------------------------------------

// fp32 importance -> unsigned key with the same order; NaN ranks below
// -inf, -0 equals +0.
__device__ inline uint32_t order_key(float f) {
    const uint32_t b = __float_as_uint(f + 0.0f);  // -0 + 0 = +0
    return f != f ? 0u : b ^ ((uint32_t)((int32_t)b >> 31) | 0x80000000u);
}

// Middle token i's rank key: importance, then position (the later token
// wins a tie, so a constant or position-valued importance gives the
// recency partition).
__device__ inline uint64_t rank_key(const float* row, int pos) {
    return ((uint64_t)order_key(row[pos]) << 32) | (uint32_t)pos;
}

constexpr int kPartThreads = 1024;
constexpr int kPartWaves = kPartThreads / kWave;

// Fixed slots of a near index row: sinks, window, headroom.
__device__ inline void fixed_slots(int32_t* nrow, int S, const fkv_tiers& tb, int tid) {
    const int k = tb.near_from_mid;
    for (int i = tid; i < tb.n_near_padded; i += kPartThreads) {
        if (i < tb.n_sinks) nrow[i] = i;
        else if (i >= tb.n_sinks + k && i < tb.r_actual) nrow[i] = S - tb.window + (i - tb.n_sinks - k);
        else if (i >= tb.r_actual) nrow[i] = -1;
    }
}

// No instruction: keeps what is computed from x after this point after it.
// (Over R registers the compiler otherwise computes every lane mask of a loop
// first, or keeps one loop's for the next, and spills them.)
#define PART_PIN(x) asm volatile("" : "+v"(x))

constexpr int kPartRegs = 64;  // most tokens per thread held in registers
constexpr int kPartBits = 11, kPartBins = 1 << kPartBits, kPartCopies = 4;

// Partition of a (batch, head) whose middle fits the workgroup's registers,
// q of R tokens per thread (the fewest that hold it).  Bound by one CU's
// vector instructions, not by memory, so the row is read once and as little
// as possible is done per token: wave w holds order_key of the middle's
// tokens w * q * 64 .. in position order (register r: 64 consecutive
// tokens).  A radix select of 11 + 11 + 10 bits over the registers (LDS
// histograms, one per wave modulo kPartCopies; one per lane modulo 16, free
// of bank conflicts, was no faster) finds the near_from_mid-th largest key v
// and how many tokens equal to it stay near (the last ones in position
// order: the later token wins a tie, which is what the 64-bit rank key
// orders by).  The compaction needs no block step per chunk: a token's far
// row is its position less the near tokens before it, and those follow from
// one scan of the waves' counts and ballots.  Registers from q on take no
// part (a test of a scalar): as padding their histogram adds all met in one
// bin (16,385 tokens in 64 registers per thread 73 us; 53 with the 8-bit
// passes below, 22 with q; 32,768 tokens 61, 97 and 24).  The fewer than 1,024 places past the middle in
// the others hold the lowest key: they come after every token in position
// order, so they only take part in a tie at that key, where they are counted
// out, and their places lie past the near and far rows (a range test per
// token and pass made half of the instructions).  64K tokens x 8 heads: 190
// us with 8-bit passes that each re-read the row and a block scan per 1,024
// tokens, 53 us with the range tests (and their lane masks spilled), 40 us
// here.
template <int R>
__global__ __launch_bounds__(kPartThreads) void partition_regs_kernel(const float* __restrict__ imp, int S,
                                                                     fkv_tiers tb, int32_t* __restrict__ near_idx,
                                                                     int32_t* __restrict__ far_idx) {
    __shared__ uint32_t hist[kPartCopies][kPartBins];
    __shared__ uint32_t wtot[kPartWaves], wgt[kPartWaves], weq[kPartWaves];
    __shared__ uint32_t s_bin, s_rem, s_cnt;
    const int bh = blockIdx.x, tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave), lane = tid % kWave;
    const int npad = tb.n_near_padded, F = tb.far_count, m0 = tb.mid_start;
    const int mlen = tb.mid_end > tb.mid_start ? tb.mid_end - tb.mid_start : 0;
    const int k = tb.near_from_mid;
    int32_t* nrow = near_idx + (int64_t)bh * npad;
    int32_t* frow = far_idx + (int64_t)bh * F;
    fixed_slots(nrow, S, tb, tid);
    if (k >= mlen || k <= 0) {  // the whole middle is near, or far
        for (int i = tid; i < mlen; i += kPartThreads) {
            if (k > 0) nrow[tb.n_sinks + i] = m0 + i;
            else if (i < F) frow[i] = m0 + i;
        }
        return;
    }
    constexpr int C = R < 16 ? 1 : 4;  // registers per test of q
    const int q = (mlen + C * kPartThreads - 1) / (C * kPartThreads) * C;  // at most R
    // whether chunk c's registers are in use (tested anew each time: kept, the
    // results of all chunks would be spilled)
    auto used = [&](int c) {
        int qc = q;
        asm volatile("" : "+s"(qc));
        return c < qc;
    };
    const int i0 = wave * q * kWave + lane;  // the lane's first token of the middle
    const float* row = imp + (int64_t)bh * S + m0;
    uint32_t key[R];
    {
        float f[R] = {};
#pragma unroll
        for (int c = 0; c < R; c += C)
            if (used(c))
#pragma unroll
                for (int r = c; r < c + C; r++) f[r] = row[min(i0 + r * kWave, mlen - 1)];
#pragma unroll
        for (int r = 0; r < R; r++) key[r] = order_key(f[r]);
        if ((wave + 1) * q * kWave > mlen)
#pragma unroll
            for (int r = 0; r < R; r++)
                if (i0 + r * kWave >= mlen) key[r] = 0;
    }
    uint32_t v = 0, rem = k;
    constexpr int shift[3] = {32 - kPartBits, 32 - 2 * kPartBits, 0};
    constexpr int bits[3] = {kPartBits, kPartBits, 32 - 2 * kPartBits};
#pragma unroll
    for (int p = 0; p < 3; p++) {
        for (int i = tid; i < kPartCopies * kPartBins; i += kPartThreads) (&hist[0][0])[i] = 0;
        __syncthreads();
        uint32_t* const h = hist[wave % kPartCopies];
#pragma unroll
        for (int c = 0; c < R; c += C) {
            if (!used(c)) break;
#pragma unroll
            for (int r = c; r < c + C; r++) {
                PART_PIN(key[r]);
                if (p == 0 || (key[r] ^ v) >> (shift[p] + bits[p]) == 0)  // the digits already known
                    atomicAdd(&h[(key[r] >> shift[p]) & ((1u << bits[p]) - 1)], 1u);
            }
        }
        __syncthreads();
        // thread t takes bins top - 2t and top - 2t - 1: an inclusive scan
        // over the threads counts the keys from the top bin down
        const int hi = kPartBins - 1 - 2 * tid;
        uint32_t c1 = 0, c0 = 0;
#pragma unroll
        for (int q = 0; q < kPartCopies; q++) {
            c1 += hist[q][hi];
            c0 += hist[q][hi - 1];
        }
        uint32_t inc = c1 + c0;
#pragma unroll
        for (int d = 1; d < kWave; d <<= 1) {
            const uint32_t t = __shfl_up(inc, d, kWave);
            if (lane >= d) inc += t;
        }
        if (lane == kWave - 1) wtot[wave] = inc;
        __syncthreads();
        uint32_t above = inc - c1 - c0;
#pragma unroll
        for (int w = 0; w < kPartWaves; w++)
            if (w < wave) above += wtot[w];
        if (above < rem && above + c1 >= rem) {
            s_bin = hi;
            s_rem = rem - above;
            s_cnt = c1;
        } else if (above + c1 < rem && above + c1 + c0 >= rem) {
            s_bin = hi - 1;
            s_rem = rem - above - c1;
            s_cnt = c0;
        }
        __syncthreads();
        v |= (uint32_t)__builtin_amdgcn_readfirstlane((int)s_bin) << shift[p];
        rem = (uint32_t)__builtin_amdgcn_readfirstlane((int)s_rem);
    }
    // tokens equal to v that stay far (the places past the middle are not tokens)
    const uint32_t equal_far = s_cnt - (v == 0 ? (uint32_t)(kPartThreads * q - mlen) : 0u) - rem;
    // lane r: which of register r's tokens lie above v (near) and at v
    static_assert(R <= kWave, "a lane per register");
    uint32_t nlo = 0, nhi = 0, elo = 0, ehi = 0;
#pragma unroll
    for (int c = 0; c < R; c += C) {
        if (!used(c)) break;
#pragma unroll
        for (int r = c; r < c + C; r++) {
            PART_PIN(key[r]);
            const uint64_t g = __ballot(key[r] > v), e = __ballot(key[r] == v);
            // (a select per lane would need R lane masks; the wait states are those
            // of a scalar register written by a compare and read here)
            asm volatile("s_nop 1\n\tv_writelane_b32 %0, %4, %8\n\tv_writelane_b32 %1, %5, %8\n\t"
                         "v_writelane_b32 %2, %6, %8\n\tv_writelane_b32 %3, %7, %8"
                         : "+v"(nlo), "+v"(nhi), "+v"(elo), "+v"(ehi)
                         : "s"((uint32_t)g), "s"((uint32_t)(g >> 32)), "s"((uint32_t)e), "s"((uint32_t)(e >> 32)), "n"(r));
        }
    }
    // inclusive sums over the wave's registers
    auto lane_scan = [&](uint32_t x) {
#pragma unroll
        for (int d = 1; d < kWave; d <<= 1) {
            const uint32_t t = __shfl_up(x, d, kWave);
            if (lane >= d) x += t;
        }
        return x;
    };
    uint64_t near = ((uint64_t)nhi << 32) | nlo, at_v = ((uint64_t)ehi << 32) | elo;
    const uint32_t eq = __popcll(at_v), eq_upto = lane_scan(eq);
    const uint32_t gt_all = lane_scan(__popcll(near));
    if (lane == kWave - 1) {
        wgt[wave] = gt_all;
        weq[wave] = eq_upto;
    }
    __syncthreads();
    uint32_t near_before = 0, eq_before = 0;  // in the waves before this one
#pragma unroll
    for (int w = 0; w < kPartWaves; w++)
        if (w < wave) {
            near_before += wgt[w];
            eq_before += weq[w];
        }
    near_before += eq_before > equal_far ? eq_before - equal_far : 0u;
    // the first equal_far tokens at v are far: this register's share of them
    const uint32_t eq_first = eq_before + eq_upto - eq;
    for (uint32_t n = min(equal_far > eq_first ? equal_far - eq_first : 0u, eq); n > 0; n--) at_v &= at_v - 1;
    near |= at_v;
    nlo = (uint32_t)near;
    nhi = (uint32_t)(near >> 32);
    const uint32_t upto = near_before + lane_scan(__popcll(near)), first = upto - __popcll(near);
    nrow += tb.n_sinks;
#pragma unroll 4
    for (int r = 0; r < q; r++) {
        const uint32_t lo = __builtin_amdgcn_readlane(nlo, r), hi = __builtin_amdgcn_readlane(nhi, r);
        const int before = (int)__builtin_amdgcn_readlane(first, r) +
                           (int)__builtin_amdgcn_mbcnt_hi(hi, __builtin_amdgcn_mbcnt_lo(lo, 0u));
        const int i = i0 + r * kWave;
        if (((((uint64_t)hi << 32) | lo) >> lane) & 1) {
            if (before < k) nrow[before] = m0 + i;
        } else if (i - before < F) {
            frow[i - before] = m0 + i;
        }
    }
}

// One workgroup per (batch, head).  The near_from_mid-th largest rank key
// is found by an 8-pass MSB-first radix select (256-bin LDS histograms);
// then the middle is compacted in position order into near slots
// n_sinks.. and far slots 0.. with a block-wide scan per 1024-token chunk.
// For middles of more than kPartThreads * kPartRegs tokens, which do not fit
// partition_regs_kernel's registers: eight passes over the row (8 heads: 181
// us for 65,537 tokens where 65,536 in registers take 38; 350 us for 131,072).
__global__ __launch_bounds__(kPartThreads) void partition_kernel(const float* __restrict__ imp, int S, fkv_tiers tb,
                                                                int32_t* __restrict__ near_idx,
                                                                int32_t* __restrict__ far_idx) {
    constexpr int NW = kPartWaves;
    __shared__ uint32_t hist[NW][256];  // one histogram per wave (less atomic contention)
    __shared__ uint64_t s_prefix;
    __shared__ int s_rem;
    __shared__ int wcount[2][NW];
    const int bh = blockIdx.x, tid = threadIdx.x;
    const int wave = tid / 64, lane = tid % 64;
    const float* row = imp + (int64_t)bh * S;
    const int npad = tb.n_near_padded, F = tb.far_count;
    const int m0 = tb.mid_start;
    const int mlen = tb.mid_end > tb.mid_start ? tb.mid_end - tb.mid_start : 0;
    const int k = tb.near_from_mid;
    int32_t* nrow = near_idx + (int64_t)bh * npad;
    int32_t* frow = far_idx + (int64_t)bh * F;
    fixed_slots(nrow, S, tb, tid);
    const bool all = k >= mlen, none = k <= 0;
    uint64_t thr = 0;  // near <=> rank key >= thr
    if (!all && !none) {
        uint64_t prefix = 0, mask = 0;
        int rem = k;
        for (int p = 7; p >= 0; p--) {
            for (int i = tid; i < NW * 256; i += kPartThreads) (&hist[0][0])[i] = 0;
            __syncthreads();
            for (int i = tid; i < mlen; i += kPartThreads) {
                const uint64_t key = rank_key(row, m0 + i);
                if ((key & mask) == prefix) atomicAdd(&hist[wave][(key >> (8 * p)) & 255], 1u);
            }
            __syncthreads();
            if (wave == 0) {
                // lane l holds bins 4l..4l+3; the bin holding the rem-th largest
                // key is the one where the count of larger keys crosses rem
                uint32_t c[4] = {0, 0, 0, 0};
                for (int w = 0; w < NW; w++)
#pragma unroll
                    for (int e = 0; e < 4; e++) c[e] += hist[w][4 * lane + e];
                const uint32_t tot = c[0] + c[1] + c[2] + c[3];
                uint32_t suf = tot;  // inclusive suffix sum over lanes >= l
#pragma unroll
                for (int d = 1; d < 64; d <<= 1) {
                    const uint32_t t = __shfl_down(suf, d, 64);
                    if (lane + d < 64) suf += t;
                }
                uint32_t cum = suf - tot;  // keys in bins above this lane's
#pragma unroll
                for (int e = 3; e >= 0; e--) {
                    if (cum < (uint32_t)rem && cum + c[e] >= (uint32_t)rem) {
                        s_prefix = prefix | ((uint64_t)(4 * lane + e) << (8 * p));
                        s_rem = rem - (int)cum;
                    }
                    cum += c[e];
                }
            }
            __syncthreads();
            prefix = s_prefix;
            rem = s_rem;
            mask |= (uint64_t)255 << (8 * p);
        }
        thr = prefix;
    }
    // compaction in position order
    int near_base = 0, far_base = 0;
    for (int c0 = 0; c0 < mlen; c0 += kPartThreads) {
        const int i = c0 + tid;
        const bool valid = i < mlen;
        const bool nf = valid && (all || (!none && rank_key(row, m0 + i) >= thr));
        const bool ff = valid && !nf;
        const uint64_t bn = __ballot(nf), bf = __ballot(ff);
        const uint64_t below = lane ? (~0ull >> (64 - lane)) : 0ull;
        const int rn = __popcll(bn & below), rf = __popcll(bf & below);
        if (lane == 0) {
            wcount[0][wave] = __popcll(bn);
            wcount[1][wave] = __popcll(bf);
        }
        __syncthreads();
        int wn = 0, wf = 0, tn = 0, tf = 0;
        for (int w = 0; w < NW; w++) {
            if (w < wave) {
                wn += wcount[0][w];
                wf += wcount[1][w];
            }
            tn += wcount[0][w];
            tf += wcount[1][w];
        }
        if (nf) {
            const int slot = tb.n_sinks + near_base + wn + rn;
            if (slot < tb.n_sinks + k) nrow[slot] = m0 + i;
        }
        if (ff) {
            const int f = far_base + wf + rf;
            if (f < F) frow[f] = m0 + i;
        }
        near_base += tn;
        far_base += tf;
        __syncthreads();  // wcount is rewritten by the next chunk
    }
}

// Compression from explicit index sets: output row r < Npad is near slot r
// (source near_idx, zeros for headroom / -1 / out-of-range indices), row
// Npad + f is far row f (source far_idx; an out-of-range index encodes a
// zero row).
template <int D, int VG, bool NT>
__global__ __launch_bounds__(256) void compress_gather_kernel(CompressArgs a, const int32_t* __restrict__ near_idx,
                                                              const int32_t* __restrict__ far_idx) {
    constexpr int LPR = D / 8;
    constexpr int RPB = 256 / LPR;
    const fkv_tiers& tb = a.tb;
    const int bh = blockIdx.y;
    const int r = blockIdx.x * RPB + threadIdx.x / LPR;
    const int sub = threadIdx.x % LPR;
    if (blockIdx.x == 0 && threadIdx.x == 0 && bh < a.H) a.near_valid[bh] = tb.r_actual;
    const int npad = tb.n_near_padded;
    const int F = tb.far_count;
    if (r >= npad + F) return;  // whole row group leaves together
    uint4 kw = make_uint4(0, 0, 0, 0), vw = kw;
    const bool near = r < npad;
    int t = -1;
    if (near) t = r < tb.r_actual ? near_idx[(int64_t)bh * npad + r] : -1;
    else t = far_idx[(int64_t)bh * F + (r - npad)];
    if (t >= 0 && t < a.S) {
        const int64_t src = ((int64_t)bh * a.S + t) * D + sub * 8;
        kw = load8(a.k, a.dtype, src, a.nt_in);
        vw = load8(a.v, a.dtype, src, a.nt_in);
    }
    if (near) {
        const int64_t o = ((int64_t)bh * npad + r) * D + sub * 8;
        store16<NT>(a.near_k + o, kw);
        store16<NT>(a.near_v + o, vw);
        return;
    }
    far_row<D, VG, NT>(a, bh, (int64_t)bh * F + (r - npad), sub, kw, vw);
}

// The recency partition's index sets, one element per thread (an
// importance partition of position-valued importance gives the same).
__global__ void tier_index_kernel(fkv_tiers tb, int S, int64_t bh_n, int32_t* __restrict__ near_idx,
                                  int32_t* __restrict__ far_idx) {
    const int npad = tb.n_near_padded, F = tb.far_count, row = npad + F;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < bh_n * row; i += (int64_t)gridDim.x * blockDim.x) {
        const int64_t bh = i / row;
        const int e = (int)(i % row), mid = e - tb.n_sinks, win = mid - tb.near_from_mid;
        if (e >= npad) far_idx[bh * F + e - npad] = tb.mid_start + e - npad;
        else near_idx[bh * npad + e] = mid < 0           ? e
                                       : win < 0         ? tb.near_mid_start + mid
                                       : win < tb.window ? S - tb.window + win
                                                         : -1;
    }
}

}  // namespace fkv

namespace {

// Shared argument checks and CompressArgs of the compress entry points.
int compress_setup(const char* fn, const fkv_tier_config* cfg, const void* keys, const void* values,
                   int32_t in_dtype, int32_t B, int32_t H, int32_t S, int32_t D, void* near_k, void* near_v,
                   uint8_t* far_k, uint8_t* far_v, void* far_v_scale, void* far_v_zero, int32_t* near_valid,
                   void* archive_k, void* archive_v, fkv::CompressArgs& a, bool archive_only = false) {
    using fkv::set_error;
    const std::string name(fn);
    if (!cfg) return set_error(name + ": cfg is NULL");
    if (B <= 0 || H <= 0 || S < 0) return set_error(name + ": bad shape");
    if (D != 64 && D != 128) return set_error(name + ": head dim must be 64 or 128, got " + std::to_string(D));
    if (in_dtype < FKV_F16 || in_dtype > FKV_F32) return set_error(name + ": unsupported dtype");
    if (cfg->v_group != 0 && cfg->v_group != 32)
        return set_error(name + ": v_group must be 0 (per token) or 32, got " + std::to_string(cfg->v_group));
    if (cfg->k_scale != 0 && cfg->k_scale != 1)
        return set_error(name + ": k_scale must be 0 (unscaled) or 1 (per head), got " + std::to_string(cfg->k_scale));
    fkv_tiers tb;
    if (int rc = fkv_tier_boundaries(cfg, S, &tb)) return rc;
    if ((S > 0 && (!keys || !values)) || !near_k || !near_v || !near_valid ||
        (tb.far_count > 0 && (archive_only ? !archive_k || !archive_v : !far_k || !far_v || !far_v_scale || !far_v_zero)))
        return set_error(name + ": NULL output/input");
    a.k = keys;
    a.v = values;
    a.dtype = in_dtype;
    a.B = B;
    a.H = H;
    a.S = S;
    a.tb = tb;
    a.near_k = (uint16_t*)near_k;
    a.near_v = (uint16_t*)near_v;
    a.far_k = far_k;
    a.far_v = far_v;
    a.fvs = (uint16_t*)far_v_scale;
    a.fvz = (uint16_t*)far_v_zero;
    a.near_valid = near_valid;
    a.arc_k = (uint16_t*)archive_k;
    a.arc_v = (uint16_t*)archive_v;
    a.kscale = nullptr;
    a.nt_in = true;
    return FKV_OK;
}

// Recency (near_idx == NULL) or indexed compress of one layer, with the
// per-head key scales computed first when cfg->k_scale is set.
int compress_launch(const char* fn, const fkv_tier_config* cfg, fkv::CompressArgs& a, int D, const int32_t* near_idx,
                    const int32_t* far_idx, float* far_k_scale, hipStream_t st) {
    const int B = a.B, H = a.H;
    const bool g32 = cfg->v_group == 32;
    if (cfg->k_scale) {
        if (!far_k_scale) return fkv::set_error(std::string(fn) + ": k_scale needs far_k_scale");
        const int F = a.tb.far_count;
        const int32_t* idx = near_idx ? far_idx : nullptr;
        auto pick = [&](auto ONE) {
            constexpr bool one = ONE.value;
            return a.dtype == FKV_F16    ? (D == 128 ? fkv::kscale_kernel<128, FKV_F16, one> : fkv::kscale_kernel<64, FKV_F16, one>)
                   : a.dtype == FKV_BF16 ? (D == 128 ? fkv::kscale_kernel<128, FKV_BF16, one> : fkv::kscale_kernel<64, FKV_BF16, one>)
                                         : (D == 128 ? fkv::kscale_kernel<128, FKV_F32, one> : fkv::kscale_kernel<64, FKV_F32, one>);
        };
        if (fkv::kscale_one(F, D)) {
            hipLaunchKernelGGL(pick(std::true_type{}), dim3(1, (unsigned)(B * H)), dim3(fkv::kScaleOneThreads), 0, st, a,
                               idx, far_k_scale);
        } else {
            // the far code buffer holds the workgroups' maxima until they are
            // reduced (the compress launch then writes the codes over them)
            const int parts = fkv::kscale_parts(F, D, B * H);
            float* part_max = (float*)a.far_k;
            hipLaunchKernelGGL(pick(std::false_type{}), dim3((unsigned)parts, (unsigned)(B * H)), dim3(fkv::kScaleThreads),
                               0, st, a, idx, part_max);
            hipLaunchKernelGGL(fkv::kscale_finish_kernel, dim3((unsigned)(B * H)), dim3(fkv::kWave), 0, st, part_max, parts,
                               far_k_scale);
        }
        a.kscale = far_k_scale;
    }
    const int rpb = 256 / (D / 8);
    // K and V are read once and the archive is written for later: both pass
    // the caches by, which leaves the tiers in the 256 MB last-level cache for
    // the blob packing that follows (4 x 8 heads x 8,192 tokens: compress 62 ->
    // 58 us, packing 32 -> 25). Tiers that would not stay there pass it by as
    // well (8 x 8 x 16K, 262 MB: 215 us with plain stores, 211 with the first
    // rule alone, 204 with both; 132 MB of tiers 121 with the first, 125 with
    // both): from three quarters of the cache on.
    const size_t tiers = (size_t)B * H * ((size_t)a.tb.n_near_padded * D * 4 + (size_t)a.tb.far_count * (D + D / 2));
    const bool nt = tiers > ((size_t)192 << 20);
    // the same line for float32 K and V, whose rows take two loads per lane:
    // what stays in that cache is better read through it (126 MB: 38 us, 43-45
    // past it, 42 before either; 150 MB 43-48, 52 and 48; 250 MB 79-80, 78 and
    // 86; 512 MB 162, 154 and 171)
    a.nt_in = (size_t)B * H * a.S * D * 8 > ((size_t)192 << 20);
    if (!near_idx) {
        const int rows = a.S + a.tb.headroom;
        dim3 grid((unsigned)fkv::cdiv(rows > 0 ? rows : 1, rpb), (unsigned)(B * H));
        auto pick = [&](auto NT) {
            return D == 128 ? (g32 ? fkv::compress_kernel<128, 32, NT.value> : fkv::compress_kernel<128, 0, NT.value>)
                            : (g32 ? fkv::compress_kernel<64, 32, NT.value> : fkv::compress_kernel<64, 0, NT.value>);
        };
        hipLaunchKernelGGL(nt ? pick(std::true_type{}) : pick(std::false_type{}), grid, dim3(256), 0, st, a);
        return fkv::check_hip(hipGetLastError(), "compress_kernel launch");
    }
    const int rows = a.tb.n_near_padded + a.tb.far_count;
    dim3 grid((unsigned)fkv::cdiv(rows > 0 ? rows : 1, rpb), (unsigned)(B * H));
    auto pick = [&](auto NT) {
        return D == 128 ? (g32 ? fkv::compress_gather_kernel<128, 32, NT.value> : fkv::compress_gather_kernel<128, 0, NT.value>)
                        : (g32 ? fkv::compress_gather_kernel<64, 32, NT.value> : fkv::compress_gather_kernel<64, 0, NT.value>);
    };
    hipLaunchKernelGGL(nt ? pick(std::true_type{}) : pick(std::false_type{}), grid, dim3(256), 0, st, a, near_idx,
                       far_idx);
    return fkv::check_hip(hipGetLastError(), "compress_gather_kernel launch");
}

}  // namespace

extern "C" int fkv_compress_layer(const fkv_tier_config* cfg, const void* keys, const void* values,
                                  int32_t in_dtype, int32_t B, int32_t H, int32_t S, int32_t D,
                                  void* near_k, void* near_v, uint8_t* far_k, uint8_t* far_v,
                                  void* far_v_scale, void* far_v_zero, int32_t* near_valid,
                                  void* archive_k, void* archive_v, void* stream) {
    fkv::CompressArgs a;
    if (int rc = compress_setup("fkv_compress_layer", cfg, keys, values, in_dtype, B, H, S, D, near_k, near_v, far_k,
                                far_v, far_v_scale, far_v_zero, near_valid, archive_k, archive_v, a))
        return rc;
    if (cfg->k_scale) return fkv::set_error("fkv_compress_layer: k_scale needs fkv_compress_layer_ex (far_k_scale)");
    return compress_launch("fkv_compress_layer", cfg, a, D, nullptr, nullptr, nullptr, (hipStream_t)stream);
}

extern "C" int fkv_partition_importance(const fkv_tier_config* cfg, const float* importance, int32_t B, int32_t H,
                                        int32_t S, int32_t* near_idx, int32_t* far_idx, void* stream) {
    using fkv::set_error;
    if (!cfg) return set_error("fkv_partition_importance: cfg is NULL");
    if (B <= 0 || H <= 0 || S < 0) return set_error("fkv_partition_importance: bad shape");
    fkv_tiers tb;
    if (int rc = fkv_tier_boundaries(cfg, S, &tb)) return rc;
    if ((S > 0 && !importance) || !near_idx || (tb.far_count > 0 && !far_idx))
        return set_error("fkv_partition_importance: NULL argument");
    // tokens per thread: the smallest compiled count that holds the middle
    // (a larger one adds a scalar test per empty register to every pass)
    const int64_t per = fkv::cdiv(tb.mid_end - tb.mid_start, fkv::kPartThreads);
    auto* kern = per <= 4    ? fkv::partition_regs_kernel<4>
                 : per <= 16 ? fkv::partition_regs_kernel<16>
                 : per <= fkv::kPartRegs ? fkv::partition_regs_kernel<fkv::kPartRegs>
                                         : fkv::partition_kernel;
    hipLaunchKernelGGL(kern, dim3((unsigned)(B * H)), dim3(fkv::kPartThreads), 0, (hipStream_t)stream, importance, S,
                       tb, near_idx, far_idx);
    return fkv::check_hip(hipGetLastError(), "partition_kernel launch");
}

extern "C" int fkv_tier_index_rows(const fkv_tiers* tiers, int32_t B, int32_t H, int32_t S, int32_t* near_idx,
                                   int32_t* far_idx, void* stream) {
    using fkv::set_error;
    if (!tiers) return set_error("fkv_tier_index_rows: tiers is NULL");
    const fkv_tiers tb = *tiers;
    if (B < 0 || H < 0 || S < 0 || tb.n_near_padded < 0 || tb.far_count < 0)
        return set_error("fkv_tier_index_rows: bad shape");
    const int64_t n = (int64_t)B * H * ((int64_t)tb.n_near_padded + tb.far_count);
    if (n == 0) return FKV_OK;
    if ((tb.n_near_padded > 0 && !near_idx) || (tb.far_count > 0 && !far_idx))
        return set_error("fkv_tier_index_rows: NULL argument");
    const int64_t blocks = fkv::cdiv(n, 256);
    hipLaunchKernelGGL(fkv::tier_index_kernel, dim3((unsigned)(blocks < 65536 ? blocks : 65536)), dim3(256), 0,
                       (hipStream_t)stream, tb, S, (int64_t)B * H, near_idx, far_idx);
    return fkv::check_hip(hipGetLastError(), "tier_index_kernel launch");
}

extern "C" int fkv_compress_layer_indexed(const fkv_tier_config* cfg, const void* keys, const void* values,
                                          int32_t in_dtype, int32_t B, int32_t H, int32_t S, int32_t D,
                                          const int32_t* near_idx, const int32_t* far_idx, void* near_k,
                                          void* near_v, uint8_t* far_k, uint8_t* far_v, void* far_v_scale,
                                          void* far_v_zero, int32_t* near_valid, void* archive_k, void* archive_v,
                                          void* stream) {
    fkv::CompressArgs a;
    if (int rc = compress_setup("fkv_compress_layer_indexed", cfg, keys, values, in_dtype, B, H, S, D, near_k, near_v,
                                far_k, far_v, far_v_scale, far_v_zero, near_valid, archive_k, archive_v, a))
        return rc;
    if (!near_idx || (a.tb.far_count > 0 && !far_idx))
        return fkv::set_error("fkv_compress_layer_indexed: NULL index array");
    if (cfg->k_scale)
        return fkv::set_error("fkv_compress_layer_indexed: k_scale needs fkv_compress_layer_ex (far_k_scale)");
    return compress_launch("fkv_compress_layer_indexed", cfg, a, D, near_idx, far_idx, nullptr, (hipStream_t)stream);
}

extern "C" int fkv_compress_layer_ex(const fkv_tier_config* cfg, const void* keys, const void* values,
                                     int32_t in_dtype, int32_t B, int32_t H, int32_t S, int32_t D,
                                     const int32_t* near_idx, const int32_t* far_idx, void* near_k, void* near_v,
                                     uint8_t* far_k, uint8_t* far_v, void* far_v_scale, void* far_v_zero,
                                     float* far_k_scale, int32_t* near_valid, void* archive_k, void* archive_v,
                                     void* stream) {
    fkv::CompressArgs a;
    if (int rc = compress_setup("fkv_compress_layer_ex", cfg, keys, values, in_dtype, B, H, S, D, near_k, near_v,
                                far_k, far_v, far_v_scale, far_v_zero, near_valid, archive_k, archive_v, a))
        return rc;
    if (!near_idx != !far_idx && a.tb.far_count > 0)
        return fkv::set_error("fkv_compress_layer_ex: near_idx and far_idx are both given or both NULL");
    return compress_launch("fkv_compress_layer_ex", cfg, a, D, near_idx, near_idx ? far_idx : nullptr, far_k_scale,
                           (hipStream_t)stream);
}

extern "C" int fkv_archive_layer(const fkv_tier_config* cfg, const void* keys, const void* values, int32_t in_dtype,
                                 int32_t B, int32_t H, int32_t S, int32_t D, const int32_t* near_idx,
                                 const int32_t* far_idx, void* near_k, void* near_v, int32_t* near_valid,
                                 void* archive_k, void* archive_v, void* stream) {
    fkv::CompressArgs a;
    if (int rc = compress_setup("fkv_archive_layer", cfg, keys, values, in_dtype, B, H, S, D, near_k, near_v, nullptr,
                                nullptr, nullptr, nullptr, near_valid, archive_k, archive_v, a, true))
        return rc;
    if (!near_idx != !far_idx && a.tb.far_count > 0)
        return fkv::set_error("fkv_archive_layer: near_idx and far_idx are both given or both NULL");
    if (cfg->k_scale) return fkv::set_error("fkv_archive_layer: there are no far keys to scale");
    return compress_launch("fkv_archive_layer", cfg, a, D, near_idx, near_idx ? far_idx : nullptr, nullptr,
                           (hipStream_t)stream);
}
