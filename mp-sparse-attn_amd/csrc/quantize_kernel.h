// The MX quantizer's per-workgroup body and its argument block, shared by quantize.hip (the stand-alone entry
// points) and prepare.hip (the one-launch operand preparation of the attention path).  The scheme is described at
// the top of quantize.hip.
#pragma once
#include "mpsa_common.h"
#include "mx_codec.h"
#include "midpoints.h"


struct QuantArgs {
    const void* x;
    const void* sub;           // optional [B,H,D] of x's dtype, subtracted (and the difference rounded to that dtype) first
    int64_t sb, sh, sn;        // element strides of x
    int n, d;                  // valid rows, row length
    int out_rows;              // rows per (b,h) in the outputs
    float pre;
    int sure4;                 // mpsa_e2m1_sure(pre, ...)
    int emax4, emax8;
    uint8_t *codes4, *scales4, *codes8, *scales8;
    int spread;                // 4-bit codes one per byte
    int scales5d;              // scales as [rows/128, D/128, 32, 4, 4] (rows and D in multiples of 128)
};

// host side, defined in quantize.hip
int mpsa_quantize_setup(const void* x, int x_dtype, int64_t B, int64_t H, int64_t N, int64_t D, const int64_t* xs,
                        const void* sub, float pre, bool do4, int emax4, bool do8, int fmt8, int emax8,
                        uint8_t* c4, uint8_t* s4, uint8_t* c8, uint8_t* s8, int64_t out_rows, QuantArgs* out, unsigned* blocks);
bool mpsa_quantize_sw_encoders();

namespace {


template <int DPP_CTRL>
__device__ __forceinline__ uint32_t dpp_u32(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, DPP_CTRL, 0xf, 0xf, true);
}

template <int FMT8, bool SW8>
__device__ __forceinline__ uint32_t fp8_pack4(float y0, float y1, float y2, float y3) {
    if constexpr (SW8) {
        if constexpr (FMT8 == MPSA_FMT_E4M3)
            return e4m3_encode_sw(y0) | (e4m3_encode_sw(y1) << 8) | (e4m3_encode_sw(y2) << 16) | (e4m3_encode_sw(y3) << 24);
        else
            return e5m2_encode_sw(y0) | (e5m2_encode_sw(y1) << 8) | (e5m2_encode_sw(y2) << 16) | (e5m2_encode_sw(y3) << 24);
    } else {
        int w = 0;
        if constexpr (FMT8 == MPSA_FMT_E4M3) {
            w = __builtin_amdgcn_cvt_pk_fp8_f32(y0, y1, w, false);
            w = __builtin_amdgcn_cvt_pk_fp8_f32(y2, y3, w, true);
        } else {
            w = __builtin_amdgcn_cvt_pk_bf8_f32(y0, y1, w, false);
            w = __builtin_amdgcn_cvt_pk_bf8_f32(y2, y3, w, true);
        }
        return (uint32_t)w;
    }
}

template <int XDT>
__device__ __forceinline__ void unpack8(const uint4& raw, float (&x)[8]) {
    const uint32_t w[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        if constexpr (XDT == MPSA_BF16) {
            x[2 * i] = mpsa_u2f(w[i] << 16);
            x[2 * i + 1] = mpsa_u2f(w[i] & 0xFFFF0000u);
        } else {
            x[2 * i] = (float)__builtin_bit_cast(_Float16, (unsigned short)(w[i] & 0xFFFFu));
            x[2 * i + 1] = (float)__builtin_bit_cast(_Float16, (unsigned short)(w[i] >> 16));
        }
    }
}

// round a float32 to the 16-bit dtype XDT (nearest even) and back
template <int XDT>
__device__ __forceinline__ float round16(float v) {
    if constexpr (XDT == MPSA_BF16) {
        const uint32_t u = mpsa_f2u(v);
        return mpsa_u2f((u + 0x7FFFu + ((u >> 16) & 1u)) & 0xFFFF0000u);
    } else {
        return (float)(_Float16)v;
    }
}

// Eight E2M1 codes (one packed word, element i in nibble i) of x[0..7] / 2^se.
// Fast path: v_cvt_scalef32_pk_fp4_f32 divides by the power of two and rounds to nearest, ties to even.  The
// reference's rule (argmin of float32 distances with 1e-6 taken off the even-mantissa candidate, e2m1_index in
// mx_codec.h) differs from that only for a value within about 1e-6 of the midpoint between two E2M1 values.
// The midpoints (0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5) have nothing but zeros below their first two mantissa bits, and dividing
// by a power of two leaves the mantissa alone: a value close to one shows in the low 21 bits of x itself.  A value whose bits
// are 128 units or more away from such a pattern is at least 1.9e-6 away from every midpoint (the smallest, 0.25, from below:
// 128 * 2^-26), and the conversion is the result.  That is one shift-and-add an element and half a minimum; converting
// the inputs twice, nudged down and up by 2^-17 of themselves, which this replaces, took two products and half a conversion (32 heads
// of 8192 x 128 14.9 -> 14.5 us).
// The pattern is that of the E2M1 values and of zero as well; so a lane that finds it converts the nudged inputs, and if
// they differ (a rounding boundary lies between) it takes the explicit rule.  (2^-17 of a value near a midpoint - the
// smallest is 0.25 - is at least 1.9e-6.)  Small scales, where x may be subnormal, take the explicit rule as well.
// Which values have the pattern the host can tell from the pre-scale: a product's mantissa depends on the two mantissas alone, and
// a 16-bit value has 128 or 1024 of them.  Where none has (63 of 64 pre-scales for bfloat16, seven of eight for float16), or the pre-scale is a
// power of two -- 16-bit inputs times a power of two, at most 11 significant bits, are either exactly a midpoint, where the two
// rules agree (both take the even mantissa), or at least 2^-12 away from one --, the check is skipped (`sure`).  It would otherwise
// fire on every exact tie, and on every zero: with half of the inputs zeros it did, 32 heads of 8192 x 128 16.5 us, with the check
// on other inputs 14.5, without it 14.0 either way.
constexpr int SMALLEST_SE = -100;      // x below 2^-126 is less than 2^-26 of a unit then: it rounds to zero in every format

__device__ __forceinline__ uint32_t e2m1_convert8(const float (&x)[8], int se, float f) {
    const float sc = mpsa_u2f((uint32_t)(se + 127) << 23);
    uint32_t w = 0;
    w = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(w, x[0] * f, x[1] * f, sc, 0);
    w = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(w, x[2] * f, x[3] * f, sc, 1);
    w = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(w, x[4] * f, x[5] * f, sc, 2);
    return __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(w, x[6] * f, x[7] * f, sc, 3);
}

// What a lane does whose conversion may not be the rule's result.  The explicit rule is rolled up (a hundred instructions, not
// seven hundred) and stands behind ONE branch instead of early returns and conditional blocks for every word.
__device__ __forceinline__ uint32_t e2m1_pack8_explicit(const float (&x)[8], int se) {
    float y[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) y[i] = x[i];
    uint32_t word = 0;
#pragma unroll 1
    for (int i = 0; i < 8; ++i) {
        word = (word >> 4) | (e2m1_encode(ldexpf(y[0], -se)) << 28);
#pragma unroll
        for (int j = 0; j + 1 < 8; ++j) y[j] = y[j + 1];
    }
    return word;
}

__device__ __forceinline__ uint32_t e2m1_pack8_rule(const float (&x)[8], int se) {
    // no boundary between the two nudged values: the value itself converts to the same codes
    const uint32_t w = e2m1_convert8(x, se, 1.0f - 0x1p-17f);
    if (se >= SMALLEST_SE && w == e2m1_convert8(x, se, 1.0f + 0x1p-17f)) return w;
    return e2m1_pack8_explicit(x, se);
}

// the conversion, and whether e2m1_pack8_rule has to look at it instead.  STRAIGHT: the check is made and not used instead of
// branched around.
template <bool STRAIGHT = false>
__device__ __forceinline__ uint32_t e2m1_try8(const float (&x)[8], int se, bool sure, bool& rule) {
    rule = se < SMALLEST_SE;
    if (STRAIGHT || !sure) {
        uint32_t nearest = ~0u;
#pragma unroll
        for (int i = 0; i < 8; ++i) nearest = min(nearest, (mpsa_f2u(x[i]) << 11) + MIDPOINT_NEAR);
        rule |= nearest < 2 * MIDPOINT_NEAR && !sure;
    }
    return e2m1_convert8(x, se, 1.0f);
}

// Eight FP8 codes of x[0..7] / 2^se.  The scaled conversion divides and rounds in one instruction a pair.  With the formats' own
// emax (7) a finite block's values lie below 256 and never meet the format's maximum; what does -- a NaN, or a larger value
// under another emax -- shows in the codes (fp8_past).
template <int FMT8>
__device__ __forceinline__ uint2 fp8_convert8(const float (&x)[8], int se) {
    typedef short v2s __attribute__((ext_vector_type(2)));
    const float sc = mpsa_u2f((uint32_t)(se + 127) << 23);
    v2s lo = {0, 0}, hi = {0, 0};
    if constexpr (FMT8 == MPSA_FMT_E4M3) {
        lo = __builtin_amdgcn_cvt_scalef32_pk_fp8_f32(lo, x[0], x[1], sc, false);
        lo = __builtin_amdgcn_cvt_scalef32_pk_fp8_f32(lo, x[2], x[3], sc, true);
        hi = __builtin_amdgcn_cvt_scalef32_pk_fp8_f32(hi, x[4], x[5], sc, false);
        hi = __builtin_amdgcn_cvt_scalef32_pk_fp8_f32(hi, x[6], x[7], sc, true);
    } else {
        lo = __builtin_amdgcn_cvt_scalef32_pk_bf8_f32(lo, x[0], x[1], sc, false);
        lo = __builtin_amdgcn_cvt_scalef32_pk_bf8_f32(lo, x[2], x[3], sc, true);
        hi = __builtin_amdgcn_cvt_scalef32_pk_bf8_f32(hi, x[4], x[5], sc, false);
        hi = __builtin_amdgcn_cvt_scalef32_pk_bf8_f32(hi, x[6], x[7], sc, true);
    }
    return make_uint2(__builtin_bit_cast(uint32_t, lo), __builtin_bit_cast(uint32_t, hi));
}

// Whether a code is the format's NaN or E5M2's infinity: three instructions a word, where clamping first takes one an element.
template <int FMT8>
__device__ __forceinline__ bool fp8_past(const uint2& w) {
    constexpr uint32_t UP = FMT8 == MPSA_FMT_E4M3 ? 0x01010101u : 0x04040404u;       // the first such code to 0x80
    return ((((w.x & 0x7F7F7F7Fu) + UP) | ((w.y & 0x7F7F7F7Fu) + UP)) & 0x80808080u) != 0u;
}

// the same one step at a time, with the clamp to the format's maximum: infinities and larger values saturate there, a NaN at
// its negative
template <int FMT8, bool SW8>
__device__ __forceinline__ uint2 fp8_careful8(const float (&x)[8], int se) {
    const float lim = (FMT8 == MPSA_FMT_E4M3) ? 448.0f : 57344.0f;
    float y[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) y[i] = __builtin_fminf(__builtin_fmaxf(ldexpf(x[i], -se), -lim), lim);
    return make_uint2(fp8_pack4<FMT8, SW8>(y[0], y[1], y[2], y[3]), fp8_pack4<FMT8, SW8>(y[4], y[5], y[6], y[7]));
}

// whether a block of largest magnitude 2^e or more wants fp8_careful8 whatever its codes: infinities, and scales that are no
// normal float32
__device__ __forceinline__ bool fp8_odd(int e, int se) { return e >= 128 || se < SMALLEST_SE || se > 127; }

// floor(log2(amax)) of a block's largest magnitude, subnormals included; -1 for a block of zeros (whose codes and scale are
// zero whatever it says)
__device__ __forceinline__ int block_exponent(float amax) {
    const int biased = (int)(mpsa_f2u(amax) >> 23), tiny = __builtin_amdgcn_frexp_expf(amax) - 1;
    return biased ? biased - 127 : tiny;
}

// One lane's eight elements (a quarter of an MX block; the quad's other lanes hold the rest): codes and the block's scale
// bytes in the formats asked for.  x comes back multiplied by `pre`, e is the block's exponent.  Where `again` comes back
// true, the caller has quantize_again finish the chunk: several chunks in a row share one branch that way, and run interleaved.
// CLAMP8: the 8-bit codes are the careful ones at once, and never a reason for `again`: what quantize_straight's callers take rare
// blocks to.
template <bool DO4, bool DO8, int FMT8, bool SW8, bool CLAMP8 = false>
__device__ __forceinline__ void quantize_most(float (&x)[8], float pre, bool sure, int emax4, int emax8, uint32_t& w4, int& s4, uint2& w8, int& s8, bool& again, int& e) {
    float amax = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        x[i] = x[i] * pre;
        amax = __builtin_fmaxf(amax, __builtin_fabsf(x[i]));
    }
    // magnitudes order like their bits
    uint32_t ab = mpsa_f2u(amax);
    ab = max(ab, dpp_u32<0xB1>(ab));                      // quad_perm [1,0,3,2]
    ab = max(ab, dpp_u32<0x4E>(ab));                      // quad_perm [2,3,0,1]
    const bool zero = ab == 0u;
    e = block_exponent(mpsa_u2f(ab));
    w4 = 0u; s4 = 0;
    w8 = make_uint2(0u, 0u); s8 = 0;
    again = SW8;
    if constexpr (DO4) {
        const int se = e - emax4;
        if constexpr (!SW8) {
            w4 = e2m1_try8(x, se, sure, again);
            w4 = zero ? 0u : w4;
        }
        s4 = zero ? 0 : min(max(se + 127, 0), 254);
    }
    if constexpr (DO8) {
        const int se = e - emax8;
        if constexpr (!SW8) {
            w8 = CLAMP8 ? fp8_careful8<FMT8, false>(x, se) : fp8_convert8<FMT8>(x, se);
            w8.x = zero ? 0u : w8.x;
            w8.y = zero ? 0u : w8.y;
            if constexpr (!CLAMP8) again |= fp8_odd(e, se) || fp8_past<FMT8>(w8);
        }
        s8 = zero ? 0 : min(max(se + 127, 0), 254);
    }
    again &= !zero;
}

template <bool DO4, bool DO8, int FMT8, bool SW8>
__device__ __forceinline__ void quantize_again(const float (&x)[8], int e, int emax4, int emax8, bool sure, uint32_t& w4, uint2& w8) {
    if constexpr (DO4) {
        bool rule = true;
        if constexpr (DO8 && !SW8) (void)e2m1_try8(x, e - emax4, sure, rule);
        if (rule) w4 = SW8 ? e2m1_pack8_explicit(x, e - emax4) : e2m1_pack8_rule(x, e - emax4);
    }
    if constexpr (DO8) {
        if (SW8 || fp8_odd(e, e - emax8) || fp8_past<FMT8>(w8)) w8 = fp8_careful8<FMT8, SW8>(x, e - emax8);
    }
}

template <bool DO4, bool DO8, int FMT8, bool SW8, bool CLAMP8>
__device__ __forceinline__ void quantize_chunk(float (&x)[8], float pre, bool sure, int emax4, int emax8, uint32_t& w4, int& s4, uint2& w8, int& s8) {
    bool again;
    int e;
    quantize_most<DO4, DO8, FMT8, SW8, CLAMP8>(x, pre, sure, emax4, emax8, w4, s4, w8, s8, again, e);
    if (again) quantize_again<DO4, DO8 && !CLAMP8, FMT8, SW8>(x, e, emax4, emax8, sure, w4, w8);
}

// What nearly every block is, without a branch: the shared exponents from the bits of the largest magnitude, by a maximum that NaN goes
// through.  `rare`: a NaN, an infinity, or a scale so small that elements may be subnormal; nothing else here is to be used then.
// The scale bytes of the others need no clamp, and their 8-bit codes stay below the format's maximum (emax 7).
struct BlockScale {
    static constexpr int EMAX4 = 3, EMAX8 = 7;
    int biased;
    bool zero, rare;
    __device__ __forceinline__ int se4() const { return biased - EMAX4 - 127; }
    __device__ __forceinline__ int se8() const { return biased - EMAX8 - 127; }
    __device__ __forceinline__ int s4() const { return zero ? 0 : biased - EMAX4; }
    __device__ __forceinline__ int s8() const { return zero ? 0 : biased - EMAX8; }
};
__device__ __forceinline__ BlockScale block_scale(uint32_t amax_bits) {
    constexpr uint32_t LOW = (uint32_t)(SMALLEST_SE + 127 + BlockScale::EMAX8) << 23;
    return {(int)(amax_bits >> 23), amax_bits == 0u, amax_bits != 0u && amax_bits - LOW >= 0x7F800000u - LOW};
}

// quantize_most that way, with half of its instructions (60 and 115 a chunk in both formats), so that several chunks run interleaved:
// x holds products with the pre-scale; that none is near a midpoint is the caller's to know (`sure`).  Where `rare` comes back true
// the caller takes the whole wave's chunks to quantize_chunk.  Whole calls, us: 32 query heads over 8, D = 128, causal, diag, 400 tokens
// 12.8 -> 12.3, 1500 32.4 -> 31.1; 2 x 16 heads, 4096 queries over 333 keys, 8-bit, 39.1 -> 37.7.
template <bool DO4, bool DO8, int FMT8>
__device__ __forceinline__ void quantize_straight(const float (&x)[8], uint32_t& w4, int& s4, uint2& w8, int& s8, bool& rare) {
    float amax = __builtin_fabsf(x[0]);
#pragma unroll
    for (int i = 1; i < 8; ++i) amax = __builtin_elementwise_maximum(amax, __builtin_fabsf(x[i]));
    uint32_t ab = mpsa_f2u(amax);
    ab = max(ab, dpp_u32<0xB1>(ab));                      // quad_perm [1,0,3,2]
    ab = max(ab, dpp_u32<0x4E>(ab));                      // quad_perm [2,3,0,1]
    const BlockScale b = block_scale(ab);
    rare = b.rare;
    if constexpr (DO4) {
        s4 = b.s4();
        w4 = e2m1_convert8(x, b.se4(), 1.0f);
        w4 = b.zero ? 0u : w4;
    }
    if constexpr (DO8) {
        s8 = b.s8();
        w8 = fp8_convert8<FMT8>(x, b.se8());
        w8.x = b.zero ? 0u : w8.x;
        w8.y = b.zero ? 0u : w8.y;
    }
}

// x, but nothing that is computed from it can be computed elsewhere: what only a rare path wants stays in it
__device__ __forceinline__ uint4 only_here(uint4 x) {
    asm("" : "+v"(x.x), "+v"(x.y), "+v"(x.z), "+v"(x.w));
    return x;
}

// The chunk of 16 bytes that a thread quantizes: number c of a head's, in the outputs; rows past the last count as zeros.
struct QuantChunk {
    uint32_t c, row, col8;
    uint4 raw;
    __device__ __forceinline__ QuantChunk(const QuantArgs& a, uint32_t number) : c(number) {
        const uint32_t cpr = (uint32_t)a.d >> 3;                          // 16-byte chunks per row
        row = c / cpr;
        col8 = c - row * cpr;
    }
    __device__ __forceinline__ bool inside(const QuantArgs& a) const { return row < (uint32_t)a.n; }
    __device__ __forceinline__ const uint4* at(const QuantArgs& a, uint32_t r, uint32_t hh, uint32_t bb) const {
        return reinterpret_cast<const uint4*>(static_cast<const char*>(a.x) + 2 * ((int64_t)bb * a.sb + (int64_t)hh * a.sh + (int64_t)r * a.sn + 8 * (int64_t)col8));
    }
    // from a head with a row; what lies past the last one is left to quantize_chunks
    __device__ __forceinline__ void request(const QuantArgs& a, uint32_t hh, uint32_t bb) { raw = *at(a, min(row, (uint32_t)a.n - 1u), hh, bb); }
};

// head: the flat (batch, head)
template <bool DO4, bool DO8>
__device__ __forceinline__ void store_chunk(const QuantArgs& a, const QuantChunk& q, int64_t head, uint32_t w4, int s4, uint2 w8, int s8) {
    const uint32_t cpr = (uint32_t)a.d >> 3, chunks = (uint32_t)a.out_rows * cpr;
    const int64_t oc = head * chunks + q.c;                               // flat output chunk
    int64_t os = oc >> 2;                                                 // and scale
    if (a.scales5d) {
        const uint32_t kc = cpr >> 4, block = q.col8 >> 2;
        os = head * (chunks >> 2) + (((int64_t)(q.row >> 7) * kc + (block >> 2)) << 9) + ((q.row & 31) << 4) + ((q.row >> 5 & 3) << 2) + (block & 3);
    }
    const bool quad_leader = (threadIdx.x & 3u) == 0u;
    // an output set that is not wanted has no pointer (one side of a mixed preparation: 8-bit Q, 4-bit K)
    if (DO4 && a.codes4) {
        if (a.spread) reinterpret_cast<uint2*>(a.codes4)[oc] = make_uint2(spread_nibbles(w4 & 0xFFFFu), spread_nibbles(w4 >> 16));
        else          reinterpret_cast<uint32_t*>(a.codes4)[oc] = w4;
        if (quad_leader) a.scales4[os] = (uint8_t)s4;
    }
    if (DO8 && a.codes8) {
        reinterpret_cast<uint2*>(a.codes8)[oc] = w8;
        if (quad_leader) a.scales8[os] = (uint8_t)s8;
    }
}

// Several chunks of a thread, straight through (the formats' own emax): the preparation's form.
// subtract(head, col8, x): what is taken off a row's chunk before anything else.
template <int XDT, bool DO4, bool DO8, int FMT8, int N, typename Subtract>
__device__ __forceinline__ void quantize_chunks(const QuantArgs& a, const QuantChunk (&q)[N], int64_t head, Subtract subtract) {
    uint32_t w4[N];
    uint2 w8[N];
    int s4[N], s8[N];
    bool again = DO4 && !a.sure4;
    if (!again) {
        bool rare = false;
#pragma unroll
        for (int i = 0; i < N; ++i) {
            float x[8];
            bool r;
            unpack8<XDT>(q[i].raw, x);
            subtract(head, q[i].col8, x);
            const float pre = q[i].inside(a) ? a.pre : 0.0f;
#pragma unroll
            for (int e = 0; e < 8; ++e) x[e] *= pre;
            w4[i] = 0; s4[i] = 0; w8[i] = make_uint2(0, 0); s8[i] = 0;
            quantize_straight<DO4, DO8, FMT8>(x, w4[i], s4[i], w8[i], s8[i], r);
            rare |= r;
        }
        again = __ballot(rare) != 0;
    }
    if (again) {
#pragma unroll
        for (int i = 0; i < N; ++i) {
            float x[8];
            unpack8<XDT>(only_here(q[i].raw), x);
            subtract(head, q[i].col8, x);
#pragma unroll
            for (int e = 0; e < 8; ++e) x[e] = q[i].inside(a) ? x[e] : 0.0f;
            quantize_chunk<DO4, DO8, FMT8, false, true>(x, a.pre, a.sure4 != 0, a.emax4, a.emax8, w4[i], s4[i], w8[i], s8[i]);
        }
    }
    const uint32_t chunks = (uint32_t)a.out_rows * ((uint32_t)a.d >> 3);
#pragma unroll
    for (int i = 0; i < N; ++i)
        if (q[i].c < chunks) store_chunk<DO4, DO8>(a, q[i], head, w4[i], s4[i], w8[i], s8[i]);       // (whole waves)
}

// x - m in the inputs' 16-bit type
template <int XDT>
__device__ __forceinline__ void less_mean(float (&x)[8], const uint4& mean) {
    float m[8];
    unpack8<XDT>(mean, m);
#pragma unroll
    for (int i = 0; i < 8; ++i) x[i] = round16<XDT>(x[i] - m[i]);
}

// takes the mean that the caller has at hand off a chunk (quantize_chunks)
template <int XDT>
__device__ __forceinline__ void less_given(const QuantArgs& a, int64_t head, uint32_t col8, float (&x)[8]) {
    if (a.sub) less_mean<XDT>(x, *reinterpret_cast<const uint4*>(static_cast<const char*>(a.sub) + 2 * (head * a.d + 8 * (int64_t)col8)));
}

// One workgroup's share in the stand-alone kernels: 256 consecutive 16-byte chunks, starting at chunk 256*bx, of head hh of batch bb
// (nh heads).
template <int XDT, bool DO4, bool DO8, int FMT8, bool SW8>
__device__ __forceinline__ void quantize_block(const QuantArgs& a, uint32_t bx, uint32_t hh, uint32_t bb, uint32_t nh) {
    QuantChunk q(a, bx * 256u + threadIdx.x);
    if (q.c >= (uint32_t)a.out_rows * ((uint32_t)a.d >> 3)) return;       // whole quads leave together (d % 32 == 0)
    const int64_t head = (int64_t)bb * nh + hh;                           // flat (b,h)
    float x[8];
    if (q.inside(a)) {
        unpack8<XDT>(*q.at(a, q.row, hh, bb), x);
        less_given<XDT>(a, head, q.col8, x);
    } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) x[i] = 0.0f;
    }
    uint32_t w4;
    uint2 w8;
    int s4, s8;
    quantize_chunk<DO4, DO8, FMT8, SW8, false>(x, a.pre, a.sure4 != 0, a.emax4, a.emax8, w4, s4, w8, s8);
    store_chunk<DO4, DO8>(a, q, head, w4, s4, w8, s8);
}

template <int XDT, bool DO4, bool DO8, int FMT8, bool SW8>
__global__ __launch_bounds__(256) void quantize_kernel(QuantArgs a) {
    // two 256-chunk blocks per workgroup: both loads are in flight before either block is converted
    quantize_block<XDT, DO4, DO8, FMT8, SW8>(a, 2 * blockIdx.x, blockIdx.y, blockIdx.z, gridDim.y);
    quantize_block<XDT, DO4, DO8, FMT8, SW8>(a, 2 * blockIdx.x + 1, blockIdx.y, blockIdx.z, gridDim.y);
}

}  // namespace
