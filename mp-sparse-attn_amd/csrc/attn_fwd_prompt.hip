// Fused attention forward for the shortest sequences (gfx950): from unquantized Q, K and V in one launch.
//
// What bounds a call over a few hundred keys is launches: the preparation of K and V and the kernel that waits for it each take
// a few microseconds of a wait for memory, and the host as long for either.  Here a workgroup makes its operands itself: it quantizes
// its queries and all of the keys it will see into LDS, each block of 32 keys in the one precision its queries want, and V's elements go
// straight from their rows into the operand order of the P.V product.  Every workgroup of a head does that again, which is what
// bounds the number of keys that pay (attn_prompt_supported).
// Workgroups, splits, arithmetic and merge are those of the four-split kernel of attn_fwd_short.hip, and so are the bits: four
// waves share 32 queries, wave s takes the key blocks s, s + 4, ...  What does not come here: mpsa_prepare_operands and attn_fwd_short.hip.
// The keys are quantized together, and by eight waves, two a SIMD, half of which end with that: a lone wave issues little more than half
// as many instructions as two.  Kernels alone, us (32 heads over 8, causal, diag, 160 tokens; the preparation and the four-split kernel
// 8.6): 7.2; quantized by four waves 8.9; by every wave for itself, in registers, 9.2 (16 bytes of every 64 a lane are
// read, and one wave has two blocks to do where three have one).  Whole calls, two launches -> one: 160 tokens, 32 heads over 8, diag 10.8 ->
// 7.8, 4-bit 11.0 -> 7.8, 256 tokens 10.8 -> 8.7; 24 heads, 300 queries over 256 keys, 8-bit, 10.6 -> 8.6; 1000 queries over 77 keys, 8 heads 10.6 -> 7.9.
// These are calls repeated on the same tensors, one queued behind the other; a call that is waited for, with its inputs in memory instead
// of the caches, 18.1 -> 15.1 (4-bit, 160 tokens).  What bounds the 7.8 is the kernel again (a call that allocates no workspace takes as long).  Its
// longest wave takes 14 200 clocks: 2 100 until all loads are asked for, 650 for its queries, 3 000 for five blocks of keys, 1 100 to the first
// scores, 2 300 for two blocks of scores, one after the other, and 2 800 for the merge; with inputs in memory 16 500.
#include "attn_common.h"
#include "seq_mean_kernel.h"
#include "reciprocal.h"

namespace {

struct PromptArgs : AttnArgs {
    const char *k_raw, *v_raw;
    int64_t k_sb, k_sh, k_sn, v_sb, v_sh, v_sn;
    Reciprocal by_units, by_group, by_hkv;
    int units, group, nqb, k_sure;
    float inv_n;
};

constexpr int KS = 4, D = 128, UNITS = D / 16 / KS;              // splits; 16-dim units each split finishes
constexpr int THREADS = 512;                                     // a chunk of eight elements each of 32 rows; only the first KS waves go on to the scores
constexpr int MAX_BLOCKS = 8;                                    // of 32 keys
constexpr int PART = (KS - 1) * UNITS * 2 * 64;                  // 16-byte words of partial output a wave leaves

// Operands of the score product in LDS: rows of 64 (4-bit) or 128 bytes, 16-byte pieces swizzled so that 16 consecutive rows lie in
// different banks, then four scale bytes a row.  Queries of both widths, then blocks of 32 keys, each of one width.
template <int MODE> struct Prompt {
    static constexpr bool DIAG = MODE == MPSA_MODE_DIAG, MIXED = MODE == MPSA_MODE_MIXED;
    static constexpr bool Q4 = MODE == MPSA_MODE_MXFP4 || DIAG, Q8 = MODE != MPSA_MODE_MXFP4, K4 = MODE != MPSA_MODE_MXFP8, K8 = DIAG || !K4;
    static constexpr int ROWS4 = 32 * 64, ROWS8 = 32 * 128, SCALES = 32 * 4;
    static constexpr int Q8AT = Q4 ? ROWS4 + SCALES : 0, KAT = Q8AT + (Q8 ? ROWS8 + SCALES : 0), KBLOCK = (K8 ? ROWS8 : ROWS4) + SCALES;
    static constexpr int OPERANDS = KAT + MAX_BLOCKS * KBLOCK, MERGE = KS * PART * 16;
    static constexpr int SMEM = OPERANDS > MERGE ? OPERANDS : MERGE;
};
// the four bytes of a chunk of eight 4-bit codes, or the eight of 8-bit ones, chunk c of row r
__device__ __forceinline__ int at4(int r, int c) { return r * 64 + (((c >> 2) ^ ((r >> 2) & 3)) << 4) + 4 * (c & 3); }
__device__ __forceinline__ int at8(int r, int c) { return r * 128 + (((c >> 1) ^ ((r >> 1) & 7)) << 4) + 8 * (c & 1); }

template <int PVT, int FMT8, int MODE, bool SMOOTH>
__global__ __launch_bounds__(THREADS, 2) void attn_prompt_kernel(PromptArgs a) {
    typedef PV<PVT> P;
    typedef Prompt<MODE> G;
    __shared__ __attribute__((aligned(16))) uint8_t smem[G::SMEM];
    __shared__ float ml[KS * 64];                                // [split][maximum, sum][query]
    __shared__ __attribute__((aligned(16))) uint16_t mean[SMOOTH ? D : 8];
    v4f* const parts = reinterpret_cast<v4f*>(smem);
    const int tid = threadIdx.x, lane = tid & 63, split = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int h = lane >> 5, r = lane & 31;
    // one (batch, KV head)'s workgroups on one XCD where their number allows it; causal: long rows first
    const int row = divide_by((int)blockIdx.x, a.by_units), unit = (int)blockIdx.x - row * a.units;
    const int rank = divide_by(row, a.by_group), sub = row - rank * a.group;
    const int b = divide_by(unit, a.by_hkv), kvh = unit - b * a.Hkv, hq = kvh * a.group + sub;
    const int qb = a.causal ? a.nqb - 1 - rank : rank;
    const int nb = (a.n + 31) / 32, mine = a.causal ? min(qb + 1, nb) : nb;
    const int masked_kb = a.causal ? qb : (a.n & 31) ? nb - 1 : -1;
    const int own_first = a.tile == 128 ? qb & ~3 : qb & ~1, own_end = own_first + a.tile / 32;

    const char* const kg = a.k_raw + 2 * ((int64_t)b * a.k_sb + (int64_t)kvh * a.k_sh);
    const char* const vg = a.v_raw + 2 * ((int64_t)b * a.v_sb + (int64_t)kvh * a.v_sh) + 4 * r;
    // thread t takes chunk t % 16 (eight elements) of row t / 16 of a block of 32
    const int crow = tid >> 4, chunk = tid & 15;
    auto request = [&](const char* base, int64_t sn, int row0, int n) __attribute__((always_inline)) {
        return *reinterpret_cast<const uint4*>(base + 2 * (int64_t)min(row0 + crow, n - 1) * sn + 16 * chunk);
    };
    auto request_k = [&](int kb) __attribute__((always_inline)) { return request(kg, a.k_sn, 32 * kb, a.n); };
    // V: lane r holds dims 64 g + 2 r and the next one of the keys that the P.V product's k index wants from its half
    auto key_at = [&](int kb, int c, int t) { return 32 * kb + 16 * c + 4 * h + 8 * (t >> 2) + (t & 3); };
    auto request_v = [&](int kb, uint32_t (&v)[2][2][8]) __attribute__((always_inline)) {
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int t = 0; t < 8; ++t) {
                const char* const p = vg + 2 * (int64_t)min(key_at(kb, c, t), a.n - 1) * a.v_sn;
#pragma unroll
                for (int g = 0; g < 2; ++g) v[c][g][t] = *reinterpret_cast<const uint32_t*>(p + 128 * g);
            }
    };

    const uint4 q = request(static_cast<const char*>(a.q_raw) + 2 * ((int64_t)b * a.q_sb + (int64_t)hq * a.q_sh), a.q_sn, 32 * qb, a.nq);
    uint4 k[MAX_BLOCKS];
#pragma unroll
    for (int x = 0; x < MAX_BLOCKS; ++x)
        if (x < mine) k[x] = request_k(x);
    uint32_t v[2][2][8], v_next[2][2][8];
    if (split < KS && split < mine) request_v(split, v);
    if (split < KS && split + KS < mine) request_v(split + KS, v_next);
    MeanChunk<D> head;
    if (SMOOTH && tid < 256) head.request(kg, a.k_sn, 0, a.n, tid);
    __builtin_amdgcn_sched_barrier(0);

    // ---- the mean over the head's keys: the additions of mpsa_seq_mean, one chunk of MEAN_ROWS, in their order ----
    if constexpr (SMOOTH) {
        static_assert(32 * MAX_BLOCKS <= MEAN_ROWS && sizeof(float[256][9]) <= G::SMEM, "one chunk; its sums lie where the operands will");
        float (&part)[256][9] = *reinterpret_cast<float (*)[256][9]>(smem);
        if (tid < 256) head.template add<PVT>(part, 0, a.n, tid);
        __syncthreads();
        if (tid < D) mean[tid] = mean_bits<PVT>((0.0f + MeanChunk<D>::total(part, tid)) * a.inv_n);
        __syncthreads();
    }

    // ---- operands of the score product into LDS: straight through, and where a wave has a rare chunk, or 4-bit codes are the rule's
    //      to look at, again the careful way (quantize_kernel.h).  Rows past the last are zeros, like the quantizer's padding. ----
    auto put = [&](auto do4, auto do8, auto key, const uint4& y, int row0, int n, float pre, bool sure, uint8_t* to4, uint8_t* to8) __attribute__((always_inline)) {
        constexpr bool DO4 = decltype(do4)::value, DO8 = decltype(do8)::value;
        const bool inside = row0 + crow < n;
        auto values = [&](const uint4& raw, float (&x)[8]) __attribute__((always_inline)) {
            unpack8<PVT>(raw, x);
            if constexpr (SMOOTH && decltype(key)::value) less_mean<PVT>(x, *reinterpret_cast<const uint4*>(mean + 8 * chunk));
#pragma unroll
            for (int e = 0; e < 8; ++e) x[e] = inside ? x[e] : 0.0f;
        };
        float x[8];
        uint32_t w4 = 0;
        uint2 w8 = make_uint2(0, 0);
        int s4 = 0, s8 = 0;
        bool again = DO4 && !sure;
        if (!again) {
            bool rare;
            values(y, x);
#pragma unroll
            for (int e = 0; e < 8; ++e) x[e] *= pre;
            quantize_straight<DO4, DO8, FMT8>(x, w4, s4, w8, s8, rare);
            again = __ballot(rare) != 0;
        }
        if (again) {
            values(only_here(y), x);
            quantize_chunk<DO4, DO8, FMT8, false, true>(x, pre, sure, 3, 7, w4, s4, w8, s8);
        }
        if constexpr (DO4) {
            *reinterpret_cast<uint32_t*>(to4 + at4(crow, chunk)) = w4;
            to4[G::ROWS4 + 4 * crow + (chunk >> 2)] = (uint8_t)s4;
        }
        if constexpr (DO8) {
            *reinterpret_cast<uint2*>(to8 + at8(crow, chunk)) = w8;
            to8[G::ROWS8 + 4 * crow + (chunk >> 2)] = (uint8_t)s8;
        }
    };
    put(std::bool_constant<G::Q4>{}, std::bool_constant<G::Q8>{}, std::false_type{}, q, 32 * qb, a.nq, a.q_pre, a.q_sure != 0, smem, smem + G::Q8AT);
#pragma unroll 1
    for (int kb = 0; kb < mine; ++kb) {
        uint8_t* const to = smem + G::KAT + kb * G::KBLOCK;
        if (!G::K4 || (G::DIAG && kb >= own_first && kb < own_end)) put(std::false_type{}, std::true_type{}, std::true_type{}, k[0], 32 * kb, a.n, 1.0f, true, nullptr, to);
        else if constexpr (G::K4)                                   put(std::true_type{}, std::false_type{}, std::true_type{}, k[0], 32 * kb, a.n, 1.0f, a.k_sure != 0, to, nullptr);
#pragma unroll
        for (int x = 0; x < MAX_BLOCKS - 1; ++x) k[x] = k[x + 1];
    }
    __syncthreads();
    if (split >= KS) return;                                     // (the barriers below wait for the waves that are left)
    // row r's operand of step s, and its scale word
    auto load4 = [&](const uint8_t* from, v8i (&y)[2], uint32_t& scales) __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const v4i x = *reinterpret_cast<const v4i*>(from + at4(r, 4 * (2 * s + h)));
            y[s] = (v8i){x[0], x[1], x[2], x[3], 0, 0, 0, 0};
        }
        scales = *reinterpret_cast<const uint32_t*>(from + G::ROWS4 + 4 * r) >> (8 * h);
    };
    auto load8 = [&](const uint8_t* from, v8i (&y)[2], uint32_t& scales) __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const v4i x0 = *reinterpret_cast<const v4i*>(from + at8(r, 2 * (4 * s + h))), x1 = *reinterpret_cast<const v4i*>(from + at8(r, 2 * (4 * s + h + 2)));
            y[s] = (v8i){x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]};
        }
        scales = *reinterpret_cast<const uint32_t*>(from + G::ROWS8 + 4 * r) >> (8 * h);
    };
    v8i q4f[2], q8f[2];
    uint32_t qs4 = 0, qs8 = 0;
    if constexpr (G::Q4) load4(smem, q4f, qs4);
    if constexpr (G::Q8) load8(smem + G::Q8AT, q8f, qs8);

    // lane (h, r): acc[2 g + x][e] is dim 64 g + 2 i + x of query r, i = 8 (e >> 2) + 4 h + (e & 3)
    v16f acc[4], minus_m;
#pragma unroll
    for (int d = 0; d < 4; ++d)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[d][e] = 0.0f;
#pragma unroll
    for (int e = 0; e < 16; ++e) minus_m[e] = 0.0f;
    float m_run = 0.0f, l_run = 0.0f;
#pragma unroll 1
    for (int kb = split; kb < mine; kb += KS) {
        // ---- scores ----
        v16f st = minus_m;
        const uint8_t* const from = smem + G::KAT + kb * G::KBLOCK;
        v8i kf[2];
        uint32_t ks;
        if (!G::K4 || (G::DIAG && kb >= own_first && kb < own_end)) {
            load8(from, kf, ks);
#pragma unroll
            for (int s = 0; s < 2; ++s) st = score_mfma8<FMT8>(kf[s], q8f[s], st, s, (int)ks, (int)qs8);
        } else if constexpr (G::K4) {
            load4(from, kf, ks);
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                if constexpr (G::MIXED) st = score_mfma48<FMT8>(kf[s], q8f[s], st, s, (int)ks, (int)qs8);
                else                    st = score_mfma4(kf[s], q4f[s], st, s, (int)ks, (int)qs4);
            }
        }
        // ---- V's operands, while the scores are on their way ----
        typename P::vec vf[2][4];
        const bool ragged = 32 * kb + 32 > a.n;
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int g = 0; g < 2; ++g) {
                uint32_t (&two)[8] = v[c][g];
                if (ragged) {
#pragma unroll
                    for (int t = 0; t < 8; ++t) two[t] = key_at(kb, c, t) < a.n ? two[t] : 0u;
                }
                v4i even, odd;
#pragma unroll
                for (int y = 0; y < 4; ++y) {
                    even[y] = (int)__builtin_amdgcn_perm(two[2 * y + 1], two[2 * y], 0x05040100u);
                    odd[y] = (int)__builtin_amdgcn_perm(two[2 * y + 1], two[2 * y], 0x07060302u);
                }
                vf[c][2 * g] = __builtin_bit_cast(typename P::vec, even);
                vf[c][2 * g + 1] = __builtin_bit_cast(typename P::vec, odd);
            }
        // ---- probabilities: against the old maximum at once; maximum first in a wave's first block, in a masked one, and where a
        //      row sum shows a score far above the old one ----
        v4i pk[2];
        float ps;
        auto probabilities = [&]() __attribute__((always_inline)) {
            float s0 = 0.0f, s1 = 0.0f;
#pragma unroll
            for (int e = 0; e < 16; e += 2) {
                const float p0 = __builtin_amdgcn_exp2f(st[e]), p1 = __builtin_amdgcn_exp2f(st[e + 1]);
                s0 += p0;
                s1 += p1;
                pk[e >> 3][(e & 7) >> 1] = __builtin_bit_cast(int, P::pack(p0, p1));
            }
            ps = s0 + s1;
        };
        bool careful = kb == split || kb == masked_kb;
        if (!careful) {
            probabilities();
            careful = __ballot(!(ps < P::OPTIMISTIC_LIMIT)) != 0;
        }
        if (careful) {
            if (kb == masked_kb) {
                const int kmax = a.causal ? r : a.n - 1 - masked_kb * 32;                                     // last visible key of the block
#pragma unroll
                for (int e = 0; e < 16; ++e)
                    if (8 * (e >> 2) + 4 * h + (e & 3) > kmax) st[e] = -__builtin_inff();
            }
            float mx = st[0];
#pragma unroll
            for (int e = 1; e < 16; ++e) mx = __builtin_fmaxf(mx, st[e]);
            mx = max_lane_pair(mx);
            if (kb == split || __any(mx > P::REBASE)) {
                const float delta = kb == split ? mx : __builtin_fmaxf(mx, 0.0f);
                m_run += delta;
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    st[e] -= delta;
                    minus_m[e] = -m_run;
                }
                if (kb > split) {
                    const float alpha = __builtin_amdgcn_exp2f(-delta);
                    l_run *= alpha;
#pragma unroll
                    for (int d = 0; d < 4; ++d)
#pragma unroll
                        for (int e = 0; e < 16; ++e) acc[d][e] *= alpha;
                }
            }
            probabilities();
        }
        l_run += ps;
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int d = 0; d < 4; ++d) acc[d] = P::mfma(vf[c][d], __builtin_bit_cast(typename P::vec, pk[c]), acc[d]);
        // two blocks at most
#pragma unroll
        for (int x = 0; x < 32; ++x) v[x >> 4][x >> 3 & 1][x & 7] = v_next[x >> 4][x >> 3 & 1][x & 7];
    }

    static_assert(MAX_BLOCKS <= 2 * KS, "a wave has two blocks at most");
    // ---- merge, as in attn_fwd_short.hip: split s finishes the s-th share of the dims ----
    const float l_own = sum_lane_pair(l_run);
    __syncthreads();                                             // the operands have been read
    // dims 16 u + 8 h + 4 x .. + 3
    auto piece = [&](int u, int x) {
        const v16f &even = acc[2 * (u >> 2)], &odd = acc[2 * (u >> 2) + 1];
        const int e = 4 * (u & 3) + 2 * x;
        return (v4f){even[e], odd[e], even[e + 1], odd[e + 1]};
    };
    if (lane < 32) {
        ml[split * 64 + r] = mine > split ? m_run : -__builtin_inff();
        ml[split * 64 + 32 + r] = l_own;
    }
    v4f sum[2 * UNITS];
    auto part = [&](int from, int to) { return parts + from * PART + (to < from ? to : to - 1) * (UNITS * 2 * 64) + lane; };
    auto finish = [&](auto mine_c) __attribute__((always_inline)) {
        constexpr int S = decltype(mine_c)::value;
#pragma unroll
        for (int to = 0; to < KS; ++to)
#pragma unroll
            for (int x = 0; x < 2 * UNITS; ++x)
                if (to != S) part(S, to)[x * 64] = piece(to * UNITS + (x >> 1), x & 1);
#pragma unroll
        for (int x = 0; x < 2 * UNITS; ++x) sum[x] = piece(S * UNITS + (x >> 1), x & 1);
    };
    if (split == 0) finish(std::integral_constant<int, 0>{});
    if (split == 1) finish(std::integral_constant<int, 1>{});
    if (split == 2) finish(std::integral_constant<int, 2>{});
    if (split == 3) finish(std::integral_constant<int, 3>{});
    __syncthreads();
    float mall = ml[r], lall = 0.0f;
#pragma unroll
    for (int y = 1; y < KS; ++y) mall = __builtin_fmaxf(mall, ml[y * 64 + r]);
    const float own = __builtin_amdgcn_exp2f(ml[split * 64 + r] - mall);
#pragma unroll
    for (int x = 0; x < 2 * UNITS; ++x) sum[x] = sum[x] * own;
#pragma unroll
    for (int d = 0; d < KS; ++d) {                     // sums in split order; the outputs start from the wave's own
        const int y = (split + d) & (KS - 1);
        lall += ml[d * 64 + 32 + r] * __builtin_amdgcn_exp2f(ml[d * 64 + r] - mall);
        if (d == 0) continue;
        const float factor = __builtin_amdgcn_exp2f(ml[y * 64 + r] - mall);
        const v4f* p = part(y, split);
#pragma unroll
        for (int x = 0; x < 2 * UNITS; ++x) sum[x] += p[x * 64] * factor;
    }
    const float inv = 1.0f / lall;
    const int query = 32 * qb + r;
    if (query >= a.nq) return;
    const int64_t at = (int64_t)b * a.o_sb + (int64_t)hq * a.o_sh + (int64_t)query * a.o_sn + 16 * split * UNITS + 8 * h;
    typedef v4i v4i_8 __attribute__((aligned(8)));
#pragma unroll
    for (int u = 0; u < UNITS; ++u) {
        const v4f x = sum[2 * u] * inv, y = sum[2 * u + 1] * inv;
        auto halves = [&](auto type_c) __attribute__((always_inline)) {
            typedef PV<decltype(type_c)::value> T;
            *reinterpret_cast<v4i_8*>(static_cast<uint16_t*>(a.o) + at + 16 * u) =
                (v4i){__builtin_bit_cast(int, T::pack(x[0], x[1])), __builtin_bit_cast(int, T::pack(x[2], x[3])),
                      __builtin_bit_cast(int, T::pack(y[0], y[1])), __builtin_bit_cast(int, T::pack(y[2], y[3]))};
        };
        if (a.o_dtype == MPSA_F32) {
            v4f* const to = reinterpret_cast<v4f*>(static_cast<float*>(a.o) + at + 16 * u);
            to[0] = x;
            to[1] = y;
        } else if (a.o_dtype == MPSA_BF16) halves(std::integral_constant<int, MPSA_BF16>{});
        else                               halves(std::integral_constant<int, MPSA_F16>{});
    }
}

template <int PVT, int FMT8, int MODE>
void launch(const PromptArgs& a, bool smooth, unsigned grid, hipStream_t st) {
    if (smooth) hipLaunchKernelGGL((attn_prompt_kernel<PVT, FMT8, MODE, true>), dim3(grid), dim3(THREADS), 0, st, a);
    else        hipLaunchKernelGGL((attn_prompt_kernel<PVT, FMT8, MODE, false>), dim3(grid), dim3(THREADS), 0, st, a);
}

template <int PVT, int FMT8>
void launch_mode(const PromptArgs& a, bool smooth, unsigned grid, hipStream_t st) {
    if (a.mode == MPSA_MODE_MIXED)      launch<PVT, FMT8, MPSA_MODE_MIXED>(a, smooth, grid, st);
    else if (a.mode == MPSA_MODE_MXFP8) launch<PVT, FMT8, MPSA_MODE_MXFP8>(a, smooth, grid, st);
    else                                launch<PVT, FMT8, MPSA_MODE_DIAG>(a, smooth, grid, st);
}

template <int PVT>
void launch_fmt(const PromptArgs& a, bool smooth, unsigned grid, hipStream_t st) {
    if (a.mode == MPSA_MODE_MXFP4)        launch<PVT, MPSA_FMT_E4M3, MPSA_MODE_MXFP4>(a, smooth, grid, st);
    else if (a.fmt8 == MPSA_FMT_E5M2)     launch_mode<PVT, MPSA_FMT_E5M2>(a, smooth, grid, st);
    else                                  launch_mode<PVT, MPSA_FMT_E4M3>(a, smooth, grid, st);
}

}  // namespace

// The bytes from a [B,H,N,128] tensor's first element to its last
struct Extent { uintptr_t first, end; };
static Extent extent_of(const void* p, int64_t B, int64_t H, int64_t N, const int64_t* strides, int64_t bytes) {
    int64_t lo = 0, hi = 128;
    const int64_t steps[3] = {(B - 1) * strides[0], (H - 1) * strides[1], (N - 1) * strides[2]};
    for (int64_t step : steps) (step < 0 ? lo : hi) += step;
    return {reinterpret_cast<uintptr_t>(p) + (uintptr_t)(lo * bytes), reinterpret_cast<uintptr_t>(p) + (uintptr_t)(hi * bytes)};
}
static bool apart(const Extent& x, const Extent& y) { return x.end <= y.first || y.end <= x.first; }

// For calls that are the four-split kernel's.  Up to 256 keys:
// every key block costs each workgroup 0.25 us and every second one of a wave 0.5, and at 256 causal ones the kernels' time alone is that of the two
// launches (8.3 and 8.9 us; 201 tokens 8.0 and 8.7); whole calls gain more (10.8 -> 8.7), since the host's launch is saved too.  More than
// eight blocks would not fit the registers that hold every block's chunk from the start, nor the two blocks of V a wave.  With a mean to take off K, every workgroup reads all of the head's keys a
// second time: 160 tokens, diag, 11.3 -> 9.7 us a call, kernels 10.2 -> 9.3; 201 tokens 11.4 -> 10.6, 10.5 -> 10.3; 256 tokens, 4-bit, 11.2 -> 10.7 but
// the kernels 10.2 -> 10.6, so up to 224.  And up to 256 workgroups, one a CU, which is as far as the choice takes four splits at all.  Past that,
// for callers that name the kernel, a second round quantizes everything again: with a mean that loses, 340 queries over 224 keys 15.7 -> 18.0 us (264
// workgroups), 31 keys 27.3 -> 29.9 (1512); without one it still gains, less and less, 160 tokens, diag, 13.6 -> 9.9 (320), 18.7 -> 15.6 (640), 31 keys
// 26.4 -> 25.0 (1512), 256 keys 14.9 -> 14.7 (264), and is left to the two launches with the rest.
bool attn_prompt_supported(const mpsa_attn_desc* d, int kernel, const void* q, const void* k, const void* v, const void* o) {
    if (kernel != MPSA_ATTN_SHORT4 || d->D != 128 || d->skip || d->nk > (d->smooth_k ? 224 : 32 * MAX_BLOCKS)) return false;
    if (mpsa_quantize_sw_encoders()) return false;
    // rows on 16 bytes (V: elements two at a time), as the kernel reads them; the other path copes with the rest or refuses it
    const int64_t* const qs = d->q_strides; const int64_t* const ks = d->k_strides; const int64_t* const vs = d->v_strides; const int64_t* const os = d->o_strides;
    if (qs[3] != 1 || ks[3] != 1 || vs[3] != 1 || os[3] != 1 || ((qs[0] | qs[1] | qs[2] | ks[0] | ks[1] | ks[2]) & 7) || ((vs[0] | vs[1] | vs[2]) & 1) || ((os[0] | os[1] | os[2]) & 3)) return false;
    if (!mpsa_aligned16(q) || !mpsa_aligned16(k) || (reinterpret_cast<uintptr_t>(v) & 3) || !mpsa_aligned16(o)) return false;
    if ((d->dtype != MPSA_BF16 && d->dtype != MPSA_F16) || (d->o_dtype != MPSA_BF16 && d->o_dtype != MPSA_F16 && d->o_dtype != MPSA_F32)) return false;
    if (d->mode == MPSA_MODE_ROUTED || (d->mode != MPSA_MODE_MXFP4 && d->fmt8 != MPSA_FMT_E4M3 && d->fmt8 != MPSA_FMT_E5M2)) return false;
    if (d->nq != d->nk && (d->causal || d->mode == MPSA_MODE_DIAG)) return false;
    if (d->B > 256 || d->Hq > 256 || d->nq > 256 * 32 || d->B * d->Hq * ((d->nq + 31) / 32) > 256) return false;
    // an output over K's or V's memory: there one workgroup would store what another has yet to read, where the preparation reads all of
    // both before the attention kernel stores anything
    const Extent to = extent_of(o, d->B, d->Hq, d->nq, os, d->o_dtype == MPSA_F32 ? 4 : 2);
    return apart(to, extent_of(k, d->B, d->Hkv, d->nk, ks, 2)) && apart(to, extent_of(v, d->B, d->Hkv, d->nk, vs, 2));
}

int attn_prompt_launch(const mpsa_attn_desc* d, const void* q, const void* k, const void* v, void* o, hipStream_t st) {
    PromptArgs a{};
    a.q_raw = q; a.q_sb = d->q_strides[0]; a.q_sh = d->q_strides[1]; a.q_sn = d->q_strides[2];
    a.k_raw = static_cast<const char*>(k); a.k_sb = d->k_strides[0]; a.k_sh = d->k_strides[1]; a.k_sn = d->k_strides[2];
    a.v_raw = static_cast<const char*>(v); a.v_sb = d->v_strides[0]; a.v_sh = d->v_strides[1]; a.v_sn = d->v_strides[2];
    a.o = o; a.o_sb = d->o_strides[0]; a.o_sh = d->o_strides[1]; a.o_sn = d->o_strides[2];
    a.q_pre = d->pre_scale_q;
    a.q_sure = mpsa_e2m1_sure(d->pre_scale_q, d->dtype) ? 1 : 0;
    a.k_sure = mpsa_e2m1_sure(1.0f, d->dtype) ? 1 : 0;
    a.B = (int)d->B; a.Hq = (int)d->Hq; a.Hkv = (int)d->Hkv; a.n = (int)d->nk; a.nq = (int)d->nq;
    a.causal = d->causal ? 1 : 0; a.mode = d->mode; a.fmt8 = d->fmt8; a.o_dtype = d->o_dtype; a.tile = d->tile;
    a.inv_n = 1.0f / (float)d->nk;
    a.units = a.B * a.Hkv; a.group = a.Hq / a.Hkv; a.nqb = (a.nq + 31) / 32;
    a.by_units = reciprocal_of((uint32_t)a.units); a.by_group = reciprocal_of((uint32_t)a.group); a.by_hkv = reciprocal_of((uint32_t)a.Hkv);
    const unsigned grid = (unsigned)(a.units * a.group * a.nqb);
    if (d->dtype == MPSA_BF16) launch_fmt<MPSA_BF16>(a, d->smooth_k != 0, grid, st);
    else                       launch_fmt<MPSA_F16>(a, d->smooth_k != 0, grid, st);
    MPSA_CHECK_LAUNCH("attn (prompt)");
    return MPSA_OK;
}
