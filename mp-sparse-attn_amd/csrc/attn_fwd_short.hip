// Fused attention forward for short sequences (gfx950): the math of attn_fwd_kernel.h, mapped for latency.
//
// What bounds a short prompt on the tile kernels is the serial chain of one workgroup: a paired-tile workgroup takes 256
// queries through a 28 000-clock prologue and epilogue and 3 600 clocks a tile, and there are 32 of them (160 tokens, 32
// heads) or 128 (1000 tokens) for 256 CUs.  Here a workgroup owns 32 queries and its four waves split the KEYS between
// them: wave w takes the 32-key blocks w, w + 4, ... with a running maximum, row sum and output of its own, and the four
// partial results are merged through LDS at the end (in wave order: results do not depend on timing).  Nothing is shared
// in the loop, so there is no barrier in it: a block's K rows and V fragments come into LDS buffers of the wave's own, one
// block ahead.
// Q may arrive unquantized (QRAW): the workgroup quantizes its 32 rows cooperatively into LDS, eight elements per lane, with the
// quantizer's own code -- the bits of mpsa_quantize_mx.
// What bounds it: a fixed 5 us per workgroup (two share a CU; Q and the first block from memory, quantization, merge) and
// 1300 clocks a block and wave.  A 160-token prefill (32 heads) takes 5 us where the paired-tile kernel takes 12.8, 512
// tokens 8 where it takes 17.  The price is traffic, 40 KiB of K and V per 128 keys and 32 queries, four times the tile
// kernels': long sequences stay there.  Two query blocks per wave (half the traffic) took 2.5 us longer up to 1000 tokens
// and were no faster than the tile kernels beyond.
#include "attn_common.h"
#include "quantize_kernel.h"

namespace {

struct ShortArgs : AttnArgs {
    int group, per_unit;                          // query heads per KV head; workgroups per (batch, KV head)
    uint32_t m_units, m_per_unit, m_group, m_hkv; // reciprocals
};

template <int D, int MODE>
struct Short {
    static constexpr int SST = D / 64;            // score matrix instructions along D
    static constexpr int NDB = D / 32;            // 32-wide output dim blocks
    static constexpr int ROW4 = D / 2, ROW8 = D;  // bytes per K row
    static constexpr int CPR4 = ROW4 / 16, CPR8 = ROW8 / 16;
    static constexpr int SH4 = CPR4 == 2 ? 3 : 2, SH8 = CPR8 == 4 ? 2 : 1;      // log2(rows per 256 bytes)
    static constexpr int KBUF = 32 * (MODE == MPSA_MODE_MXFP8 ? ROW8 : ROW4);
    static constexpr int VBUF = 32 * D * 2;
    static constexpr int MINE = KBUF + VBUF;      // a wave's buffers
    // quantized Q: codes and scales of both widths
    static constexpr int Q4 = 4 * MINE, QS4 = Q4 + 32 * ROW4, Q8 = QS4 + 32 * NDB, QS8 = Q8 + 32 * ROW8, LOOP = QS8 + 32 * NDB;
    static constexpr int PART = 4 * (NDB / 2) * 16 * 64 * 4, MERGE = PART + 4 * 2 * 32 * 4;    // half of the dim blocks at a time
    static constexpr int SMEM = LOOP > MERGE ? LOOP : MERGE;
};

// x / d with the host's ceil(2^32 / d), exact while x * d < 2^32; 0 stands for d = 1
__device__ __forceinline__ int by_reciprocal(int x, uint32_t m) { return m ? (int)(((uint64_t)(uint32_t)x * m) >> 32) : x; }

template <int D, int PVT, int FMT8, int MODE, bool QRAW>
__global__ __launch_bounds__(256, D == 128 ? 3 : 4) void attn_short_kernel(ShortArgs a) {
    typedef Short<D, MODE> G;
    typedef PV<PVT> P;
    constexpr bool MIXED = MODE == MPSA_MODE_MIXED, DIAG = MODE == MPSA_MODE_DIAG;
    constexpr bool MAIN8 = MODE == MPSA_MODE_MXFP8;                        // the plain blocks' K is 8 bits wide
    constexpr bool Q4 = !MAIN8 && !MIXED, Q8 = MODE != MPSA_MODE_MXFP4;    // Q in which formats
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int h = lane >> 5, r = lane & 31;

    // ---- which (batch, kv head, query head, query rows): one KV head's query heads per XCD, long causal rows first.  Fewer
    //      heads than XCDs, or an uneven number: the rows of a head are dealt out over all of them.  Divisions by the host's
    //      reciprocals: three in integer arithmetic took a quarter of a microsecond of every workgroup. ----
    const int nqb = (a.nq + 31) / 32, units = a.B * a.Hkv;
    int unit, row;                                        // (batch, kv head); query rows times query heads of the group
    if (units & 7) {
        row = by_reciprocal(blockIdx.x, a.m_units);
        unit = blockIdx.x - row * units;
    } else {
        const int L = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
        unit = by_reciprocal(L, a.m_per_unit);
        row = L - unit * a.per_unit;
    }
    const int rank = by_reciprocal(row, a.m_group), sub = row - rank * a.group;
    const int b = by_reciprocal(unit, a.m_hkv), kvh = unit - b * a.Hkv, hq = kvh * a.group + sub;
    const int qb = a.causal ? nqb - 1 - rank : rank;
    const int64_t krow0 = ((int64_t)b * a.Hkv + kvh) * a.n_pad;

    // ---- this wave's key blocks: first the plain ones (main precision, no mask), then the one that needs a mask (the causal
    //      diagonal, a ragged end), last the block of the query's own tile in a diag run (8-bit; often the same one) ----
    const int nb = min(a.causal ? qb + 1 : 0x7fffffff, (a.n + 31) / 32);
    const int count = nb > w ? (nb - w + 3) / 4 : 0;
    const int last_kb = w + 4 * (count - 1);
    const bool last_masked = count > 0 && (a.causal ? last_kb >= qb : last_kb == nb - 1 && (a.n & 31) != 0);
    const int own_first = a.tile == 128 ? qb & ~3 : qb & ~1;
    const int own_t = own_first / 4, own_kb = 4 * own_t + w;
    const bool has_own = DIAG && own_kb >= own_first && own_kb < own_first + a.tile / 32 && own_kb < nb;
    const bool last_apart = last_masked && !(has_own && own_t == count - 1);
    const int plain = count - (has_own ? 1 : 0) - (last_apart ? 1 : 0);
    auto block_at = [&](int i) {
        if (i < plain) return w + 4 * (i + (has_own && i >= own_t ? 1 : 0));
        return last_apart && i == plain ? last_kb : own_kb;
    };
    auto block_is8 = [&](int i) { return MAIN8 || (DIAG && has_own && i == count - 1); };

    // ---- a block's operands: K rows (swizzled) and V fragments into this wave's buffers, the lane's K scale word ----
    uint8_t* const kbuf = smem + w * G::MINE;
    uint8_t* const vbuf = kbuf + G::KBUF;
    uint32_t ks_next = 0;
    auto fetch = [&](int i) __attribute__((always_inline)) {
        const int kb = block_at(i);
        const bool is8 = block_is8(i);
        auto rows = [&](const uint8_t* src, int row_bytes, int cpr, int sh) __attribute__((always_inline)) {
#pragma unroll
            for (int c = 0; c < row_bytes * 32 / 1024; ++c) {
                const int p = c * 64 + lane, row = p / cpr, slot = p % cpr;
                load16_to_lds_sv((uint32_t)(row * row_bytes + (slot ^ ((row >> sh) & (cpr - 1))) * 16), src, kbuf + c * 1024);
            }
        };
        if constexpr (MAIN8) rows(a.k8 + (krow0 + kb * 32) * G::ROW8, G::ROW8, G::CPR8, G::SH8);
        else if (!is8)       rows(a.k4 + (krow0 + kb * 32) * G::ROW4, G::ROW4, G::CPR4, G::SH4);
        const uint8_t* sp = (is8 ? a.ks8 : a.ks4) + (krow0 + kb * 32) * (D / 32);
        ks_next = (D == 128) ? reinterpret_cast<const uint32_t*>(sp)[r] : (uint32_t)reinterpret_cast<const uint16_t*>(sp)[r];
        const uint8_t* vb = static_cast<const uint8_t*>(a.v) + (krow0 + kb * 32) * (D * 2);
#pragma unroll
        for (int x = 0; x < 2 * G::NDB; ++x) load16_to_lds_sv((uint32_t)lane * 16u, vb + x * 1024, vbuf + x * 1024);
    };
    if (count > 0) fetch(0);

    // ---- this workgroup's queries, quantized, into LDS ----
    uint8_t* const qlds = smem;
    const int64_t qrow0 = ((int64_t)b * a.Hq + hq) * a.nq_pad + 32 * qb;
#pragma unroll
    for (int q = 0; q < D / 64; ++q) {
        const int c = q * 256 + tid, row = c / (D / 8), col8 = c % (D / 8);
        uint32_t w4 = 0;
        uint2 w8 = make_uint2(0u, 0u);
        int s4 = 0, s8 = 0;
        if constexpr (QRAW) {
            float x[8];
            if (32 * qb + row < a.nq) {
                load8<PVT>(static_cast<const char*>(a.q_raw) + 2 * ((int64_t)b * a.q_sb + (int64_t)hq * a.q_sh + (int64_t)(32 * qb + row) * a.q_sn + 8 * col8), x);
            } else {
#pragma unroll
                for (int i = 0; i < 8; ++i) x[i] = 0.0f;
            }
            quantize_chunk<Q4, Q8, FMT8, false>(x, a.q_pre, a.q_exact16 != 0, 3, 7, w4, s4, w8, s8);
        } else {
            if constexpr (Q4) {
                w4 = reinterpret_cast<const uint32_t*>(a.q4 + qrow0 * G::ROW4)[c];
                s4 = a.qs4[qrow0 * G::NDB + (c >> 2)];
            }
            if constexpr (Q8) {
                w8 = reinterpret_cast<const uint2*>(a.q8 + qrow0 * G::ROW8)[c];
                s8 = a.qs8[qrow0 * G::NDB + (c >> 2)];
            }
        }
        if constexpr (Q4) {
            *reinterpret_cast<uint32_t*>(qlds + G::Q4 + c * 4) = w4;
            if ((tid & 3) == 0) qlds[G::QS4 + (c >> 2)] = (uint8_t)s4;
        }
        if constexpr (Q8) {
            *reinterpret_cast<uint2*>(qlds + G::Q8 + c * 8) = w8;
            if ((tid & 3) == 0) qlds[G::QS8 + (c >> 2)] = (uint8_t)s8;
        }
    }
    __syncthreads();
    auto scale_word = [&](int off) { return D == 128 ? *reinterpret_cast<const uint32_t*>(qlds + off + r * 4) : (uint32_t)*reinterpret_cast<const uint16_t*>(qlds + off + r * 2); };
    v8i qf[G::SST];                                       // fragments of the precision in use; a diag run re-reads them for its own tile
    auto load_q = [&](bool is8) __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < G::SST; ++s) {
            if (Q8 && (is8 || !Q4)) {
                const v4i x0 = *reinterpret_cast<const v4i*>(qlds + G::Q8 + r * G::ROW8 + s * 64 + h * 16);
                const v4i x1 = *reinterpret_cast<const v4i*>(qlds + G::Q8 + r * G::ROW8 + s * 64 + h * 16 + 32);
                qf[s] = (v8i){x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]};
            } else {
                const v4i x0 = *reinterpret_cast<const v4i*>(qlds + G::Q4 + r * G::ROW4 + (2 * s + h) * 16);
                qf[s] = (v8i){x0[0], x0[1], x0[2], x0[3], 0, 0, 0, 0};
            }
        }
    };
    const int qs8 = Q8 ? (int)(scale_word(G::QS8) >> (8 * h)) : 0, qs = Q4 ? (int)(scale_word(G::QS4) >> (8 * h)) : qs8;
    load_q(false);

    v16f acc[G::NDB];
#pragma unroll
    for (int d = 0; d < G::NDB; ++d)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[d][e] = 0.0f;
    float m_run = 0.0f, l_run = 0.0f;                     // lazily moved reference maximum and row sum, as in attn_fwd_kernel.h

    // One block.  CAREFUL takes the maximum first (a wave's first block sets its reference maximum, masked blocks come once);
    // otherwise the exponentials are taken against the old maximum at once and a row sum that shows a score far above it sends
    // the wave back to do the block the careful way -- no reduction and no branch between the scores and the exponentials.
    auto step = [&](int i, auto is8_c, auto masked_c, auto careful_c) __attribute__((always_inline)) {
        constexpr bool IS8 = decltype(is8_c)::value, MASKED = decltype(masked_c)::value, CAREFUL = decltype(careful_c)::value;
        const int kb = block_at(i);
        // the one 8-bit block of a diag run goes straight into registers, when its turn comes: a step ahead its fragments would
        // hold registers throughout (two fewer workgroups' worth), in LDS its rows twice the buffer
        v4i k8[IS8 && DIAG ? 2 * G::SST : 1];
        if constexpr (IS8 && DIAG) {
#pragma unroll
            for (int s = 0; s < 2 * G::SST; ++s) k8[s] = *reinterpret_cast<const v4i*>(a.k8 + (krow0 + kb * 32 + r) * G::ROW8 + h * 16 + s * 32);
        }
        // the block has landed; its fragments go into registers, and the buffers take the next one
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        const int ks = (int)(ks_next >> (8 * h));
        v8i kf[G::SST];
#pragma unroll
        for (int s = 0; s < G::SST; ++s) {
            if constexpr (IS8 && DIAG) {
                const v4i x0 = k8[2 * s], x1 = k8[2 * s + 1];
                kf[s] = (v8i){x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]};
            } else if constexpr (IS8) {
                const int f = (r >> G::SH8) & (G::CPR8 - 1);
                const v4i x0 = *reinterpret_cast<const v4i*>(kbuf + r * G::ROW8 + (((4 * s + h) ^ f) * 16));
                const v4i x1 = *reinterpret_cast<const v4i*>(kbuf + r * G::ROW8 + (((4 * s + h + 2) ^ f) * 16));
                kf[s] = (v8i){x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]};
            } else {
                const int f = (r >> G::SH4) & (G::CPR4 - 1);
                const v4i x = *reinterpret_cast<const v4i*>(kbuf + r * G::ROW4 + (((2 * s + h) ^ f) * 16));
                kf[s] = (v8i){x[0], x[1], x[2], x[3], 0, 0, 0, 0};
            }
        }
        typename P::vec vf[2][G::NDB];
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int d = 0; d < G::NDB; ++d) vf[c][d] = *reinterpret_cast<const typename P::vec*>(vbuf + (c * G::NDB + d) * 1024 + lane * 16);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        if (i + 1 < count) fetch(i + 1);
        __builtin_amdgcn_sched_barrier(0);

        auto scores = [&]() __attribute__((always_inline)) {
            v16f st;
#pragma unroll
            for (int e = 0; e < 16; ++e) st[e] = -m_run;
#pragma unroll
            for (int s = 0; s < G::SST; ++s) {
                if constexpr (IS8)        st = score_mfma8<FMT8>(kf[s], qf[s], st, s, ks, qs8);
                else if constexpr (MIXED) st = score_mfma48<FMT8>(kf[s], qf[s], st, s, ks, qs8);
                else                      st = score_mfma4(kf[s], qf[s], st, s, ks, qs);
            }
            if constexpr (MASKED) {
                const int kmax = a.causal ? (kb == qb ? r : 31) : min(31, a.n - 1 - kb * 32);      // last visible key of the block
#pragma unroll
                for (int e = 0; e < 16; ++e)
                    if (8 * (e >> 2) + 4 * h + (e & 3) > kmax) st[e] = -__builtin_inff();
            }
            return st;
        };
        v4i pk[2];
        float ps;
        auto exponentials = [&](const v16f& st) __attribute__((always_inline)) {
            float ps0 = 0.0f, ps1 = 0.0f;
#pragma unroll
            for (int c = 0; c < 2; ++c)
#pragma unroll
                for (int e = 0; e < 8; e += 2) {
                    const float p0 = __builtin_amdgcn_exp2f(st[8 * c + e]), p1 = __builtin_amdgcn_exp2f(st[8 * c + e + 1]);
                    pk[c][e >> 1] = __builtin_bit_cast(int, P::pack(p0, p1));
                    ps0 += p0;
                    ps1 += p1;
                }
            ps = ps0 + ps1;
        };
        auto careful = [&]() __attribute__((always_inline)) {
            v16f st = scores();
            float mx = st[0];
#pragma unroll
            for (int e = 1; e < 16; ++e) mx = __builtin_fmaxf(mx, st[e]);
            mx = max_lane_pair(mx);
            if (i == 0 || __any(mx > P::REBASE)) {
                const float delta = i == 0 ? mx : __builtin_fmaxf(mx, 0.0f);
                const float alpha = i == 0 ? 1.0f : __builtin_amdgcn_exp2f(-delta);
                m_run += delta;
#pragma unroll
                for (int e = 0; e < 16; ++e) st[e] -= delta;
                l_run *= alpha;
#pragma unroll
                for (int d = 0; d < G::NDB; ++d)
#pragma unroll
                    for (int e = 0; e < 16; ++e) acc[d][e] *= alpha;
            }
            exponentials(st);
        };
        if constexpr (CAREFUL) {
            careful();
        } else {
            exponentials(scores());
            if (__any(!(ps < P::OPTIMISTIC_LIMIT))) careful();
        }
        l_run += ps;
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int d = 0; d < G::NDB; ++d) acc[d] = P::mfma(vf[c][d], __builtin_bit_cast(typename P::vec, pk[c]), acc[d]);
    };
    typedef std::integral_constant<bool, MAIN8> Main;
    if (plain > 0) step(0, Main{}, std::false_type{}, std::true_type{});
    for (int i = 1; i < plain; ++i) step(i, Main{}, std::false_type{}, std::false_type{});
    if (last_apart) step(plain, Main{}, std::true_type{}, std::true_type{});
    if (has_own) {
        load_q(true);
        step(count - 1, std::integral_constant<bool, MAIN8 || DIAG>{}, std::true_type{}, std::true_type{});
    }

    // ---- merge: every wave's output is brought to the common maximum; wave d adds up and stores dim block d ----
    __syncthreads();                                      // everybody is through with the buffers
    v4f* const part = reinterpret_cast<v4f*>(smem);       // [wave][dim block][quarter of its registers][lane]
    float* const ml = reinterpret_cast<float*>(smem + G::PART);       // [wave][maximum, sum][query]
    const float l_own = sum_lane_pair(l_run);
    if (lane < 32) {
        ml[w * 64 + r] = count > 0 ? m_run : -__builtin_inff();
        ml[w * 64 + 32 + r] = l_own;
    }
    __syncthreads();
    float mall = ml[r];
#pragma unroll
    for (int y = 1; y < 4; ++y) mall = __builtin_fmaxf(mall, ml[y * 64 + r]);
    float lall = 0.0f;
#pragma unroll
    for (int y = 0; y < 4; ++y) lall += ml[y * 64 + 32 + r] * __builtin_amdgcn_exp2f(ml[y * 64 + r] - mall);
    const float scale = count > 0 ? __builtin_amdgcn_exp2f(m_run - mall) : 0.0f;
    // half of the dim blocks at a time; wave w stores dims 16 (w & 1) .. + 15 of block w / 2 of the half
    constexpr int HD = G::NDB / 2;
#pragma unroll
    for (int half = 0; half < 2; ++half) {
#pragma unroll
        for (int d = 0; d < HD; ++d)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const v16f& x = acc[half * HD + d];
                part[((w * HD + d) * 4 + e) * 64 + lane] = (v4f){x[4 * e], x[4 * e + 1], x[4 * e + 2], x[4 * e + 3]} * scale;
            }
        __syncthreads();
        const int d = w >> 1, u = w & 1;
        if (d < HD) {
            v4f o[2];
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                o[e] = part[(d * 4 + 2 * u + e) * 64 + lane];
#pragma unroll
                for (int y = 1; y < 4; ++y) o[e] += part[((y * HD + d) * 4 + 2 * u + e) * 64 + lane];
            }
            store_16_dims(a, b, hq, 32 * qb + r, 32 * (half * HD + d) + 16 * u, h, o[0], o[1], 1.0f / lall);
        }
        if (half == 0) __syncthreads();
    }
}

template <int D, int PVT, int FMT8, int MODE, bool QRAW>
struct ShortLds {
    static inline const bool registered = mpsa_register_lds_kernel(reinterpret_cast<const void*>(attn_short_kernel<D, PVT, FMT8, MODE, QRAW>), Short<D, MODE>::SMEM);
};

template <int D, int PVT, int FMT8, int MODE, bool QRAW>
int launch_one(const AttnArgs& a, hipStream_t st) {
    if (!ShortLds<D, PVT, FMT8, MODE, QRAW>::registered) return mpsa_fail(MPSA_ELAUNCH, "attn: kernel not registered");
    const int rc = mpsa_ensure_init();
    if (rc != MPSA_OK) return rc;
    ShortArgs s;
    static_cast<AttnArgs&>(s) = a;
    const int units = a.B * a.Hkv;
    s.group = a.Hq / a.Hkv;
    s.per_unit = s.group * ((a.nq + 31) / 32);
    auto reciprocal = [](int d) { return d == 1 ? 0u : (uint32_t)(((uint64_t(1) << 32) + d - 1) / d); };
    s.m_units = reciprocal(units); s.m_per_unit = reciprocal(s.per_unit); s.m_group = reciprocal(s.group); s.m_hkv = reciprocal(a.Hkv);
    hipLaunchKernelGGL((attn_short_kernel<D, PVT, FMT8, MODE, QRAW>), dim3((unsigned)(units * s.per_unit)), dim3(256), (Short<D, MODE>::SMEM), st, s);
    MPSA_CHECK_LAUNCH("attn (short)");
    return MPSA_OK;
}

template <int D, int PVT, int FMT8, int MODE>
int launch_q(const AttnArgs& a, hipStream_t st) {
    return a.q_raw ? launch_one<D, PVT, FMT8, MODE, true>(a, st) : launch_one<D, PVT, FMT8, MODE, false>(a, st);
}

template <int D, int PVT, int FMT8>
int launch_mode(const AttnArgs& a, hipStream_t st) {
    if (a.mode == MPSA_MODE_MIXED) return launch_q<D, PVT, FMT8, MPSA_MODE_MIXED>(a, st);
    if (a.mode == MPSA_MODE_MXFP8) return launch_q<D, PVT, FMT8, MPSA_MODE_MXFP8>(a, st);
    return launch_q<D, PVT, FMT8, MPSA_MODE_DIAG>(a, st);
}

template <int D, int PVT>
int launch_fmt(const AttnArgs& a, hipStream_t st) {
    if (a.mode == MPSA_MODE_MXFP4) return launch_q<D, PVT, MPSA_FMT_E4M3, MPSA_MODE_MXFP4>(a, st);
    return a.fmt8 == MPSA_FMT_E5M2 ? launch_mode<D, PVT, MPSA_FMT_E5M2>(a, st) : launch_mode<D, PVT, MPSA_FMT_E4M3>(a, st);
}

}  // namespace

int attn_short_launch(const AttnArgs& a, int pv_dtype, hipStream_t st) {
    if (a.d == 128) return pv_dtype == MPSA_BF16 ? launch_fmt<128, MPSA_BF16>(a, st) : launch_fmt<128, MPSA_F16>(a, st);
    return pv_dtype == MPSA_BF16 ? launch_fmt<64, MPSA_BF16>(a, st) : launch_fmt<64, MPSA_F16>(a, st);
}
