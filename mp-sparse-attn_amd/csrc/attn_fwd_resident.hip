// Fused attention forward for many queries over few keys (gfx950): the short-sequence kernel with one split
// (attn_fwd_short.hip), where all of a head's K and V fit one CU's LDS; D = 128, 8-bit Q (mxfp8, mixed), no mask, unquantized Q.
//
// A workgroup of the short-sequence kernel takes 128 queries: it waits for them from memory, brings K and V through a ring with a
// barrier every 32 keys and is gone after a dozen of them.  Here a workgroup of eight waves brings K and V of one head into LDS
// once and its waves take blocks of 32 queries one after the other, each at its own pace: no ring, no barrier but the first, and a
// wave's next queries are on their way while it works on these.  Its arithmetic is the short-sequence kernel's, operation by
// operation, and so are its bits: which of the two a call takes can depend on the batch.
// Clock stamps in a copy of this kernel, 2 x 16 heads, 4096 queries over 333 keys, 8-bit (two blocks of queries a wave): 15 900 until
// K, V and the first queries are there (16.8 MB of queries from memory in one go), then a block 4600 for Q (8 a lane and
// instruction, two waves a SIMD; with a branch in it), 11 400 for eleven blocks of keys (510 a block of one SIMD: matrix 384, exponentials 256) and 1800
// for the store.  Whole calls, the streaming kernel -> this one: that shape 42.6 -> 39.9 us; 2 x 8 heads, 10000 over 256, 40.1 ->
// 36.9; 24 heads, 32000 over 333, mixed, 175 -> 157; 16 heads, 16000 over 352, 64.8 -> 58.3; 24 heads, 30000 over 77, 104 -> 98.
// Few blocks of queries a head, few altogether or few keys do not pay the way into LDS back (resident_choice.h); with 4-bit Q the
// streaming kernel has three waves a SIMD and wins (2 x 24 heads, 8000 over 200, 66.4 -> 75.8), and with D = 64 four (2 x 24 heads,
// 3000 over 512, 37.4 -> 39.6).
#include "attn_common.h"
#include "quantize_kernel.h"
#include "reciprocal.h"
#include "resident_choice.h"

namespace {

struct ResidentArgs : AttnArgs {
    Reciprocal by_units, by_hkv, by_nqb;
    int units, group, nqb, tasks, step, nb;               // tasks: blocks of 32 queries of a (batch, KV head); step: waves that share them; nb: blocks of 32 keys
};

constexpr int D = 128, RW = RESIDENT_WAVES;

template <int MODE>
struct Resident {
    static constexpr bool MAIN8 = MODE == MPSA_MODE_MXFP8;
    static constexpr int SST = D / 64, NDB = D / 32;
    static constexpr int ROW = MAIN8 ? D : D / 2, CPR = ROW / 16, SH = CPR == 4 ? 2 : 1;         // bytes, 16-byte pieces of a K row; log2(rows per 256 bytes)
    static constexpr int KBLOCK = 32 * ROW, VBLOCK = 32 * D * 2, SBLOCK = 32 * NDB;              // of 32 keys: codes, V, scale bytes
    static constexpr int QROWS = 16, QBYTES = QROWS * (D + NDB);                                 // a wave's quantized queries, so many rows at a time
    // LDS: K, V, scales, queries
    static int lds(int nb) { return nb * (KBLOCK + VBLOCK) + (nb * SBLOCK + 255) / 256 * 256 + RW * QBYTES; }
};

template <int PVT, int FMT8, int MODE>
__global__ __launch_bounds__(RW * 64, 1) void attn_resident_kernel(ResidentArgs a) {
    typedef Resident<MODE> G;
    typedef PV<PVT> P;
    constexpr bool MAIN8 = G::MAIN8;
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int h = lane >> 5, r = lane & 31;
    const int share = divide_by((int)blockIdx.x, a.by_units), unit = (int)blockIdx.x - share * a.units;
    const int b = divide_by(unit, a.by_hkv), kvh = unit - b * a.Hkv;
    const int64_t krow0 = (int64_t)unit * a.n_pad;
    const int nb = a.nb;
    uint8_t* const vl = smem + nb * G::KBLOCK;
    uint8_t* const sl = vl + nb * G::VBLOCK;
    uint8_t* const ql = sl + (nb * G::SBLOCK + 255) / 256 * 256 + w * G::QBYTES;

    // ---- a block of queries: head and rows, and its 16-bit elements, eight a lane and chunk ----
    constexpr int CHUNKS = 32 * D / 8 / 64;
    int hq, row0;
    auto place = [&](int t) {
        const int sub = divide_by(t, a.by_nqb);
        hq = kvh * a.group + sub;
        row0 = 32 * (t - sub * a.nqb);
    };
    uint4 raw[CHUNKS];
    auto fetch_q = [&]() __attribute__((always_inline)) {
        const char* const base = static_cast<const char*>(a.q_raw) + 2 * ((int64_t)b * a.q_sb + (int64_t)hq * a.q_sh);
#pragma unroll
        for (int q = 0; q < CHUNKS; ++q) {
            const int c = q * 64 + lane, src = min(row0 + c / (D / 8), a.nq - 1);
            raw[q] = *reinterpret_cast<const uint4*>(base + 2 * ((int64_t)src * a.q_sn + 8 * (c % (D / 8))));
        }
    };
    int t = share * RW + w;
    place(t);
    if (t < a.tasks) fetch_q();
    __builtin_amdgcn_sched_barrier(0);

    // ---- K (rows swizzled), V fragments and scale words of the whole head ----
    {
        const uint8_t* const kg = (MAIN8 ? a.k8 : a.k4) + krow0 * G::ROW;
        const uint8_t* const vg = static_cast<const uint8_t*>(a.v) + krow0 * (D * 2);
        const uint8_t* const sg = (MAIN8 ? a.ks8 : a.ks4) + krow0 * G::NDB;
        for (int p = w; p < nb * (G::KBLOCK / 1024); p += RW) {
            const int at = p * 64 + lane, krow = at / G::CPR, chunk = at % G::CPR;
            load16_to_lds_sv((uint32_t)(krow * G::ROW + (chunk ^ ((krow >> G::SH) & (G::CPR - 1))) * 16), kg, smem + p * 1024);
        }
        for (int p = w; p < (nb * G::SBLOCK + 255) / 256; p += RW) load4_to_lds_sv((uint32_t)min(p * 256 + lane * 4, nb * G::SBLOCK - 4), sg, sl + p * 256);
        for (int p = w; p < nb * (G::VBLOCK / 1024); p += RW) load16_to_lds_sv((uint32_t)(p * 1024 + lane * 16), vg, vl + p * 1024);
    }
    __builtin_amdgcn_s_waitcnt(0x0F70);
    __syncthreads();

    const int masked_at = (a.n & 31) ? nb - 1 : -1;
#pragma unroll 1
    for (; t < a.tasks; t += a.step) {
        // ---- quantize: the quantizer's own code, through LDS into the matrix operand's layout ----
        const int hq_now = hq, row_now = row0;
        v8i qf[G::SST];
        int qs;
        {
            constexpr int BATCH = 4;
            uint32_t scale = 0;
#pragma unroll
            for (int q0 = 0; q0 < CHUNKS; q0 += BATCH) {
                // straight through; a wave with a rare chunk does the batch again (rows past the last are zeros, as in the streaming kernel)
                auto inside = [&](int q) { return row_now + ((q0 + q) * 64 + lane) / (D / 8) < a.nq; };
                auto put = [&](int q, const uint2& w8, int s8) __attribute__((always_inline)) {
                    const int at = ((q0 + q) * 64 + lane) % (G::QROWS * (D / 8));
                    *reinterpret_cast<uint2*>(ql + at * 8) = w8;
                    ql[G::QROWS * D + (at >> 2)] = (uint8_t)s8;
                };
                uint32_t none;
                uint2 w8;
                int no, s8;
                bool rare = false;
#pragma unroll
                for (int q = 0; q < BATCH; ++q) {
                    float x[8];
                    bool r1;
                    unpack8<PVT>(raw[q0 + q], x);
                    const float pre = inside(q) ? a.q_pre : 0.0f;
#pragma unroll
                    for (int i = 0; i < 8; ++i) x[i] *= pre;
                    quantize_straight<false, true, FMT8>(x, none, no, w8, s8, r1);
                    rare |= r1;
                    put(q, w8, s8);
                }
                if (__ballot(rare) != 0) {
#pragma unroll
                    for (int q = 0; q < BATCH; ++q) {
                        float x[8];
                        unpack8<PVT>(inside(q) ? only_here(raw[q0 + q]) : make_uint4(0, 0, 0, 0), x);
                        quantize_chunk<false, true, FMT8, false, true>(x, a.q_pre, false, 3, 7, none, no, w8, s8);
                        put(q, w8, s8);
                    }
                }
                // so many rows are there: the lanes that own them take them
                constexpr int AT_ONCE = G::QROWS * (D / 8) / 64;         // chunks
                if ((q0 + BATCH) % AT_ONCE == 0) {
                    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // this wave's own writes, in front of its reads
                    const int from = r - ((q0 + BATCH) / AT_ONCE - 1) * G::QROWS;
                    if (from >= 0 && from < G::QROWS) {
#pragma unroll
                        for (int s = 0; s < G::SST; ++s) {
                            const v4i x0 = *reinterpret_cast<const v4i*>(ql + from * D + s * 64 + h * 16);
                            const v4i x1 = *reinterpret_cast<const v4i*>(ql + from * D + s * 64 + h * 16 + 32);
                            qf[s] = (v8i){x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]};
                        }
                        scale = *reinterpret_cast<const uint32_t*>(ql + G::QROWS * D + from * G::NDB);
                    }
                    asm volatile("" ::: "memory");
                }
            }
            if (t + a.step < a.tasks) {
                place(t + a.step);
                fetch_q();
            }
            qs = (int)(scale >> (8 * h));
        }

        v16f acc[G::NDB], minus_m;
#pragma unroll
        for (int d = 0; d < G::NDB; ++d)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[d][e] = 0.0f;
#pragma unroll
        for (int e = 0; e < 16; ++e) minus_m[e] = 0.0f;
        float m_run = 0.0f, l_run = 0.0f, ps;
        v4i pk[2];
        typename P::vec vf[2][G::NDB];
        v8i kf[G::SST];
        uint32_t ks_word;
        auto load_k = [&](int j) __attribute__((always_inline)) {
            const uint8_t* const kb = smem + j * G::KBLOCK + r * G::ROW;
            const int f = (r >> G::SH) & (G::CPR - 1);
            ks_word = *reinterpret_cast<const uint32_t*>(sl + (j * 32 + r) * G::NDB);
#pragma unroll
            for (int s = 0; s < G::SST; ++s) {
                if constexpr (MAIN8) {
                    const v4i x0 = *reinterpret_cast<const v4i*>(kb + (((4 * s + h) ^ f) * 16));
                    const v4i x1 = *reinterpret_cast<const v4i*>(kb + (((4 * s + h + 2) ^ f) * 16));
                    kf[s] = (v8i){x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]};
                } else {
                    const v4i x = *reinterpret_cast<const v4i*>(kb + (((2 * s + h) ^ f) * 16));
                    kf[s] = (v8i){x[0], x[1], x[2], x[3], 0, 0, 0, 0};
                }
            }
        };
        auto load_v = [&](int j, int c) __attribute__((always_inline)) {
            const uint8_t* const vb = vl + j * G::VBLOCK + lane * 16;
#pragma unroll
            for (int d = 0; d < G::NDB; ++d) vf[c][d] = *reinterpret_cast<const typename P::vec*>(vb + (c * G::NDB + d) * 1024);
        };
        auto scores = [&]() __attribute__((always_inline)) {
            v16f st = minus_m;
            const int ks = (int)(ks_word >> (8 * h));
#pragma unroll
            for (int s = 0; s < G::SST; ++s) {
                if constexpr (MAIN8) st = score_mfma8<FMT8>(kf[s], qf[s], st, s, ks, qs);
                else                 st = score_mfma48<FMT8>(kf[s], qf[s], st, s, ks, qs);
            }
            return st;
        };
        auto probability = [&](const v16f& st, int e, float& s0, float& s1) __attribute__((always_inline)) {
            const float p0 = __builtin_amdgcn_exp2f(st[e]), p1 = __builtin_amdgcn_exp2f(st[e + 1]);
            s0 += p0;
            s1 += p1;
            return __builtin_bit_cast(int, P::pack(p0, p1));
        };
        // maximum first
        auto careful = [&](v16f& st, int j) __attribute__((always_inline)) {
            if (j == masked_at) {
                const int kmax = a.n - 1 - j * 32;                                                            // last visible key of the block
#pragma unroll
                for (int e = 0; e < 16; ++e)
                    if (8 * (e >> 2) + 4 * h + (e & 3) > kmax) st[e] = -__builtin_inff();
            }
            float mx = st[0];
#pragma unroll
            for (int e = 1; e < 16; ++e) mx = __builtin_fmaxf(mx, st[e]);
            mx = max_lane_pair(mx);
            if (j == 0 || __any(mx > P::REBASE)) {
                const float delta = j == 0 ? mx : __builtin_fmaxf(mx, 0.0f);
                m_run += delta;
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    st[e] -= delta;
                    minus_m[e] = -m_run;
                }
                if (j > 0) {
                    const float alpha = __builtin_amdgcn_exp2f(-delta);
                    l_run *= alpha;
#pragma unroll
                    for (int d = 0; d < G::NDB; ++d)
#pragma unroll
                        for (int e = 0; e < 16; ++e) acc[d][e] *= alpha;
                }
            }
            float s0 = 0.0f, s1 = 0.0f;
#pragma unroll
            for (int e = 0; e < 16; e += 2) pk[e >> 3][(e & 7) >> 1] = probability(st, e, s0, s1);
            ps = s0 + s1;
        };
        load_k(0);
        v16f st = scores();
        load_k(nb > 1 ? 1 : 0);
        careful(st, 0);
        l_run = ps;
        st = scores();
        // block j's exponentials go with the P.V product of block j - 1, instruction by instruction, and block j + 1's scores
        // follow; the exponentials are taken against the old maximum, and a row sum that shows a score far above it, or a mask,
        // sends the wave back to do the block with the maximum first
#pragma unroll 1
        for (int j = 1; j < nb; ++j) {
            load_v(j - 1, 0);
            load_k(min(j + 1, nb - 1));
            __builtin_amdgcn_sched_barrier(0);
            v4i pn[2];
            float s0 = 0.0f, s1 = 0.0f;
            constexpr int PER = 16 / (2 * G::NDB);        // exponentials per P.V instruction
#pragma unroll
            for (int x = 0; x < 2 * G::NDB; ++x) {
                const int c = x / G::NDB, d = x % G::NDB;
                if (x > 0) acc[d] = P::mfma(vf[c][d], __builtin_bit_cast(typename P::vec, pk[c]), acc[d]);
#pragma unroll
                for (int e = x * PER; e < (x + 1) * PER; e += 2) pn[e >> 3][(e & 7) >> 1] = probability(st, e, s0, s1);
                __builtin_amdgcn_sched_barrier(0);
                if (x == 0) {
                    acc[d] = P::mfma(vf[c][d], __builtin_bit_cast(typename P::vec, pk[c]), acc[d]);
                    load_v(j - 1, 1);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            ps = s0 + s1;
            pk[0] = pn[0];
            pk[1] = pn[1];
            if ((__ballot(!(ps < P::OPTIMISTIC_LIMIT)) | (j == masked_at ? 1ull : 0ull)) != 0) careful(st, j);
            l_run += ps;
            st = scores();
            __builtin_amdgcn_sched_barrier(0);
        }
        load_v(nb - 1, 0);
        load_v(nb - 1, 1);
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int d = 0; d < G::NDB; ++d) acc[d] = P::mfma(vf[c][d], __builtin_bit_cast(typename P::vec, pk[c]), acc[d]);
        const float inv = 1.0f / sum_lane_pair(l_run);
        store_output<2 * G::NDB>(a, b, hq_now, row_now + r, 0, h, [&](int x) __attribute__((always_inline)) {
            const v16f& o = acc[x >> 2];
            const int e = 4 * (x & 3);
            return (v4f){o[e], o[e + 1], o[e + 2], o[e + 3]};
        }, inv);
    }
}

template <int PVT, int FMT8, int MODE>
struct ResidentLds {
    static inline const bool registered = mpsa_register_lds_kernel(reinterpret_cast<const void*>(attn_resident_kernel<PVT, FMT8, MODE>), 163840);
};

template <int PVT, int FMT8, int MODE>
int launch_one(const ResidentArgs& s, unsigned grid, hipStream_t st) {
    if (!ResidentLds<PVT, FMT8, MODE>::registered) return mpsa_fail(MPSA_ELAUNCH, "attn: kernel not registered");
    const int rc = mpsa_ensure_init();
    if (rc != MPSA_OK) return rc;
    const unsigned lds = (unsigned)(Resident<MODE>::lds(s.nb));
    hipLaunchKernelGGL((attn_resident_kernel<PVT, FMT8, MODE>), dim3(grid), dim3(RW * 64), lds, st, s);
    MPSA_CHECK_LAUNCH("attn (resident)");
    return MPSA_OK;
}

template <int PVT>
int launch_mode(const ResidentArgs& s, unsigned grid, hipStream_t st) {
    const bool e5 = s.fmt8 == MPSA_FMT_E5M2;
    if (s.mode == MPSA_MODE_MXFP8) return e5 ? launch_one<PVT, MPSA_FMT_E5M2, MPSA_MODE_MXFP8>(s, grid, st) : launch_one<PVT, MPSA_FMT_E4M3, MPSA_MODE_MXFP8>(s, grid, st);
    return e5 ? launch_one<PVT, MPSA_FMT_E5M2, MPSA_MODE_MIXED>(s, grid, st) : launch_one<PVT, MPSA_FMT_E4M3, MPSA_MODE_MIXED>(s, grid, st);
}

}  // namespace

int attn_resident_shares(const AttnArgs& a) {
    if (!a.q_raw || a.causal || a.d != D || (a.mode != MPSA_MODE_MXFP8 && a.mode != MPSA_MODE_MIXED)) return 0;
    const int64_t nb = ((int64_t)a.n + 31) / 32;
    if (nb > 64 || (a.mode == MPSA_MODE_MXFP8 ? Resident<MPSA_MODE_MXFP8>::lds((int)nb) : Resident<MPSA_MODE_MIXED>::lds((int)nb)) > 163840) return 0;
    return (int)resident_choice(a.B, a.Hq, a.Hkv, a.nq, a.n);
}

int attn_resident_launch(const AttnArgs& a, int pv_dtype, int shares, hipStream_t st) {
    ResidentArgs s;
    static_cast<AttnArgs&>(s) = a;
    s.units = a.B * a.Hkv;
    s.group = a.Hq / a.Hkv;
    s.nqb = (a.nq + 31) / 32;
    s.tasks = s.group * s.nqb;
    s.nb = (a.n + 31) / 32;
    s.step = shares * RW;
    s.by_units = reciprocal_of(s.units); s.by_hkv = reciprocal_of(a.Hkv); s.by_nqb = reciprocal_of(s.nqb);
    const unsigned grid = (unsigned)((int64_t)s.units * shares);
    return pv_dtype == MPSA_BF16 ? launch_mode<MPSA_BF16>(s, grid, st) : launch_mode<MPSA_F16>(s, grid, st);
}
