// Fused attention forward for short and middle sequences (gfx950): the math of attn_fwd_kernel.h, mapped for latency.
//
// What bounds a short prompt is one workgroup's serial chain: a paired-tile workgroup takes 256 queries through a prologue and
// an epilogue of 28 000 clocks and 3 600 clocks a tile, and there are 32 of them (160 tokens, 32 heads) for 256 CUs.  Here a
// workgroup of four waves owns 32, 64 or 128 queries, a wave 32 of them, and KS = 4, 2 or 1 waves split the KEYS of the same
// queries: split s takes the 32-key blocks s, s + KS, ... with a running maximum, row sum and output of its own, and the
// partial results are merged through LDS (in a fixed order: results do not depend on timing).  Many splits make short chains
// and many workgroups for few queries; few splits share a stage's K and V between more queries.
// A stage is KS blocks.  K and V arrive two stages ahead in LDS rings of three; the scores of a stage are taken together with
// the P.V product of the stage before, so that a wave's exponentials run under its own matrix instructions.  Clock stamps in a
// copy of this kernel, D = 128, 333 keys, 8 bits: with one wave a SIMD a stage takes 1120 clocks, of which 290 are loads and
// barrier and 290 LDS reads and scores; with two, 660 each.  Before the loop Q's quantization takes 3600 clocks (5300 with two
// waves) of the workgroup's 25 000, after it the last P.V product and the store 3100.  Two of these workgroups share a CU (80
// KiB of LDS, 190 registers); four splits take it whole.
// Q may arrive unquantized (a.q_raw): the workgroup quantizes its rows into LDS, eight elements per lane, with the quantizer's
// own code -- the bits of mpsa_quantize_mx.
// With 32 heads, 8 KV heads, causal, D = 128 (us of this kernel in a kernel trace; tile kernels): 160 tokens 6.8 (12.8), 1000
// tokens 17 (25).  Many queries over keys that fit LDS may go on to attn_fwd_resident.hip.
#include "attn_common.h"
#include "quantize_kernel.h"
#include "reciprocal.h"

namespace {

struct ShortArgs : AttnArgs {
    Reciprocal by_split, by_group, by_hkv;        // first: they arrive with the end of AttnArgs, the first thing a workgroup needs
    int group, per_unit, nqb, np;                 // query heads per KV head; workgroups per (batch, KV head); 32-query blocks, workgroups per head
    int dealt, slice;                             // rows dealt out over the XCDs; else (batch, KV head) pairs per XCD
    int rows_first, split_by;                     // whether a pair's rows follow each other; the divisor of a workgroup's place
    int longest, shortest;                        // causal: row blocks from the long end that come first, then those from the short end; the rest, long ones first
};

template <int D, int MODE, int KS>
struct Short {
    static constexpr bool MAIN8 = MODE == MPSA_MODE_MXFP8;
    static constexpr bool Q4USED = !MAIN8 && MODE != MPSA_MODE_MIXED, Q8USED = MODE != MPSA_MODE_MXFP4;
    static constexpr int QW = 4 / KS, QR = 32 * QW;                             // query blocks, query rows of a workgroup
    static constexpr int SST = D / 64;            // score matrix instructions along D
    static constexpr int NDB = D / 32;            // 32-wide output dim blocks
    static constexpr int ROW4 = D / 2, ROW8 = D;  // bytes per K row
    static constexpr int CPR4 = ROW4 / 16, CPR8 = ROW8 / 16;
    static constexpr int SH4 = CPR4 == 2 ? 3 : 2, SH8 = CPR8 == 4 ? 2 : 1;      // log2(rows per 256 bytes)
    static constexpr int ROW = MAIN8 ? ROW8 : ROW4, CPR = MAIN8 ? CPR8 : CPR4, SH = MAIN8 ? SH8 : SH4;
    // a stage: KS blocks of 32 keys, K rows and V fragments, in rings of three.  In LDS: V 0, V 1, K 0, K 1, K 2, V 2
    static constexpr int KBLOCK = 32 * ROW, VBLOCK = 32 * D * 2, KBUF = KS * KBLOCK, VBUF = KS * VBLOCK, RINGS = 3 * (KBUF + VBUF);
    static constexpr int KI = KBUF / 1024, VI = VBUF / 1024;                    // load instructions of a stage
    static constexpr int LOADS = (KI >= 4 ? KI / 4 : 0) + VI / 4 + 1;           // of which every wave has issued at least this many
    // quantized Q, codes and scales of both widths, lies where K 2 and V 2 will be: it is in registers by then
    static constexpr int Q4 = 2 * VBUF + 2 * KBUF, QS4 = Q4 + (Q4USED ? QR * ROW4 : 0), Q8 = QS4 + (Q4USED ? QR * NDB : 0), QS8 = Q8 + (Q8USED ? QR * ROW8 : 0);
    static constexpr int QEND = QS8 + (Q8USED ? QR * NDB : 0);
    // K scale words of three stages, a copy per wave; a diag run's own rows, 8 bits wide, and their scales
    static constexpr int KSC = QEND > RINGS ? QEND : RINGS, OWN = KSC + 3 * 1024;
    static constexpr int OWN_ROWS = MODE == MPSA_MODE_DIAG ? 128 : 0, OWNSC = OWN + OWN_ROWS * ROW8, LOOP = OWNSC + OWN_ROWS * NDB;
    // the merge: partial outputs, then every wave's maxima and sums
    static constexpr int UNITS = D / 16 / KS;                                   // 16-dim units each split finishes
    static constexpr int PART = (KS - 1) * UNITS * 2 * 64 * 16, ML = 4 * PART, MERGE = KS > 1 ? ML + 1024 : 0;
    static constexpr int SMEM = LOOP > MERGE ? LOOP : MERGE;
};

template <int D, int PVT, int FMT8, int MODE, int KS>
__global__ __launch_bounds__(256, D == 128 ? 2 : 3) void attn_short_kernel(ShortArgs a) {
    typedef Short<D, MODE, KS> G;
    typedef PV<PVT> P;
    constexpr bool MIXED = MODE == MPSA_MODE_MIXED, DIAG = MODE == MPSA_MODE_DIAG, MAIN8 = G::MAIN8, Q4 = G::Q4USED, Q8 = G::Q8USED;
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int h = lane >> 5, r = lane & 31, qw = w / KS, split = w % KS;

    // ---- which (batch, kv head, query head, query rows): one KV head's query heads per XCD; fewer heads than XCDs, or an uneven
    //      number: the rows of a head are dealt out over all of them.  Divisions by the host's reciprocals, and no branches: the
    //      arguments arrive in one go. ----
    const int place = a.dealt ? (int)blockIdx.x : (int)(blockIdx.x >> 3);
    const int quot = divide_by(place, a.by_split), rest = place - quot * a.split_by;
    const int row = a.rows_first ? rest : quot;           // query rows times query heads of the group
    const int unit = (a.dealt ? 0 : (int)(blockIdx.x & 7) * a.slice) + (a.rows_first ? quot : rest);     // (batch, kv head)
    const int rank = divide_by(row, a.by_group), sub = row - rank * a.group;
    const int b = divide_by(unit, a.by_hkv), kvh = unit - b * a.Hkv, hq = kvh * a.group + sub;
    const int p = !a.causal ? rank : rank < a.longest ? a.np - 1 - rank : rank < a.longest + a.shortest ? rank - a.longest : a.np - 1 - rank + a.shortest;
    const int64_t krow0 = (int64_t)unit * a.n_pad;

    // ---- this workgroup's queries, quantized, into LDS: their loads go out in front of the first stage's, which nobody waits
    //      for before the queries are through ----
    constexpr int CHUNKS = G::QR * D / 8 / 256;          // of eight elements, per thread
    auto raw_chunk = [&](int q) __attribute__((always_inline)) {
        const int c = q * 256 + tid, src = min(G::QR * p + c / (D / 8), a.nq - 1);
        return *reinterpret_cast<const uint4*>(static_cast<const char*>(a.q_raw) + 2 * ((int64_t)b * a.q_sb + (int64_t)hq * a.q_sh + (int64_t)src * a.q_sn + 8 * (c % (D / 8))));
    };
    uint4 raw[CHUNKS];
    if (a.q_raw) {
#pragma unroll
        for (int q = 0; q < CHUNKS; ++q) raw[q] = raw_chunk(q);
    }
    __builtin_amdgcn_sched_barrier(0);

    // ---- this wave's key blocks: KS j + split of stage j, up to its query block (causal) ----
    const int nb = (a.n + 31) / 32, qb = G::QW * p + qw, qb_last = min(G::QW * p + G::QW, a.nqb) - 1;
    const int mine = qb >= a.nqb ? 0 : a.causal ? min(qb + 1, nb) : nb;
    const int blocks = mine > split ? (mine - split + KS - 1) / KS : 0;
    // with four splits a wave loads what it reads itself
    const int stages = KS == 4 ? blocks : ((a.causal ? min(qb_last + 1, nb) : nb) + KS - 1) / KS;
    const int masked_kb = a.causal ? qb : (a.n & 31) ? nb - 1 : -1;
    const int own_first = a.tile == 128 ? qb & ~3 : qb & ~1;
    const int masked_at = masked_kb >= 0 && masked_kb % KS == split ? masked_kb / KS : -1;      // as stages
    const int own_at = (own_first - split + KS - 1) / KS, own_end = (own_first + a.tile / 32 - split + KS - 1) / KS;

    // ---- a stage's operands into LDS: K rows (swizzled) and V fragments, a quarter of the loads per wave, and the wave's own K
    //      scale words.  Sources only move forward, ring places turn: few scalar instructions, which a lone wave feels. ----
    constexpr int KPER = G::KI >= 4 ? G::KI / 4 : 1, VPER = G::VI / 4;
    const uint8_t* kg = (MAIN8 ? a.k8 : a.k4) + krow0 * G::ROW + w * (KPER * 1024);
    const uint8_t* vg = static_cast<const uint8_t*>(a.v) + krow0 * (D * 2) + w * (VPER * 1024);
    const uint8_t* ksg = (MAIN8 ? a.ks8 : a.ks4) + (krow0 + 32 * split) * G::NDB;
    uint32_t k_lane[KPER];
#pragma unroll
    for (int x = 0; x < KPER; ++x) {
        const int at = (w * KPER + x) * 64 + lane, krow = at / G::CPR, chunk = at % G::CPR;
        k_lane[x] = (krow - w * (KPER * 64 / G::CPR) - x * (64 / G::CPR)) * G::ROW + (chunk ^ ((krow >> G::SH) & (G::CPR - 1))) * 16;
    }
    const uint32_t v_lane = lane * 16, ks_lane = D == 128 ? r * 4 : (r >> 1) * 4;
    auto fetch_k = [&](int slot) __attribute__((always_inline)) {
        uint8_t* const to = smem + 2 * G::VBUF + slot * G::KBUF + w * (KPER * 1024);
        if (G::KI >= 4 || w < G::KI) {
#pragma unroll
            for (int x = 0; x < KPER; ++x) load16_to_lds_sv(k_lane[x], kg + x * 1024, to + x * 1024);
        }
        load4_to_lds_sv(ks_lane, ksg, smem + G::KSC + slot * 1024 + w * 256);
        kg += G::KBUF;
        ksg += KS * 32 * G::NDB;
    };
    auto v_at = [&](int slot) { return smem + slot * G::VBUF + (slot == 2 ? 3 * G::KBUF : 0); };
    auto fetch_v = [&](int slot) __attribute__((always_inline)) {
        uint8_t* const to = v_at(slot) + w * (VPER * 1024);
#pragma unroll
        for (int x = 0; x < VPER; x += 4) load16n_to_lds_sv<(VPER < 4 ? VPER : 4)>(v_lane, vg + x * 1024, to + x * 1024);
        vg += G::VBUF;
    };
    // the rows of a diag run's own tile (all of this workgroup's: one tile, or with 128 queries and tiles of 64 two)
    const int own_rows = max(a.tile, G::QR), own_base = G::QR * p & ~(own_rows - 1);
    auto fetch_own = [&]() __attribute__((always_inline)) {
        const uint8_t* const k8 = a.k8 + (krow0 + own_base) * G::ROW8;
        const uint8_t* const ks8 = a.ks8 + (krow0 + own_base) * G::NDB;
        const int last = a.n_pad - 1 - own_base;
#pragma unroll
        for (int x = 0; x < 128 * G::ROW8 / 4096; ++x) {
            const int c = w * (128 * G::ROW8 / 4096) + x, at = c * 64 + lane, krow = at / G::CPR8, chunk = at % G::CPR8;
            load16_to_lds_sv((uint32_t)(min(krow, last) * G::ROW8 + (chunk ^ ((krow >> G::SH8) & (G::CPR8 - 1))) * 16), k8, smem + G::OWN + c * 1024);
        }
        if (w < 2 * G::NDB / 4) {
            const int at = (w * 64 + lane) * 4;
            load4_to_lds_sv((uint32_t)min(at, last * G::NDB & ~3), ks8, smem + G::OWNSC + w * 256);
        }
    };
    if (KS < 4 || stages > 0) fetch_k(0);
    __builtin_amdgcn_sched_barrier(0);

    auto put_q = [&](int c, uint32_t w4, int s4, uint2 w8, int s8) __attribute__((always_inline)) {
        // (the four lanes of an MX block all write its scale byte: no branch)
        if constexpr (Q4) {
            *reinterpret_cast<uint32_t*>(smem + G::Q4 + c * 4) = w4;
            smem[G::QS4 + (c >> 2)] = (uint8_t)s4;
        }
        if constexpr (Q8) {
            *reinterpret_cast<uint2*>(smem + G::Q8 + c * 8) = w8;
            smem[G::QS8 + (c >> 2)] = (uint8_t)s8;
        }
    };
    if (a.q_raw) {
        // Straight through, without a branch between the chunks.  A wave with a rare chunk does all of its own again, and so do all
        // where the 4-bit codes are the rule's to look at.  Rows past the last are zeros: nobody reads their results, but a maximum
        // that moves moves for the whole wave.
        bool again = Q4 && a.q_sure == 0;
        auto inside = [&](int q) { return G::QR * p + (q * 256 + tid) / (D / 8) < a.nq; };
        if (!again) {
            bool rare = false;
#pragma unroll
            for (int q = 0; q < CHUNKS; ++q) {
                float x[8];
                uint32_t w4 = 0;
                uint2 w8 = make_uint2(0, 0);
                int s4 = 0, s8 = 0;
                bool r1;
                unpack8<PVT>(raw[q], x);
                const float pre = inside(q) ? a.q_pre : 0.0f;
#pragma unroll
                for (int i = 0; i < 8; ++i) x[i] *= pre;
                quantize_straight<Q4, Q8, FMT8>(x, w4, s4, w8, s8, r1);
                rare |= r1;
                put_q(q * 256 + tid, w4, s4, w8, s8);
            }
            again = __ballot(rare) != 0;
        }
        if (again) {
#pragma unroll
            for (int q = 0; q < CHUNKS; ++q) {
                float x[8];
                uint32_t w4;
                uint2 w8;
                int s4, s8;
                unpack8<PVT>(inside(q) ? only_here(raw[q]) : make_uint4(0, 0, 0, 0), x);
                quantize_chunk<Q4, Q8, FMT8, false, true>(x, a.q_pre, a.q_sure != 0, 3, 7, w4, s4, w8, s8);
                put_q(q * 256 + tid, w4, s4, w8, s8);
            }
        }
    } else {
        // rows up to nq_pad exist (zeros beyond nq); a last workgroup may reach past them
        const int64_t chunk0 = (((int64_t)b * a.Hq + hq) * a.nq_pad + G::QR * p) * (D / 8);
        const int left = (a.nq_pad - G::QR * p) * (D / 8);
#pragma unroll 2
        for (int q = 0; q < CHUNKS; ++q) {
            const int c = q * 256 + tid;
            uint32_t w4 = 0;
            uint2 w8 = make_uint2(0, 0);
            int s4 = 0, s8 = 0;
            if (c < left) {
                if constexpr (Q4) { w4 = reinterpret_cast<const uint32_t*>(a.q4)[chunk0 + c]; s4 = a.qs4[(chunk0 + c) >> 2]; }
                if constexpr (Q8) { w8 = reinterpret_cast<const uint2*>(a.q8)[chunk0 + c]; s8 = a.qs8[(chunk0 + c) >> 2]; }
            }
            put_q(c, w4, s4, w8, s8);
        }
    }
    if (DIAG) fetch_own();
    if (stages > 1) fetch_k(1);
    if (KS < 4 || stages > 0) fetch_v(0);
    __syncthreads();
    const int qrow = 32 * qw + r;
    auto scale_word = [&](int off, int row) { return D == 128 ? *reinterpret_cast<const uint32_t*>(smem + off + row * 4) : (uint32_t)*reinterpret_cast<const uint16_t*>(smem + off + row * 2); };
    auto load_q = [&](v8i (&q)[G::SST], bool is8) __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < G::SST; ++s) {
            if (is8) {
                const v4i x0 = *reinterpret_cast<const v4i*>(smem + G::Q8 + qrow * G::ROW8 + s * 64 + h * 16);
                const v4i x1 = *reinterpret_cast<const v4i*>(smem + G::Q8 + qrow * G::ROW8 + s * 64 + h * 16 + 32);
                q[s] = (v8i){x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]};
            } else {
                const v4i x0 = *reinterpret_cast<const v4i*>(smem + G::Q4 + qrow * G::ROW4 + (2 * s + h) * 16);
                q[s] = (v8i){x0[0], x0[1], x0[2], x0[3], 0, 0, 0, 0};
            }
        }
    };
    v8i qf[G::SST], q8f[DIAG ? G::SST : 1];
    load_q(qf, !Q4);
    const int qs = (int)(scale_word(Q4 ? G::QS4 : G::QS8, qrow) >> (8 * h));
    int qs8 = 0;
    if constexpr (DIAG) {
        load_q(q8f, true);
        qs8 = (int)(scale_word(G::QS8, qrow) >> (8 * h));
    }

    v16f acc[G::NDB], minus_m;                            // scores start from minus the reference maximum
#pragma unroll
    for (int d = 0; d < G::NDB; ++d)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[d][e] = 0.0f;
#pragma unroll
    for (int e = 0; e < 16; ++e) minus_m[e] = 0.0f;
    float m_run = 0.0f, l_run = 0.0f;                     // lazily moved reference maximum and row sum, as in attn_fwd_kernel.h
    v4i pk[2];

    int now = 0, next = 1, last = 2;                      // ring places of stages j, j + 1 and j + 2 (or j - 1)
    // stage j's K and the V of the one before have landed (the next may be on its way), and nobody reads older ones any more
    auto turn = [&](int j) __attribute__((always_inline)) {
        if (j > 0) {
            const int t = now;
            now = next;
            next = last;
            last = t;
        }
        if (j + 1 < stages) __builtin_amdgcn_s_waitcnt(0x0F70 | (G::LOADS & 15) | (G::LOADS >> 4 << 14));
        else                __builtin_amdgcn_s_waitcnt(0x0F70);
        if (KS < 4 || j == 0) __syncthreads();
        __builtin_amdgcn_sched_barrier(0);
        if (j + 2 < stages) fetch_k(last);
        if (j + 1 < stages) fetch_v(next);
        __builtin_amdgcn_sched_barrier(0);
    };
    typename P::vec vf[2][G::NDB];
    auto load_v = [&](int c) __attribute__((always_inline)) {
        const uint8_t* const vbuf = v_at(last) + split * G::VBLOCK + lane * 16;
#pragma unroll
            for (int d = 0; d < G::NDB; ++d) vf[c][d] = *reinterpret_cast<const typename P::vec*>(vbuf + (c * G::NDB + d) * 1024);
    };
    auto scores = [&](int j, auto with_v) __attribute__((always_inline)) {
        const uint8_t* const kbuf = smem + 2 * G::VBUF + now * G::KBUF + split * G::KBLOCK;
        v16f st = minus_m;
        if (DIAG && j >= own_at && j < own_end) {
            const int krow = (KS * j + split) * 32 - own_base + r, f = (krow >> G::SH8) & (G::CPR8 - 1);
            const int ks = (int)(scale_word(G::OWNSC, krow) >> (8 * h));
            v8i kf[G::SST];
#pragma unroll
            for (int s = 0; s < G::SST; ++s) {
                const v4i x0 = *reinterpret_cast<const v4i*>(smem + G::OWN + krow * G::ROW8 + (((4 * s + h) ^ f) * 16));
                const v4i x1 = *reinterpret_cast<const v4i*>(smem + G::OWN + krow * G::ROW8 + (((4 * s + h + 2) ^ f) * 16));
                kf[s] = (v8i){x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]};
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int s = 0; s < G::SST; ++s) st = score_mfma8<FMT8>(kf[s], q8f[DIAG ? s : 0], st, s, ks, qs8);
            // 20 wait states lie between an 8-bit product and the use of its result, 12 behind a 4-bit one; where the two paths meet
            // the compiler counted 12 for both
            asm volatile("s_nop 7" : "+v"(st));
        } else {
            const uint32_t ks_word = *reinterpret_cast<const uint32_t*>(smem + G::KSC + now * 1024 + w * 256 + lane * 4) >> (D == 128 ? 0 : 16 * (r & 1));
            const int ks = (int)(ks_word >> (8 * h)), f = (r >> G::SH) & (G::CPR - 1);
            v8i kf[G::SST];
#pragma unroll
            for (int s = 0; s < G::SST; ++s) {
                if constexpr (MAIN8) {
                    const v4i x0 = *reinterpret_cast<const v4i*>(kbuf + r * G::ROW + (((4 * s + h) ^ f) * 16));
                    const v4i x1 = *reinterpret_cast<const v4i*>(kbuf + r * G::ROW + (((4 * s + h + 2) ^ f) * 16));
                    kf[s] = (v8i){x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]};
                } else {
                    const v4i x = *reinterpret_cast<const v4i*>(kbuf + r * G::ROW + (((2 * s + h) ^ f) * 16));
                    kf[s] = (v8i){x[0], x[1], x[2], x[3], 0, 0, 0, 0};
                }
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int s = 0; s < G::SST; ++s) {
                if constexpr (MAIN8)      st = score_mfma8<FMT8>(kf[s], qf[s], st, s, ks, qs);
                else if constexpr (MIXED) st = score_mfma48<FMT8>(kf[s], qf[s], st, s, ks, qs);
                else                      st = score_mfma4(kf[s], qf[s], st, s, ks, qs);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (decltype(with_v)::value) load_v(0);
        __builtin_amdgcn_sched_barrier(0);
        return st;
    };
    float ps;
    auto probability = [&](const v16f& st, int e, float& s0, float& s1) __attribute__((always_inline)) {
        const float p0 = __builtin_amdgcn_exp2f(st[e]), p1 = __builtin_amdgcn_exp2f(st[e + 1]);
        s0 += p0;
        s1 += p1;
        return __builtin_bit_cast(int, P::pack(p0, p1));
    };
    // maximum first
    auto careful = [&](v16f& st, int j) __attribute__((always_inline)) {
        if (j == masked_at) {
            const int kmax = a.causal ? r : a.n - 1 - masked_kb * 32;                                     // last visible key of the block
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
    turn(0);
    if (blocks > 0) {
        v16f st = scores(0, std::false_type{});
        careful(st, 0);
        l_run = ps;
    }
    // The scores of stage j and the P.V product of stage j - 1 go together: while the vector units take the exponentials of the
    // one, the matrix cores do the other, instruction by instruction.  The exponentials are taken against the old maximum at
    // once, and a row sum that shows a score far above it sends the wave back to do the block with the maximum first, as does
    // a mask: no reduction and no branch between the scores and the exponentials.
    // Alone on its SIMD a wave feels where its instructions lie: in steps of a word the loop's place moves 8 heads of 128 queries over
    // 16384 keys, 4-bit, between 56.7 and 59.4 us, with a period of 32 bytes (59.0 where the code in front of it had left it), and 8
    // heads of 1024 x 64, causal, diag, between 7.14 and 7.31 (7.27).  The other modes gain less than 1 % or lose.
    if constexpr (KS == 4 && (D == 128 ? MODE == MPSA_MODE_MXFP4 : DIAG)) asm volatile(".p2align 5\n\t.fill 2, 4, 0xBF800000");      // s_nop 0
#pragma unroll 1
    for (int j = 1; j < blocks; ++j) {
        turn(j);
        v16f st = scores(j, std::true_type{});
        v4i pn[2];
        float s0 = 0.0f, s1 = 0.0f;
        constexpr int PER = 16 / (2 * G::NDB);            // exponentials per P.V instruction
#pragma unroll
        for (int x = 0; x < 2 * G::NDB; ++x) {
            const int c = x / G::NDB, d = x % G::NDB;
            if (x > 0) acc[d] = P::mfma(vf[c][d], __builtin_bit_cast(typename P::vec, pk[c]), acc[d]);
#pragma unroll
            for (int e = x * PER; e < (x + 1) * PER; e += 2) pn[e >> 3][(e & 7) >> 1] = probability(st, e, s0, s1);
            __builtin_amdgcn_sched_barrier(0);
            if (x == 0) {
                acc[d] = P::mfma(vf[c][d], __builtin_bit_cast(typename P::vec, pk[c]), acc[d]);
                load_v(1);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        ps = s0 + s1;
        pk[0] = pn[0];
        pk[1] = pn[1];
        if ((__ballot(!(ps < P::OPTIMISTIC_LIMIT)) | (j == masked_at ? 1ull : 0ull)) != 0) careful(st, j);
        l_run += ps;
    }
    if (blocks > 0) {
        turn(blocks);
        load_v(0);
        load_v(1);
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int d = 0; d < G::NDB; ++d) acc[d] = P::mfma(vf[c][d], __builtin_bit_cast(typename P::vec, pk[c]), acc[d]);
    }
#pragma unroll 1
    for (int j = blocks + 1; KS < 4 && j <= stages; ++j) turn(j);
    __builtin_amdgcn_s_waitcnt(0x0F70);                   // no load into LDS may outlive this point

    const float l_own = sum_lane_pair(l_run);
    auto piece = [&](int u, int q) { const v16f& x = acc[u >> 1]; const int e = 8 * (u & 1) + 4 * q; return (v4f){x[e], x[e + 1], x[e + 2], x[e + 3]}; };
    if constexpr (KS == 1) {
        const float inv = 1.0f / l_own;
        store_output<G::UNITS>(a, b, hq, 32 * qb + r, 0, h, [&](int x) __attribute__((always_inline)) { return piece(x >> 1, x & 1); }, inv);
    } else {
        // ---- merge: split s finishes the s-th share of the dims.  Every wave leaves the other shares of its partial output in
        //      LDS, then brings the splits' pieces of its own share to their common maximum and adds them in split order. ----
        float* const ml = reinterpret_cast<float*>(smem + G::ML) + qw * KS * 64;          // [split][maximum, sum][query]
        __syncthreads();
        if (lane < 32) {
            ml[split * 64 + r] = mine > split ? m_run : -__builtin_inff();
            ml[split * 64 + 32 + r] = l_own;
        }
        v4f o[G::UNITS][2];
        auto part = [&](int from, int to) { return reinterpret_cast<v4f*>(smem + (qw * KS + from) * G::PART) + (to < from ? to : to - 1) * (G::UNITS * 2 * 64) + lane; };
        auto finish = [&](auto mine_c) __attribute__((always_inline)) {
            constexpr int S = decltype(mine_c)::value;
#pragma unroll
            for (int to = 0; to < KS; ++to)
#pragma unroll
                for (int x = 0; x < 2 * G::UNITS; ++x)
                    if (to != S) part(S, to)[x * 64] = piece(to * G::UNITS + (x >> 1), x & 1);
#pragma unroll
            for (int x = 0; x < 2 * G::UNITS; ++x) o[x >> 1][x & 1] = piece(S * G::UNITS + (x >> 1), x & 1);
        };
        if (split == 0) finish(std::integral_constant<int, 0>{});
        if (split == 1) finish(std::integral_constant<int, 1>{});
        if constexpr (KS == 4) {
            if (split == 2) finish(std::integral_constant<int, 2>{});
            if (split == 3) finish(std::integral_constant<int, 3>{});
        }
        __syncthreads();
        float mall = ml[r], lall = 0.0f;
#pragma unroll
        for (int y = 1; y < KS; ++y) mall = __builtin_fmaxf(mall, ml[y * 64 + r]);
        const float own = __builtin_amdgcn_exp2f(ml[split * 64 + r] - mall);
        v4f sum[G::UNITS][2];
#pragma unroll
        for (int x = 0; x < 2 * G::UNITS; ++x) sum[x >> 1][x & 1] = o[x >> 1][x & 1] * own;
#pragma unroll
        for (int d = 0; d < KS; ++d) {                     // sums in split order; the outputs start from the wave's own
            const int y = (split + d) & (KS - 1);
            lall += ml[d * 64 + 32 + r] * __builtin_amdgcn_exp2f(ml[d * 64 + r] - mall);
            if (d == 0) continue;
            const float factor = __builtin_amdgcn_exp2f(ml[y * 64 + r] - mall);
            const v4f* q = part(y, split);
#pragma unroll
            for (int x = 0; x < 2 * G::UNITS; ++x) sum[x >> 1][x & 1] += q[x * 64] * factor;
        }
        const float inv = 1.0f / lall;
        store_output<G::UNITS>(a, b, hq, 32 * qb + r, 16 * split * G::UNITS, h, [&](int x) __attribute__((always_inline)) { return sum[x >> 1][x & 1]; }, inv);
    }
}

template <int D, int PVT, int FMT8, int MODE, int KS>
struct ShortLds {
    static inline const bool registered = mpsa_register_lds_kernel(reinterpret_cast<const void*>(attn_short_kernel<D, PVT, FMT8, MODE, KS>), Short<D, MODE, KS>::SMEM);
};

template <int D, int PVT, int FMT8, int MODE, int KS>
int launch_one(const AttnArgs& a, hipStream_t st) {
    if (!ShortLds<D, PVT, FMT8, MODE, KS>::registered) return mpsa_fail(MPSA_ELAUNCH, "attn: kernel not registered");
    const int rc = mpsa_ensure_init();
    if (rc != MPSA_OK) return rc;
    ShortArgs s;
    static_cast<AttnArgs&>(s) = a;
    const int units = a.B * a.Hkv;
    s.group = a.Hq / a.Hkv;
    s.nqb = (a.nq + 31) / 32;
    s.np = (s.nqb + 4 / KS - 1) / (4 / KS);
    s.per_unit = s.group * s.np;
    s.dealt = (units & 7) != 0;
    s.slice = units / 8;
    const int total = units * s.per_unit, heads = a.B * a.Hq;
    s.rows_first = !s.dealt && !(a.causal && total <= 1536);
    s.split_by = s.rows_first ? s.per_unit : s.dealt ? units : s.slice;
    const int layer = max(1, 256 / heads);
    s.longest = s.rows_first || !a.causal ? s.np : min(s.np, layer);
    s.shortest = min(s.np - s.longest, total <= 512 ? s.np : layer);
    s.by_split = reciprocal_of(s.split_by); s.by_group = reciprocal_of(s.group); s.by_hkv = reciprocal_of(a.Hkv);
    hipLaunchKernelGGL((attn_short_kernel<D, PVT, FMT8, MODE, KS>), dim3((unsigned)(units * s.per_unit)), dim3(256), (Short<D, MODE, KS>::SMEM), st, s);
    MPSA_CHECK_LAUNCH("attn (short)");
    return MPSA_OK;
}

template <int D, int PVT, int FMT8, int MODE>
int launch_split(const AttnArgs& a, int splits, hipStream_t st) {
    if (splits == 4) return launch_one<D, PVT, FMT8, MODE, 4>(a, st);
    if (splits == 2) return launch_one<D, PVT, FMT8, MODE, 2>(a, st);
    return launch_one<D, PVT, FMT8, MODE, 1>(a, st);
}

template <int D, int PVT, int FMT8>
int launch_mode(const AttnArgs& a, int splits, hipStream_t st) {
    if (a.mode == MPSA_MODE_MIXED) return launch_split<D, PVT, FMT8, MPSA_MODE_MIXED>(a, splits, st);
    if (a.mode == MPSA_MODE_MXFP8) return launch_split<D, PVT, FMT8, MPSA_MODE_MXFP8>(a, splits, st);
    return launch_split<D, PVT, FMT8, MPSA_MODE_DIAG>(a, splits, st);
}

template <int D, int PVT>
int launch_fmt(const AttnArgs& a, int splits, hipStream_t st) {
    if (a.mode == MPSA_MODE_MXFP4) return launch_split<D, PVT, MPSA_FMT_E4M3, MPSA_MODE_MXFP4>(a, splits, st);
    return a.fmt8 == MPSA_FMT_E5M2 ? launch_mode<D, PVT, MPSA_FMT_E5M2>(a, splits, st) : launch_mode<D, PVT, MPSA_FMT_E4M3>(a, splits, st);
}

}  // namespace

int attn_short_launch(const AttnArgs& a, int pv_dtype, int splits, hipStream_t st) {
    if (const int shares = splits == 1 ? attn_resident_shares(a) : 0) return attn_resident_launch(a, pv_dtype, shares, st);
    if (a.d == 128) return pv_dtype == MPSA_BF16 ? launch_fmt<128, MPSA_BF16>(a, splits, st) : launch_fmt<128, MPSA_F16>(a, splits, st);
    return pv_dtype == MPSA_BF16 ? launch_fmt<64, MPSA_BF16>(a, splits, st) : launch_fmt<64, MPSA_F16>(a, splits, st);
}
