// Fused attention forward with one 128-query tile a workgroup and the softmax inside the P.V product (gfx950; D = 128, 128x128
// tiles, every mode, masked or not, any lengths, visiting lists).
//
// The math is that of attn_fwd.hip, a step's order that of attn_fwd_pp.hip: the scores of tile t + 1, then the 32 matrix
// instructions of P.V(t) with the exponentials, sums and conversions of tile t + 1 in the gaps between them, against the old
// maximum and looked at afterwards.  That step is bound by the vector and matrix instructions that a SIMD issues, and by the clock
// that the power limit leaves (attn_fwd_pp.hip).  What differs is that a workgroup of four waves and 80 KiB of LDS owns one query
// tile, so that two workgroups share a CU and each may walk key tiles of its own: visiting lists (two query tiles a workgroup
// would walk the union of theirs), and half as large pieces of work where pairs do not fill the chip evenly.  It reads K and V
// twice as often as a pair: 40 heads of 32760 tokens, diag, 11.64 ms (pairs 11.56), 32 of 8192 under the mask 345 us (324).
// Lists, 40 heads of 32760 tokens with 8 % of the tiles in 8 bits, whole call: 13.2 -> 12.0 ms; 8 heads, a third of the tiles left
// out, 1547 -> 1427 us: before, on the general kernel (attn_fwd_kernel.h), whose exponentials and P.V products take turns.
//
// 80 KiB hold two V tiles and two 4-bit K tiles.  A K tile's fragments are in registers a step before its scores, so its
// buffer takes the tile two steps on; the tile that has to be done again is read from memory.  An 8-bit tile takes both K
// buffers: its fragments are read at its scores, and a second barrier says that everybody has them.
// No register is to spare: 241 to 256 without spills.  A spilled register in a long loop costs more than its reload: the wait for
// it waits for the tiles that are on their way as well (40 heads of 32760 tokens, diag, 12.7 ms with three of them, 11.7 without).
#include "attn_q_raw.h"

namespace {

constexpr int D = 128, TILE = 128;
constexpr int KB = TILE / 32, SST = D / 64, NDB = D / 32;
constexpr int ROW4 = D / 2, ROW8 = D, CPR4 = ROW4 / 16, CPR8 = ROW8 / 16;
constexpr int K4_BYTES = TILE * ROW4, K8_BYTES = TILE * ROW8, V_BYTES = TILE * D * 2;
constexpr int SMEM = 2 * K4_BYTES + 2 * V_BYTES;      // two 4-bit K tiles or one 8-bit one, and two V tiles: half of a CU's LDS
static_assert(K8_BYTES == 2 * K4_BYTES && SMEM == 80 * 1024, "two workgroups share a CU's LDS");

template <int PVT, int FMT8, int MODE, bool QRAW>
__global__ __launch_bounds__(256, 2) void attn_tile_kernel(AttnArgs a) {
    typedef PV<PVT> P;
    constexpr bool ROUTED = MODE == MPSA_MODE_ROUTED, MIXED = MODE == MPSA_MODE_MIXED, DIAG = MODE == MPSA_MODE_DIAG;
    constexpr bool HAS4 = MODE != MPSA_MODE_MXFP8, HAS8 = MODE == MPSA_MODE_MXFP8 || ROUTED || DIAG;
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const int tid = threadIdx.x, lane = tid & 63, h = lane >> 5, r = lane & 31;
    // What only the prologue and the epilogue want of the arguments is read from memory there: kept in scalar registers across
    // the loops it is spilled into vector registers, of which there are none to spare.
    typedef const __attribute__((address_space(4))) AttnArgs* Kept;
    auto kept = [&]() __attribute__((always_inline)) {
        Kept p = (Kept)__builtin_amdgcn_kernarg_segment_ptr();
        asm volatile("" : "+s"(p));
        return p;
    };
    const int wu = __builtin_amdgcn_readfirstlane(tid >> 6);

    // ---- which (batch, kv head, query head, query tile) -- XCD-aware, heavy causal tiles first ----
    const int group = a.Hq / a.Hkv, units = a.B * a.Hkv;
    int unit, rem;
    if (a.causal & ROWS_DEALT) {            // every XCD gets long and short rows
        rem = blockIdx.x / units;
        unit = blockIdx.x - rem * units;
    } else {
        const int total = a.B * a.Hq * a.ntq, per_unit = group * a.ntq;
        int L = blockIdx.x;
        if ((total & 7) == 0) L = (L & 7) * (total >> 3) + (L >> 3);      // XCD x gets one contiguous logical range
        unit = L / per_unit;
        rem = L - unit * per_unit;
    }
    const int rank = rem / group;
    const int b = unit / a.Hkv, kvh = unit - b * a.Hkv, hq = kvh * group + (rem - rank * group);
    int i = rank;
    if (a.causal) {
        // 512 workgroups or fewer, two a CU, are all there at once: the second layer in reverse, a long row beside a short one
        const int heads = a.B * a.Hq, layer = max(1, 256 / heads), end = heads * a.ntq <= 512 ? min(2 * layer, a.ntq) : 0;
        i = a.ntq - 1 - (rank >= layer && rank < end ? layer + end - 1 - rank : rank);
    }
    const int64_t krow0 = (int64_t)unit * a.n_pad;
    const uint8_t *const k4 = a.k4 + krow0 * ROW4, *const k8 = a.k8 + krow0 * ROW8, *const vt = static_cast<const uint8_t*>(a.v) + krow0 * (D * 2);
    const uint8_t *const ks4 = a.ks4 + krow0 * (D / 32), *const ks8 = a.ks8 + krow0 * (D / 32);
    // What a step in the long loops does not use is made from the lane's number where it is used, for the same reason.
    auto lane_now = []() __attribute__((always_inline)) {
        int x;
        asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(x));
        return x;
    };
    auto query_of = [&](int ln) __attribute__((always_inline)) { return i * TILE + 32 * wu + (ln & 31); };

    // ---- the key tiles in four runs: 4-bit, 4-bit with a mask, 8-bit, 8-bit with a mask.  Softmax does not care about the order. ----
    const int64_t list = ((int64_t)b * a.Hq + hq) * a.ntq + i;
    const int32_t* const ord = ROUTED ? a.order + list * a.nt : nullptr;
    const bool tail = a.n < a.n_pad;
    int r4p, r4, r8p, nsteps;
    if constexpr (ROUTED) {                 // clamped: a malformed list cannot take the kernel outside its buffers
        const int32_t* cn = a.counts + list * 4;
        r4p = min(max(cn[0], 0), a.nt);
        r4 = r4p + min(max(cn[1], 0), a.nt - r4p);
        r8p = r4 + min(max(cn[2], 0), a.nt - r4);
        nsteps = r8p + min(max(cn[3], 0), a.nt - r8p);
    } else {
        nsteps = a.causal ? i + 1 : a.nt;
        const int masked = a.causal || tail ? 1 : 0;
        if constexpr (DIAG) {               // the query tile's own key tile comes last
            r4 = r8p = nsteps - 1;
            r4p = r4 - (tail && !a.causal && i != a.nt - 1 ? 1 : 0);
        } else if constexpr (HAS4) {
            r4 = r8p = nsteps;
            r4p = nsteps - masked;
        } else {
            r4p = r4 = 0;
            r8p = nsteps - masked;
        }
    }
    const int nt = a.nt;
    // key tile of step t; past the last one any valid tile
    auto tile_at = [&](int t) __attribute__((always_inline)) {
        if constexpr (ROUTED) return t < nsteps ? min(max(scalar_load(ord + t), 0), nt - 1) : 0;
        else if constexpr (DIAG) return t < r4p ? t + (t >= i ? 1 : 0) : t < r4 ? nt - 1 : i;
        else return min(t, nt - 1);
    };
    // those of steps t .. t + 3, t being the step in progress, in scalar registers
    int j0 = tile_at(0), j1 = tile_at(1), j2 = tile_at(2), j3 = tile_at(3);
    auto shift = [&](int j4) __attribute__((always_inline)) { j0 = j1; j1 = j2; j2 = j3; j3 = j4; };
    // keys from the limit on are dead: those after the query, and those beyond the sequence
    auto limit_of = [&](int j) __attribute__((always_inline)) {
        const int end = j == a.nt - 1 ? a.n - j * TILE : TILE;
        return a.causal && j == i ? min(32 * wu + (lane_now() & 31) + 1, end) : end;
    };

    // ---- staging: every wave its share of each tile ----
    uint8_t* const kbuf = smem;
    uint8_t* const vbuf = smem + 2 * K4_BYTES;
    // the lane's byte offsets into: a V fragment, a wave's piece of a 4-bit K tile (swizzled rows), a 32-key block of such a tile
    // for its fragments of MX blocks 0 and 1
    const uint32_t lane16 = lane * 16;
    const uint32_t koff = (uint32_t)(lane / CPR4 * ROW4 + ((lane % CPR4) ^ ((lane / CPR4 >> 2) & (CPR4 - 1))) * 16);
    const uint32_t kfoff = (uint32_t)(r * ROW4 + ((h ^ ((r >> 2) & (CPR4 - 1))) * 16));
    auto issue_k4 = [&](int t, int j) __attribute__((always_inline)) {
        load16n_to_lds_sv<2>(koff, k4 + (int64_t)j * K4_BYTES + wu * 2048, kbuf + (t & 1) * K4_BYTES + wu * 2048);
    };
    auto issue_k8 = [&](int j) __attribute__((always_inline)) {                  // the one 8-bit tile
        const uint8_t* src = k8 + (int64_t)j * K8_BYTES + wu * 4096;
        const int ln = HAS4 ? lane_now() : lane;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const int row = 8 * c + ln / CPR8, slot = ln % CPR8;
            load16_to_lds_sv((uint32_t)(row * ROW8 + (slot ^ ((row >> 1) & (CPR8 - 1))) * 16), src, kbuf + wu * 4096 + c * 1024);
        }
    };
    auto issue_v = [&](int t, int j) __attribute__((always_inline)) {
        const uint8_t* src = vt + (int64_t)j * V_BYTES + wu * 8192;
        uint8_t* dst = vbuf + (t & 1) * V_BYTES + wu * 8192;
        load16n_to_lds_sv<4>(lane16, src, dst);
        load16n_to_lds_sv<4>(lane16, src + 4096, dst + 4096);
    };
    // K for the steps after t: the 4-bit tile of step t + 3 into the buffer of step t + 1, whose fragments are in registers, and
    // the first 8-bit tile as soon as the last 4-bit one is
    auto issue_k = [&](int t, int j_8, int j_4) __attribute__((always_inline)) {
        if constexpr (HAS4) {
            if (t + 3 < r4) issue_k4(t + 3, j_4);
            if constexpr (HAS8) {
                if (t + 2 == r4 && r4 < nsteps) issue_k8(j_8);
            }
        }
    };
    // step t's V and the K that its scores or its fragment reads want have landed, everybody's; then the next loads go out
    auto turn = [&](int t) __attribute__((always_inline)) {
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_waitcnt(0x0070);               // vmcnt(0), lgkmcnt(0)
        __syncthreads();
        __builtin_amdgcn_sched_barrier(0);
        if (t + 1 < nsteps) issue_v(t + 1, j1);
        issue_k(t, j2, j3);
    };

    // ---- operands in registers ----
    v8i qf[SST];
    int qsc = 0;                                          // Q's scale bytes in bytes 0 and 2
    v4i kf4[KB][SST];
    int ksc[KB];
    auto ask_q = [&](uint4 (&raw)[2][4]) __attribute__((always_inline)) {       // rows beyond the sequence read the last row and become zeros
        const Kept p = kept();
        const int ln = lane_now();
        const int64_t src = min(query_of(ln), p->nq - 1);
        load_query(static_cast<const char*>(p->q_raw) + 2 * ((int64_t)b * p->q_sb + (int64_t)hq * p->q_sh + src * p->q_sn), ln >> 5, raw);
    };
    auto take_q = [&](const uint4 (&raw)[2][4], auto is8_c) __attribute__((always_inline)) {
        constexpr bool IS8 = decltype(is8_c)::value;
        const Kept p = kept();
        uint32_t s4, s8;
        v8i none[SST];
        if constexpr (IS8) quantize_query_careful<PVT, FMT8, false, true>(raw, p->q_pre, p->q_sure != 0, none, s4, qf, s8);
        else               quantize_query_careful<PVT, FMT8, true, false>(raw, p->q_pre, p->q_sure != 0, qf, s4, none, s8);
        qsc = (int)(IS8 ? s8 : s4);
        const int nq = p->nq;
        if (i * TILE + 32 * wu + 31 >= nq) {              // a wave of the ragged last tile: its padding rows are zeros, as the quantizer pads them
            const bool ok = query_of(lane_now()) < nq;
#pragma unroll
            for (int s = 0; s < SST; ++s)
#pragma unroll
                for (int e = 0; e < (IS8 ? 8 : 4); ++e) qf[s][e] = ok ? qf[s][e] : 0;
            qsc = ok ? qsc : 0;
        }
    };
    auto read_q = [&](bool is8) __attribute__((always_inline)) {
        const Kept p = kept();
        const int ln = lane_now(), h = ln >> 5;
        const int64_t q_row = ((int64_t)b * p->Hq + hq) * p->nq_pad + query_of(ln);
        if (is8) {
#pragma unroll
            for (int s = 0; s < SST; ++s) {
                // 8-bit operand: registers 0-3 hold 16 bytes of MX block 2s, registers 4-7 of block 2s+1
                const v4i x0 = *reinterpret_cast<const v4i*>(p->q8 + q_row * D + s * 64 + h * 16);
                const v4i x1 = *reinterpret_cast<const v4i*>(p->q8 + q_row * D + s * 64 + h * 16 + 32);
                qf[s] = (v8i){x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]};
            }
        } else {
#pragma unroll
            for (int s = 0; s < SST; ++s) {
                const v4i x = *reinterpret_cast<const v4i*>(p->q4 + q_row * (D / 2) + (2 * s + h) * 16);
                qf[s] = (v8i){x[0], x[1], x[2], x[3], 0, 0, 0, 0};
            }
        }
        qsc = (int)(*reinterpret_cast<const uint32_t*>((is8 ? p->qs8 : p->qs4) + q_row * (D / 32)) >> (8 * h));
    };
    auto load_kscales = [&](int j, bool is8) __attribute__((always_inline)) {
        const uint8_t* sp = (is8 ? ks8 : ks4) + (int64_t)j * (TILE * D / 32);
        uint32_t at = lane16;                             // not to be kept as a pointer a lane
        asm volatile("" : "+v"(at));
        const uint32_t row = at / 4 & 124, shift = at / 64 & 8;
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) ksc[kb] = (int)(*reinterpret_cast<const uint32_t*>(sp + row + kb * 32 * (D / 32)) >> shift);
    };
    auto kfrag = [&](int t, int kb, int s) __attribute__((always_inline)) {
        kf4[kb][s] = *reinterpret_cast<const v4i*>(kbuf + (t & 1) * K4_BYTES + kb * 32 * ROW4 + (kfoff ^ (32 * s)));
    };
    auto read_kf4 = [&](int t) __attribute__((always_inline)) {
#pragma unroll
        for (int kb = 0; kb < KB; ++kb)
#pragma unroll
            for (int s = 0; s < SST; ++s) kfrag(t, kb, s);
    };

    // ---- per-query state ----
    v16f acc[NDB];
#pragma unroll
    for (int d = 0; d < NDB; ++d)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[d][e] = 0.0f;
    float l_run = 0.0f;
    v16f negm;
#pragma unroll
    for (int e = 0; e < 16; ++e) negm[e] = 0.0f;
    v16f st[KB];
    v4i pk[KB][2];

    auto scores4 = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int kb = 0; kb < KB; ++kb)
#pragma unroll
            for (int s = 0; s < SST; ++s) {
                const v4i x = kf4[kb][s];
                const v8i k = (v8i){x[0], x[1], x[2], x[3], 0, 0, 0, 0};
                if constexpr (MIXED) st[kb] = score_mfma48<FMT8>(k, qf[s], s == 0 ? negm : st[kb], s, ksc[kb], qsc);
                else                 st[kb] = score_mfma4(k, qf[s], s == 0 ? negm : st[kb], s, ksc[kb], qsc);
            }
    };
    auto scores8 = [&](const uint8_t* rows, bool swizzled) __attribute__((always_inline)) {
        const int ln = HAS4 ? lane_now() : lane, h = ln >> 5, r = ln & 31;
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) {
            const int krow = 32 * kb + r, f = swizzled ? (krow >> 1) & (CPR8 - 1) : 0;
#pragma unroll
            for (int s = 0; s < SST; ++s) {
                const v4i x0 = *reinterpret_cast<const v4i*>(rows + krow * ROW8 + (((4 * s + h) ^ f) * 16));
                const v4i x1 = *reinterpret_cast<const v4i*>(rows + krow * ROW8 + (((4 * s + h + 2) ^ f) * 16));
                const v8i k = (v8i){x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]};
                st[kb] = score_mfma8<FMT8>(k, qf[s], s == 0 ? negm : st[kb], s, ksc[kb], qsc);
            }
        }
    };
    // everybody has the 8-bit tile's fragments: the next one may come
    auto hand_over8 = [&](bool more, int j) __attribute__((always_inline)) {
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_waitcnt(0xC07F);               // lgkmcnt(0)
        __syncthreads();
        __builtin_amdgcn_sched_barrier(0);
        if (more) issue_k8(j);
    };
    auto rebase = [&](float delta, float alpha) __attribute__((always_inline)) {
#pragma unroll
        for (int e = 0; e < 16; ++e) negm[e] -= delta;
#pragma unroll
        for (int kb = 0; kb < KB; ++kb)
#pragma unroll
            for (int e = 0; e < 16; ++e) st[kb][e] -= delta;
        l_run *= alpha;
#pragma unroll
        for (int d = 0; d < NDB; ++d)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[d][e] *= alpha;
    };
    auto row_max = [&]() __attribute__((always_inline)) {
        float mx = st[0][0];
#pragma unroll
        for (int kb = 0; kb < KB; ++kb)
#pragma unroll
            for (int e = 0; e < 16; ++e) mx = __builtin_fmaxf(mx, st[kb][e]);
        return max_lane_pair(mx);
    };
    // P = exp2(S - m), rounded to 16 bits for P.V; the row sum adds the float32 values, as the reference does
    // (ours/mxfp_attn_kernel.py:324-327)
    auto exponentials = [&]() __attribute__((always_inline)) {
        float ps0 = 0.0f, ps1 = 0.0f;
#pragma unroll
        for (int g = 0; g < 2 * KB; ++g)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float p0 = __builtin_amdgcn_exp2f(st[g >> 1][8 * (g & 1) + 2 * j]), p1 = __builtin_amdgcn_exp2f(st[g >> 1][8 * (g & 1) + 2 * j + 1]);
                pk[g >> 1][g & 1][j] = __builtin_bit_cast(int, P::pack(p0, p1));
                ps0 += p0;
                ps1 += p1;
            }
        return ps0 + ps1;
    };
    auto softmax = [&](bool first, int limit) __attribute__((always_inline)) {
        if (__any(limit < TILE)) {
            int past = limit - 4 * (lane_now() >> 5);
#pragma unroll
            for (int kb = 0; kb < KB; ++kb)
#pragma unroll
                for (int e = 0; e < 16; e += 2) {
                    // Two comparisons, then their two selections: left alone the compiler makes all 64 masks first, more than there
                    // are scalar registers, and four at a time spill one of the diag mode's.  The statements hold no instruction, so the
                    // waits between matrix instructions, comparisons and selections are the compiler's.
                    const int key = 32 * kb + 8 * (e >> 2) + (e & 3);
                    asm volatile("" : "+v"(past));
                    uint64_t live0 = __builtin_amdgcn_ballot_w64(key < past), live1 = __builtin_amdgcn_ballot_w64(key + 1 < past);
                    asm volatile("" : "+s"(live0), "+s"(live1));
                    float x0 = __builtin_amdgcn_inverse_ballot_w64(live0) ? st[kb][e] : -__builtin_inff();
                    float x1 = __builtin_amdgcn_inverse_ballot_w64(live1) ? st[kb][e + 1] : -__builtin_inff();
                    asm volatile("" : "+v"(x0), "+v"(x1));
                    st[kb][e] = x0;
                    st[kb][e + 1] = x1;
                }
        }
        const float mx = row_max();
        if (first || __any(mx > P::REBASE)) {
            const float delta = first ? mx : __builtin_fmaxf(mx, 0.0f);
            rebase(delta, first ? 1.0f : __builtin_amdgcn_exp2f(-delta));
        }
        l_run += exponentials();
    };

    // P.V(t); OVERLAP: with the exponentials of the coming tile, whose scores are in st, in the gaps
    auto pv = [&](int t, auto overlap_c, auto kfrag_c) __attribute__((always_inline)) {
        constexpr int NV = KB * 2 * NDB;       // matrix instructions
        constexpr bool OVERLAP = decltype(overlap_c)::value, KFRAG = decltype(kfrag_c)::value;
        constexpr int PRE = 8;
        const uint8_t* vl = vbuf + (t & 1) * V_BYTES + lane16;
        typename P::vec vf[PRE];
#pragma unroll
        for (int x = 0; x < PRE; ++x) vf[x] = *reinterpret_cast<const typename P::vec*>(vl + x * 1024);
        float ps0 = 0.0f, ps1 = 0.0f;
        auto do_exp = [&](int e) __attribute__((always_inline)) {
            const int g = e >> 2, j = e & 3, kb = g >> 1, c = g & 1;
            st[kb][8 * c + 2 * j] = __builtin_amdgcn_exp2f(st[kb][8 * c + 2 * j]);
            st[kb][8 * c + 2 * j + 1] = __builtin_amdgcn_exp2f(st[kb][8 * c + 2 * j + 1]);
        };
        auto do_add = [&](int e) __attribute__((always_inline)) {
            const int g = e >> 2, j = e & 3, kb = g >> 1, c = g & 1;
            ps0 += st[kb][8 * c + 2 * j];
            ps1 += st[kb][8 * c + 2 * j + 1];
        };
        auto do_cvt = [&](int e) __attribute__((always_inline)) {
            const int g = e >> 2, j = e & 3, kb = g >> 1, c = g & 1;
            int word = __builtin_bit_cast(int, P::pack(st[kb][8 * c + 2 * j], st[kb][8 * c + 2 * j + 1]));
            // pin the conversion here, between the matrix instructions: the redo path overwrites pk, so the compiler
            // would otherwise sink all 32 conversions behind the check, where nothing overlaps them
            asm volatile("" : "+v"(word));
            pk[kb][c][j] = word;
        };
#pragma unroll
        for (int idx = 0; idx < NV; ++idx) {
            const int d = idx % NDB, kc = idx / NDB;
            const typename P::vec cur = vf[idx % PRE];
            if (idx + PRE < NV) vf[idx % PRE] = *reinterpret_cast<const typename P::vec*>(vl + (idx + PRE) * 1024);
            acc[d] = P::mfma(cur, __builtin_bit_cast(typename P::vec, pk[kc >> 1][kc & 1]), acc[d]);
            if constexpr (OVERLAP) {
                do_exp(idx);
                if (idx >= 1) do_add(idx - 1);
                if (idx >= NDB) do_cvt(idx - NDB);
                if (KFRAG && kc >= KB && d < SST) kfrag(t + 2, kc - KB, d);      // K fragments of step t + 2
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x400, 2, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, 3, 0);
            }
        }
        if constexpr (OVERLAP) {
            do_add(NV - 1);
#pragma unroll
            for (int e = NV - NDB; e < NV; ++e) do_cvt(e);
            asm volatile("" : "+v"(ps0), "+v"(ps1));      // the sums stay here, too
        }
        return ps0 + ps1;
    };
    // The exponentials were taken without looking for the tile's maximum first; where the row sum shows a score far above the
    // running maximum, the tile (j_now) is done again, from its K rows in memory.
    auto settle = [&](int t, float tot, int j_now, int j_next, auto is8_c) __attribute__((always_inline)) {
        constexpr bool IS8 = decltype(is8_c)::value;
        if (__any(!(tot < P::OPTIMISTIC_LIMIT))) {
            load_kscales(j_now, IS8);
            if constexpr (IS8) {
                scores8(k8 + (int64_t)j_now * K8_BYTES, false);
            } else {
                const uint8_t* rows = k4 + (int64_t)j_now * K4_BYTES;
                const int ln = lane_now(), at = (ln & 31) * ROW4 + (ln >> 5) * 16;
#pragma unroll
                for (int kb = 0; kb < KB; ++kb)
#pragma unroll
                    for (int s = 0; s < SST; ++s) kf4[kb][s] = *reinterpret_cast<const v4i*>(rows + (uint32_t)at + kb * 32 * ROW4 + s * 32);
                scores4();
            }
            const float delta = __builtin_fmaxf(row_max(), 0.0f);
            rebase(delta, __builtin_amdgcn_exp2f(-delta));
            tot = exponentials();
            load_kscales(j_next, IS8);                    // back to the operands of the next step
            if constexpr (!IS8) read_kf4(t + 2);
        }
        l_run += tot;
    };
    typedef std::true_type Yes;
    typedef std::false_type No;

    if (!ROUTED || nsteps > 0) {
        // ---- prologue: V(0), K(0), K(1) on their way; Q into registers; step 0's scores and softmax ----
        const bool first8 = HAS8 && (!HAS4 || r4 == 0);
        uint4 raw[SST][4];
        if constexpr (QRAW) {
            ask_q(raw);
            __builtin_amdgcn_sched_barrier(0);
        }
        if (first8) {
            if constexpr (HAS8) issue_k8(j0);
        } else {
            issue_k4(0, j0);
            if (r4 > 1) issue_k4(1, j1);
        }
        issue_v(0, j0);
        load_kscales(j0, first8);
        if constexpr (QRAW) {
            if constexpr (MIXED || !HAS4) {
                take_q(raw, Yes{});
            } else {
                if (first8) take_q(raw, Yes{});
                else        take_q(raw, No{});
            }
        } else {
            read_q(first8 || MIXED);
        }
        __builtin_amdgcn_s_waitcnt(0x0F70);
        __syncthreads();
        if (first8) {
            if constexpr (HAS8) {
                scores8(kbuf, true);
                hand_over8(nsteps > 1, j1);
            }
        } else {
            read_kf4(0);
            scores4();
            __builtin_amdgcn_sched_barrier(0);
            __builtin_amdgcn_s_waitcnt(0xC07F);
            __syncthreads();
            __builtin_amdgcn_sched_barrier(0);
            issue_k(-1, j1, j2);
        }
        softmax(true, limit_of(j0));
        if (HAS4 && r4 > 1) {
            load_kscales(j1, false);
            read_kf4(1);
        } else if (HAS8 && HAS4 == false) {
            load_kscales(j1, true);
        }

        // ---- step t: P.V of its tile, scores and softmax of the next one's ----
        int t = 0;
        if constexpr (HAS4) {
            for (; t + 1 < r4p; ++t) {
                turn(t);
                scores4();
                const int j4 = tile_at(t + 4);
                load_kscales(j2, false);
                const float tot = pv(t, Yes{}, Yes{});
                settle(t, tot, j1, j2, No{});
                shift(j4);
            }
            for (; t + 1 < r4; ++t) {
                turn(t);
                pv(t, No{}, No{});
                scores4();
                softmax(false, limit_of(j1));
                const int j4 = tile_at(t + 4);
                load_kscales(j2, false);
                read_kf4(t + 2);
                shift(j4);
            }
        }
        if constexpr (HAS8) {
            if constexpr (DIAG) {
                if (t + 1 < nsteps) {                      // the own tile, with Q in 8 bits, which arrives during P.V
                    turn(t);
                    if constexpr (QRAW) ask_q(raw);
                    else                read_q(true);
                    load_kscales(j1, true);
                    __builtin_amdgcn_sched_barrier(0);
                    pv(t, No{}, No{});
                    if constexpr (QRAW) take_q(raw, Yes{});
                    scores8(kbuf, true);
                    softmax(false, limit_of(j1));
                    ++t;
                    shift(j3);
                }
            } else {
                if (HAS4 && t + 1 < nsteps) {
                    if (r4 > 0) read_q(true);              // from 4 to 8 bits
                    load_kscales(j1, true);
                }
                for (; t + 1 < r8p; ++t) {
                    turn(t);
                    scores8(kbuf, true);
                    const int j4 = tile_at(t + 4);
                    hand_over8(t + 2 < nsteps, j2);
                    load_kscales(j2, true);
                    const float tot = pv(t, Yes{}, No{});
                    settle(t, tot, j1, j2, Yes{});
                    shift(j4);
                }
                for (; t + 1 < nsteps; ++t) {
                    turn(t);
                    scores8(kbuf, true);
                    const int j4 = tile_at(t + 4);
                    hand_over8(t + 2 < nsteps, j2);
                    load_kscales(j2, true);
                    pv(t, No{}, No{});
                    softmax(false, limit_of(j1));
                    shift(j4);
                }
            }
        }
        turn(t);
        pv(t, No{}, No{});
        __builtin_amdgcn_s_waitcnt(0x0F70);                // no direct-to-LDS load may outlive the workgroup
    }

    // ---- epilogue: O = acc / l ; register e of lane (h, r): dim 32*db + 8*(e/4) + 4*h + e%4 of query r ----
    const float l_tot = sum_lane_pair(l_run);
    const float inv = (ROUTED && !(l_tot > 0.0f)) ? 0.0f : 1.0f / l_tot;       // lists: a row with every tile skipped gives zeros
    AttnArgs out;
    {
        const Kept p = kept();
        out.o = p->o; out.o_sb = p->o_sb; out.o_sh = p->o_sh; out.o_sn = p->o_sn; out.nq = p->nq; out.o_dtype = p->o_dtype;
    }
    const int ln = lane_now();
    store_output<2 * NDB>(out, b, hq, query_of(ln), 0, ln >> 5, [&](int x) __attribute__((always_inline)) {
        const v16f& v = acc[x >> 2];
        const int e = 4 * (x & 3);
        return (v4f){v[e], v[e + 1], v[e + 2], v[e + 3]};
    }, inv);
}

template <int PVT, int FMT8, int MODE, bool QRAW>
struct TileLds {
    static inline const bool registered = mpsa_register_lds_kernel(reinterpret_cast<const void*>(attn_tile_kernel<PVT, FMT8, MODE, QRAW>), SMEM);
};

template <int PVT, int FMT8, int MODE, bool QRAW>
int launch_tile(const AttnArgs& a, hipStream_t st) {
    if (!TileLds<PVT, FMT8, MODE, QRAW>::registered) return mpsa_fail(MPSA_ELAUNCH, "attn: kernel not registered");
    const int rc = mpsa_ensure_init();
    if (rc != MPSA_OK) return rc;
    hipLaunchKernelGGL((attn_tile_kernel<PVT, FMT8, MODE, QRAW>), dim3((unsigned)(a.B * a.Hq * a.ntq)), dim3(256), SMEM, st, a);
    MPSA_CHECK_LAUNCH("attn (tile)");
    return MPSA_OK;
}

template <int PVT, int FMT8>
int launch_mode(const AttnArgs& a, hipStream_t st) {
    const bool raw = a.q_raw != nullptr;
    if (a.mode == MPSA_MODE_ROUTED) return launch_tile<PVT, FMT8, MPSA_MODE_ROUTED, false>(a, st);
    if (a.mode == MPSA_MODE_MIXED) return raw ? launch_tile<PVT, FMT8, MPSA_MODE_MIXED, true>(a, st) : launch_tile<PVT, FMT8, MPSA_MODE_MIXED, false>(a, st);
    if (a.mode == MPSA_MODE_MXFP8) return raw ? launch_tile<PVT, FMT8, MPSA_MODE_MXFP8, true>(a, st) : launch_tile<PVT, FMT8, MPSA_MODE_MXFP8, false>(a, st);
    return raw ? launch_tile<PVT, FMT8, MPSA_MODE_DIAG, true>(a, st) : launch_tile<PVT, FMT8, MPSA_MODE_DIAG, false>(a, st);
}

template <int PVT>
int launch_fmt(const AttnArgs& a, hipStream_t st) {
    if (a.mode == MPSA_MODE_MXFP4) return a.q_raw ? launch_tile<PVT, MPSA_FMT_E4M3, MPSA_MODE_MXFP4, true>(a, st) : launch_tile<PVT, MPSA_FMT_E4M3, MPSA_MODE_MXFP4, false>(a, st);
    return a.fmt8 == MPSA_FMT_E5M2 ? launch_mode<PVT, MPSA_FMT_E5M2>(a, st) : launch_mode<PVT, MPSA_FMT_E4M3>(a, st);
}

}  // namespace

int attn_tile_launch(const AttnArgs& a, int pv_dtype, hipStream_t st) {
    return pv_dtype == MPSA_BF16 ? launch_fmt<MPSA_BF16>(a, st) : launch_fmt<MPSA_F16>(a, st);
}
