// Block-scaled NT matmul on the CDNA4 scaled matrix cores (gfx950).
//
//   C[m][n] = sum over 32-wide K blocks kb of  2^(sa[m][kb]-127) * 2^(sb[n][kb]-127) * sum_{k in kb} a[m][k] * b[n][k]
//
// the computation of the reference's block_scaled_matmul_kernel (ours/block_scaled_matmul.py:154-267)
// whose torch statement is ours/block_scaled_matmul.py:382-392.  Operands arrive as the quantizer
// leaves them: row-major packed codes and row-major E8M0 bytes (one per 32 elements of K).
//
// Mapping.  A workgroup of four waves owns a 256x256 tile of C; each wave owns 128x128 as a 4x4 grid of
// v_mfma_scale_f32_32x32x64_f8f6f4 accumulators (256 accumulator registers).  For that instruction
// lane (h = lane/32, r = lane%32) supplies 32 K elements of row r of its operand and the E8M0 byte of MX
// block h of the 64-element step.  With 4-bit elements the lane's four registers are exactly block h;
// with 8-bit elements registers 0-3 of the two lane halves together are block 0 and registers 4-7 block 1
// (each half holds 16 bytes of either block).  Either way fragments are plain 16-byte pieces of the
// row-major HBM layout.  K advances 64 bytes of codes per row per stage (128 E2M1 or 64 8-bit elements).
//
// Staging.  Codes go HBM/L2 -> LDS with direct-to-LDS loads (no registers, no LDS-write instructions) into a
// ring of four stages.  The vector memory path moves cache lines: a wave instruction that takes 64 bytes from each
// of 16 rows uses half of every 128-byte line it touches and runs at half the rate of one that takes 128 bytes
// from each of 8 rows (measured L2 -> LDS: 17 against 31 TB/s chip-wide).  So the ring is refilled two stages -- one "unit"
// of 128 bytes per row -- at a time: the unit's LDS image has a 128-byte row pitch, one workgroup barrier per unit, one unit in
// flight while the other is multiplied.
// With an odd number of stages (ODD: 4-bit codes, K % 256 == 128) every other row starts in the middle of a line, and whole units
// gain less.  With row-major scales such runs end in half a unit (HALF; they take the EDGE form, whose loads have their rows apart
// from the place in a row); with packed ones they keep a stage-by-stage ring (RING), three stages in flight while one is
// multiplied: 4096 x 4096 x 4224 47.5 us, with units 50.3, 256 x 256 x 4224 27.3 and 29.4.
// The 16-byte pieces of a row are XOR-swizzled with the row index so that the 128-bit operand reads of 16 consecutive rows hit
// 16 distinct 4-bank groups, and wave tiles of 128x128 keep LDS reads at 8 operand fragments per 16 matrix instructions.
//
// Scale bytes.  A row's scale bytes for one stage are 4 (or 2) bytes in a line of their own, so fetching them
// stage by stage costs the vector memory path one cache-line access per row per stage - as many accesses as
// the codes themselves.  The kernel instead fetches 16 scale bytes per row at a
// time (a "group" of 4 stages of 4-bit codes, 8 stages of 8-bit codes) into a double-buffered LDS area, one
// group ahead: 16 bytes a lane when K is a multiple of 512, else (WORDS) a word a lane, four lanes a row.
// The step from one 4-byte load per row per stage, which K % 512 != 0 had: 3396 x 15872 x 9856, 8-bit x 4-bit, 579 -> 432 us;
// 1000 x 14336 x 4224 65.6 -> 50.5; 4096 x 4096 x 4224, 8-bit, 74.7 -> 60.3; 4096 x 4096 x 4352, 4-bit, 47.3 -> 40.7.
// With the scales in the reference's packed form [rows/128, K/128, 32, 4, 4] (ours/mxfp_attn_kernel.py:56-57) the
// scale bytes of 128 rows x 128 elements of K are one contiguous 512-byte chunk: a stage's scales are four chunks,
// one 32-lane load per wave, and a lane reads its scale words for all four row blocks with one 128-bit LDS read.
//
// Ragged edges.  EDGE runs take any M and N: rows past the matrix are fetched from its last row (a lane's row offset is
// capped with one comparison per load) and not stored.  Their own instantiations, so that whole tiles pay nothing; 1000 x
// 14336 x 4096 and 1024 rows of it take the same, 40.2 and 39.7 us 4-bit, 52.7 and 52.4 8-bit x 4-bit, 58.2 and 59.4 8-bit, a kernel
// after the other and weights from memory (the general kernel: 102, 106 the first two).
#pragma once
#include "gemm_mx_args.h"

namespace {

constexpr int BM = 256, BN = 256;       // workgroup tile
constexpr int ROWB = 64;                // code bytes per row per stage
constexpr int NSTAGE = 4;               // LDS ring depth: two units of two stages
constexpr int OP_BYTES = BM * ROWB;     // one operand's codes per stage (16 KiB)
constexpr int SC_BYTES = BM * 4;        // packed scales: one operand's scale bytes per stage (4 per row)
constexpr int SCG_BYTES = BM * 16;      // row-major scales: one operand's scale bytes per group (16 per row)
constexpr int CODE_LOADS = 2 * (OP_BYTES / 1024 / 4);   // direct-to-LDS code instructions per wave per stage (8)

template <bool PK> constexpr int stage_bytes() { return PK ? 2 * OP_BYTES + 2 * SC_BYTES : 2 * OP_BYTES; }
template <bool PK> constexpr int smem_bytes() { return NSTAGE * stage_bytes<PK>() + (PK ? 0 : 4 * SCG_BYTES); }

// s_waitcnt immediate: vmcnt(vm), lgkmcnt(0), expcnt untouched
constexpr int wait_imm(int vm) { return 0x0070 | (vm & 15) | ((vm >> 4) << 14); }

// Direct-to-LDS load written as inline assembly: lane L's BYTES bytes at wave_base + lane_off land at
// lds_wave_base + L*BYTES (M0 carries the wave-uniform LDS base; the global address is a scalar base plus a
// 32-bit lane offset, so advancing along K costs scalar additions only).  The compiler's own builtin for this instruction makes it wait for
// every outstanding load (vmcnt(0)) before the next barrier or LDS read, which would drain the ring each stage;
// as assembly the loads are invisible to that bookkeeping and the kernel's explicit partial waits stand.
template <int BYTES>
__device__ __forceinline__ void load_to_lds(uint32_t lane_off, const uint8_t* wave_base, uint8_t* lds_wave_base) {
    // address = wave-uniform base (scalar registers) + the lane's unsigned 32-bit byte offset
    // the low 32 bits of a generic pointer into LDS are the LDS byte address (a cast to the LDS address space
    // would add a null check per load)
    const uint32_t base = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)lds_wave_base);
    const uint64_t gb = (uint64_t)(uintptr_t)wave_base;
    if constexpr (BYTES == 16)
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(base), "v"(lane_off), "s"(gb) : "memory", "m0");
    else
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" ::"s"(base), "v"(lane_off), "s"(gb) : "memory", "m0");
}

// FMT: element format of A (and of B, unless FMTB says otherwise).  FMTB == E2M1 under an 8-bit FMT is the reference's
// "mixed" type (ours/block_scaled_matmul.py:318-324): everything follows the 8-bit geometry -- a stage is 64 elements
// of K, a unit 128 -- except B's codes, which are half as wide: 32 bytes per row and stage, a unit's image 64-byte rows.
template <int FMT, int FMTB, typename OutT, bool WORDS, bool PK, bool EDGE, bool ODD>
__global__ __launch_bounds__(256, 1) void gemm_mx_kernel(GemmArgs g) {
    static_assert(!WORDS || !PK, "words: row-major scales whose rows do not lie on 16 bytes");
    static_assert(!ODD || FMT == MPSA_FMT_E2M1, "an odd number of stages: 4-bit codes, K % 256 == 128");
    constexpr bool RING = ODD && PK, HALF = ODD && !PK;
    static_assert(!HALF || (WORDS && EDGE), "half a unit at the end");
    static_assert(NSTAGE == 4, "the ring is two units of two stages");
    constexpr bool FP4 = (FMT == MPSA_FMT_E2M1);
    constexpr bool B4 = !FP4 && (FMTB == MPSA_FMT_E2M1);       // 8-bit A against 4-bit B
    static_assert(FMT == FMTB || B4, "the operands share a format, or A is 8-bit and B is E2M1");
    constexpr int STAGE_BYTES = stage_bytes<PK>();
    constexpr int GROUP = FP4 ? 4 : 8;                 // stages covered by 16 scale bytes of a row
    const int row_bytes = FP4 ? g.K / 2 : g.K;         // code bytes per matrix row (of A)
    const int row_bytes_b = B4 ? g.K / 2 : row_bytes;  // and of B
    const int srow_bytes = g.K / 32;
    const int KT = row_bytes / ROWB;

    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    uint8_t* const scg = smem + NSTAGE * STAGE_BYTES;  // row-major scales: [group parity][operand][row][16]

    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);   // the wave index, known to be uniform
    const int wm = wave >> 1, wn = wave & 1;
    const int h = lane >> 5, r = lane & 31;

    // XCD-aware tile order.  Consecutive workgroup ids go to different XCDs (8 of them, each with its own L2) and
    // an XCD starts its workgroups in id order.  Give XCD x one block of a 2 x 4 split of the tile grid and walk
    // that block in panels four tile rows high, column by column: the workgroups running together on an XCD
    // then cover a few tile rows by a few tile columns and share both operands' K-slices in that L2.
    const int tiles_m = EDGE ? (g.M + BM - 1) / BM : g.M / BM, tiles_n = EDGE ? (g.N + BN - 1) / BN : g.N / BN;
    int tm, tn;
    if (tiles_m % 2 == 0 && tiles_n % 4 == 0) {
        const int x = blockIdx.x & 7, j = blockIdx.x >> 3;
        const int rm = tiles_m / 2, rn = tiles_n / 4;
        const int ph = rm % 4 == 0 ? 4 : (rm % 2 == 0 ? 2 : 1);
        const int panel = j / (ph * rn), jj = j % (ph * rn);
        tm = (x >> 2) * rm + panel * ph + jj % ph;
        tn = (x & 3) * rn + jj / ph;
    } else {
        tm = blockIdx.x / tiles_n;
        tn = blockIdx.x % tiles_n;
    }
    const int m0 = tm * BM;
    const int n0 = tn * BN;

    // ---- direct-to-LDS staging ----
    // batched runs (blockIdx.y): operands of this batch entry; grouped heads share a B operand
    const int bz = blockIdx.y;
    const int bb = bz / g.heads_a, ha = bz - bb * g.heads_a;
    const int64_t zb = (int64_t)bb * g.heads_b + ha / (g.heads_a / g.heads_b);
    g.a += (int64_t)bz * g.M * row_bytes;
    g.sa += (int64_t)bz * g.M * srow_bytes;
    g.b += zb * g.N * row_bytes_b;
    g.sb += zb * g.N * srow_bytes;
    // lane offsets inside a tile's operand (the same for A and B) and inside its scale rows; tile bases are scalar
    // a unit = two consecutive stages = 128 code bytes per row, fetched as whole cache lines: an instruction
    // of a wave covers 8 rows x 128 B (half-used lines move at half the rate through the vector memory path).  The
    // unit's LDS image has a 128-byte row pitch; row's 16-byte piece c sits at slot c ^ ((row >> 1) & 7), so that
    // 16 consecutive rows' reads of one piece fall into 16 distinct 4-bank groups.  Instruction x of the unit
    // (wave * 8 + c2, c2 = 0..7) covers rows 8x .. 8x+7: only the parity of c2 enters the lane's swizzle.
    // EDGE: the tile's last row inside the matrix, of either operand, and its byte offset
    const int last_a = EDGE ? min(BM - 1, g.M - 1 - m0) : BM - 1, last_b = EDGE ? min(BN - 1, g.N - 1 - n0) : BN - 1;
    const uint32_t cap_a = (uint32_t)last_a * (uint32_t)row_bytes, cap_b = (uint32_t)last_b * (uint32_t)row_bytes_b;
    uint32_t lo[2];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
        const int cb = (lane & 7) ^ (4 * e + ((lane >> 4) & 3));
        lo[e] = (EDGE ? 0u : (uint32_t)(lane >> 3) * (uint32_t)row_bytes) + cb * 16;
    }
    // a unit of a mixed product's B, and a stage of the stage-by-stage ring, is 64 bytes per row: four instructions per wave, 16
    // rows each, row's piece c at slot c ^ ((row >> 2) & 3)
    uint32_t lo64a[4] = {0, 0, 0, 0}, lo64b[4] = {0, 0, 0, 0};
    if constexpr (B4 || RING) {
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const int p = (wave * 4 + c) * 64 + lane;
            const int row = p >> 2, slot = p & 3;
            const uint32_t piece = (uint32_t)(slot ^ ((row >> 2) & 3)) * 16u;
            lo64a[c] = (uint32_t)min(row, last_a) * (uint32_t)row_bytes + piece;
            lo64b[c] = EDGE || B4 ? (uint32_t)min(row, last_b) * (uint32_t)row_bytes_b + piece : lo64a[c];
        }
    }
    const uint32_t los_a = (uint32_t)min(wave * 64 + lane, last_a) * (uint32_t)srow_bytes;
    const uint32_t los_b = EDGE ? (uint32_t)min(wave * 64 + lane, last_b) * (uint32_t)srow_bytes : los_a;
    const uint32_t lrow = (uint32_t)(lane >> 3) * (uint32_t)row_bytes;      // EDGE: this lane's row inside a load's eight
    const uint8_t* const a_base = g.a + (int64_t)m0 * row_bytes;
    const uint8_t* const b_base = g.b + (int64_t)n0 * row_bytes_b;
    const uint8_t* const sa_base = g.sa + (int64_t)m0 * srow_bytes;
    const uint8_t* const sb_base = g.sb + (int64_t)n0 * srow_bytes;
    // packed scales (the reference's [rows/128, K/128, 32, 4, 4] form, ours/mxfp_attn_kernel.py:56-57): the scale bytes
    // of 128 rows x 128 elements of K are one 512-byte chunk, byte (row%32)*16 + (row/32)*4 + k.  A stage needs two
    // chunks per operand: waves 0, 1 bring A's, waves 2, 3 B's, each with its first 32 lanes.
    const int kchunks = g.K / 128;
    const uint32_t pko = (uint32_t)((lane & 31) * 16);
    // (EDGE: the second chunk of the last tile may not exist: the first one again)
    const int chunk = EDGE ? min(wave & 1, (wave < 2 ? last_a : last_b) >> 7) : wave & 1;
    const uint8_t* const s_pk = (wave < 2 ? g.sa + (int64_t)(m0 / 128) * kchunks * 512 : g.sb + (int64_t)(n0 / 128) * kchunks * 512) +
                                (int64_t)chunk * kchunks * 512;
    // Part `part` of unit u's loads: four code instructions, two per operand (mixed formats: two and one), and the packed scale
    // bytes with the last.  In four parts so that they can be spread between the matrix instructions of a step.
    // Unit u lives in ring half u & 1: [A codes 32 KiB][B codes 32 KiB][packed: scale bytes of its two stages]
    auto unit_base = [&](int u) __attribute__((always_inline)) { return smem + (u & 1) * 2 * STAGE_BYTES; };
    auto issue_unit_part = [&](int u, int part) __attribute__((always_inline)) {
        const int NU = HALF ? (KT + 1) / 2 : KT / 2;
        const int uc = u < NU ? u : NU - 1;               // past the end: re-load the last unit
        // HALF: the last unit has its first 64 bytes a row, and twice
        const uint32_t inside = HALF && uc == NU - 1 ? ~64u : ~0u;
        uint8_t* ub = unit_base(u);
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const int c2 = part * 2 + q, x = wave * 8 + c2;
            if constexpr (EDGE) {
                const uint32_t row = (uint32_t)(x * 8) * (uint32_t)row_bytes + lrow;
                load_to_lds<16>(min(row, cap_a) + (HALF ? lo[q] & inside : lo[q]), a_base + (int64_t)uc * (2 * ROWB), ub + x * 1024);
                if constexpr (!B4) load_to_lds<16>(min(row, cap_b) + (HALF ? lo[q] & inside : lo[q]), b_base + (int64_t)uc * (2 * ROWB), ub + 2 * OP_BYTES + x * 1024);
            } else {
                const int64_t go = (int64_t)uc * (2 * ROWB) + (int64_t)x * 8 * row_bytes;
                load_to_lds<16>(lo[q], a_base + go, ub + x * 1024);
                if constexpr (!B4) load_to_lds<16>(lo[q], b_base + go, ub + 2 * OP_BYTES + x * 1024);
            }
        }
        if constexpr (B4) load_to_lds<16>(lo64b[part], b_base + (int64_t)uc * ROWB, ub + 2 * OP_BYTES + (wave * 4 + part) * 1024);
        if (part != 3) return;
        uint8_t* sc = ub + 4 * OP_BYTES;
        if constexpr (PK) {
            // 4-bit codes: the unit's two stages are two consecutive 512-byte chunks -- one 64-lane load; 8-bit
            // codes: one chunk covers the unit, the odd stage takes its scale words from the even stage's registers
            if constexpr (FP4) load_to_lds<16>((uint32_t)lane * 16u, s_pk + (int64_t)uc * 1024, sc + wave * 1024);
            else if (lane < 32) load_to_lds<16>(pko, s_pk + (int64_t)uc * 512, sc + wave * 1024);
        }
    };
    // the same for stage kt of the stage-by-stage ring: one instruction per operand and part
    auto issue_stage_part = [&](int kt, int part) __attribute__((always_inline)) {
        const int kc = kt < KT ? kt : KT - 1;             // past the end: re-load the last stage (keeps the count uniform)
        uint8_t* st = smem + (kt % NSTAGE) * STAGE_BYTES;
        load_to_lds<16>(lo64a[part], a_base + (int64_t)kc * ROWB, st + (wave * 4 + part) * 1024);
        load_to_lds<16>(lo64b[part], b_base + (int64_t)kc * ROWB, st + OP_BYTES + (wave * 4 + part) * 1024);
        if (part == 3 && lane < 32) load_to_lds<16>(pko, s_pk + (int64_t)kc * 512, st + 2 * OP_BYTES + wave * 512);
    };
    auto issue_unit = [&](int u) __attribute__((always_inline)) {
#pragma unroll
        for (int part = 0; part < 4; ++part) issue_unit_part(u, part);
    };
    // row-major scales: the 16 scale bytes per row of group grp (two instructions per wave).  WORDS (K is no multiple of 512: rows of
    // scale bytes start on words, and the last group is cut): a word a lane, four neighbouring lanes a row, 16 rows an
    // instruction; words past the row's end are its last one.
    auto issue_scales = [&](int grp) __attribute__((always_inline)) {
        const int ng = (KT + GROUP - 1) / GROUP;
        const int gc = grp < ng ? grp : ng - 1;
        uint8_t* dst = scg + (grp & 1) * 2 * SCG_BYTES + wave * 1024;
        if constexpr (WORDS) {
            const uint32_t w = (uint32_t)(min(4 * gc + (lane & 3), g.K / 128 - 1) * 4);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int row = wave * 64 + q * 16 + (lane >> 2);
                load_to_lds<4>((uint32_t)min(row, last_a) * (uint32_t)srow_bytes + w, sa_base, dst + q * 256);
                load_to_lds<4>((uint32_t)min(row, last_b) * (uint32_t)srow_bytes + w, sb_base, dst + SCG_BYTES + q * 256);
            }
        } else {
            load_to_lds<16>(los_a, sa_base + gc * 16, dst);
            load_to_lds<16>(los_b, sb_base + gc * 16, dst + SCG_BYTES);
        }
    };

    v16f acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;

    if constexpr (!PK) issue_scales(0);
    if constexpr (RING) {
#pragma unroll
        for (int s = 0; s < NSTAGE; ++s)
#pragma unroll
            for (int part = 0; part < 4; ++part) issue_stage_part(s, part);
    } else {
        issue_unit(0);
        issue_unit(1);
    }

    // LDS offsets of this lane's operand rows (128-byte rows; 64-byte ones in the ring and of a mixed product's B; swizzled pieces)
    int offa[4], offb[4], swz_a[4], swz_b[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int ra_ = wm * 128 + i * 32 + r, rb_ = wn * 128 + i * 32 + r;
        offa[i] = ra_ * (RING ? ROWB : 2 * ROWB); swz_a[i] = RING ? (ra_ >> 2) & 3 : (ra_ >> 1) & 7;
        offb[i] = rb_ * (RING || B4 ? ROWB : 2 * ROWB); swz_b[i] = RING || B4 ? (rb_ >> 2) & 3 : (rb_ >> 1) & 7;
    }

    // One matrix-instruction step's operands: 4 + 4 fragments and their scale bytes.  Two sets alternate: while
    // the 16 instructions of one set run, the LDS reads of the next set are in flight.
    // Scale bytes: the four bytes of a row's aligned scale word cover an even step and the odd step after it
    // (bytes h and 2+h of the lane half h).  The word is read once, with the even step's operands, shifted right by
    // 8h when that step starts, and handed on to the odd step's set, whose instructions select byte 2.
    struct Frag { v8i a[4], b[4]; int sa[4], sb[4]; uint32_t ra[4], rb[4]; };
    // Row-major scales, 4-bit codes: a row's 16 scale bytes of the current group are read from LDS ONCE per group with one
    // 128-bit read per row (16 consecutive rows x 16 bytes are conflict-free; a 32-bit read per step pair at this
    // 16-byte row pitch is a four-way bank conflict, and those conflicts were 38 % of the kernel's LDS cycles).
    // Dword k of a row covers step pair k of the group.  With 8-bit codes the operand sets fill the register file:
    // 32 (or, reading half a group at a time, 16) more registers spill and the kernel gets slower, so that path
    // keeps the 32-bit read per step pair.
    constexpr bool GREAD = !PK && FP4;
    v4i w_a[4], w_b[4];

    // reads operands of step s of stage kt out of the ring: part 0 the B fragments and their scale bytes,
    // part 1 the A fragments and theirs.  grp >= 0 (GREAD): also this part's scale rows of group grp.
    auto read_part = [&](Frag& f, const Frag& even, int kt, int s, int part, bool fresh, int grp) __attribute__((always_inline)) {
        const bool isb = part == 0;
        const int hh = kt & 1;                             // which stage of its unit
        const uint8_t* st = RING ? smem + (kt % NSTAGE) * STAGE_BYTES : unit_base(kt >> 1);
        const uint8_t* lx = isb ? st + (RING ? 1 : 2) * OP_BYTES : st;
        const int c0 = RING ? 0 : 4 * hh;                  // first 16-byte piece of this stage inside the LDS row
        // the row's scale word of this step pair (paths without the per-group read)
        const uint8_t* sc = RING ? st + 2 * OP_BYTES + (isb ? 1024 : 0)
                          : PK ? st + 4 * OP_BYTES + hh * 512 + (isb ? 2048 : 0)
                               : scg + ((kt / GROUP) & 1) * 2 * SCG_BYTES + 4 * (FP4 ? kt % GROUP : (kt % GROUP) >> 1) + (isb ? SCG_BYTES : 0);
        const uint8_t* sg = scg + (grp & 1) * 2 * SCG_BYTES + (isb ? SCG_BYTES : 0);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int row = (isb ? wn : wm) * 128 + i * 32 + r;
            const int off = isb ? offb[i] : offa[i], swz = isb ? swz_b[i] : swz_a[i];
            v8i& fx = isb ? f.b[i] : f.a[i];
            if constexpr (GREAD) {
                if (grp >= 0) (isb ? w_b[i] : w_a[i]) = *reinterpret_cast<const v4i*>(sg + row * 16);
                if (!fresh) {
                    if (isb) f.sb[i] = even.sb[i]; else f.sa[i] = even.sa[i];
                }
            } else if (fresh) {
                if constexpr (PK) {
                    // one conflict-free 128-bit read: the scale words of this lane's row in all four row blocks
                    if (i == 0) {
                        const v4i wsc = *reinterpret_cast<const v4i*>(sc + (isb ? wn : wm) * (RING ? 512 : 1024) + r * 16);
#pragma unroll
                        for (int q = 0; q < 4; ++q) (isb ? f.rb[q] : f.ra[q]) = (uint32_t)wsc[q];
                    }
                } else {
                    (isb ? f.rb[i] : f.ra[i]) = *reinterpret_cast<const uint32_t*>(sc + row * 16);
                }
            } else {
                if (isb) f.sb[i] = even.sb[i]; else f.sa[i] = even.sa[i];
            }
            if constexpr (FP4) {
                const v4i x = *reinterpret_cast<const v4i*>(lx + off + (((c0 + 2 * s + h) ^ swz) * 16));
                fx = (v8i){x[0], x[1], x[2], x[3], 0, 0, 0, 0};
            } else if (B4 && isb) {
                // the 4-bit operand of a mixed product: stage hh of the unit is pieces 2hh, 2hh + 1 of the 64-byte row
                const v4i x = *reinterpret_cast<const v4i*>(lx + off + (((2 * hh + h) ^ swz) * 16));
                fx = (v8i){x[0], x[1], x[2], x[3], 0, 0, 0, 0};
            } else {
                // 8-bit operands: registers 0-3 of both lane halves form MX block 0 (scaled by the byte
                // lane half 0 supplies), registers 4-7 form block 1 (scaled by lane half 1's byte)
                const v4i x0 = *reinterpret_cast<const v4i*>(lx + off + (((c0 + h) ^ swz) * 16));
                const v4i x1 = *reinterpret_cast<const v4i*>(lx + off + (((c0 + h + 2) ^ swz) * 16));
                fx = (v8i){x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]};
            }
        }
    };
    // the four matrix instructions of accumulator row i
    auto multiply_row = [&](const Frag& f, int i, bool odd) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (odd) acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(f.a[i], f.b[j], acc[i][j], FMT, FMTB, 2, f.sa[i], 2, f.sb[j]);
            else     acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(f.a[i], f.b[j], acc[i][j], FMT, FMTB, 0, f.sa[i], 0, f.sb[j]);
        }
    };
    // One step: the 16 matrix instructions on operand set `cur`, in four rows.  Between them go the LDS reads
    // that fill the other set `nxt` with step ns of stage nkt (rows 0 and 1) and, when `refill` is set, the
    // loads of the unit of stage lkt into the buffer of the unit before last (two per operand and row; where a group of scale
    // bytes is due they follow the last), so that the matrix pipe keeps running while they issue.
    // `odd`: cur is the odd step of its pair (its scale words were handed on by the even step's set)
    // row-major scales: `fetch_grp` >= 0: the refill also fetches that group's scale bytes.  GREAD: `kd` = which dword of the
    // group's scale rows an even step uses; `read_grp` >= 0: the operand reads also bring that group's scale rows into
    // registers (the step after the group's last even step, so the registers are free)
    auto step = [&](Frag& cur, Frag& nxt, int nkt, int ns, bool refill, int lkt, bool odd, int kd, int fetch_grp, int read_grp) __attribute__((always_inline)) {
        constexpr int PER = FP4 ? 2 : 3;                   // LDS reads issued behind each matrix instruction
        if (!odd) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if constexpr (GREAD) {
                    cur.sa[i] = (int)((uint32_t)w_a[i][kd] >> (8 * h));
                    cur.sb[i] = (int)((uint32_t)w_b[i][kd] >> (8 * h));
                } else {
                    cur.sa[i] = (int)(cur.ra[i] >> (8 * h));
                    cur.sb[i] = (int)(cur.rb[i] >> (8 * h));
                }
            }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (refill) {
                if constexpr (RING) issue_stage_part(lkt, i);
                else issue_unit_part(lkt >> 1, i);         // lkt: first stage of the unit to fetch
                if constexpr (!PK) {
                    if (i == 3 && fetch_grp >= 0) issue_scales(fetch_grp);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            if (i < 2) read_part(nxt, cur, nkt, ns, i, odd, read_grp);   // the step after an odd one starts a new pair
            multiply_row(cur, i, odd);
            if (i < 2) {
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);      // one matrix instruction
                    __builtin_amdgcn_sched_group_barrier(0x100, PER, 0);    // PER LDS reads
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    // Called once per unit, after its second stage has been read into registers: wait for the loads in flight -- the next unit's,
    // and possibly a scale group's, all of which must have landed before that unit is read -- and meet the other waves; after
    // that this unit's buffer may be refilled.
    // Ring: once per stage, after it has been read: wait for the next stage, everything but the loads of the two issued last.
    auto publish = [&]() __attribute__((always_inline)) {
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_waitcnt(wait_imm(RING ? 2 * (CODE_LOADS + 1) : 0));
        __syncthreads();
        __builtin_amdgcn_sched_barrier(0);
    };

    Frag f0, f1;
    {
        // unit 1 stays in flight (its code loads and, packed, its scale load), in the ring the stages after the first
        constexpr int KEEP = RING ? (NSTAGE - 1) * (CODE_LOADS + 1) : (B4 ? CODE_LOADS + CODE_LOADS / 2 : 2 * CODE_LOADS) + (PK ? 1 : 0);
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_waitcnt(wait_imm(KEEP));
        __syncthreads();
        __builtin_amdgcn_sched_barrier(0);
    }
    read_part(f0, f0, 0, 0, 0, true, GREAD ? 0 : -1);
    read_part(f0, f0, 0, 0, 1, true, GREAD ? 0 : -1);
    if constexpr (GREAD) {
        // a stage is two steps: the second step's operands load under the first step's instructions, and the next stage's first
        // operands under the second step's; barrier and refill after a unit's second stage.  One trip = one scale group.
        for (int grp = 0; grp < KT / GROUP; ++grp) {
#pragma unroll
            for (int u = 0; u < GROUP; ++u) {
                const int kt = grp * GROUP + u;            // written so that the stage's parity is a constant
                step(f0, f1, kt, 1, false, 0, false, u, -1, -1);
                if (u & 1) publish();
                step(f1, f0, kt + 1, 0, (u & 1) != 0, kt + 3, true, 0, u == 1 ? grp + 1 : -1, u == GROUP - 1 ? grp + 1 : -1);
            }
        }
        if (WORDS && (KT & 2)) {                           // the last group is one unit (and HALF: half a one)
            const int kt = KT & ~3;
            step(f0, f1, kt, 1, false, 0, false, 0, -1, -1);
            step(f1, f0, kt + 1, 0, false, 0, true, 0, -1, -1);
            step(f0, f1, kt + 1, 1, false, 0, false, 1, -1, -1);
            if (HALF) publish();
            step(f1, f0, HALF ? kt + 2 : kt, 0, false, 0, true, 0, -1, -1);
        }
        if constexpr (HALF) {
            if (KT & 2) {                                  // its scale words: the third of the group, or the first
#pragma unroll
                for (int i = 0; i < 4; ++i) { w_a[i][0] = w_a[i][2]; w_b[i][0] = w_b[i][2]; }
            }
            step(f0, f1, KT - 1, 1, false, 0, false, 0, -1, -1);
            step(f1, f0, KT - 1, 0, false, 0, true, 0, -1, -1);
        }
    } else if constexpr (RING) {
        for (int kt = 0; kt < KT; ++kt) {
            step(f0, f1, kt, 1, false, 0, false, 0, -1, -1);
            publish();
            step(f1, f0, kt + 1, 0, true, kt + NSTAGE, true, 0, -1, -1);
        }
    } else if constexpr (FP4) {
        for (int u2 = 0; u2 < KT / 2; ++u2) {
            const int kt = 2 * u2;
            step(f0, f1, kt, 1, false, 0, false, 0, -1, -1);
            step(f1, f0, kt + 1, 0, false, 0, true, 0, -1, -1);
            step(f0, f1, kt + 1, 1, false, 0, false, 0, -1, -1);
            publish();
            step(f1, f0, kt + 2, 0, true, kt + 4, true, 0, -1, -1);
        }
    } else {
        // a stage is one step.  The group whose scale bytes the refill of stage kt also fetches:
        auto fetch_at = [&](int kt) { return !PK && kt % GROUP == 1 ? kt / GROUP + 1 : -1; };
        for (int u2 = 0; u2 < KT / 2; ++u2) {
            const int kt = 2 * u2;
            step(f0, f1, kt + 1, 0, false, 0, false, 0, -1, -1);
            publish();
            step(f1, f0, kt + 2, 0, true, kt + 4, true, 0, fetch_at(kt + 1), -1);
        }
    }
    __builtin_amdgcn_s_waitcnt(0x0F70);                // no direct-to-LDS load may outlive the workgroup

    // epilogue: accumulator register e of lane (h, r) is C[8*(e/4) + 4*h + e%4][r] of its 32x32 block
    OutT* c = static_cast<OutT*>(g.c) + (int64_t)bz * g.M * g.ldc;
    if constexpr (EDGE && sizeof(OutT) == 2) {         // whole tiles gain nothing by it: 8192^3 0.98 to 1.014 of the time; in one or two rounds a row less, stored this way, 0.98 to 1.02
        if (rows16_aligned(g)) {
            __syncthreads();                           // the ring is free: everybody has read it, and nothing is on its way into it
#pragma unroll
            for (int i = 0; i < 4; ++i)
                store_rows16<4, OutT, EDGE>(acc[i], smem + wave * rows16_bytes<4>(), c, g.ldc, m0 + wm * 128 + i * 32, n0 + wn * 128, g.M, g.N, lane);
            return;
        }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int col = n0 + wn * 128 + j * 32 + r;
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int row = m0 + wm * 128 + i * 32 + 8 * (e >> 2) + 4 * h + (e & 3);
                if (!EDGE || (row < g.M && col < g.N)) c[(int64_t)row * g.ldc + col] = cvt_out<OutT>(acc[i][j][e]);
            }
        }
}

template <int FMT, int FMTB, typename OutT, bool WORDS, bool PK, bool EDGE, bool ODD>
struct GemmLds {
    static inline const bool registered =
        mpsa_register_lds_kernel(reinterpret_cast<const void*>(gemm_mx_kernel<FMT, FMTB, OutT, WORDS, PK, EDGE, ODD>), smem_bytes<PK>());
};

template <int FMT, int FMTB, typename OutT, bool WORDS, bool PK, bool EDGE, bool ODD = false>
void launch_kernel(const GemmArgs& g, dim3 grid, hipStream_t st) {
    if (!GemmLds<FMT, FMTB, OutT, WORDS, PK, EDGE, ODD>::registered) return;
    hipLaunchKernelGGL((gemm_mx_kernel<FMT, FMTB, OutT, WORDS, PK, EDGE, ODD>), grid, dim3(256), smem_bytes<PK>(), st, g);
}


}  // namespace
