// A query's row of unquantized Q, MX-quantized in registers into the fragments of the score product: with the quantizer's own
// device functions, so that the bits are those mpsa_quantize_mx would have written (ours/quant_mxint8.py:276-351, :164-219 with
// sm_scale*log2(e) folded in, :479-494), but the codes and scales never travel through HBM.  Shared by the tile kernels.
#pragma once
#include "attn_common.h"
#include "quantize_kernel.h"

namespace {

// lane half h owns MX blocks h and 2 + h of its row's four (the 4-bit operand layout)
__device__ __forceinline__ void load_query(const char* row, int h, uint4 (&raw)[2][4]) {
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int c = 0; c < 4; ++c) raw[s][c] = *reinterpret_cast<const uint4*>(row + 2 * (32 * (2 * s + h) + 8 * c));
}

// The 8-bit codes of block 2s + h, w8[0..3] its bytes 0-15 and w8[4..7] 16-31, into the operand's registers: lane half 0 keeps its
// low half in registers 0-3 and takes block 2s + 1's low half from its partner into 4-7; lane half 1 keeps its high half in 4-7 and
// takes block 2s's high half into 0-3: swap (lanes 32-63 of register i) with (lanes 0-31 of register 4 + i).
__device__ __forceinline__ v8i trade_halves(int (&w8)[8]) {
#pragma unroll
    for (int q = 0; q < 4; ++q)
        asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1" : "+v"(w8[q]), "+v"(w8[4 + q]));
    return (v8i){w8[0], w8[1], w8[2], w8[3], w8[4], w8[5], w8[6], w8[7]};
}

// Both precisions from one pass over the lane's blocks: a block's maximum and shared exponent are lane-local and serve both
// formats (the element exponent limits differ: 3 and 7).  The 8-bit operand wants 16 bytes of EVERY block in each lane half
// (registers 0-3: block 2s, 4-7: block 2s + 1), so the two lanes of a query trade halves of their blocks afterwards: one
// v_permlane32_swap per register pair.  sc4 / sc8: the scale bytes of blocks h and 2 + h in bytes 0 and 2.
template <int PVT, int FMT8, bool WANT4, bool WANT8>
__device__ __forceinline__ void quantize_query_careful(const uint4 (&raw)[2][4], float pre, bool sure, v8i (&q4f)[2], uint32_t& sc4, v8i (&q8f)[2], uint32_t& sc8) {
#pragma clang fp contract(off)        // the quantizer's arithmetic, operation by operation
    sc4 = sc8 = 0;
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        float x[4][8];
        float amax = 0.0f;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            unpack8<PVT>(raw[s][c], x[c]);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                x[c][e] = x[c][e] * pre;
                amax = __builtin_fmaxf(amax, __builtin_fabsf(x[c][e]));
            }
        }
        const bool zero = mpsa_f2u(amax) == 0u;
        const int ex = block_exponent(amax);
        const int se = ex - 3, se8 = ex - 7;             // emax of E2M1: ours/quant_mxint8.py:303; of the 8-bit formats: :191
        int w[4];
        int w8[8];
        bool rule[4], odd = false, again = false;        // chunks, and the block, that the conversions may not be right for
        if constexpr (WANT4) {
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                w[c] = (int)e2m1_try8<true>(x[c], se, sure, rule[c]);
                again |= rule[c];
            }
        }
        if constexpr (WANT8) {
            odd = fp8_odd(ex, se8);
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const uint2 y = fp8_convert8<FMT8>(x[c], se8);
                w8[2 * c] = (int)y.x;
                w8[2 * c + 1] = (int)y.y;
                odd |= fp8_past<FMT8>(y);
            }
            again |= odd;
        }
        if (again && !zero) {
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                if (WANT4 && rule[c]) w[c] = (int)e2m1_pack8_rule(x[c], se);
                if (WANT8 && odd) {
                    const uint2 y = fp8_careful8<FMT8, false>(x[c], se8);
                    w8[2 * c] = (int)y.x;
                    w8[2 * c + 1] = (int)y.y;
                }
            }
        }
        if constexpr (WANT4) {
            q4f[s] = (v8i){zero ? 0 : w[0], zero ? 0 : w[1], zero ? 0 : w[2], zero ? 0 : w[3], 0, 0, 0, 0};
            sc4 |= (uint32_t)(zero ? 0 : min(max(se + 127, 0), 254)) << (16 * s);
        }
        if constexpr (WANT8) {
#pragma unroll
            for (int c = 0; c < 8; ++c) w8[c] = zero ? 0 : w8[c];
            q8f[s] = trade_halves(w8);
            // lane half h hands the matrix core the scale byte of block 2s + h: its own
            sc8 |= (uint32_t)(zero ? 0 : min(max(se8 + 127, 0), 254)) << (16 * s);
        }
    }
}

// The same, straight through for rows without rare blocks (quantize_straight, quantize_kernel.h, says which); a wave with one does
// its rows again the careful way, and so do all whose 4-bit codes are the rule's to look at.  For workgroups that own their CU, whose
// prologue hides behind nothing: the paired-tile kernel, 32 heads, causal, diag, 2048 tokens 45.7 -> 45.2 us a call, 8192 335.5 -> 333.5.
// Two workgroups a CU (the tile kernel) do not feel it: 0.99 to 1.02.
template <int PVT, int FMT8, bool WANT4, bool WANT8>
__device__ __forceinline__ void quantize_query(const uint4 (&raw)[2][4], float pre, bool sure, v8i (&q4f)[2], uint32_t& sc4, v8i (&q8f)[2], uint32_t& sc8) {
#pragma clang fp contract(off)
    bool again = WANT4 && !sure;
    if (!again) {
        bool rare = false;
        sc4 = sc8 = 0;
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            float x[4][8];
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                unpack8<PVT>(raw[s][c], x[c]);
#pragma unroll
                for (int e = 0; e < 8; ++e) x[c][e] = x[c][e] * pre;
            }
            float amax = __builtin_fabsf(x[0][0]);
#pragma unroll
            for (int i = 1; i < 32; ++i) amax = __builtin_elementwise_maximum(amax, __builtin_fabsf(x[i >> 3][i & 7]));
            const BlockScale b = block_scale(mpsa_f2u(amax));
            rare |= b.rare;
            if constexpr (WANT4) {
                int w[4];
#pragma unroll
                for (int c = 0; c < 4; ++c) w[c] = (int)e2m1_convert8(x[c], b.se4(), 1.0f);
                q4f[s] = (v8i){b.zero ? 0 : w[0], b.zero ? 0 : w[1], b.zero ? 0 : w[2], b.zero ? 0 : w[3], 0, 0, 0, 0};
                sc4 |= (uint32_t)b.s4() << (16 * s);
            }
            if constexpr (WANT8) {
                int w8[8];
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    const uint2 y = fp8_convert8<FMT8>(x[c], b.se8());
                    w8[2 * c] = b.zero ? 0 : (int)y.x;
                    w8[2 * c + 1] = b.zero ? 0 : (int)y.y;
                }
                q8f[s] = trade_halves(w8);
                sc8 |= (uint32_t)b.s8() << (16 * s);
            }
        }
        again = __ballot(rare) != 0;
    }
    if (again) {
        uint4 y[2][4];
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int c = 0; c < 4; ++c) y[s][c] = only_here(raw[s][c]);
        quantize_query_careful<PVT, FMT8, WANT4, WANT8>(y, pre, sure, q4f, sc4, q8f, sc8);
    }
}

}  // namespace
