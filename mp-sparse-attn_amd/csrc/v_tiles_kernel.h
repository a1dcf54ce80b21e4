// The value-tile repack's per-workgroup body, shared by v_tiles.hip and prepare.hip (layout: top of v_tiles.hip).
#pragma once
#include "mpsa_common.h"


struct VTArgs {
    const unsigned short* v;
    int64_t sb, sh, sn;
    int n, nt;
    int pairs;                 // two neighbouring elements of a row are four aligned bytes
    unsigned short* out;
};

// host side, defined in v_tiles.hip: validates and fills the argument block; *blocks = workgroups per (batch, head)
int mpsa_v_tiles_setup(const void* v, int v_dtype, int64_t B, int64_t H, int64_t N, int64_t D, const int64_t* v_strides,
                       int tile, void* v_tiles, VTArgs* out, unsigned* blocks);

namespace {


// One workgroup's share: 2 THREADS consecutive 16-byte output words, starting at word 2*THREADS*bx, of head hh of batch bb: two a thread,
// neighbours, whose elements lie side by side in V's rows.  Eight loads of four bytes, all in flight at once, where two words a
// thread one after the other took sixteen of two bytes (figures: prepare.hip).
template <int TILE, int D, int THREADS>
__device__ __forceinline__ void v_tiles_block(const VTArgs& a, uint32_t bx, uint32_t hh, uint32_t bb, uint32_t nh) {
    constexpr int NDB = D / 32;
    constexpr int KB = TILE / 32;
    const uint32_t per_head = (uint32_t)a.nt * (TILE * D / 8);
    const uint32_t o = bx * (2u * THREADS) + 2u * threadIdx.x;
    if (o >= per_head) return;
    const uint32_t lane = o & 63u;
    uint32_t rest = o >> 6;
    const uint32_t db = rest % NDB; rest /= NDB;
    const uint32_t c = rest & 1u;   rest >>= 1;
    const uint32_t kb = rest % KB;
    const uint32_t it = rest / KB;
    const uint32_t h = lane >> 5, r = lane & 31u;
    const uint32_t key0 = TILE * it + 32u * kb + 16u * c + 4u * h;
    const unsigned short* src = a.v + (int64_t)bb * a.sb + (int64_t)hh * a.sh + (32u * db + r);
    uint32_t two[8];
#pragma unroll
    for (int t = 0; t < 8; ++t) {
        const unsigned short* const p = src + (int64_t)min(key0 + 8u * (t >> 2) + (t & 3), (uint32_t)a.n - 1u) * a.sn;
        two[t] = a.pairs ? *reinterpret_cast<const uint32_t*>(p) : p[0] | (uint32_t)p[1] << 16;
    }
    if (key0 + 11u >= (uint32_t)a.n) {
#pragma unroll
        for (int t = 0; t < 8; ++t)
            if (key0 + 8u * (t >> 2) + (t & 3) >= (uint32_t)a.n) two[t] = 0;
    }
    uint4 even, odd;
    even.x = __builtin_amdgcn_perm(two[1], two[0], 0x05040100u); odd.x = __builtin_amdgcn_perm(two[1], two[0], 0x07060302u);
    even.y = __builtin_amdgcn_perm(two[3], two[2], 0x05040100u); odd.y = __builtin_amdgcn_perm(two[3], two[2], 0x07060302u);
    even.z = __builtin_amdgcn_perm(two[5], two[4], 0x05040100u); odd.z = __builtin_amdgcn_perm(two[5], two[4], 0x07060302u);
    even.w = __builtin_amdgcn_perm(two[7], two[6], 0x05040100u); odd.w = __builtin_amdgcn_perm(two[7], two[6], 0x07060302u);
    const int64_t head = (int64_t)bb * nh + hh;
    uint4* const to = reinterpret_cast<uint4*>(a.out) + head * per_head + o;
    to[0] = even;
    to[1] = odd;
}

template <int TILE, int D>
__global__ __launch_bounds__(256) void v_tiles_kernel(VTArgs a) {
    v_tiles_block<TILE, D, 256>(a, blockIdx.x, blockIdx.y, blockIdx.z, gridDim.y);
}

}  // namespace

