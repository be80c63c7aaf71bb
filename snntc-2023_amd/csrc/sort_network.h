// Bitonic sorting network over the threads of a workgroup, shared by the segmented sort and by the scan
// that orders its own rows.
#pragma once
#include "snntc_common.h"

namespace snntc {
namespace {

typedef unsigned long long u64;

__device__ __forceinline__ uint32_t float_to_key(float f) {
    uint32_t u = __float_as_uint(f);
    if (u == 0x80000000u) u = 0u;                         // -0 sorts together with +0
    return u ^ ((u >> 31) ? 0xffffffffu : 0x80000000u);
}

__device__ __forceinline__ float key_to_float(uint32_t k) {
    return __uint_as_float(k ^ ((k >> 31) ? 0x80000000u : 0xffffffffu));
}

// The value of `v` in lane `lane ^ d`.  Distances 1, 2 and 8 are lane patterns the vector unit applies
// by itself while it moves a register (quad permutes, rotation of a row of 16 by 8); the others go
// through the LDS crossbar, which the four SIMDs of a CU share.  (Distance 4 as two masked shifts and 16 and 32 as
// permlane swaps instead: 8192 rows of 100 9.6 -> 11.3 us, 4096 of 1521 71 -> 76, the others unchanged.)
__device__ __forceinline__ u64 lane_xor(u64 v, int d) {
    const int lo = (int)(uint32_t)v, hi = (int)(uint32_t)(v >> 32);
    int olo, ohi;
    if (d == 1) {
        olo = __builtin_amdgcn_mov_dpp(lo, 0xB1, 0xf, 0xf, true);      // quad_perm:[1,0,3,2]
        ohi = __builtin_amdgcn_mov_dpp(hi, 0xB1, 0xf, 0xf, true);
    } else if (d == 2) {
        olo = __builtin_amdgcn_mov_dpp(lo, 0x4E, 0xf, 0xf, true);      // quad_perm:[2,3,0,1]
        ohi = __builtin_amdgcn_mov_dpp(hi, 0x4E, 0xf, 0xf, true);
    } else if (d == 8) {
        olo = __builtin_amdgcn_mov_dpp(lo, 0x128, 0xf, 0xf, true);     // row_ror:8
        ohi = __builtin_amdgcn_mov_dpp(hi, 0x128, 0xf, 0xf, true);
    } else {
        return __shfl_xor(v, d, kWave);
    }
    return ((u64)(uint32_t)ohi << 32) | (uint32_t)olo;
}

// Ascending order of the EPT * G keys of G consecutive threads (a power of two; EPT consecutive ones each, tseg: the thread's place
// among them).  Where G is larger than a wavefront, keys change wavefronts through xchg[EPT * G], and every thread of the
// workgroup calls this at the same time; EPT * G keys of every group of G threads then have a part of xchg of their own.
template <int EPT, int G>
__device__ __forceinline__ void bitonic_sort(u64 (&v)[EPT], int tseg, u64* xchg) {
    constexpr int NPAD = EPT * G;
#pragma unroll
    for (int k = 2; k <= NPAD; k <<= 1) {
        // partners in other threads: element distance j >= EPT
#pragma unroll
        for (int j = k >> 1; j >= EPT; j >>= 1) {
            const int d = j / EPT;
            const bool lower = (tseg & d) == 0;
            const bool up = ((tseg * EPT) & k) == 0;
            const bool keep_min = (lower == up);
            if (d >= kWave) {
                __syncthreads();
#pragma unroll
                for (int r = 0; r < EPT; ++r) xchg[r * G + tseg] = v[r];
                __syncthreads();
#pragma unroll
                for (int r = 0; r < EPT; ++r) {
                    const u64 o = xchg[r * G + (tseg ^ d)];
                    const bool take = (o < v[r]) == keep_min;
                    v[r] = take ? o : v[r];
                }
            } else {
#pragma unroll
                for (int r = 0; r < EPT; ++r) {
                    const u64 o = lane_xor(v[r], d);
                    const bool take = (o < v[r]) == keep_min;
                    v[r] = take ? o : v[r];
                }
            }
        }
        // partners inside the thread: element distance j < EPT
#pragma unroll
        for (int j = (EPT >> 1); j >= 1; j >>= 1) {
            if (j <= (k >> 1)) {
#pragma unroll
                for (int r = 0; r < EPT; ++r) {
                    if ((r & j) == 0) {
                        const bool up = ((tseg * EPT + r) & k) == 0;
                        const u64 a = v[r], b = v[r | j];
                        const bool sw = (a > b) == up;
                        v[r] = sw ? b : a;
                        v[r | j] = sw ? a : b;
                    }
                }
            }
        }
    }
}

}  // namespace
}  // namespace snntc
