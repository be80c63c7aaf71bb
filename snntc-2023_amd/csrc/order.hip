// Stable ascending order of every conv patch, shared between overlapping patches.
//
// Stands where the reference calls cub::DeviceSegmentedSort::SortPairs on an im2col tensor
// (snntc/snncv_kernels.cu.cc:112-166).  Patches overlap: with 3x3 kernels an input belongs to nine of them.  A
// workgroup takes a tile of th x tw neighbouring patches and ranks the inputs of the image region they cover
// ONCE; ranks are unique whole numbers, consistent with (value, kh, kw, c) in every patch, so a patch's order
// is then a matter of counting: set a bit per input at its rank, and an input's place is the number of bits
// below it.  No comparison, no dependent chain and no sorted copy of the pixels is left per patch.
//
// Ranking a region of n inputs (a few thousand): a histogram over the leading bits of the value range (1024 coarse
// buckets) gives every coarse bucket 16 bits of a bitmap per input it holds, shared out evenly over the bucket's range, so
// inputs spread over the bitmap whatever their distribution (spike times crowd in one octave and trail off over four
// decades).  An input's rank is the number of inputs before its 32-bit word plus the bits below its own.  About one input
// in eight lies in a word where two share a bit; these go to a list, are gathered by word and compared with the two or three
// others there.  Inputs that never spiked all carry the same largest time: they keep their index order behind the others,
// by a prefix count.  Where another value repeats (or values crowd) so that more than ORDER_BUCKET_LIMIT inputs share a word,
// the region's inputs are ranked by a stable radix sort instead, eight bits a pass.
//
// A patch's bitmap is the union of its pixels' (patches of 32 channels and more; built once per region) or is set bit by bit.
// Patches of up to 1152 inputs belong to a wavefront, which needs no barrier for them; longer ones to the workgroup.
//
// What bounds it: vector instructions, LDS cycles and stores in about equal parts (65 536 patches of 576 inputs: 53, 46 and
// 50 us of 83 to 93, by card).  An input costs some 110 / (patches over it) + 19 vector and 1 + 5 LDS instructions per 64; the 8
// bytes per input it writes are 302 MB there.  Measured against pixels sorted by a network of their own and patches put together
// from them by merge path (chains of dependent LDS reads), in us: those 65 536 patches 188 -> 83, 100 352 of 576 297 -> 124,
// 25 088 of 1152 227 -> 86, 6272 of 2304 144 -> 54, 1568 of 4608 79 -> 42; 401 408 of 147 (7x7x3, stride 2), sorted patch by patch
// before, 438 -> 137.
//
// Ties, on 8-bit images (as they are / a third of the rows saturated / smooth / one value), us between events, next to continuous values and to
// the order by networks and merges that this replaced (any values): 65 536 patches of 576 inputs 158 / 174 / 182 / 194 (88; 205),
// 401 408 of 147 177 / 228 / 240 / 319 (138; 430), 131 072 of 75 43 / 52 / 51 / 58 (41; 89), 6272 of 2304 109 / 119 / 133 / 134 (50; 140);
// above it only at few long and at short strided patches: 1568 of 4608 88 / 115 / 108 / 96 (39; 77), 16 384 of 180 33 / 52 / 38 / 45
// (18; 33).  A bitonic network over the region in the radix sort's place took 173 / 420 / 469 / 724 for the first.  With up to
// 64 inputs compared per word instead of 16 they take up to 37 % longer (smooth 248), with 8 the continuous ones do (96).
#include <algorithm>
#include <atomic>
#include <iterator>

#include "snntc_common.h"
#include "sort_network.h"

namespace snntc {
namespace {

constexpr int ORDER_COARSE = 1024;
constexpr int ORDER_COARSE_BITS = 10;
constexpr int ORDER_BUCKET_LIMIT = 16;                       // inputs of a word that are still compared with each other
constexpr int ORDER_EPT = 16;                              // region inputs per thread at most
constexpr int ORDER_ROW_BUCKET_LIMIT = 32;                   // ... of a dense row
constexpr int ORDER_GROUP_PITCH = ORDER_COARSE + 1;          // counts of a pair of wavefronts: buckets, and the largest time
constexpr int ORDER_RADIX_PITCH = 260;                     // 256 digit counts and a shift of the banks
constexpr int ORDER_LDS_BYTES = 160 * 1024;

struct OrderGeom {
    int H, W, C, Kh, Kw, Sh, Sw, Nh, Nw, P;
    int th, tw, tiles_y, tiles_x;
    int n_cap;                                             // inputs of the region of a full tile
    int words;                                             // bitmap words, n_cap / 32 rounded up
    int region_pixels;                                     // of a full tile; 0: patches set their bits themselves
    int stride;                                            // entries per output row
    float max_cmp;
    uint32_t per_image_magic, tiles_x_magic, kw_len_magic, c_magic, row_magic[2];       // [1]: the last tile of a row
};

// x / d for x * d < 2^32, from 2^32 / d rounded up (d = 1: 2^32 - 1)
inline uint32_t order_magic(int d) { return d > 1 ? 0xffffffffu / (uint32_t)d + 1 : 0xffffffffu; }
__device__ __forceinline__ int order_divide(int x, int d, uint32_t magic) {
    int q = (int)__umulhi((uint32_t)x, magic);
    if (q * d > x) --q;
    if (x - q * d >= d) ++q;
    return q;
}

__device__ __forceinline__ uint32_t order_key(uint32_t u) { return u ^ ((u >> 31) ? 0xffffffffu : 0x80000000u); }

// Inclusive prefix sum / maximum over the wavefront (the maximum arrives in lane 63 and is returned in all).
template <int CTRL, int ROWS>
__device__ __forceinline__ uint32_t dpp(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROWS, 0xf, false);
}
__device__ __forceinline__ uint32_t wave_prefix(uint32_t s) {
    s += dpp<0x111, 0xf>(s);      // row_shr:1
    s += dpp<0x112, 0xf>(s);      // row_shr:2
    s += dpp<0x114, 0xf>(s);      // row_shr:4
    s += dpp<0x118, 0xf>(s);      // row_shr:8
    s += dpp<0x142, 0xa>(s);      // row_bcast:15 into rows 1 and 3
    s += dpp<0x143, 0xc>(s);      // row_bcast:31 into rows 2 and 3
    return s;
}
__device__ __forceinline__ uint32_t wave_max(uint32_t v) {
    v = max(v, dpp<0x111, 0xf>(v));
    v = max(v, dpp<0x112, 0xf>(v));
    v = max(v, dpp<0x114, 0xf>(v));
    v = max(v, dpp<0x118, 0xf>(v));
    v = max(v, dpp<0x142, 0xa>(v));
    v = max(v, dpp<0x143, 0xc>(v));
    return (uint32_t)__builtin_amdgcn_readlane((int)v, kWave - 1);
}
__device__ __forceinline__ uint32_t lanes_below(uint64_t m) {
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0));
}

__device__ __forceinline__ void lds_order() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Byte offset in LDS <-> pointer
typedef __attribute__((address_space(3))) uint32_t lds_u32;
__device__ __forceinline__ uint32_t lds_offset(uint32_t* p) { return (uint32_t)(uintptr_t)(lds_u32*)p; }

// Ranks as they lie in LDS, two halves at a time: byte offset of the word among 8-byte words | bit << 11 (up to 8192 inputs).
__device__ __forceinline__ uint32_t pack_ranks(uint32_t r) { return ((r >> 2) & 0x07f807f8u) | ((r << 11) & 0xf800f800u); }

// LDS: values [n_cap] u32, ranks [n_cap] u16, then -- one after the other -- the ranking's tables or the patches' bitmaps
// and staging buffers.
inline size_t order_lds_bytes(int n_cap, int threads, int stride, int waves, int patches, int region_pixels) {
    const size_t bit_len = ((size_t)(n_cap + 31) / 32 + 3) / 4 * 4;
    const size_t head = ((size_t)n_cap * 6 + 15) / 16 * 16;
    const size_t list_cap = ((size_t)n_cap + 4 * threads - 1) / (4 * threads) * (4 * threads);
    size_t tables = (ORDER_COARSE + kWave) * 4 + (((size_t)n_cap + 7) / 8 * 4 + kWave) * 8 + ((size_t)n_cap + 1) / 2 * 4 + list_cap * 2 + 64;
    const size_t radix = ((size_t)n_cap + 3) / 4 * 16 + (size_t)threads / kWave * ORDER_RADIX_PITCH * 4;
    if (tables < radix) tables = radix;
    const size_t per_patch = waves ? (size_t)waves * (bit_len * 8 + (size_t)stride * 4)             // a patch per wavefront
                                   : (size_t)patches * bit_len * 8 + (size_t)stride * 8;
    const size_t after = (size_t)region_pixels * bit_len * 4 + per_patch;
    return head + (tables > after ? tables : after);
}

// ROWS > 0: the region is one dense row of up to ROWS inputs and its only patch: an input's rank is its place.  Where values
// repeat, see there; where more than ORDER_ROW_BUCKET_LIMIT inputs share a word all the same, the row is sorted by a network.
// T threads; ITERS inputs per lane (WAVE: a patch belongs to a wavefront) or per thread (a patch belongs to
// the workgroup) of a patch; VEC = 4: rows of the image are read in aligned groups of four (C a multiple of four).
template <int T, bool WAVE, int ITERS, int FULL, int VEC, bool PIXELS, int ROWS = 0>
__global__ void __launch_bounds__(T)
order_patches_kernel(const float* __restrict__ xpad, float* __restrict__ sorted, int32_t* __restrict__ perm,
                     int32_t* __restrict__ n_real, OrderGeom g) {
    extern __shared__ __align__(16) uint32_t lds[];
    constexpr int EPT = ROWS > 0 ? (ROWS + 4 * T - 1) / (4 * T) * 4 : ORDER_EPT;         // region inputs per thread at most
    constexpr int WAVES = T / kWave, ROUNDS = EPT / 4;
    constexpr uint32_t kNone = ~0u, kFrequent = ~0u - 1, kNegZero = 0x80000000u;
    __shared__ uint4 red[WAVES];
    __shared__ uint32_t bases[2][WAVES];
    __shared__ uint32_t overflow, several;
    const int tid = threadIdx.x, lane = tid % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int block = xcd_contiguous(blockIdx.x, gridDim.x);
    const int per_image = g.tiles_y * g.tiles_x;
    const int image = order_divide(block, per_image, g.per_image_magic), tile = block - image * per_image;
    const int ty = order_divide(tile, g.tiles_x, g.tiles_x_magic), tx = tile - ty * g.tiles_x;
    const int nh0 = ty * g.th, nw0 = tx * g.tw;
    const int n_ph = min(g.th, g.Nh - nh0), n_pw = min(g.tw, g.Nw - nw0);
    const int row_len = ((n_pw - 1) * g.Sw + g.Kw) * g.C;                // inputs of one image row of the region
    const int n = ((n_ph - 1) * g.Sh + g.Kh) * row_len;
    const uint32_t row_magic = g.row_magic[n_pw < g.tw];                 // e / row_len == umulhi(e, row_magic) for e < n unless row_len is 1

    uint32_t* value = lds;
    uint16_t* rank = reinterpret_cast<uint16_t*>(lds + g.n_cap);
    uint32_t* area = lds + (((size_t)g.n_cap * 6 + 15) / 16 * 4);
    uint32_t* coarse = area;                                             // + one spare entry per lane
    uint2* words = reinterpret_cast<uint2*>(area + ORDER_COARSE + kWave);            // + one spare word per lane
    const int n_words = (n + 7) / 8 * 4;                    // they are counted in fours
    uint16_t* slots = reinterpret_cast<uint16_t*>(words + (g.n_cap + 7) / 8 * 4 + kWave);
    uint16_t* dirty_list = slots + (g.n_cap + 1) / 2 * 2 + wave * ((n + 4 * T - 1) / (4 * T)) * 4 * kWave;       // (a list per wavefront)

    // input j of a thread's round
    bool tied = false, counted = false;                     // ROWS: values repeat; and nothing else is left to rank
    auto begun = [&](int round) { return VEC == 4 ? (round * T + wave * kWave) * 4 < n : round * 4 * T + wave * kWave < n; };      // wave-uniform
    auto input = [&](int round, int j) { return VEC == 4 ? (round * T + tid) * 4 + j : (round * 4 + j) * T + tid; };

    // ---- the region's inputs ---------------------------------------------------------------------------------------
    const float* __restrict__ origin = xpad + (((size_t)image * g.H + (size_t)nh0 * g.Sh) * g.W + (size_t)nw0 * g.Sw) * g.C;
    const uint32_t image_row = (uint32_t)(g.W * g.C);
    const uint32_t key_cmp = order_key(__float_as_uint(g.max_cmp));
    for (int i = tid; i < ORDER_COARSE / 4; i += T) reinterpret_cast<uint4*>(coarse)[i] = make_uint4(0, 0, 0, 0);
    for (int i = tid; i < (n_words + kWave) / 2; i += T) reinterpret_cast<uint4*>(words)[i] = make_uint4(0, 0, 0, 0);
    uint32_t d[EPT];                                                     // key, then distance from the smallest key, then position
#pragma unroll
    for (int round = 0; round < ROUNDS; ++round) {
        if (!begun(round)) break;
        if constexpr (VEC == 4) {
            const uint32_t e = (uint32_t)min(input(round, 0), n - 4), r = __umulhi(e, row_magic);
            const uint4 q = *reinterpret_cast<const uint4*>(origin + (r * image_row + (e - r * (uint32_t)row_len)));
            d[round * 4] = q.x; d[round * 4 + 1] = q.y; d[round * 4 + 2] = q.z; d[round * 4 + 3] = q.w;
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const uint32_t e = (uint32_t)min(input(round, j), n - 1), r = row_len > 1 ? __umulhi(e, row_magic) : e;
                d[round * 4 + j] = __float_as_uint(origin[r * image_row + (e - r * (uint32_t)row_len)]);
            }
        }
    }
    uint32_t k_low = ~0u, k_max = 0;                        // (a thread past the end repeats an input of the region)
#pragma unroll
    for (int round = 0; round < ROUNDS; ++round) {
        if (!begun(round)) break;
        uint32_t* u = d + round * 4;
        if (__builtin_amdgcn_ballot_w64(u[0] == kNegZero || u[1] == kNegZero || u[2] == kNegZero || u[3] == kNegZero))
#pragma unroll
            for (int j = 0; j < 4; ++j) u[j] = u[j] == kNegZero ? 0u : u[j];          // -0 sorts together with +0
        if constexpr (VEC == 4) {
            if (input(round, 0) < n) *reinterpret_cast<uint4*>(value + input(round, 0)) = make_uint4(u[0], u[1], u[2], u[3]);
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (input(round, j) < n) value[input(round, j)] = u[j];
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            u[j] = order_key(u[j]);
            k_low = min(k_low, u[j]);
            k_max = max(k_max, u[j]);
        }
    }
    k_low = ~wave_max(~k_low);
    k_max = wave_max(k_max);
    uint32_t k_high = k_max, idle = 0;                      // the largest key up to key_cmp, and how many lie above
    if (k_max > key_cmp) {
        k_high = 0;
#pragma unroll
        for (int round = 0; round < ROUNDS; ++round) {
            if (!begun(round)) break;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const uint32_t k = d[round * 4 + j];
                k_high = max(k_high, k <= key_cmp ? k : 0u);
                idle += (uint32_t)__builtin_popcountll(__builtin_amdgcn_ballot_w64(k > key_cmp && input(round, j) < n));
            }
        }
        k_high = wave_max(k_high);
    }
    if (lane == 0) red[wave] = make_uint4(k_low, k_max, k_high, idle);
    if (tid == 0) overflow = 0;
    __syncthreads();
    idle = 0;
#pragma unroll
    for (int v = 0; v < WAVES; ++v) {
        const uint4 q = red[v];
        k_low = min(k_low, q.x);
        k_max = max(k_max, q.y);
        k_high = max(k_high, q.z);
        idle += q.w;
    }
    const uint32_t k_min = (uint32_t)__builtin_amdgcn_readfirstlane((int)k_low);
    k_max = (uint32_t)__builtin_amdgcn_readfirstlane((int)k_max);
    const uint32_t range = (uint32_t)__builtin_amdgcn_readfirstlane((int)(max(k_high, k_min) - k_min));
    const uint32_t reals = (uint32_t)n - (uint32_t)__builtin_amdgcn_readfirstlane((int)idle);        // inputs that take part in a scan
    const bool has_last = k_max > key_cmp;                  // inputs of the largest time: behind all others, in index order
    const int sh = range >> (ORDER_COARSE_BITS + 1) ? 32 - __builtin_clz(range) - ORDER_COARSE_BITS : 1;
    const uint32_t d_limit = sh + ORDER_COARSE_BITS >= 32 ? kFrequent - 1 : ((uint32_t)ORDER_COARSE << sh) - 1;

    // ---- positions: 16 bits of a bitmap per input, shared out evenly over the coarse buckets ---------------------------
    // PLAIN: no input of the largest time and whole groups of four; threads past the end stay out.  Otherwise inputs of
    // the largest time, and threads past the end, go through the motions on entries of no consequence.
    uint32_t* last = reinterpret_cast<uint32_t*>(slots);    // inputs of the largest time before a wavefront's round
    const bool plain = VEC == 4 && !has_last;
    auto coarse_of = [&](uint32_t dist) { return dist >= kFrequent ? (uint32_t)(ORDER_COARSE + lane) : dist >> sh; };
    const uint32_t spare = (uint32_t)(n_words + lane);      // a word of no consequence
    auto last_of = [&](int round, int j) { return __builtin_amdgcn_ballot_w64(d[round * 4 + j] == kNone && input(round, j) < n); };
    if (plain) {
#pragma unroll
        for (int round = 0; round < ROUNDS; ++round) {
            if (!begun(round)) break;
            if (input(round, 0) < n)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    d[round * 4 + j] -= k_min;
                    atomicAdd(&coarse[d[round * 4 + j] >> sh], 1u);
                }
        }
    } else {
#pragma unroll
        for (int round = 0; round < ROUNDS; ++round) {
            if (!begun(round)) break;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int q = round * 4 + j;
                const bool none = input(round, j) >= n || (has_last && d[q] == k_max);
                d[q] = none ? kNone : min(d[q] - k_min, d_limit);
                atomicAdd(&coarse[coarse_of(d[q])], 1u);
            }
        }
        if (has_last) {
#pragma unroll
            for (int round = 0; round < ROUNDS; ++round) {
                if (round * 4 * T >= n) break;
                uint32_t c = 0;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    if constexpr (VEC == 1) c = 0;
                    if (begun(round)) c += (uint32_t)__builtin_popcountll(last_of(round, j));
                    if constexpr (VEC == 1) if (lane == 0) last[(round * 4 + j) * WAVES + wave] = c;
                }
                if constexpr (VEC == 4) if (lane == 0) last[round * WAVES + wave] = c;
            }
        }
    }
    __syncthreads();
    // coarse: inputs before the bucket << 19 | inputs in it
    constexpr int HELD = ORDER_COARSE / T;
    uint32_t held[HELD], held_sum = 0;
#pragma unroll
    for (int q = 0; q < HELD; ++q) held_sum += held[q] = coarse[tid * HELD + q];
    if constexpr (ROWS > 0)                                 // in the upper half: buckets in use
#pragma unroll
        for (int q = 0; q < HELD; ++q) held_sum += held[q] ? 1u << 16 : 0u;
    uint32_t before = wave_prefix(held_sum);
    if (lane == kWave - 1) bases[0][wave] = before;
    before -= held_sum;
    uint32_t most = 0;                                      // ROWS: inputs of the thread's fullest bucket << 10 | the bucket
    if constexpr (ROWS > 0) {
#pragma unroll
        for (int q = 0; q < HELD; ++q) most = max(most, held[q] << ORDER_COARSE_BITS | (uint32_t)(tid * HELD + q));
        if (most >> ORDER_COARSE_BITS > max((uint32_t)ORDER_BUCKET_LIMIT, (uint32_t)n / 192)) overflow = 1;
    }
    if (has_last && wave == 0) {
        const int m = (n + 4 * T - 1) / (4 * T) * WAVES * (VEC == 1 ? 4 : 1);
        uint32_t carry = 0;
        for (int i0 = 0; i0 < m; i0 += kWave) {
            const uint32_t v = i0 + lane < m ? last[i0 + lane] : 0, s = wave_prefix(v);
            if (i0 + lane < m) last[i0 + lane] = carry + s - v;
            carry += (uint32_t)__builtin_amdgcn_readlane((int)s, kWave - 1);
        }
    }
    __syncthreads();
    uint32_t n_first = 0;                                   // inputs before the ones of the largest time
#pragma unroll
    for (int v = 0; v < WAVES; ++v) {
        const uint32_t b = bases[0][v];
        if (v < wave) before += b;
        n_first += b;
    }
    // Values repeat (or crowd): a bucket holds more inputs, or fewer buckets are in use, than evenly spread values make of it.
    if constexpr (ROWS > 0) {
        const uint32_t used = n_first >> 16;
        n_first &= 0xffffu;
        before &= 0xffffu;
        tied = __builtin_amdgcn_readfirstlane((int)(overflow | (used * 5 < min(n_first, (range >> sh) + 1) * 3))) != 0;
    }
#pragma unroll
    for (int q = 0; q < HELD; ++q) {
        coarse[tid * HELD + q] = before << 19 | held[q];
        before += held[q];
    }
    uint32_t last_before[VEC == 1 ? EPT : ROUNDS];
    if (has_last) {
#pragma unroll
        for (int q = 0; q < (VEC == 1 ? EPT : ROUNDS); ++q)
            last_before[q] = q * (VEC == 1 ? 1 : 4) * T < n ? last[q * WAVES + wave] : 0;
    }
    __syncthreads();
    // A position: how many inputs come before, as far as the coarse bucket and the place in it tell, times 2^19.  Two inputs
    // make a word of the bitmap.
    auto position = [&](uint32_t dist, uint32_t c) {
        return __umul24((dist << (32 - sh)) >> 13, c & 0x3fffu) + (c & 0xfff80000u);
    };
    auto enter = [&](uint32_t at) {
        uint2* w = words + (at >> 20);
        atomicOr(&w->x, 1u << ((at >> 15) & 31));
        atomicAdd(&w->y, 1u);
    };
    // Rows whose values repeat.  Where every bucket holds a single value, an input's place among its equals is all that is missing:
    // a wavefront takes a run of inputs, 64 at a time, and counts them per bucket (a pair of wavefronts shares a word), which makes the ranks.
    // Where one value repeats among others, its inputs stay out of the bitmap and keep their index order between the
    // smaller and the larger ones, by a prefix count.
    uint32_t k_frequent = 0, n_frequent = 0, n_lower = 0;   // the value that stays out, inputs of it and of smaller values
    uint32_t frequent_before[VEC == 1 ? EPT : ROUNDS];
    if constexpr (ROWS > 0) {
        if (tied) {
            uint16_t* one = slots + (g.n_cap + 1) / 2 * 2;  // an input of every bucket, where the lists will stand (1024 or more entries)
            auto each = [&](auto&& f) {
#pragma unroll
                for (int round = 0; round < ROUNDS; ++round) {
                    if (!begun(round)) break;
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        if (input(round, j) < n && d[round * 4 + j] != kNone) f((uint32_t)input(round, j), d[round * 4 + j] >> sh);
                }
            };
            most = wave_max(most);
            if (lane == 0) bases[1][wave] = most;
            if (tid == 0) overflow = several = 0;
            each([&](uint32_t e, uint32_t b) { one[b] = (uint16_t)e; });
            __syncthreads();
#pragma unroll
            for (int v = 0; v < WAVES; ++v) most = max(most, bases[1][v]);
            const uint32_t frequent = value[one[most & (ORDER_COARSE - 1)]];             // (any, where the bucket holds several)
            k_frequent = order_key(frequent);
            uint32_t counts = 0;                            // inputs of it, and of smaller values << 16
            bool differs = false;
            each([&](uint32_t e, uint32_t b) {
                const uint32_t v = value[e];
                counts += v == frequent ? 1u : order_key(v) < k_frequent ? 1u << 16 : 0u;
                differs |= v != value[one[b]];
            });
            counts = wave_prefix(counts);
            if (lane == kWave - 1) bases[0][wave] = counts;
            if (__builtin_amdgcn_ballot_w64(differs) != 0 && lane == 0) several = 1;
            __syncthreads();
            counts = 0;
#pragma unroll
            for (int v = 0; v < WAVES; ++v) counts += bases[0][v];
            n_lower = counts >> 16;
            n_frequent = counts & 0xffffu;
            counted = __builtin_amdgcn_readfirstlane((int)several) == 0;
            tied = __builtin_amdgcn_readfirstlane((int)n_frequent) > ORDER_ROW_BUCKET_LIMIT;
        }
        if (counted) {
            uint32_t* counter = reinterpret_cast<uint32_t*>(words);                      // [pair of wavefronts][bucket]
            for (int i = tid; i < WAVES / 2 * ORDER_GROUP_PITCH; i += T) counter[i] = 0;
            __syncthreads();
            constexpr int RUNS = ROWS / T;
            const int runs = (n + T - 1) / T, half = wave % 2 * 16;
            uint32_t place[RUNS];                           // bucket << 16 | inputs of it before, in the wavefront
#pragma unroll
            for (int r = 0; r < RUNS; ++r) {
                const int e = (wave * runs + r) * kWave + lane;
                if (r >= runs || e - lane >= n) break;
                const uint32_t k = order_key(value[min(e, n - 1)]);
                const uint32_t b = has_last && k == k_max ? (uint32_t)ORDER_COARSE : min(k - k_min, d_limit) >> sh;
                const uint64_t some = __builtin_amdgcn_ballot_w64(e < n);
                uint32_t lo = (uint32_t)some, hi = (uint32_t)(some >> 32);               // lanes of the same bucket
#pragma unroll
                for (int bit = 0; bit <= ORDER_COARSE_BITS; ++bit) {
                    const uint32_t unset = ((b >> bit) & 1) - 1;
                    const uint64_t set = __builtin_amdgcn_ballot_w64(unset == 0);
                    lo &= (uint32_t)set ^ unset;
                    hi &= (uint32_t)(set >> 32) ^ unset;
                }
                const uint64_t same = (uint64_t)hi << 32 | lo;
                const uint32_t ahead = lanes_below(same);
                uint32_t before_run = 0;
                if (e < n && ahead == 0)
                    before_run = atomicAdd(&counter[wave / 2 * ORDER_GROUP_PITCH + b], (uint32_t)__builtin_popcountll(same) << half);
                before_run = (uint32_t)__shfl((int)before_run, e < n ? __builtin_ctzll(same) : lane, kWave);
                place[r] = b << 16 | (((before_run >> half) & 0xffffu) + ahead);
            }
            __syncthreads();
#pragma unroll
            for (int r = 0; r < RUNS; ++r) {
                const int e = (wave * runs + r) * kWave + lane;
                if (r >= runs || e - lane >= n) break;
                if (e >= n) continue;
                const uint32_t b = place[r] >> 16;
                uint32_t at = (place[r] & 0xffffu) + (b == (uint32_t)ORDER_COARSE ? n_first : coarse[b] >> 19);
                for (int p = 0; p < wave / 2; ++p) {
                    const uint32_t c = counter[p * ORDER_GROUP_PITCH + b];
                    at += (c & 0xffffu) + (c >> 16);
                }
                if (half) at += counter[wave / 2 * ORDER_GROUP_PITCH + b] & 0xffffu;
                rank[e] = (uint16_t)pack_ranks(at);
            }
        } else if (tied) {
#pragma unroll
            for (int round = 0; round < ROUNDS; ++round) {
                uint32_t c = 0;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int q = round * 4 + j, e = input(round, j);
                    d[q] = e >= n ? kNone : d[q] != kNone && order_key(value[min(e, n - 1)]) == k_frequent ? kFrequent : d[q];
                    if constexpr (VEC == 1) c = 0;
                    c += (uint32_t)__builtin_popcountll(__builtin_amdgcn_ballot_w64(d[q] == kFrequent));
                    if constexpr (VEC == 1) if (lane == 0) last[q * WAVES + wave] = c;
                }
                if constexpr (VEC == 4) if (lane == 0) last[round * WAVES + wave] = c;
            }
            __syncthreads();
            constexpr int COUNTS = (VEC == 1 ? EPT : ROUNDS) * WAVES, TURNS = (COUNTS + kWave - 1) / kWave;
            uint32_t prefix[TURNS], sum = n_lower;
#pragma unroll
            for (int t = 0; t < TURNS; ++t) {
                const uint32_t v = t * kWave + lane < COUNTS ? last[t * kWave + lane] : 0, s = wave_prefix(v);
                prefix[t] = sum + s - v;
                sum += (uint32_t)__builtin_amdgcn_readlane((int)s, kWave - 1);
            }
#pragma unroll
            for (int q = 0; q < (VEC == 1 ? EPT : ROUNDS); ++q)                          // (WAVES divides 64)
                frequent_before[q] = (uint32_t)__builtin_amdgcn_readlane((int)prefix[q * WAVES / kWave], q * WAVES % kWave + wave);
        }
    }
    const bool whole = plain && !(ROWS > 0 && tied);        // every group of four as it is
    if (counted) {
    } else if (whole) {
#pragma unroll
        for (int round = 0; round < ROUNDS; ++round) {
            if (!begun(round)) break;
            if (input(round, 0) < n) {
                uint32_t c[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) c[j] = coarse[d[round * 4 + j] >> sh];
#pragma unroll
                for (int j = 0; j < 4; ++j) enter(d[round * 4 + j] = position(d[round * 4 + j], c[j]));
            }
        }
    } else {
#pragma unroll
        for (int round = 0; round < ROUNDS; ++round) {
            if (!begun(round)) break;
            uint32_t c[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) c[j] = coarse[coarse_of(d[round * 4 + j])];      // (those that stay out as well)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int q = round * 4 + j;
                if (d[q] < kFrequent) enter(d[q] = min(position(d[q], c[j]), kFrequent - 1));
            }
        }
    }
    if (!counted) {
        __syncthreads();
        // words: the bitmap and, behind it, the number of inputs before the word | inputs share a bit in it << 31
        constexpr int STEPS = (EPT + 7) / 8;
        const int steps = (n_words + 4 * T - 1) / (4 * T);
        uint32_t count_of[STEPS][4];
        uint32_t carry = 0, fullest = 0;
#pragma unroll
        for (int st = 0; st < STEPS; ++st) {
            if (st >= steps) break;
            const int w = ((wave * steps + st) * kWave + lane) * 4;
            uint4 q[2] = {make_uint4(0, 0, 0, 0), make_uint4(0, 0, 0, 0)};
            if (w < n_words) {
                q[0] = *reinterpret_cast<const uint4*>(words + w);
                q[1] = *reinterpret_cast<const uint4*>(words + w + 2);
            }
            const uint32_t sum = q[0].y + q[0].w + q[1].y + q[1].w, s = carry + wave_prefix(sum);
            fullest = max(max(fullest, max(q[0].y, q[0].w)), max(q[1].y, q[1].w));
            count_of[st][0] = (s - sum) | ((uint32_t)__builtin_popcount(q[0].x) != q[0].y ? 1u << 31 : 0u);
            count_of[st][1] = (s - sum + q[0].y) | ((uint32_t)__builtin_popcount(q[0].z) != q[0].w ? 1u << 31 : 0u);
            count_of[st][2] = (s - q[1].y - q[1].w) | ((uint32_t)__builtin_popcount(q[1].x) != q[1].y ? 1u << 31 : 0u);
            count_of[st][3] = (s - q[1].w) | ((uint32_t)__builtin_popcount(q[1].z) != q[1].w ? 1u << 31 : 0u);
            carry = (uint32_t)__builtin_amdgcn_readlane((int)s, kWave - 1);
        }
        if (lane == 0) bases[1][wave] = carry;
        if (__builtin_amdgcn_ballot_w64(fullest > (ROWS > 0 ? ORDER_ROW_BUCKET_LIMIT : ORDER_BUCKET_LIMIT)) != 0 && lane == 0) overflow = 1;
        __syncthreads();
        const bool give_up = __builtin_amdgcn_readfirstlane((int)overflow) != 0;
        if (!give_up) {
            uint32_t base = 0;
#pragma unroll
            for (int v = 0; v < WAVES; ++v)
                if (v < wave) base += bases[1][v];
#pragma unroll
            for (int st = 0; st < STEPS; ++st) {
                if (st >= steps) break;
                const int w = ((wave * steps + st) * kWave + lane) * 4;
                if (w < n_words)
#pragma unroll
                    for (int t = 0; t < 4; ++t) words[w + t].y = count_of[st][t] + base;
            }
            __syncthreads();

            // ---- ranks ---------------------------------------------------------------------------------------------------
            uint32_t n_listed = 0;
#pragma unroll
            for (int round = 0; round < ROUNDS; ++round) {
                if (!begun(round)) break;
                uint2 w[4];
                uint32_t r[4];
                uint64_t dirty[4];
                if (whole) {
#pragma unroll
                    for (int j = 0; j < 4; ++j) w[j].y = 0;
                    if (input(round, 0) < n)
#pragma unroll
                        for (int j = 0; j < 4; ++j) w[j] = words[d[round * 4 + j] >> 20];
                } else {
#pragma unroll
                    for (int j = 0; j < 4; ++j) w[j] = words[d[round * 4 + j] >= kFrequent ? spare : d[round * 4 + j] >> 20];
                }
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    r[j] = (uint32_t)__builtin_popcount(__builtin_amdgcn_ubfe(w[j].x, 0, d[round * 4 + j] >> 15)) + (w[j].y & 0xffffu);
                    dirty[j] = __builtin_amdgcn_ballot_w64((int)w[j].y < 0);
                }
                if (has_last) {
                    uint64_t l[4];
#pragma unroll
                    for (int j = 0; j < 4; ++j) l[j] = last_of(round, j);
                    uint32_t below = 0;
                    if constexpr (VEC == 4)
                        below = n_first + last_before[round] + lanes_below(l[0]) + lanes_below(l[1]) + lanes_below(l[2]) + lanes_below(l[3]);
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        if constexpr (VEC == 1) below = n_first + last_before[round * 4 + j] + lanes_below(l[j]);
                        const bool mine = __builtin_amdgcn_inverse_ballot_w64(l[j]);
                        r[j] = mine ? below : r[j];
                        if constexpr (VEC == 4) below += mine ? 1u : 0u;
                    }
                }
                if constexpr (ROWS > 0)
                    if (tied) {
                        uint64_t f[4];
#pragma unroll
                        for (int j = 0; j < 4; ++j) f[j] = __builtin_amdgcn_ballot_w64(d[round * 4 + j] == kFrequent);
                        uint32_t below = 0;
                        if constexpr (VEC == 4)
                            below = frequent_before[round] + lanes_below(f[0]) + lanes_below(f[1]) + lanes_below(f[2]) + lanes_below(f[3]);
#pragma unroll
                        for (int j = 0; j < 4; ++j) {
                            if constexpr (VEC == 1) below = frequent_before[round * 4 + j] + lanes_below(f[j]);
                            const bool mine = __builtin_amdgcn_inverse_ballot_w64(f[j]);
                            const bool above = d[round * 4 + j] < kFrequent && order_key(value[min(input(round, j), n - 1)]) > k_frequent;
                            r[j] = mine ? below : above ? r[j] + n_frequent : r[j];
                            if constexpr (VEC == 4) below += mine ? 1u : 0u;
                        }
                    }
                if constexpr (VEC == 4) {
                    if (input(round, 0) < n)
                        *reinterpret_cast<uint2*>(rank + input(round, 0)) =
                            make_uint2(pack_ranks(r[0] | r[1] << 16), pack_ranks(r[2] | r[3] << 16));
                } else {
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        if (input(round, j) < n) rank[input(round, j)] = (uint16_t)pack_ranks(r[j]);
                }
                // inputs of words in which a bit is shared: a list per wavefront
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    if (__builtin_amdgcn_inverse_ballot_w64(dirty[j])) dirty_list[n_listed + lanes_below(dirty[j])] = (uint16_t)input(round, j);
                    n_listed += (uint32_t)__builtin_popcountll(dirty[j]);
                }
            }
            // ... which are gathered by word and counted among themselves
            lds_order();
            auto gather = [&](uint32_t e, uint32_t& k, uint32_t*& word) {
                k = order_key(value[e]);
                const uint32_t dist = min(k - k_min, d_limit);
                word = &words[min(position(dist, coarse[dist >> sh]), kFrequent - 1) >> 20].y;
            };
            auto count = [&](uint32_t e, uint32_t k, const uint32_t* word) {
                const uint32_t m = *word, s0 = m & 0xffffu, s1 = s0 + ((m >> 16) & 0x7fffu);
                const uint64_t mine = (uint64_t)k << 32 | e;
                uint32_t r = s0;
                for (uint32_t q = s0; q < s1; q += 4) {
                    uint32_t o[4], ko[4];
#pragma unroll
                    for (int t = 0; t < 4; ++t) o[t] = slots[min(q + t, s1 - 1)];
#pragma unroll
                    for (int t = 0; t < 4; ++t) ko[t] = order_key(value[o[t]]);
#pragma unroll
                    for (int t = 0; t < 4; ++t) r += (q + t < s1) & (((uint64_t)ko[t] << 32 | o[t]) < mine);
                }
                if constexpr (ROWS > 0) r += tied && k > k_frequent ? n_frequent : 0;
                rank[e] = (uint16_t)pack_ranks(r);
            };
            auto arrive = [&](uint32_t e, uint32_t* word) {
                const uint32_t m = atomicAdd(word, 1u << 16);
                slots[(m & 0xffffu) + ((m >> 16) & 0x7fffu)] = (uint16_t)e;
            };
            uint32_t e0 = 0, k0 = 0, *word0 = nullptr;          // the first 64 of the list stay in registers, most often all
            if (lane < (int)n_listed) {
                e0 = dirty_list[lane];
                gather(e0, k0, word0);
                arrive(e0, word0);
            }
            for (uint32_t i = kWave + lane; i < n_listed; i += kWave) {
                uint32_t e = dirty_list[i], k, *word;
                gather(e, k, word);
                arrive(e, word);
            }
            __syncthreads();
            if (lane < (int)n_listed) count(e0, k0, word0);
            for (uint32_t i = kWave + lane; i < n_listed; i += kWave) {
                uint32_t e = dirty_list[i], k, *word;
                gather(e, k, word);
                count(e, k, word);
            }
        } else if constexpr (ROWS > 0) {
            constexpr int KEYS = ROWS / T;
            u64 v[KEYS];
#pragma unroll
            for (int q = 0; q < KEYS; ++q) {
                const int e = tid * KEYS + q;
                v[q] = (u64)(e < n ? order_key(value[e]) : ~0u) << 32 | (uint32_t)e;
            }
            bitonic_sort<KEYS, T>(v, tid, reinterpret_cast<u64*>(area));
#pragma unroll
            for (int q = 0; q < KEYS; ++q)
                if (const uint32_t e = (uint32_t)v[q]; e < (uint32_t)n) rank[e] = (uint16_t)pack_ranks((uint32_t)(tid * KEYS + q));
        } else {
            // a value repeats too often: stable radix sort of the inputs' indexes, eight bits of the distance from the
            // smallest key a pass; the last pass leaves ranks.  A wavefront takes a run of inputs, 64 at a time.
            constexpr int DIGITS = 256, PITCH = ORDER_RADIX_PITCH, GROUP = WAVES / 4;
            const int rounds = (n + T - 1) / T, half = (g.n_cap + 3) / 4 * 4;
            uint16_t* item = reinterpret_cast<uint16_t*>(area);                              // [2][half], from pass to pass
            uint32_t* count = area + half;                      // [wavefront][digit]
            uint32_t* own = count + wave * PITCH;
            const uint32_t spread = k_max - k_min;
            int shift = 0;
            do {
                const bool last_pass = spread >> shift < DIGITS;
                const uint16_t* from = item + ((shift / 8) & 1) * half;
                uint16_t* to = item + ((shift / 8 + 1) & 1) * half;
                auto index_at = [&](int at) { return shift == 0 ? (uint32_t)at : (uint32_t)from[at]; };
                auto digit_of = [&](uint32_t e) { return ((order_key(value[e]) - k_min) >> shift) & (DIGITS - 1); };
                reinterpret_cast<uint4*>(own)[lane] = make_uint4(0, 0, 0, 0);
                lds_order();
#pragma unroll 1
                for (int r = 0; r < rounds; ++r) {
                    const int at = (wave * rounds + r) * kWave + lane;
                    if (at < n) atomicAdd(&own[digit_of(index_at(at))], 1u);
                }
                __syncthreads();
                // inputs before the ones of a wavefront and digit: in order of (digit, wavefront), four wavefronts per thread
                const int digit = tid / GROUP, first = tid % GROUP * 4;
                uint32_t c[4], sum = 0;
#pragma unroll
                for (int q = 0; q < 4; ++q) sum += c[q] = count[(first + q) * PITCH + digit];
                uint32_t at_or_below = wave_prefix(sum);
                if (lane == kWave - 1) bases[0][wave] = at_or_below;
                __syncthreads();
                uint32_t start = at_or_below - sum;
#pragma unroll 1
                for (int v = 0; v < wave; ++v) start += bases[0][v];
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    count[(first + q) * PITCH + digit] = start;
                    start += c[q];
                }
                __syncthreads();
#pragma unroll 1
                for (int r = 0; r < rounds; ++r) {
                    const int at = (wave * rounds + r) * kWave + lane;
                    const uint32_t e = at < n ? index_at(at) : 0, dg = digit_of(e);
                    const uint64_t some = __builtin_amdgcn_ballot_w64(at < n);
                    uint32_t lo = (uint32_t)some, hi = (uint32_t)(some >> 32);               // lanes with the same digit
#pragma unroll 4
                    for (int b = 0; b < 8; ++b) {               // (in two goes: all eight at once cost every launch 12 registers)
                        const uint32_t unset = ((dg >> b) & 1) - 1;
                        const uint64_t set = __builtin_amdgcn_ballot_w64(unset == 0);
                        lo &= (uint32_t)set ^ unset;
                        hi &= (uint32_t)(set >> 32) ^ unset;
                    }
                    const uint64_t same = (uint64_t)hi << 32 | lo;
                    if (at < n) {
                        const uint32_t before = own[dg], place = before + lanes_below(same);
                        if ((same >> lane) == 1) own[dg] = place + 1;                        // the last of them
                        if (last_pass) rank[e] = (uint16_t)pack_ranks(place);
                        else to[place] = (uint16_t)e;
                    }
                    lds_order();
                }
                __syncthreads();
                shift += 8;
            } while (shift < 32 && spread >> shift);
        }
    }
    __syncthreads();                                        // ranks are in place, the tables are free

    if constexpr (ROWS > 0) {
        uint32_t* at = area;                                // the input at every place of the row, 0 behind its end
        for (int e = tid; e < n; e += T) {
            const uint32_t r = rank[e];
            at[(r & 0x7ffu) * 4 + (r >> 11)] = (uint32_t)e;
        }
        for (int i = n + tid; i < g.stride; i += T) at[i] = 0;
        // inputs that take part: keys below that of -inf are NaN, which do not (those above key_cmp are out already)
        uint32_t nans = 0;
        if (k_min < order_key(0xff800000u)) {
            for (int e = tid; e < n; e += T) nans += order_key(value[e]) < order_key(0xff800000u);
            nans = (uint32_t)__builtin_amdgcn_readlane((int)wave_prefix(nans), kWave - 1);
            if (lane == 0) bases[1][wave] = nans;
        }
        __syncthreads();
        if (tid == 0) {
            uint32_t m = reals;
            if (k_min < order_key(0xff800000u))
                for (int v = 0; v < WAVES; ++v) m -= bases[1][v];
            n_real[image] = (int)m;
        }
        float* __restrict__ zs = sorted + (size_t)image * g.stride;
        int32_t* __restrict__ ps = perm + (size_t)image * g.stride;
        for (int i = tid * 4; i < g.stride; i += T * 4) {
            const uint4 q = *reinterpret_cast<const uint4*>(at + i);
            uint4 z = make_uint4(value[q.x], value[q.y], value[q.z], value[q.w]);
            if (i >= n) z.x = 0x7f800000u;
            if (i + 1 >= n) z.y = 0x7f800000u;
            if (i + 2 >= n) z.z = 0x7f800000u;
            if (i + 3 >= n) z.w = 0x7f800000u;
            *reinterpret_cast<uint4*>(zs + i) = z;
            *reinterpret_cast<uint4*>(ps + i) = q;
        }
        return;
    }

    // ---- patches ---------------------------------------------------------------------------------------------------
    // bits[w]: a patch's inputs as bits at their ranks and, behind it, the byte offset in LDS of the stage entry that the
    // first of them takes.  An entry: patch index << 16 | byte offset in `value` from the patch's first input.
    const int bit_len = (g.words + 3) / 4 * 4;
    const int n_patches = n_ph * n_pw, pix_row = (n_pw - 1) * g.Sw + g.Kw;
    uint32_t* pixel_bits = area;                            // PIXELS: [pixel of the region][bit_len]
    uint32_t* patch_area = area + (PIXELS ? (size_t)g.region_pixels * bit_len : 0);
    constexpr int members = WAVE ? kWave : T;
    const int me = WAVE ? lane : tid;
    uint2* bits = reinterpret_cast<uint2*>(patch_area) + (WAVE ? (size_t)wave * bit_len : 0);        // one per wavefront, or one per patch
    uint32_t* stage = patch_area + (size_t)(WAVE ? WAVES : g.th * g.tw) * bit_len * 2 + (WAVE ? (size_t)wave * g.stride : 0);
    for (int i = g.P + me; i < g.stride; i += members) stage[i] = 0;
    if constexpr (!WAVE)
        for (int i = g.P + me; i < g.stride; i += members) stage[g.stride + i] = 0;
    // of the lane's inputs: the packed pair that is staged
    uint32_t off[ITERS];
    const int kw_len = g.Kw * g.C;
#pragma unroll
    for (int it = 0; it < ITERS; ++it) {
        const int i = min(it * members + me, g.P - 1);
        const int kh = kw_len > 1 ? (int)__umulhi((uint32_t)i, g.kw_len_magic) : i;
        off[it] = (uint32_t)(kh * row_len + (i - kh * kw_len)) * 4 | (uint32_t)i << 16;
    }
    auto first_of_patch = [&](int ph, int pw) { return (uint32_t)(ph * g.Sh * row_len + pw * g.Sw * g.C); };
    // completes the words of a patch staged at `to`, by one wavefront
    auto count_bits = [&](uint2* b, uint32_t* to, auto word_pair) {
        uint32_t carry = lds_offset(to);
        for (int i0 = 0; i0 < bit_len / 2; i0 += kWave) {
            const int i = i0 + lane;
            uint2 q = make_uint2(0, 0);
            if (i < bit_len / 2) q = word_pair(i);
            const uint32_t c0 = (uint32_t)__builtin_popcount(q.x) * 4, c = c0 + (uint32_t)__builtin_popcount(q.y) * 4;
            const uint32_t s = carry + wave_prefix(c) - c;
            if (i < bit_len / 2) reinterpret_cast<uint4*>(b)[i] = make_uint4(q.x, s, q.y, s + c0);
            carry = (uint32_t)__builtin_amdgcn_readlane((int)(s + c), kWave - 1);
        }
    };
    auto from_pixels = [&](int ph, int pw) {
        const uint32_t* p0 = pixel_bits + (size_t)(ph * g.Sh * pix_row + pw * g.Sw) * bit_len;
        return [=](int i) {
            uint2 q = make_uint2(0, 0);
            // three by three pixels at a time; repeating one does no harm
            for (int kh0 = 0; kh0 < g.Kh; kh0 += 3)
                for (int kw0 = 0; kw0 < g.Kw; kw0 += 3)
#pragma unroll
                    for (int u = 0; u < 3; ++u)
#pragma unroll
                        for (int v = 0; v < 3; ++v) {
                            const int pixel = min(kh0 + u, g.Kh - 1) * pix_row + min(kw0 + v, g.Kw - 1);
                            const uint2 t = reinterpret_cast<const uint2*>(p0 + pixel * bit_len)[i];
                            q.x |= t.x;
                            q.y |= t.y;
                        }
            return q;
        };
    };
    auto clear_bits = [&](uint2* b, int count) {
        for (int i = me; i < count / 2; i += members) reinterpret_cast<uint4*>(b)[i] = make_uint4(0, 0, 0, 0);
    };
    // whether iteration `it` of this thread is an input of the patch (the first FULL iterations always are)
    auto takes_part = [&](int it) { return it < FULL || it * members + me < g.P; };
    auto rank_at = [&](uint32_t first, uint32_t o) { return (uint32_t)rank[first + (o & 0xffffu) / 4]; };
    auto word_at = [](uint2* b, uint32_t r) { return reinterpret_cast<uint2*>(reinterpret_cast<unsigned char*>(b) + (r & 0x7ffu)); };
    auto set_bits = [&](uint2* b, uint32_t first) {
        uint32_t r[ITERS];
#pragma unroll
        for (int it = 0; it < ITERS; ++it) r[it] = rank_at(first, off[it]);
#pragma unroll
        for (int it = 0; it < ITERS; ++it)
            if (takes_part(it)) atomicOr(&word_at(b, r[it])->x, 1u << (r[it] >> 11));
    };
    auto place_inputs = [&](uint2* b, uint32_t* to, uint32_t first, size_t seg) {
        uint32_t r[ITERS];
        uint2 w[ITERS];
#pragma unroll
        for (int it = 0; it < ITERS; ++it) r[it] = rank_at(first, off[it]);
#pragma unroll
        for (int it = 0; it < ITERS; ++it) w[it] = *word_at(b, r[it]);
#pragma unroll
        for (int it = 0; it < ITERS; ++it) {
            const uint32_t below = (uint32_t)__builtin_popcount(__builtin_amdgcn_ubfe(w[it].x, 0, r[it] >> 11));
            if (takes_part(it)) *(lds_u32*)(uintptr_t)(w[it].y + below * 4) = off[it];
        }
        if (me == 0) {
            // inputs that take part in the scan: the ones ranked below the region's count of them
            int m = g.P;
            if (reals < (uint32_t)n) {
                const uint2 q = b[reals >> 5];
                m = (int)((q.y - lds_offset(to)) / 4 + (uint32_t)__builtin_popcount(__builtin_amdgcn_ubfe(q.x, 0, reals & 31)));
            }
            n_real[seg] = m;
        }
    };
    auto write_rows = [&](const uint32_t* from, uint32_t first, size_t seg) {
        float* __restrict__ zs = sorted + seg * g.stride;
        int32_t* __restrict__ ps = perm + seg * g.stride;
        const unsigned char* v = reinterpret_cast<const unsigned char*>(value + first);
        auto value_at = [&](uint32_t o) { return *reinterpret_cast<const uint32_t*>(v + (o & 0xffffu)); };
        constexpr int PASSES = (ITERS + 3) / 4;
        uint4 q[PASSES], z[PASSES];
#pragma unroll
        for (int t = 0; t < PASSES; ++t) q[t] = *reinterpret_cast<const uint4*>(from + min(4 * (t * members + me), g.stride - 4));
#pragma unroll
        for (int t = 0; t < PASSES; ++t) z[t] = make_uint4(value_at(q[t].x), value_at(q[t].y), value_at(q[t].z), value_at(q[t].w));
        if (g.stride != g.P) {                              // +inf behind the patch (the staged entry there is 0)
#pragma unroll
            for (int t = 0; t < PASSES; ++t) {
                const int i = 4 * (t * members + me);
                if (i >= g.P) z[t].x = 0x7f800000u;
                if (i + 1 >= g.P) z[t].y = 0x7f800000u;
                if (i + 2 >= g.P) z[t].z = 0x7f800000u;
                if (i + 3 >= g.P) z[t].w = 0x7f800000u;
            }
        }
#pragma unroll
        for (int t = 0; t < PASSES; ++t) {
            const uint32_t i = 4 * (t * members + me);
            if (i < (uint32_t)g.stride) {
                *reinterpret_cast<uint4*>(zs + i) = z[t];
                *reinterpret_cast<uint4*>(ps + i) = make_uint4(q[t].x >> 16, q[t].y >> 16, q[t].z >> 16, q[t].w >> 16);
            }
        }
    };
    auto segment = [&](int ph, int pw) { return ((size_t)image * g.Nh + nh0 + ph) * g.Nw + nw0 + pw; };

    if constexpr (PIXELS) {
        const int region_pixels = n / g.C;
        for (int i = tid; i < region_pixels * bit_len / 4; i += T) reinterpret_cast<uint4*>(pixel_bits)[i] = make_uint4(0, 0, 0, 0);
        __syncthreads();
#pragma unroll
        for (int round = 0; round < ROUNDS; ++round) {      // (VEC == 4: whole groups of four of one pixel)
            if (!begun(round)) break;
            if (const int e = input(round, 0); e < n) {
                const uint2 r = *reinterpret_cast<const uint2*>(rank + e);
                uint32_t* pb = pixel_bits + __umulhi((uint32_t)e, g.c_magic) * bit_len;
                atomicOr(&pb[(r.x & 0x7ffu) / 8], 1u << ((r.x >> 11) & 31));
                atomicOr(&pb[(r.x >> 16 & 0x7ffu) / 8], 1u << (r.x >> 27));
                atomicOr(&pb[(r.y & 0x7ffu) / 8], 1u << ((r.y >> 11) & 31));
                atomicOr(&pb[(r.y >> 16 & 0x7ffu) / 8], 1u << (r.y >> 27));
            }
        }
        __syncthreads();
    }
    if constexpr (WAVE) {
        int ph = 0, pw = wave;
        for (int p = wave; p < n_patches; p += WAVES, pw += WAVES) {
            for (; pw >= n_pw; pw -= n_pw) ++ph;
            const uint32_t first = first_of_patch(ph, pw);
            if constexpr (PIXELS) {
                count_bits(bits, stage, from_pixels(ph, pw));
            } else {
                clear_bits(bits, bit_len);
                lds_order();
                set_bits(bits, first);
                lds_order();
                count_bits(bits, stage, [&](int i) { return make_uint2(bits[2 * i].x, bits[2 * i + 1].x); });
            }
            lds_order();
            place_inputs(bits, stage, first, segment(ph, pw));
            lds_order();
            write_rows(stage, first, segment(ph, pw));
            lds_order();
        }
    } else {
        // all bitmaps first, a patch per wavefront; then patch by patch, between two staging buffers
        if constexpr (!PIXELS) {
            clear_bits(bits, n_patches * bit_len);
            __syncthreads();
            for (int p = 0, ph = 0, pw = 0; p < n_patches; ++p) {
                set_bits(bits + (size_t)p * bit_len, first_of_patch(ph, pw));
                if (++pw == n_pw) { pw = 0; ++ph; }
            }
            __syncthreads();
        }
        for (int p = wave, ph = 0, pw = wave; p < n_patches; p += WAVES, pw += WAVES) {
            for (; pw >= n_pw; pw -= n_pw) ++ph;
            uint2* b = bits + (size_t)p * bit_len;
            uint32_t* to = stage + (p & 1) * g.stride;
            if constexpr (PIXELS) count_bits(b, to, from_pixels(ph, pw));
            else count_bits(b, to, [=](int i) { return make_uint2(b[2 * i].x, b[2 * i + 1].x); });
        }
        __syncthreads();
        for (int p = 0, ph = 0, pw = 0; p < n_patches; ++p) {
            uint32_t* to = stage + (p & 1) * g.stride;
            place_inputs(bits + (size_t)p * bit_len, to, first_of_patch(ph, pw), segment(ph, pw));
            __syncthreads();
            write_rows(to, first_of_patch(ph, pw), segment(ph, pw));
            if (++pw == n_pw) { pw = 0; ++ph; }
        }
    }
}

typedef void (*OrderKernel)(const float*, float*, int32_t*, int32_t*, OrderGeom);
struct OrderForm {
    int threads, inputs;                                    // patches up to so many inputs ...
    bool wave;                                              // ... by a wavefront or by the workgroup
    int waves_per_cu;                                       // as far as registers go
    OrderKernel quads_pixels, quads, single;
};
template <int T, bool WAVE, int ITERS, int FULL>
constexpr OrderForm order_form() {
    return OrderForm{T, ITERS * (WAVE ? kWave : T), WAVE, ITERS <= 9 ? 28 : 20, order_patches_kernel<T, WAVE, ITERS, FULL, 4, true>,
                     order_patches_kernel<T, WAVE, ITERS, FULL, 4, false>, order_patches_kernel<T, WAVE, ITERS, FULL, 1, false>};
}
// by patch length; FULL is the number of iterations that the lengths of a form all fill
const OrderForm kOrderForms[] = {
    order_form<256, true, 1, 0>(),  order_form<256, true, 3, 1>(),  order_form<256, true, 5, 3>(),  order_form<256, true, 9, 5>(),
    order_form<256, true, 13, 9>(), order_form<256, true, 18, 13>(), order_form<512, false, 5, 2>(), order_form<1024, false, 5, 2>(),
    order_form<1024, false, 8, 5>(),
};
const OrderForm& order_form_of(int64_t P) {
    const OrderForm* f = kOrderForms;
    while (P > f->inputs) ++f;
    return *f;
}

struct OrderPlan {
    int th, tw, n_cap, region_pixels;
    size_t lds;
};

constexpr int ORDER_MAX_REGION = 8192;
constexpr int ORDER_PIXEL_CHANNELS = 32;

// LDS of a tile whose region has n inputs, 0 if the kernel does not take it.
size_t order_tile_lds(int64_t n, const OrderForm& form, int stride, int patches, int region_pixels) {
    if (n > ORDER_MAX_REGION || n > (int64_t)form.threads * ORDER_EPT) return 0;
    const size_t lds = order_lds_bytes((int)n, form.threads, stride, form.wave ? form.threads / kWave : 0, patches, region_pixels);
    return lds <= (size_t)ORDER_LDS_BYTES - 1024 ? lds : 0;
}

// Tile of a layer: the one with the smallest estimated time among the tiles that cut rows and columns evenly.  A
// workgroup issues some 450 vector instructions per wavefront, 230 per 256 inputs it ranks and 13 per 64 inputs it
// orders; alone on a CU it takes about 14000 clocks for the ranks and, per patch in turn, 1000 and 220 per 64 inputs.
// The workgroups that share a CU take about the sum of one's latency and everyone's instructions, and overlap the better
// the more they are.
OrderPlan order_best_tile(const ConvGeom& g, const OrderForm& form, bool pixels, int cus) {
    OrderPlan best{};
    float best_time = 1e30f;
    const int T = form.threads, W = T / kWave, stride = (int)padded_stride(g.P), members = form.wave ? kWave : T;
    const int iters = (int)((g.P + members - 1) / members);
    const float patch_work = form.wave ? 60.f + 13.f * iters : W * (20.f + 13.f * iters);
    const float patch_alone = 1000.f + 220.f * iters;
    for (int64_t ny = (g.Nh + 15) / 16, th = 0; ny <= g.Nh; ny = th > 1 ? (g.Nh + th - 2) / (th - 1) : g.Nh + 1) {
        th = (g.Nh + ny - 1) / ny;
        for (int64_t nx = (g.Nw + 15) / 16, tw = 0; nx <= g.Nw; nx = tw > 1 ? (g.Nw + tw - 2) / (tw - 1) : g.Nw + 1) {
            tw = (g.Nw + nx - 1) / nx;
            const int64_t px = ((th - 1) * g.Sh + g.Kh) * ((tw - 1) * g.Sw + g.Kw), n = px * g.C;
            const size_t lds = order_tile_lds(n, form, stride, (int)(th * tw), pixels ? (int)px : 0);
            if (lds == 0) continue;
            const int64_t tiles = g.B * ny * nx, fit = std::min((int64_t)(ORDER_LDS_BYTES / (lds + 512)), (int64_t)(form.waves_per_cu / W));
            const int64_t resident = std::max((int64_t)1, std::min(fit, (tiles + cus - 1) / cus));
            const float patches = (float)(th * tw), turns = form.wave ? (float)((th * tw + W - 1) / W) : patches;
            const float work = 1.1f * (450.f * W + 230.f * (float)((n + 255) / 256) + patches * patch_work);
            const float alone = 14000.f + turns * patch_alone;
            const float slots = (float)(cus * resident), rounds = (float)tiles <= slots ? 1.f : (float)tiles / slots + 0.5f;
            const float time = rounds * (alone + (float)resident * work) * (1.f + 0.6f / (float)resident);
            if (time < best_time) {
                best_time = time;
                best = OrderPlan{(int)th, (int)tw, (int)n, pixels ? (int)px : 0, lds};
            }
        }
    }
    return best;
}

// A bitmap per pixel of the region takes region^2 / C / 8 bytes: with large kernels not even a single patch's pixels fit next
// to the rest (7x7 with 164 channels, 16x16 with 32), and the patches set their bits themselves, as for fewer channels.
OrderPlan order_plan(const ConvGeom& g, const OrderForm& form, bool quads, int cus) {
    OrderPlan plan{};
    if (quads && g.C >= ORDER_PIXEL_CHANNELS) plan = order_best_tile(g, form, true, cus);
    return plan.n_cap ? plan : order_best_tile(g, form, false, cus);
}

}  // namespace

namespace {
// The kernels' LDS limits on a device, once.
int order_ready(int dev) {
    static std::atomic<bool> ready[kMaxDevices];
    if (dev < 0 || dev >= kMaxDevices) return fail(SNNTC_ERR_UNSUPPORTED, "order: device index %d not supported", dev);
    if (!ready[dev].load(std::memory_order_acquire)) {
        const int rc = order_prepare_device();
        if (rc) return rc;
        ready[dev].store(true, std::memory_order_release);
    }
    return SNNTC_OK;
}

// Dense rows by length.
struct OrderRowsForm {
    int inputs, threads;
    OrderKernel single, quads;
};
template <int T, int N>
constexpr OrderRowsForm order_rows_form() {
    return OrderRowsForm{N, T, order_patches_kernel<T, true, 1, 0, 1, false, N>, order_patches_kernel<T, true, 1, 0, 4, false, N>};
}
const OrderRowsForm kOrderRowsForms[] = {order_rows_form<256, 512>(), order_rows_form<256, 1024>(), order_rows_form<256, 2048>(),
                                         order_rows_form<512, 4096>(), order_rows_form<1024, 8192>(), order_rows_form<512, 2048>()};
constexpr int ORDER_FEW_ROWS = 256;                         // of 1025 to 2048 inputs: a workgroup per CU or none, of twice the threads

size_t order_rows_lds(int64_t I, const OrderRowsForm& form) {
    const size_t ranks = order_lds_bytes((int)I, form.threads, (int)padded_stride(I), 1, 0, 0);
    const size_t network = ((size_t)I * 6 + 15) / 16 * 16 + (size_t)form.inputs * 8;
    const size_t groups = ((size_t)I * 6 + 15) / 16 * 16 + (ORDER_COARSE + kWave + (size_t)form.threads / kWave / 2 * ORDER_GROUP_PITCH) * 4;
    return std::max({ranks, network, groups});
}
}  // namespace

// Dense rows: the sorting networks -> ranked, us between events, values all different (as they are / a tenth silent), then with repeats
// (8-bit levels / mostly background / background and different values), then crowded in a tenth of an octave with outliers:
//   16 x 1521      11.9 -> 8.7 / 9.5, 10.0 / 10.8 / 11.2, 11.3          3500 x 512     26.7 -> 17.0 / 19.8, 20.5 / 23.5 / 24.5, 22.6
//   256 x 2048     16.0 -> 12.3 / 13.1, 14.4 / 15.6 / 16.2, 14.8        5000 x 384     28.6 -> 20.6 / 23.7, 24.6 / 27.0 / 28.7, 27.7
//   400 x 1521     20.2 -> 14.0 / 15.6, 17.0 / 18.4 / 18.4, 17.8        1024 x 784     18.2 -> 13.5 / 14.4, 15.8 / 17.3 / 17.0, 16.3
//   512 x 4096     41.0 -> 24.3 / 25.4, 29.8 / 34.6 / 33.3, 32.6        4096 x 784     45.7 -> 21.9 / 25.4, 29.3 / 33.2 / 33.2, 30.5
//   512 x 8192     69.0 -> 33.0 / 37.0, 47.7 / 56.4 / 54.3, 67.2        16 384 x 784    132 -> 60 / 72, 84 / 100 / 99, 90
// A network's steps grow with the square of the length's logarithm, the ranking's do not; but up to 1024 inputs it waits for a
// workgroup's latency until several share a CU (128 x 784: 8.8 -> 8.2 / 9.2, 9.8 / 10.3 / 10.7, 10.3; 300 x 785: 11.4 -> 10.2 / 11.2,
// 11.9 / 12.7 / 12.7, 12.5; 512 x 1024: 13.7 -> 12.0 / 12.9, 13.9 / 15.0 / 15.0, 14.5), and up to 512 the network is one wavefront's,
// which a full chip hides (8192 x 512: 37.7 -> 29.3 / 33.8, 36.8 / 42.8 / 44.3, 40.9) and which rows that are read an input
// at a time hardly beat (5000 x 385: 28.9 -> 24.8 / 28.2, 27.9 / 29.7 / 31.7, 33.0; 5000 x 511: 33.4 -> 25.4 / 28.8, 28.6 / 32.3 / 33.1, 34.1;
// in fours 2048 x 300: 13.7 -> 11.3 / 12.8, 14.4 / 13.4 / 14.7, 14.8).  Different values decide, and repeats may not cost more than those gain.
// Rows with several values that repeat among others of their bucket go to a network after all, and are slower for it (a
// background with most other values close to it: 4096 x 784 45 -> 41, 512 x 4096 41 -> 47, 16 x 1521 12.0 -> 14.4).
bool order_rows_supported(int64_t S, int64_t I) {
    if (S <= 0 || I > ORDER_MAX_REGION) return false;
    if (I > 512) return I > 1024 || S >= 300;
    return I % 4 == 0 ? I > 256 && S >= 2048 && S <= 6144 : I >= 448 && S >= 3072 && S <= 5120;
}

int launch_order_rows(const float* x, float* sorted, int32_t* perm, int32_t* n_real, int64_t S, int64_t I, int64_t stride,
                      float max_cmp, hipStream_t stream) {
    int dev = 0;
    SNNTC_HIP_CHECK(hipGetDevice(&dev));
    const int rc = order_ready(dev);
    if (rc) return rc;
    const OrderRowsForm* form = kOrderRowsForms;
    while (I > form->inputs) ++form;
    if (I > 1024 && I <= 2048 && S <= ORDER_FEW_ROWS) form = std::end(kOrderRowsForms) - 1;
    OrderGeom og{};
    og.H = 1; og.W = (int)I; og.C = 1; og.Kh = 1; og.Kw = (int)I; og.Sh = 1; og.Sw = 1; og.Nh = 1; og.Nw = 1; og.P = (int)I;
    og.th = og.tw = og.tiles_y = og.tiles_x = 1;
    og.n_cap = (int)I;
    og.words = (int)((I + 31) / 32);
    og.stride = (int)stride;
    og.max_cmp = max_cmp;
    og.per_image_magic = og.tiles_x_magic = order_magic(1);
    og.kw_len_magic = og.c_magic = og.row_magic[0] = og.row_magic[1] = order_magic((int)I);
    if (S > 0x7fffffffLL) return fail(SNNTC_ERR_TOO_LARGE, "order: grid too large");
    const bool quads = I % 4 == 0 && reinterpret_cast<uintptr_t>(x) % 16 == 0;
    {
        KernelTimerScope timer_("order_rows", stream);
        hipLaunchKernelGGL(quads ? form->quads : form->single, dim3((unsigned)S), dim3(form->threads), order_rows_lds(I, *form), stream, x,
                           sorted, perm, n_real, og);
    }
    SNNTC_HIP_CHECK(hipGetLastError());
    return SNNTC_OK;
}

int order_prepare_device() {
    for (const OrderRowsForm& f : kOrderRowsForms)
        for (OrderKernel k : {f.single, f.quads})
            SNNTC_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize,
                                                ORDER_LDS_BYTES - 1024));
    for (const OrderForm& f : kOrderForms)
        for (OrderKernel k : {f.quads_pixels, f.quads, f.single})
            SNNTC_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize,
                                                ORDER_LDS_BYTES - 1024));
    return SNNTC_OK;
}

// Patches of one pixel share nothing, patches of up to 64 inputs are sorted in registers by one wavefront faster than they
// are ranked (50 176 of 27 inputs: 16.5 against 25.7 us; of 50: 25.8 / 27.5; of 72: 42.6 / 27.9), and the same holds up to
// 128 inputs while there are only a few patches per CU and the latency of one workgroup counts (784 of 72: 6.3 / 8.3 us).
// The tile that asks for least is a single patch that sets its own bits; it is among the ones order_plan looks at.
bool order_patches_supported(const ConvGeom& g) {
    return g.Kh * g.Kw > 1 && g.P > (g.S <= 4096 ? 128 : 64) && g.P <= ORDER_MAX_REGION &&
           order_tile_lds(g.P, order_form_of(g.P), (int)padded_stride(g.P), 1, 0) > 0;
}

int order_tile(const ConvGeom& g, bool aligned, int64_t tile[4]) {
    for (int i = 0; i < 4; ++i) tile[i] = 0;
    if (!order_patches_supported(g)) return SNNTC_OK;
    const OrderPlan plan = order_plan(g, order_form_of(g.P), g.C % 4 == 0 && aligned, 256);
    if (plan.n_cap == 0) return fail(SNNTC_ERR_UNSUPPORTED, "order: no tile for patches of %lld inputs", (long long)g.P);
    tile[0] = plan.th; tile[1] = plan.tw; tile[2] = plan.region_pixels; tile[3] = (int64_t)plan.lds;
    return SNNTC_OK;
}

int launch_order_patches(const float* xpad, float* sorted, int32_t* perm, int32_t* n_real, const ConvGeom& g, int64_t stride,
                         float max_cmp, hipStream_t stream) {
    int dev = 0, cus = 0;
    SNNTC_HIP_CHECK(hipGetDevice(&dev));
    const int prep = scan_prepare_device(dev, &cus);
    if (prep) return prep;
    const int rc = order_ready(dev);
    if (rc) return rc;
    const bool quads = g.C % 4 == 0 && reinterpret_cast<uintptr_t>(xpad) % 16 == 0;
    const OrderForm& form = order_form_of(g.P);
    const OrderPlan plan = order_plan(g, form, quads, cus);
    if (plan.n_cap == 0) return fail(SNNTC_ERR_UNSUPPORTED, "order: no tile for patches of %lld inputs", (long long)g.P);
    OrderGeom og;
    og.H = (int)g.H; og.W = (int)g.W; og.C = (int)g.C; og.Kh = (int)g.Kh; og.Kw = (int)g.Kw; og.Sh = (int)g.Sh; og.Sw = (int)g.Sw;
    og.Nh = (int)g.Nh; og.Nw = (int)g.Nw; og.P = (int)g.P;
    og.th = plan.th; og.tw = plan.tw;
    og.tiles_y = (int)((g.Nh + plan.th - 1) / plan.th);
    og.tiles_x = (int)((g.Nw + plan.tw - 1) / plan.tw);
    og.n_cap = plan.n_cap;
    og.words = (plan.n_cap + 31) / 32;
    og.region_pixels = plan.region_pixels;
    og.stride = (int)stride;
    og.max_cmp = max_cmp;
    og.per_image_magic = order_magic(og.tiles_y * og.tiles_x);
    og.tiles_x_magic = order_magic(og.tiles_x);
    og.kw_len_magic = order_magic((int)(g.Kw * g.C));
    og.c_magic = order_magic((int)g.C);
    og.row_magic[0] = order_magic((int)(((plan.tw - 1) * g.Sw + g.Kw) * g.C));
    og.row_magic[1] = order_magic((int)(((g.Nw - 1) % plan.tw * g.Sw + g.Kw) * g.C));
    const OrderKernel kernel = plan.region_pixels ? form.quads_pixels : quads ? form.quads : form.single;
    const int64_t blocks = g.B * og.tiles_y * og.tiles_x;
    if (blocks > 0x7fffffffLL) return fail(SNNTC_ERR_TOO_LARGE, "order: grid too large");
    {
        KernelTimerScope timer_("order_patches", stream);
        hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(form.threads), plan.lds, stream, xpad, sorted, perm, n_real, og);
    }
    SNNTC_HIP_CHECK(hipGetLastError());
    return SNNTC_OK;
}

}  // namespace snntc
