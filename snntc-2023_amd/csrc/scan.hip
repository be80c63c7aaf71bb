// Causal-set scan: for every (segment, output neuron) walk the segment's inputs in ascending
// order, accumulate sum(w) and sum(w*z), and stop at the first prefix whose weighted mean lies
// after its last input and not after the next one.
//
// Replaces SnnFcCudaOutKernel / SnnFcCudaOutKernelBias (snntc/snnfc_kernels.cu.cc:19-71,
// snntc/snncv_kernels.cu.cc:19-72) and reproduces their arithmetic step by step: bias first,
// sequential fp32 accumulation with a fused multiply-add for ysum, the division-free firing test
// |ysum| > x*|wsum| with the product rounded on its own, and y = ysum * (1/wsum).
//
// Kernels, by launch size (launch_scan_lds picks):
//   scan_filter_kernel     weight slice in LDS, one, two or four neurons per lane, and the tests of a step skipped
//                          wherever a margin test on a whole chunk of eight inputs proves that none of
//                          them can close the set;
//   scan_lds_split_kernel  fewer work items than CUs: one item per workgroup, its weights gathered
//                          into LDS in scan order first, then one wavefront accumulating and the
//                          others sharing the item's tests;
//   scan_kernel            segments so long that not even eight weight columns fit in LDS, and small launches of
//                          segments of less than a chunk: weight rows streamed from memory, one wavefront
//                          per (segment, 64 neurons).
// In all of them lanes run across neurons, so a weight row is read coalesced (or conflict-free from
// LDS), while the sorted value and the row index of a step are the same for all lanes of a segment
// (segment rows are padded to a multiple of 16 entries so that they are fetched eight at a time
// without bounds checks).
#include <algorithm>
#include <atomic>
#include <type_traits>
#include <utility>

#include "snntc_common.h"
#include "sort_network.h"

namespace snntc {
namespace {

constexpr int CHUNK = 8;

struct LaneState {
    float wsum, ysum, wa, ya;
    bool fired;
};

// One scan step for a lane that is still open.  Returns false when the causal set closes before
// consuming input x (the lane then keeps its state).
__device__ __forceinline__ bool scan_step(LaneState& s, float x, float wv) {
    if (s.fired && s.ya <= x * s.wa) return false;
    s.wsum += wv;
    s.ysum = __fmaf_rn(x, wv, s.ysum);
    s.wa = fabsf(s.wsum);
    s.ya = s.wsum < 0.0f ? -s.ysum : s.ysum;
    s.fired = s.ya > x * s.wa;
    return true;
}

template <bool WANT_K>
__global__ void __launch_bounds__(256)
scan_kernel(const float* __restrict__ sorted, const int32_t* __restrict__ perm,
            const int32_t* __restrict__ n_real, const float* __restrict__ w, float* __restrict__ y_out,
            float* __restrict__ rcp_out, int32_t* __restrict__ k_out, int64_t n_items, int I, int stride,
            int J, int j_blocks, NeuronParams np, TimeCopy copy) {
    // work item = (segment, 64-neuron block); one per wavefront
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int64_t item = (int64_t)blockIdx.x * (blockDim.x / kWave) + wave;
    if (item >= n_items) return;
    const int seg = (int)(item / j_blocks);
    const int jb = (int)(item - (int64_t)seg * j_blocks);
    const int lane = threadIdx.x % kWave;
    const int j = jb * kWave + lane;
    const bool active = j < J;
    const unsigned jc = (unsigned)(active ? j : J - 1);      // clamp so every lane reads valid memory

    const float* __restrict__ xs = sorted + (size_t)seg * stride;
    const int32_t* __restrict__ pr = perm + (size_t)seg * stride;
    const int n = n_real[seg];                                // inputs with value <= MAX-0.1

    LaneState s;
    s.wsum = -np.theta; s.ysum = 0.0f; s.wa = 0.0f; s.ya = 0.0f; s.fired = false;
    if (np.bias) {
        const float wb = (w + (size_t)I * J)[jc];
        s.wsum += wb;
        s.ysum = np.biasvolt * wb;
        s.wa = fabsf(s.wsum);
        s.ya = s.wsum < 0.0f ? -s.ysum : s.ysum;
        s.fired = s.ya > s.wa * np.biasvolt;
    }

    int kcnt = 0;
    if (active) {
        // w[row, j]: the row base is wave-uniform (scalar registers), the lane adds a 32-bit byte offset
        const unsigned joff = jc * (unsigned)sizeof(float);
        auto weight_at = [&](int32_t row) -> float {
            const char* rowp = reinterpret_cast<const char*>(w + (uint32_t)row * (uint32_t)J);
            return *reinterpret_cast<const float*>(rowp + joff);
        };

        const int n_full = n & ~(CHUNK - 1);
        float wq[CHUNK];
#pragma unroll
        for (int u = 0; u < CHUNK; ++u) wq[u] = weight_at(pr[u]);    // row padding keeps pr[0..15] readable
        bool open = true;
        for (int k0 = 0; k0 < n_full && open; k0 += CHUNK) {
            float xv[CHUNK], wc[CHUNK];
            const int kn = (k0 + CHUNK < n_full) ? k0 + CHUNK : k0;  // next chunk, or a harmless re-read
#pragma unroll
            for (int u = 0; u < CHUNK; ++u) {
                xv[u] = xs[k0 + u];
                wc[u] = wq[u];
                wq[u] = weight_at(pr[kn + u]);
            }
#pragma unroll
            for (int u = 0; u < CHUNK; ++u) {
                if (open) {
                    open = scan_step(s, xv[u], wc[u]);
                    if (WANT_K && open) kcnt = k0 + u + 1;
                }
            }
        }
        // up to CHUNK-1 trailing steps
        for (int k = n_full; k < n && open; ++k) {
            open = scan_step(s, xs[k], weight_at(pr[k]));
            if (WANT_K && open) kcnt = k + 1;
        }

        float y = np.max_time, r = 0.0f;
        if (s.fired) {
            r = 1.0f / s.wsum;
            y = s.ysum * r;
            if (y >= np.max_time) { y = np.max_time; r = 0.0f; }
        }
        const size_t o = (size_t)seg * J + j;
        y_out[o] = y;
        rcp_out[o] = r;
        if (copy.dst) copy.dst[time_copy_pixel(copy, seg) * J + j] = y;
        if (WANT_K) k_out[o] = (s.fired && r != 0.0f) ? kcnt : -1;
    }
}

// ---------------------------------------------------------------------------------------------
// Scan with the weight slice resident in LDS.
//
// Walking W rows in sorted order from memory re-reads the whole matrix once per segment (8 GB of
// cache traffic for 65 536 patches of a 3x3x64 -> 64 layer).  Here a workgroup copies the COLS
// columns it owns -- all I rows, at most 160 KB -- into LDS once and then scans many segments
// against it.  A wavefront covers 64/COLS segments at a time (lanes = segment x column), so narrow
// layers (J = 10, Kc = 32) and long segments (COLS = 8 for 4608 inputs) use the same kernel.
// Sorted values and row indices are fetched per lane (all lanes of a segment read the same
// address) eight steps at a time, one chunk ahead of the LDS reads that need them.
// ---------------------------------------------------------------------------------------------
constexpr int LDS_SCAN_THREADS = 1024;
constexpr int LDS_SCAN_BYTES = 160 * 1024;
// The widest slice that fits is taken: the register budget allows one 16-wave workgroup per CU anyway,
// and fewer slices re-read the sorted rows less often.
constexpr int FILTER_RED_BYTES = 64;                       // behind the slice: one float per wavefront for a reduction
constexpr int FILTER_STAGE_BYTES = 1024;                   // then, per wavefront, the row entries on their way to its lanes (STAGED)
// Most neurons per lane: four; two with 8-column slices (the segments of a wavefront would be too many for its row entries).
template <int COLS>
constexpr int FILTER_MAX_CH = COLS == 8 ? 2 : 4;
// STAGED: row entries reach the lanes of a segment through LDS instead of DPP broadcasts.  A vector instruction with a DPP operand
// makes the plain ones around it issue at half their rate (probe kernels, four wavefronts per SIMD: multiply-adds alone 2.0 clocks
// each, with one such move to four, sixteen, thirty-two or sixty-four of them 4.3, 3.8, 3.0 and 2.2 clocks an instruction), and an LDS read
// costs about five plain instructions whatever its width: four reads per chunk in place of sixteen broadcasts.  us with
// DPP / staged: 65 536 segments of 576 to 64 neurons 226 / 207, 100 352 329 / 299, 32 768 of 576 120 / 108.  Only with rows of 256 bytes: slices of 32,
// 16 and 8 columns read their weights with bank conflicts, and four more reads make LDS the bound (4096 rows of 784
// to 800 neurons 242 / 262, 6272 segments of 2304 to 256 365 / 405, 1568 of 4608 to 512 514 / 545), and only where the entries of all
// wavefronts fit beside the slice (launch_scan_lds): rows of up to 576 inputs.
template <int COLS>
constexpr bool FILTER_STAGES = COLS == 64;
constexpr int LDS_SCAN_TARGET = LDS_SCAN_BYTES - FILTER_RED_BYTES;

struct Chunk {
    float x[CHUNK];
    int32_t p[CHUNK];
};

// Rows are read through buffer descriptors: a scalar descriptor (first row of the work item), a
// scalar chunk offset and a per-lane byte offset that never changes during a scan.  No per-lane
// address arithmetic is left, so issuing the next loads never has to wait for those in flight.
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));

struct RowSource {
    __amdgpu_buffer_rsrc_t xs, pr;
};

__device__ __forceinline__ RowSource make_row_source(const float* xs0, const int32_t* pr0, int bytes) {
    RowSource r;
    r.xs = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(xs0), 0, bytes, 0x00020000);
    r.pr = __builtin_amdgcn_make_buffer_rsrc(const_cast<int32_t*>(pr0), 0, bytes, 0x00020000);
    return r;
}

__device__ __forceinline__ void load_chunk_flat(Chunk& c, const float* __restrict__ xs,
                                                const int32_t* __restrict__ pr, int k) {
    const float4 a = *reinterpret_cast<const float4*>(xs + k);
    const float4 b = *reinterpret_cast<const float4*>(xs + k + 4);
    const int4 pa = *reinterpret_cast<const int4*>(pr + k);
    const int4 pb = *reinterpret_cast<const int4*>(pr + k + 4);
    c.x[0] = a.x; c.x[1] = a.y; c.x[2] = a.z; c.x[3] = a.w;
    c.x[4] = b.x; c.x[5] = b.y; c.x[6] = b.z; c.x[7] = b.w;
    c.p[0] = pa.x; c.p[1] = pa.y; c.p[2] = pa.z; c.p[3] = pa.w;
    c.p[4] = pb.x; c.p[5] = pb.y; c.p[6] = pb.z; c.p[7] = pb.w;
}

#define SNNTC_SCAN_COUNT "v_add_u32_e32 %[kcnt], 1, %[kcnt]\n"
#define SNNTC_SCAN_INPUTS(XC, X)                                                                       \
    [run] "s"(run), [x0] XC(X[0]), [x1] XC(X[1]), [x2] XC(X[2]), [x3] XC(X[3]), [x4] XC(X[4]),          \
        [x5] XC(X[5]), [x6] XC(X[6]), [x7] XC(X[7]), [w0] "v"(w[0]), [w1] "v"(w[1]), [w2] "v"(w[2]),    \
        [w3] "v"(w[3]), [w4] "v"(w[4]), [w5] "v"(w[5]), [w6] "v"(w[6]), [w7] "v"(w[7])

// Eight scan steps for the lanes in `run`, written out by hand, every decision on the vector side:
// the lane carries a gate value yg = fired ? ya : +inf, the closing test `yg > x*|wsum|` writes
// EXEC directly (a lane that closes drops out of the rest of the block) and the new gate is a
// select.  Per step (x = input time, w = its weight), nine vector instructions and no branch:
//     EXEC &= yg > x*|wsum|                       (a closing lane keeps its sums)
//     wsum  += w ; ysum = fma(x, w, ysum) ; ya = wsum < 0 ? -ysum : ysum
//     yg     = ya > x*|wsum| ? ya : +inf
// No vector -> scalar -> EXEC round trips, so a step of a lone wavefront takes few cycles.  A select that reads a lane mask needs two
// wait states behind the compare that writes it: the first has the steps in between, the second AHEAD, two instructions, which
// are the next step's product x*|wsum| where there is one, the count where one is wanted, and waits.
#define SNNTC_VSCAN_PRODUCT(U) "v_mul_f32_e64 %[t], %[x" #U "], |%[wsum]|\n"
#define SNNTC_VSCAN_STEP(U, AHEAD)                                           \
    "v_cmpx_gt_f32_e32 vcc, %[yg], %[t]\n"                                   \
    "v_add_f32_e32 %[wsum], %[wsum], %[w" #U "]\n"                           \
    "v_cmp_gt_f32_e32 vcc, 0, %[wsum]\n"                                     \
    "v_fmac_f32_e32 %[ysum], %[x" #U "], %[w" #U "]\n"                       \
    SNNTC_VSCAN_PRODUCT(U)                                                   \
    "v_cndmask_b32_e64 %[ya], %[ysum], -%[ysum], vcc\n"                      \
    "v_cmp_gt_f32_e32 vcc, %[ya], %[t]\n"                                    \
    AHEAD                                                                    \
    "v_cndmask_b32_e32 %[yg], %[inf], %[ya], vcc\n"
// the steps of a chunk: FILL is the instruction next to the product, LAST what the last step has instead of both
#define SNNTC_VSCAN_CHUNK(FILL, LAST)                                                                                   \
    SNNTC_VSCAN_PRODUCT(0)                                                                                              \
    SNNTC_VSCAN_STEP(0, SNNTC_VSCAN_PRODUCT(1) FILL) SNNTC_VSCAN_STEP(1, SNNTC_VSCAN_PRODUCT(2) FILL)                   \
    SNNTC_VSCAN_STEP(2, SNNTC_VSCAN_PRODUCT(3) FILL) SNNTC_VSCAN_STEP(3, SNNTC_VSCAN_PRODUCT(4) FILL)                   \
    SNNTC_VSCAN_STEP(4, SNNTC_VSCAN_PRODUCT(5) FILL) SNNTC_VSCAN_STEP(5, SNNTC_VSCAN_PRODUCT(6) FILL)                   \
    SNNTC_VSCAN_STEP(6, SNNTC_VSCAN_PRODUCT(7) FILL) SNNTC_VSCAN_STEP(7, LAST)
#define SNNTC_VSCAN_PROLOGUE                        \
    "s_mov_b64 %[save], exec\n"                     \
    "s_mov_b64 exec, %[run]\n"
#define SNNTC_VSCAN_EPILOGUE                         \
    "s_andn2_b64 %[gone], %[run], exec\n"            \
    "s_or_b64 %[closed], %[closed], %[gone]\n"       \
    "s_mov_b64 exec, %[save]\n"
#define SNNTC_VSCAN_STATE                                                                              \
    [wsum] "+v"(wsum), [ysum] "+v"(ysum), [ya] "+v"(ya), [yg] "+v"(yg), [kcnt] "+v"(kcnt),             \
        [closed] "+s"(closed), [save] "=&s"(saved_exec), [gone] "=&s"(gone), [t] "=&v"(t)
#define SNNTC_VSCAN_INPUTS                                                                             \
    [run] "s"(run), [inf] "v"(inf), [x0] "v"(x[0]), [x1] "v"(x[1]), [x2] "v"(x[2]), [x3] "v"(x[3]),     \
        [x4] "v"(x[4]), [x5] "v"(x[5]), [x6] "v"(x[6]), [x7] "v"(x[7]), [w0] "v"(w[0]), [w1] "v"(w[1]), \
        [w2] "v"(w[2]), [w3] "v"(w[3]), [w4] "v"(w[4]), [w5] "v"(w[5]), [w6] "v"(w[6]), [w7] "v"(w[7])

template <bool WANT_K>
__device__ __forceinline__ void scan_chunk_vector(float& wsum, float& ysum, float& ya, float& yg, int& kcnt,
                                                  uint64_t& closed, uint64_t run, const float (&x)[CHUNK],
                                                  const float (&w)[CHUNK]) {
    uint64_t saved_exec, gone;
    float t;
    const float inf = INFINITY;
    if (WANT_K)
        asm volatile(SNNTC_VSCAN_PROLOGUE SNNTC_VSCAN_CHUNK(SNNTC_SCAN_COUNT, SNNTC_SCAN_COUNT "s_nop 0\n") SNNTC_VSCAN_EPILOGUE
                     : SNNTC_VSCAN_STATE : SNNTC_VSCAN_INPUTS : "vcc", "scc");
    else
        asm volatile(SNNTC_VSCAN_PROLOGUE SNNTC_VSCAN_CHUNK("s_nop 0\n", "s_nop 1\n") SNNTC_VSCAN_EPILOGUE
                     : SNNTC_VSCAN_STATE : SNNTC_VSCAN_INPUTS : "vcc", "scc");
}

// The same for scans known to be in the plain state with ysum - x*wsum above `slack` (many roundings of the sums
// of a chunk): at five instructions per input.  A lane leaves where ysum - x*wsum falls to slack, before it
// consumes x.  If its weight sum is positive then, it has fired (the value before x was above slack), and
// the reference closes it there exactly if ysum <= x*wsum, with x = x_exit; in every other case the caller
// steps the chunk through with all tests.  A lane that stays keeps the plain state: a negative weight sum with
// ysum - x*wsum > 0 has not fired.
#define SNNTC_CLOSE_STEP(U)                                                  \
    "v_mov_b32_e32 %[xe], %[x" #U "]\n"                                      \
    "v_fma_f32 %[t], %[x" #U "], %[wsum], %[slack]\n"                        \
    "v_cmpx_gt_f32_e32 vcc, %[ysum], %[t]\n"                                \
    "v_add_f32_e32 %[wsum], %[wsum], %[w" #U "]\n"                          \
    "v_fmac_f32_e32 %[ysum], %[x" #U "], %[w" #U "]\n"
#define SNNTC_CLOSE_EPILOGUE                         \
    "v_mov_b32_e32 %[stays], 1\n"                    \
    "s_mov_b64 exec, %[save]\n"
// Returns the lanes that left.  (As a vector flag turned into a mask: a statement with vector and scalar results
// has only divergent values for the compiler, and the masks would move to vector registers.)
template <bool COUNT>
__device__ __forceinline__ uint64_t close_chunk_vector(float& wsum, float& ysum, int& kcnt, float& x_exit, uint64_t run,
                                                       const float (&x)[CHUNK], const float (&w)[CHUNK], float slack) {
    uint64_t saved_exec;
    float t;
    int stays = 0;
    x_exit = 0.0f;
    if (COUNT)
        asm volatile(SNNTC_VSCAN_PROLOGUE SNNTC_CLOSE_STEP(0) SNNTC_SCAN_COUNT SNNTC_CLOSE_STEP(1) SNNTC_SCAN_COUNT
                     SNNTC_CLOSE_STEP(2) SNNTC_SCAN_COUNT SNNTC_CLOSE_STEP(3) SNNTC_SCAN_COUNT SNNTC_CLOSE_STEP(4)
                     SNNTC_SCAN_COUNT SNNTC_CLOSE_STEP(5) SNNTC_SCAN_COUNT SNNTC_CLOSE_STEP(6) SNNTC_SCAN_COUNT
                     SNNTC_CLOSE_STEP(7) SNNTC_SCAN_COUNT SNNTC_CLOSE_EPILOGUE
                     : [wsum] "+v"(wsum), [ysum] "+v"(ysum), [kcnt] "+v"(kcnt), [xe] "+v"(x_exit), [stays] "+v"(stays),
                       [save] "=&s"(saved_exec), [t] "=&v"(t)
                     : SNNTC_SCAN_INPUTS("v", x), [slack] "v"(slack) : "vcc", "scc");
    else
        asm volatile(SNNTC_VSCAN_PROLOGUE SNNTC_CLOSE_STEP(0) SNNTC_CLOSE_STEP(1) SNNTC_CLOSE_STEP(2) SNNTC_CLOSE_STEP(3)
                     SNNTC_CLOSE_STEP(4) SNNTC_CLOSE_STEP(5) SNNTC_CLOSE_STEP(6) SNNTC_CLOSE_STEP(7) SNNTC_CLOSE_EPILOGUE
                     : [wsum] "+v"(wsum), [ysum] "+v"(ysum), [xe] "+v"(x_exit), [stays] "+v"(stays),
                       [save] "=&s"(saved_exec), [t] "=&v"(t)
                     : SNNTC_SCAN_INPUTS("v", x), [slack] "v"(slack) : "vcc", "scc");
    return run & __builtin_amdgcn_ballot_w64(stays == 0);
}

// One step with all tests (an input behind the full chunks of a row).
__device__ __forceinline__ void scan_step_vector(float& wsum, float& ysum, float& ya, float& yg, int& kcnt, uint64_t run,
                                                 float x, float w) {
    uint64_t saved_exec;
    float t;
    const float inf = INFINITY;
    asm volatile(SNNTC_VSCAN_PROLOGUE SNNTC_VSCAN_PRODUCT(0) SNNTC_VSCAN_STEP(0, SNNTC_SCAN_COUNT "s_nop 0\n") "s_mov_b64 exec, %[save]\n"
                 : [wsum] "+v"(wsum), [ysum] "+v"(ysum), [ya] "+v"(ya), [yg] "+v"(yg), [kcnt] "+v"(kcnt),
                   [save] "=&s"(saved_exec), [t] "=&v"(t)
                 : [run] "s"(run), [inf] "v"(inf), [x0] "v"(x), [w0] "v"(w) : "vcc", "scc");
}

// Eight inputs added to the running sums of the lanes in `run`, no tests: what a wavefront does for
// the chunks whose tests another wavefront of its workgroup evaluates (scan_lds_split_kernel).
#define SNNTC_ACC_STEP(U)                                  \
    "v_add_f32_e32 %[wsum], %[wsum], %[w" #U "]\n"         \
    "v_fmac_f32_e32 %[ysum], %[x" #U "], %[w" #U "]\n"
__device__ __forceinline__ void accumulate_chunk(float& wsum, float& ysum, int& kcnt, uint64_t run,
                                                 const float (&x)[CHUNK], const float (&w)[CHUNK]) {
    uint64_t saved_exec;
    asm volatile("s_mov_b64 %[save], exec\n"
                 "s_mov_b64 exec, %[run]\n" SNNTC_ACC_STEP(0) SNNTC_ACC_STEP(1) SNNTC_ACC_STEP(2) SNNTC_ACC_STEP(3)
                     SNNTC_ACC_STEP(4) SNNTC_ACC_STEP(5) SNNTC_ACC_STEP(6) SNNTC_ACC_STEP(7)
                 "v_add_u32_e32 %[kcnt], 8, %[kcnt]\n"
                 "s_mov_b64 exec, %[save]\n"
                 : [wsum] "+v"(wsum), [ysum] "+v"(ysum), [kcnt] "+v"(kcnt), [save] "=&s"(saved_exec)
                 : SNNTC_SCAN_INPUTS("v", x));
}

// Eight inputs added to one sum, their factors the values that lanes FIRST ... of the row of sixteen hold.
template <int FIRST>
__device__ __forceinline__ void accumulate_row(float& acc, float x, const float (&w)[CHUNK]) {
#define SNNTC_ROW_STEP(U) "v_fmac_f32_dpp %[acc], %[x], %[w" #U "] row_newbcast:%[n" #U "] row_mask:0xf bank_mask:0xf bound_ctrl:1\n"
    if (FIRST == 0) asm volatile("s_nop 1" : "+v"(x));      // (wait states, should the compiler have moved it)
    asm(SNNTC_ROW_STEP(0) SNNTC_ROW_STEP(1) SNNTC_ROW_STEP(2) SNNTC_ROW_STEP(3) SNNTC_ROW_STEP(4) SNNTC_ROW_STEP(5)
            SNNTC_ROW_STEP(6) SNNTC_ROW_STEP(7)
        : [acc] "+v"(acc)
        : [x] "v"(x), [w0] "v"(w[0]), [w1] "v"(w[1]), [w2] "v"(w[2]), [w3] "v"(w[3]), [w4] "v"(w[4]), [w5] "v"(w[5]), [w6] "v"(w[6]),
          [w7] "v"(w[7]), [n0] "n"(FIRST), [n1] "n"(FIRST + 1), [n2] "n"(FIRST + 2), [n3] "n"(FIRST + 3), [n4] "n"(FIRST + 4),
          [n5] "n"(FIRST + 5), [n6] "n"(FIRST + 6), [n7] "n"(FIRST + 7));
}

// Copies columns [j0, j0 + COLS) of all `rows` rows of W[rows, J] into LDS as wl[row][COLS] (zeros
// past column J).  Loads are issued in batches so that a small workgroup does not pay one memory
// latency per element.
// Returns the largest |w| among the values this thread copied (NaN entries skipped).
template <int COLS>
__device__ __forceinline__ float fill_weight_slice(float* __restrict__ wl, const float* __restrict__ w, int rows,
                                                   int J, int j0) {
    const int n_fill = rows * COLS;
    float amax = 0.0f;
    if ((J & 3) == 0) {
        constexpr int C4 = COLS / 4, FILL = 4;
        for (int base = threadIdx.x; base < rows * C4; base += FILL * blockDim.x) {
            float4 v[FILL];
#pragma unroll
            for (int u = 0; u < FILL; ++u) {
                const int idx = base + u * blockDim.x;
                const int r = idx / C4, c = (idx - r * C4) * 4;
                v[u] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                if (idx < rows * C4 && j0 + c < J) v[u] = *reinterpret_cast<const float4*>(w + (size_t)r * J + j0 + c);
            }
#pragma unroll
            for (int u = 0; u < FILL; ++u) {
                const int idx = base + u * blockDim.x;
                if (idx < rows * C4) reinterpret_cast<float4*>(wl)[idx] = v[u];
                amax = fmaxf(amax, fmaxf(fmaxf(fabsf(v[u].x), fabsf(v[u].y)), fmaxf(fabsf(v[u].z), fabsf(v[u].w))));
            }
        }
    } else if (j0 == 0 && J > 1 && J < COLS && (reinterpret_cast<uintptr_t>(w) & 15) == 0 && rows * J < (1 << 24)) {
        // One slice holds every column (a 10-wide head): the source is a single run of rows*J floats.
        // It is read as aligned float4 regardless of J, eight per thread in flight, and each value
        // is dropped at [row][col]; the padding columns are zeroed first.
        for (int idx = threadIdx.x; idx < n_fill / 4; idx += blockDim.x)
            reinterpret_cast<float4*>(wl)[idx] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        __syncthreads();
        constexpr int FILL = 8;
        const int n = rows * J, n4 = n / 4;
        const unsigned magic = 0xffffffffu / (unsigned)J + 1;      // e / J == umulhi(e, magic) for e < 2^24
        for (int base = threadIdx.x; base < n4; base += FILL * blockDim.x) {
            float4 v[FILL];
#pragma unroll
            for (int u = 0; u < FILL; ++u) {
                const int idx = base + u * blockDim.x;
                if (idx < n4) v[u] = reinterpret_cast<const float4*>(w)[idx];
            }
#pragma unroll
            for (int u = 0; u < FILL; ++u) {
                const int idx = base + u * blockDim.x;
                if (idx < n4) {
                    const float q[4] = {v[u].x, v[u].y, v[u].z, v[u].w};
#pragma unroll
                    for (int t = 0; t < 4; ++t) {
                        const unsigned e = 4u * idx + t, r = __umulhi(e, magic);
                        wl[r * COLS + (e - r * J)] = q[t];
                        amax = fmaxf(amax, fabsf(q[t]));
                    }
                }
            }
        }
        if ((int)threadIdx.x < n - 4 * n4) {
            const unsigned e = 4u * n4 + threadIdx.x, r = __umulhi(e, magic);
            const float v = w[e];
            wl[r * COLS + (e - r * J)] = v;
            amax = fmaxf(amax, fabsf(v));
        }
    } else {
        constexpr int FILL = 16;
        for (int base = threadIdx.x; base < n_fill; base += FILL * blockDim.x) {
            float v[FILL];
#pragma unroll
            for (int u = 0; u < FILL; ++u) {
                const int idx = base + u * blockDim.x;
                const int r = idx / COLS, c = idx - r * COLS;
                v[u] = (idx < n_fill && j0 + c < J) ? w[(size_t)r * J + j0 + c] : 0.0f;
            }
#pragma unroll
            for (int u = 0; u < FILL; ++u) {
                const int idx = base + u * blockDim.x;
                if (idx < n_fill) wl[idx] = v[u];
                amax = fmaxf(amax, fabsf(v[u]));
            }
        }
    }
    return amax;
}

// Launches of a few dozen work items (the 10-wide head of a classifier): one item per workgroup,
// its wavefronts sharing the item instead of taking one each.  The running sums of a scan are
// inherently sequential, its tests are not, and a lone wavefront pays about five clocks for every
// instruction it issues, whatever the instruction.  So the sequential part is stripped to the two
// additions per input and the reads that feed them:
//   * before the scan all wavefronts gather the item's weights in scan order, w[lane][k] =
//     W[perm[seg][k]][j], straight from memory into LDS (every entry is independent), next to the
//     sorted rows; the scans then read times and weights as 16-byte runs with no address
//     arithmetic, and the row indices never enter LDS;
//   * wavefront 0 (the producer) only accumulates; after every chunk of eight inputs it leaves
//     the sums in LDS and advances a progress counter.  While every scan of the item still has a
//     full round of four chunks ahead no lane is masked and nothing is compared;
//   * the other wavefronts (the testers) take every SPLIT_TESTERS-th chunk: they wait for the sums before their chunk,
//     recompute the fired state from them and the last input before the chunk, and run the ordinary
//     eight-step block with all its tests.  Each tester records the first close it sees; the
//     earliest of all is the scan's (a close found in a chunk is exact as long as no earlier step
//     closed, and an earlier close wins the minimum anyway).  The producer walks the trailing
//     inputs (fewer than eight) and supplies the result of a scan that never closes.
// An item is SPLIT lanes wide: 32 lanes (the upper half of the wavefronts mirrors the lower) keep
// the gathered weights of rows of 800 inputs within LDS; 64-column slices use all 64.
// (Seven testers: leaving the wavefront that shares the producer's SIMD idle, or 11 or 15 testers,
// measured no faster.)
constexpr int SPLIT_WAVES = 8, SPLIT_TESTERS = SPLIT_WAVES - 1;
constexpr int SPLIT_THREADS = SPLIT_WAVES * kWave;
constexpr int SPLIT_STATIC_LDS = 3 * SPLIT_WAVES * kWave * 4 + 16 + 2 * 4 * CHUNK * 4;
constexpr int SPLIT_SPIN_LIMIT = 1 << 20;                  // default number of polls of the progress counter before a
                                                           // tester gives up (NeuronParams::wait_polls carries the one in force)
// Tester wavefronts that gave up since the process started: one word per device, written (a vector
// atomic) only on that path, read by read_scan_giveups().
__device__ unsigned int g_scan_giveups = 0;
constexpr int SPLIT_PAD = 4;                               // floats between the weight rows of two lanes: the 16-byte
                                                           // reads of eight neighbouring lanes fall on distinct banks
constexpr int SPLIT_ROUND = 4;                             // chunks per round of the producer
constexpr int split_lanes(int cols) { return cols == 64 ? 64 : 32; }
// Slices whose items have one or two rows can order them in the workgroup (more rows per item leave a network too few threads).
constexpr bool split_sorts(int cols) { return cols == 32 || cols == 16; }
constexpr int SPLIT_SORT_MAX = 1024;                       // inputs

// dynamic LDS of the split kernel: gathered weights [lanes][stride + pad], sorted rows [segs][stride],
// sums after every chunk [chunks + round][2][lanes].  Reads run up to a round past the end of a row
// (into whatever follows, never used); the sums behind the rows keep them inside the allocation.
__host__ __device__ inline size_t split_lds_bytes(int lanes, int segs, int stride) {
    return ((size_t)lanes * (stride + SPLIT_PAD) + (size_t)segs * stride +
            (size_t)(stride / CHUNK + SPLIT_ROUND) * 2 * lanes) * sizeof(float);
}
// Items of 32 lanes: the upper half of the producer forms the weight sums as multiply-adds with ones, a round of which stands here
// (and a round ahead, which it requests as it does of the times).
constexpr int SPLIT_ONES = 2 * SPLIT_ROUND * CHUNK;

// NPAD > 0: the workgroup orders the rows of its item itself, with a network of NPAD keys per row, from `sorted` = the input
// values as they are [S][I]; perm and n_real are not read.  Every slice orders the same rows again, on CUs that would be idle, and a
// launch (with its ramp, a store and a trip to memory) is gone: one row of 784 to 800 neurons 5.6 + 12.2 -> 15.4 us, 128 items of
// two rows of 800 6.8 + 12.4 -> 17.6.
template <int COLS, int NPAD, bool WANT_K>
__global__ void __launch_bounds__(SPLIT_THREADS)
scan_lds_split_kernel(const float* __restrict__ sorted, const int32_t* __restrict__ perm,
                      const int32_t* __restrict__ n_real, const float* __restrict__ w, float* __restrict__ y_out,
                      float* __restrict__ rcp_out, int32_t* __restrict__ k_out, int S, int I, int stride, int J,
                      int n_slices, int n_groups, NeuronParams np, TimeCopy copy) {
    extern __shared__ __align__(16) float wg[];            // [LANES][stride + SPLIT_PAD], rows, sums
    __shared__ int k_found[SPLIT_WAVES][kWave];
    __shared__ float w_found[SPLIT_WAVES][kWave], y_found[SPLIT_WAVES][kWave];
    __shared__ int progress;                               // chunks whose sums are in LDS
    __shared__ __align__(16) float ones[SPLIT_ONES];
    constexpr int LANES = split_lanes(COLS), SEGS = LANES / COLS;
    constexpr int NONE = 0x7fffffff;
    const int block = xcd_contiguous(blockIdx.x, gridDim.x);
    const int slice = block / n_groups;
    const int group = block - slice * n_groups;
    const int j0 = slice * COLS;
    const int wstride = stride + SPLIT_PAD;
    float* __restrict__ xrows = wg + LANES * wstride;      // [SEGS][stride]
    float* sums = xrows + SEGS * stride;                   // [chunk][wsum|ysum][LANES]

    const int lane = threadIdx.x % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int la = lane % LANES;                           // lanes past LANES mirror the lower ones
    const int sub = la / COLS, col = la - sub * COLS;
    const int j = j0 + col;
    const float* __restrict__ wrow = wg + la * wstride;
    const float w_bias = np.bias && j < J ? w[(size_t)I * J + j] : 0.0f;

    for (int item = group; item * SEGS < S; item += n_groups) {
        const int seg0 = item * SEGS;
        const int n_segs = S - seg0 < SEGS ? S - seg0 : SEGS;
        const int seg_raw = seg0 + sub;
        // mirror lanes scan along with the lane they mirror (same inputs, same sums, stored to the
        // same place) and only stay out of the output
        const bool scans = seg_raw < S && j < J;
        const bool live = scans && lane < LANES;
        const int seg = seg_raw < S ? seg_raw : S - 1;
        const int row = seg - seg0;                         // idle lanes shadow the item's last segment
        const float* __restrict__ xs = xrows + row * stride;
        int n = 0;
        if (NPAD == 0 && scans) n = n_real[seg];            // (requested before the rows: one round trip less)
        // row indices in LDS, where the sums will stand
        int32_t* __restrict__ own_perm = reinterpret_cast<int32_t*>(sums);
        if constexpr (NPAD > 0) {
            constexpr int G = SPLIT_THREADS / SEGS, EPT = NPAD / G;
            static_assert(EPT >= 1 && EPT * G == NPAD && G >= kWave, "a row is sorted by whole wavefronts");
            int tseg = threadIdx.x % G;
            const int own = threadIdx.x / G;
            asm volatile("" : "+v"(tseg));                  // (or the network's lane masks would be kept across items, in spilled registers)
            const float* __restrict__ p = sorted + (size_t)min(seg0 + own, S - 1) * I;
            u64 v[EPT];
#pragma unroll
            for (int r = 0; r < EPT; ++r) {
                const int e = tseg * EPT + r;
                v[r] = ((u64)(e < I ? float_to_key(p[e]) : 0xffffffffu) << 32) | (uint32_t)e;
            }
            bitonic_sort<EPT, G>(v, tseg, reinterpret_cast<u64*>(wg) + own * NPAD);       // (the weights come later)
            int below = 0;
#pragma unroll
            for (int r = 0; r < EPT; ++r) {
                const int e = tseg * EPT + r;
                const bool real = e < I;
                const float f = key_to_float((uint32_t)(v[r] >> 32));
                below += real && f <= np.max_cmp;
                if (e < stride) {
                    xrows[own * stride + e] = real ? f : INFINITY;
                    own_perm[own * stride + e] = real ? (int32_t)(uint32_t)v[r] : 0;
                }
            }
#pragma unroll
            for (int d = 1; d < kWave; d <<= 1) below += __shfl_xor(below, d, kWave);
            if (lane == 0) k_found[wave][0] = below;
            __syncthreads();
            constexpr int ROW_WAVES = G / kWave;
            for (int q = 0; q < ROW_WAVES; ++q) n += k_found[row * ROW_WAVES + q][0];
            if (!scans) n = 0;
        }
        {
            // Weights in scan order: a thread keeps its column and takes four consecutive entries of a
            // row at a time (one 16-byte read of row indices, four weights, one 16-byte LDS write);
            // COLS neighbours read one row of W together.  All row indices of a thread are requested
            // first, then the sorted rows, then all its weights: two memory round trips for the usual
            // item.  (Offsets into W as 24-bit multiply-adds: the launcher checks that rows and row
            // pitch allow it.  Groups past the end repeat the last one.)
            constexpr int KSTEP = SPLIT_THREADS / COLS, GB = 13;
            const int gc = threadIdx.x % COLS, gk = threadIdx.x / COLS;
            const bool col_live = j0 + gc < J;
            const int groups = n_segs * stride / 4;        // stride is a multiple of 16 entries
            const int4* __restrict__ gp = reinterpret_cast<const int4*>(NPAD > 0 ? own_perm : perm + (size_t)seg0 * stride);
            const __amdgpu_buffer_rsrc_t wbuf = __builtin_amdgcn_make_buffer_rsrc(
                const_cast<float*>(w), 0, (int)((size_t)(I + np.bias) * J * sizeof(float)), 0x00020000);
            const unsigned pitch = (unsigned)J * 4u, col_bytes = (unsigned)(j0 + gc) * 4u;
            const int seg_skip = COLS * wstride - stride;  // from entry k of a column to entry k of the next segment
            float* __restrict__ wcol = wg + gc * wstride;
            auto weight = [&](int32_t r) {
                return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                                                     wbuf, __umul24((unsigned)r, pitch) + col_bytes, 0, 0));
            };
            int4 pv[GB];
            auto request_rows = [&](int g0) {
#pragma unroll
                for (int t = 0; t < GB; ++t) pv[t] = gp[min(g0 + t * KSTEP, groups - 1)];
            };
            request_rows(gk);
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (NPAD == 0) {
                const float4* __restrict__ gx = reinterpret_cast<const float4*>(sorted + (size_t)seg0 * stride);
                for (int e = threadIdx.x; e < groups; e += SPLIT_THREADS) reinterpret_cast<float4*>(xrows)[e] = gx[e];
            }
            for (int g0 = gk;;) {
                float4 wv[GB];
#pragma unroll
                for (int t = 0; t < GB; ++t)
                    wv[t] = col_live ? make_float4(weight(pv[t].x), weight(pv[t].y), weight(pv[t].z), weight(pv[t].w))
                                     : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll
                for (int t = 0; t < GB; ++t) {
                    const int f = 4 * min(g0 + t * KSTEP, groups - 1);
                    int sl = 0;
#pragma unroll
                    for (int q = 1; q < SEGS; ++q) sl += f >= q * stride;
                    *reinterpret_cast<float4*>(wcol + f + sl * seg_skip) = wv[t];
                }
                g0 += GB * KSTEP;
                if (g0 >= groups) break;
                request_rows(g0);
            }
            if (threadIdx.x == 0) progress = 0;
            if (threadIdx.x < SPLIT_ONES) ones[threadIdx.x] = 1.0f;
        }
        __syncthreads();                                    // rows and weights are in place

        const int n_full = n & ~(CHUNK - 1);

        float wsum = -np.theta, ysum = 0.0f, ya = 0.0f;
        bool fired0 = false;
        if (np.bias) {
            wsum += w_bias;
            ysum = np.biasvolt * w_bias;
            ya = wsum < 0.0f ? -ysum : ysum;
            fired0 = ya > fabsf(wsum) * np.biasvolt;
        }
        int k_close = NONE, consumed = 0;
        bool fired_end = false, failed = false;

        if (wave == 0) {
            // ---- producer -----------------------------------------------------------------------
            // Chunk c is consumed from buf[c % NBUF]; after it, chunk c + NBUF is read into its place.  With 32 lanes an item
            // has a lane per sum: the lower half of the wavefront forms ysum = fma(x, w, ysum), the upper wsum = fma(1, w, wsum),
            // eight instructions a chunk instead of sixteen (98 chunks: 5.8 -> 4.6 us; the testers take 6.1, and are now what is waited
            // for: dismissing chunks by the margin test, or fifteen testers, made the launch no shorter).
            constexpr int NBUF = SPLIT_ROUND;
            constexpr bool HALVES = LANES * 2 == kWave;
            const bool ones_half = HALVES && lane >= LANES;
            float acc = ones_half ? wsum : ysum;                        // ysum alone where a lane has both sums
            const float* xp = ones_half ? ones : xs;                    // the times of the round at work
            const int xp_step = ones_half ? 0 : NBUF * CHUNK;
            float bx[NBUF][CHUNK], bw[NBUF][CHUNK];
            auto fetch = [&](float (&v)[CHUNK], const float* q) {
                const float4 a = *reinterpret_cast<const float4*>(q), b = *reinterpret_cast<const float4*>(q + 4);
                v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
            };
            // Times by DPP, where the sixteen lanes of a row scan one segment: a register holds two chunks, a lane an input (an LDS
            // request costs a lone wavefront some 14 clocks: 4.5 instead of 6 a chunk).
            constexpr bool BY_ROW = HALVES && COLS >= 16;
            float rows[NBUF / 2];
            auto fetch_rows = [&](int h, const float* q) { rows[h] = q[h * 16 + lane % 16]; };
#pragma unroll
            for (int b = 0; b < NBUF; ++b) {
                fetch(bw[b], wrow + b * CHUNK);
                if (!BY_ROW) fetch(bx[b], xp + b * CHUNK);
                else if (b % 2 == 1) fetch_rows(b / 2, xp);
                asm volatile("" ::: "memory");              // (in the loop's order: it waits for what either way in has to wait for)
            }
            // chunks of this item: the longest row decides the counter's final value, the shortest how
            // long no lane needs a mask
            int n_full_max = n_full, n_full_min = scans ? n_full : NONE;
#pragma unroll
            for (int d = kWave / 2; d > 0; d >>= 1) {
                n_full_max = max(n_full_max, __shfl_xor(n_full_max, d, kWave));
                n_full_min = min(n_full_min, __shfl_xor(n_full_min, d, kWave));
            }
            n_full_max = __builtin_amdgcn_readfirstlane(n_full_max);
            n_full_min = __builtin_amdgcn_readfirstlane(n_full_min);
            // Order inside a phase: accumulate, store the sums, move the counter to the chunks before
            // this one, then issue the reads for a later chunk.  The counter is a relaxed store and is
            // not waited for: LDS serves a wavefront's requests in order, so the sums it covers, stored
            // a phase earlier, are in place before it.  Nothing moves across a phase boundary (the
            // compiler would otherwise wait for every outstanding request before each accumulation).
            // (`also`: the sum behind the chunk before, published along)
            auto publish = [&](int k, float also, bool pair) {
                asm volatile("" ::: "memory");
                float* out = sums + (k / CHUNK) * 2 * LANES;
                if (HALVES) {
                    out[lane ^ LANES] = pair ? also : acc;              // wsum first
                    if (pair) out[2 * LANES + (lane ^ LANES)] = acc;
                } else {
                    out[la] = wsum;
                    out[LANES + la] = acc;
                }
                asm volatile("" ::: "memory");
                __hip_atomic_store(&progress, k / CHUNK, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                asm volatile("" ::: "memory");
            };
            int k0 = 0;
            for (; k0 + NBUF * CHUNK <= n_full_min; k0 += NBUF * CHUNK) {
#pragma unroll
                for (int ph = 0; ph < NBUF; ++ph) {
                    const int k = k0 + ph * CHUNK;
                    __builtin_amdgcn_sched_barrier(0);
                    if constexpr (BY_ROW) {
                        if (ph % 2 == 0) {
                            accumulate_row<0>(acc, rows[ph / 2], bw[ph]);
                            const float behind_first = acc;
                            accumulate_row<8>(acc, rows[ph / 2], bw[ph + 1]);
                            publish(k, behind_first, true);
                            fetch(bw[ph], wrow + k + NBUF * CHUNK);
                            fetch(bw[ph + 1], wrow + k + (NBUF + 1) * CHUNK);
                            fetch_rows(ph / 2, xp + NBUF * CHUNK);
                        }
                    } else {
#pragma unroll
                        for (int u = 0; u < CHUNK; ++u) {
                            if (!HALVES) wsum += bw[ph][u];
                            acc = __fmaf_rn(bx[ph][u], bw[ph][u], acc);
                        }
                        publish(k, 0.0f, false);
                        fetch(bx[ph], xp + (NBUF + ph) * CHUNK);
                        fetch(bw[ph], wrow + k + NBUF * CHUNK);
                    }
                }
                xp += xp_step;
            }
            if (BY_ROW && k0 < n_full_max)
#pragma unroll
                for (int b = 0; b < NBUF; ++b) fetch(bx[b], xp + b * CHUNK);
            for (; k0 < n_full_max; k0 += NBUF * CHUNK) {
#pragma unroll
                for (int ph = 0; ph < NBUF; ++ph) {
                    const int k = k0 + ph * CHUNK;
                    const uint64_t run = __ballot(k < n_full);
                    int unused = 0;
                    float unused_sum = 0.0f;
                    __builtin_amdgcn_sched_barrier(0);
                    accumulate_chunk(HALVES ? unused_sum : wsum, acc, unused, run, bx[ph], bw[ph]);
                    publish(k, 0.0f, false);
                    fetch(bx[ph], xp + (NBUF + ph) * CHUNK);
                    fetch(bw[ph], wrow + k + NBUF * CHUNK);
                }
                xp += xp_step;
            }
            if (HALVES) {
                wsum = __shfl(acc, lane | LANES, kWave);
                ysum = __shfl(acc, la, kWave);
            } else {
                ysum = acc;
            }
            // the last chunk's sums: wait for them, then let the counter reach its final value
            __hip_atomic_store(&progress, (n_full_max + CHUNK - 1) / CHUNK, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
            // the trailing inputs, for a scan that no tester closes
            int kcnt = n_full;
            if (scans) {
                LaneState st;
                st.wsum = wsum; st.ysum = ysum; st.wa = fabsf(wsum);
                st.ya = wsum < 0.0f ? -ysum : ysum;
                st.fired = n_full > 0 ? st.ya > xs[n_full - 1] * st.wa : fired0;
                bool open = true;
                for (int k = n_full; k < n && open; ++k) {
                    open = scan_step(st, xs[k], wrow[k]);
                    if (open) ++kcnt;
                }
                if (!open) k_close = kcnt;
                fired_end = st.fired;
                wsum = st.wsum; ysum = st.ysum;
            }
            k_found[0][lane] = k_close;
            w_found[0][lane] = wsum;
            y_found[0][lane] = ysum;
            consumed = kcnt;                                // all n inputs when nothing closed
        } else {
            // ---- tester t of SPLIT_TESTERS: chunks t, t + SPLIT_TESTERS, ... --------------------------
            uint64_t closed = 0;
            float w_close = 0.0f, y_close = 0.0f;
            float yg = fired0 ? ya : INFINITY;
            float xc[CHUNK], wc[CHUNK], xn[CHUNK], wn[CHUNK];
            auto fetch = [&](float (&x)[CHUNK], float (&wv)[CHUNK], int k) {
                const float4 x0 = *reinterpret_cast<const float4*>(xs + k), x1 = *reinterpret_cast<const float4*>(xs + k + 4);
                const float4 w0 = *reinterpret_cast<const float4*>(wrow + k), w1 = *reinterpret_cast<const float4*>(wrow + k + 4);
                x[0] = x0.x; x[1] = x0.y; x[2] = x0.z; x[3] = x0.w; x[4] = x1.x; x[5] = x1.y; x[6] = x1.z; x[7] = x1.w;
                wv[0] = w0.x; wv[1] = w0.y; wv[2] = w0.z; wv[3] = w0.w; wv[4] = w1.x; wv[5] = w1.y; wv[6] = w1.z; wv[7] = w1.w;
            };
            int c = wave - 1;
            const int last_chunk = stride - CHUNK;
            fetch(xc, wc, c * CHUNK <= last_chunk ? c * CHUNK : 0);
            for (;; c += SPLIT_TESTERS) {
                const int k = c * CHUNK;
                const uint64_t run = __ballot(k < n_full) & ~closed;
                if (run == 0) break;                        // every lane closed here or past its inputs
                const int kn = k + SPLIT_TESTERS * CHUNK;
                fetch(xn, wn, kn <= last_chunk ? kn : 0);
                if (c > 0) {
                    // Bounded wait: if the sums never arrive the tester goes on with what is there and
                    // the result is marked invalid (no early exit: every wavefront reaches the barriers).
                    // The counter and the sums are requested together and waited for once: LDS serves
                    // a wavefront's requests in order, so sums read after a counter that had reached c
                    // are the finished ones; a poll that came too early is repeated as a whole.
                    int spins = 0;
                    const float* in = sums + (c - 1) * 2 * LANES;
                    float x_prev;
                    bool arrived;
                    for (;;) {
                        const int seen = __hip_atomic_load(&progress, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                        asm volatile("" ::: "memory");
                        wsum = in[la];
                        ysum = in[LANES + la];
                        x_prev = xs[k - 1];
                        asm volatile("" ::: "memory");
                        arrived = __builtin_amdgcn_readfirstlane(seen) >= c;
                        if (arrived || spins >= np.wait_polls) break;
                        __builtin_amdgcn_s_sleep(1);
                        ++spins;
                    }
                    failed |= !arrived;
                    ya = wsum < 0.0f ? -ysum : ysum;        // fired state after input k-1, from the sums
                    yg = ya > x_prev * fabsf(wsum) ? ya : INFINITY;
                }
                const uint64_t before = closed;
                int kc = k;
                scan_chunk_vector<true>(wsum, ysum, ya, yg, kc, closed, run, xc, wc);
                if (((closed & ~before) >> lane) & 1) { k_close = kc; w_close = wsum; y_close = ysum; }
#pragma unroll
                for (int u = 0; u < CHUNK; ++u) { xc[u] = xn[u]; wc[u] = wn[u]; }
            }
            if (failed && lane == 0) atomicAdd(&g_scan_giveups, 1u);
            k_found[wave][lane] = failed ? -1 : k_close;    // -1 poisons the result below
            w_found[wave][lane] = w_close;
            y_found[wave][lane] = y_close;
        }
        __syncthreads();
        if (wave == 0 && live) {
            int best = 0, kb = k_found[0][lane];
            bool bad = false;
#pragma unroll
            for (int v = 1; v < SPLIT_WAVES; ++v) {
                const int kv = k_found[v][lane];
                bad |= kv < 0;
                if (kv < kb) { kb = kv; best = v; }
            }
            // no close anywhere: the producer went through all n inputs, fired_end is the scan's
            const bool fired = kb != NONE || fired_end;
            const float ws = w_found[best][lane], ys = y_found[best][lane];
            float y = np.max_time, r = 0.0f;
            if (fired) {
                r = 1.0f / ws;
                y = ys * r;
                if (y >= np.max_time) { y = np.max_time; r = 0.0f; }
            }
            if (bad) y = r = __builtin_nanf("");            // a tester gave up waiting: make it visible
            const size_t o = (size_t)seg * J + j;
            y_out[o] = y;
            rcp_out[o] = r;
            if (copy.dst) copy.dst[time_copy_pixel(copy, seg) * J + j] = y;
            if (WANT_K) k_out[o] = (fired && r != 0.0f) ? (kb != NONE ? kb : consumed) : -1;
        }
        __syncthreads();                                    // LDS is reused by the next item
    }
}

template <int CH>
__device__ __forceinline__ void read_columns(const float* p, float (&out)[CH]) {
    if constexpr (CH == 1) {
        out[0] = *p;
    } else if constexpr (CH == 2) {
        const float2 v = *reinterpret_cast<const float2*>(p);
        out[0] = v.x; out[1] = v.y;
    } else {
        const float4 v = *reinterpret_cast<const float4*>(p);
        out[0] = v.x; out[1] = v.y; out[2] = v.z; out[3] = v.w;
    }
}
// The same through a pointer that is known to point into LDS.
typedef float lds_float2 __attribute__((ext_vector_type(2)));
typedef float lds_float4 __attribute__((ext_vector_type(4)));
template <int CH>
__device__ __forceinline__ void read_columns(__attribute__((address_space(3))) const float* p, float (&out)[CH]) {
    static_assert(CH == 1 || CH == 2 || CH == 4, "one, two or four columns per lane");
    if constexpr (CH == 1) {
        out[0] = *p;
    } else if constexpr (CH == 2) {
        const lds_float2 v = *reinterpret_cast<__attribute__((address_space(3))) const lds_float2*>(p);
        out[0] = v.x; out[1] = v.y;
    } else {
        const lds_float4 v = *reinterpret_cast<__attribute__((address_space(3))) const lds_float4*>(p);
        out[0] = v.x; out[1] = v.y; out[2] = v.z; out[3] = v.w;
    }
}

// ---------------------------------------------------------------------------------------------
// Scan with a margin filter: the tests of a step are skipped wherever they provably cannot close.
//
// With D_k = ysum_k - x_k * wsum_k (the state after input k), consuming input k+1 leaves D
// evaluated at x_{k+1} unchanged, and moving from x_k to x_{k+1} changes it by
// -(x_{k+1} - x_k) * wsum_k.  D starts positive (theta * x_0 > 0), rises while wsum < 0 (the
// neuron cannot have fired) and falls while wsum > 0: in exact arithmetic the causal set closes
// at the first step where D reaches zero.  In fp32 the reference's own tests (products rounded
// on their own, sign-corrected compares) can disagree with the sign of D only while |D| is
// within a few ulp of the quantities compared.  So a chunk of eight inputs only accumulates,
//     wsum += w ; ysum = fma(x, w, ysum),
// and is accepted as a whole if t_u = fma(-x_u, wsum_u, ysum_u) is known to lie above
//     thr = 4u * |ysum_end| + 36u * x_last * max|w|        (u = 2^-24)
// after each of its inputs (filter_chunk bounds the eight t from the last one, see there).
// If they all are above thr (and the chunk's first input is not negative) none of the
// reference's tests before the chunk's eight inputs can close the set:
//   * wsum_{k-1} > 0: closing before input k needs ysum_{k-1} <= x_k*wsum_{k-1}*(1+u); the sums
//     after input k differ from those before by the input and two roundings, which puts D_k
//     below u*(3.01*|ysum_k| + x_k*max|w|) / (1 - 2.01u);
//   * wsum_{k-1} < 0: closing needs the neuron fired after input k-1, i.e. D_{k-1} < u*x*|wsum|
//     <= u*(|ysum_{k-1}| + D_{k-1}) -- t of the step before (the last of the previous chunk for
//     the first step; a neuron that fired on its bias alone never takes the fast path);
//   * |ysum| anywhere in the chunk is at most 1.01*(|ysum_end| + 7*x_last*max|w|).
// The running sums are then exactly those of the step-by-step scan, and the fired state is a
// function of them.  A lane whose chunk fails the test keeps the sums it had before the chunk,
// records the chunk and sits out; after the loop every lane evaluates its recorded chunk with
// the reference's tests (the eight-step block above, fed per lane), which finds the close in
// all but contrived cases, and otherwise walks on step by step.  NaN sums never pass a
// reference test and never close; a NaN bound or threshold fails the fast test.
//
// CH (1, 2 or 4) adjacent neurons per lane: one row address, one input time and one 4-, 8- or 16-byte LDS read
// serve CH scans, and a wavefront covers 64*CH/COLS segments.  Two loops:
//   * the full chip (four neurons per lane; two with eight-column slices): what bounds it is vector issue (117
//     instructions per chunk of 4 x 64 neurons) and, under it, the power limit: the same instruction stream runs
//     16 % slower on random weights than on zeros.  3x3 patches of 64 channels to 64 neurons, 65 536 segments: 310 -> 238 us;
//     128 -> 128 channels on 28x28, 32 images: 472 -> 416; 256 -> 256 on 14x14: 555 -> 440; dense 784 -> 800 at 4096 rows: 379 -> 302,
//     and with the shorter test and evenly dealt items 270;
//   * few wavefronts (LONE: one neuron per lane, two with slices of sixteen columns and more): a SIMD has a wavefront or
//     three, and each pays about 4.3 clocks for an instruction whatever it is.  52 instructions per chunk of 64 neurons
//     instead of 75: broadcasts as operands, the test's operands computed once per block of four chunks in the lanes that hold
//     it, end-of-row masks folded into them, decisions taken half a chunk later, entries kept in a ring without moves.
//     98 chunks of a lone wavefront 15.2 -> 10.9 us; whole launches: 784 -> 800 at 16 / 128 / 256 rows 24.2 / 28.0 / 38.2 -> 19.2 / 23.5 /
//     34.0; 2048 -> 512 at 16 rows 48.4 -> 36.6; 49 patches of 4608 -> 512 122 -> 88; 196 of 2304 -> 256 63 -> 49.  (Sixteen-byte
//     weight reads transposed between lane groups by permlane swaps: 29 us for the first; a swap costs 8.4 clocks.)
// ---------------------------------------------------------------------------------------------
// The fast loop does not evaluate the eight t of a chunk: it bounds them from the last one.  With the
// sums as computed, D_u = ysum_u - x_u*wsum_u obeys  D_{u-1} = D_u + (x_u - x_{u-1})*wsum_{u-1} - e_u,
// |e_u| <= u*(|ysum_u| + x_u*|wsum_u|) (the roundings of the two sums), hence for every u of the chunk
//     D_u >= D_7 + (x_7 - x_0) * min(0, wsum_0 .. wsum_7) - 7 * max|e|:
// D only falls while the weight sum is positive, and where the sum is negative it can have been lower
// earlier by at most that much.  The smallest weight sum of the chunk is not tracked but bounded from its
// two ends: none of the eight sums lies more than four weights below both, so with W = max|w| of the slice
//     min(0, wsum_0 .. wsum_7) >= min(wsum_start, wsum_7, 4W) - 4W
// (up to four roundings of a sum).  The lane evaluates t_7 and accepts the chunk if
//     fma(x_7 - x_0, min(wsum_start, wsum_7, 4W), t_7)  >  thr + (x_7 - x_0)*4W
//                                                         + 17u * 1.01 * (|ysum_7| + x_7*|wsum_7| + 18*x_7*W)
// (the last term covers the seven e_u, the roundings of the weight sums, of t_u, t_7, x_7 - x_0 and of the
// bound itself; sums inside the chunk differ from the final ones by at most seven inputs).  Every t_u then
// exceeds thr, which is the condition above.  With weight sums that stay above 4W the bound is t_7 itself;
// below, a chunk may fail although none of its inputs closes the set, by (x_7 - x_0)*4W at most.
// Two additions per input and seven vector instructions per chunk and neuron (two multiply-adds, a minimum, the compare and three
// selects), five per chunk for the operands they share.
//
// That slack is small next to ysum - x*wsum, which starts at theta*x, where weights are small and the sum soon leaves zero;
// under weights of a larger spread (the layers' own initialiser: mean 0, deviation sqrt(15 / inputs)) it stops most scans several
// times each, and every stop costs steps and another pass over the row.  There (TIGHT) the smallest weight sum of the chunk is
// tracked, one three-way minimum per two inputs, and the lane accepts if
//     fma(x_7 - x_0, min(0, wsum_0 .. wsum_7), t_7)  >  thr + the last term above.
// A workgroup decides by the largest weight of its slice, next to the threshold that ysum - x*wsum starts from; where
// a wavefront has a single item nothing hides the extra passes, and the line lies lower.  us, bounded / tracked (W / theta),
// weights of mean 4 / I and standard deviation s / sqrt(I):
//                                          s = 1             s = 1.5           s = 2             s = 3             s = 3.87
//   784 -> 800, 4096 rows            334 / 346 (0.19)  336 / 348 (0.28)  351 / 340 (0.36)  430 / 352 (0.55)  507 / 356 (0.70)
//   65 536 patches of 576, 64        230 / 252 (0.19)  238 / 252 (0.28)  260 / 254 (0.38)  342 / 262 (0.56)  448 / 288 (0.72)
//   401 408 patches of 147, 64       605 / 611 (0.35)  643 / 571 (0.51)  762 / 549 (0.68) 1278 / 555 (1.00) 1674 / 585 (1.28)
//   25 088 patches of 1152, 128      424 / 454 (0.13)  423 / 455 (0.20)  447 / 457 (0.26)  487 / 459 (0.39)  563 / 466 (0.51)
//   1568 patches of 4608, 512        652 / 656 (0.08)  656 / 662 (0.12)  656 / 660 (0.16)  672 / 667 (0.24)  692 / 679 (0.30)
//   784 -> 800, 256 rows              40 / 41  (0.19)   46 / 42  (0.28)   53 / 45  (0.36)   65 / 48  (0.55)   86 / 50  (0.70)
//   784 patches of 1152, 128          37 / 38  (0.13)   42 / 38  (0.20)   51 / 41  (0.26)   56 / 47  (0.39)   61 / 52  (0.51)
constexpr float TIGHT_FROM = 0.36f, TIGHT_FROM_SINGLE = 0.2f;
constexpr float FILTER_END_Y = 0x1p-19f;                  // 32u >= 4u + 17.2u, times |ysum_7|
constexpr float FILTER_END_XW = 0x1p-19f;                 // 32u >= 17.2u, times x_7 * |wsum_7|
constexpr float FILTER_END_W = 0x1p-15f;                  // 512u >= 36u + 310u, times x_7 * max|w| of the slice
// The fast test takes the first two terms into its operands: t_7 is evaluated at x_7 * (1 + 64u), and x_7 - x_0 is
// enlarged by 256u * x_7.  With A = 4W - min(..) >= 0 (tracked form: -min(0, ..)), passing means
// t' - dx' * A > 512u * x_7 * W, and with T = ysum_7 - x_7 * wsum_7 and dx = x_7 - x_0 <= x_7
//   wsum_7 >= 0:  T >= (1 - u) t' + 62.9u * x_7 * wsum_7 and dx' * A >= (1 + 128u) dx * A, so
//                 T - dx * A >= 126u * t' + 62.9u * x_7 * wsum_7 + 510u * x_7 * W;
//   wsum_7 < 0:   T >= (1 - u) t' - 65.2u * x_7 * |wsum_7|, and A >= |wsum_7|, so dx' * A >= (1 + 64u) dx * A +
//                 192u * x_7 * |wsum_7| and T - dx * A >= 62u * t' + 125u * x_7 * |wsum_7| + 510u * x_7 * W;
// both are above 21.2u * |ysum_7| + 17.2u * x_7 * |wsum_7| + 346u * x_7 * W, since |ysum_7| <= T + x_7 * |wsum_7|.  (What is
// left covers the roundings of t', dx', the bound and the threshold.)  Two vector instructions per neuron and chunk
// less than with a threshold of the neuron's own: 65 536 segments of 576 to 64 neurons 276 -> 265 us, 784 -> 800 at
// 4096 rows 368 -> 341, 6272 segments of 2304 to 256 neurons 423 -> 405 (kernel traces on one card).
constexpr float FILTER_AT = 1.0f + 0x1p-18f;
constexpr float FILTER_DX = 0x1p-16f;

// The test of a round: the same bound over 32 inputs at a time.  None of 32 sums lies more than sixteen weights below both ends, so
// with A = 16W - min(wsum_start, wsum_31, 16W) the scan passes if t' - dx' * A > 4096u * x_31 * W, t' evaluated at x_31 * (1 + 256u)
// and dx' = x_31 - x_0 + 1024u * x_31.  What a test of the reference inside the round needs is (31 roundings of the two sums,
// sixteen of a weight sum and six of the bound's own, sums that differ from the last ones by up to 31 inputs; compare thr above)
//   T - dx * A > 57.6u * |ysum_31| + 53.6u * x_31 * |wsum_31| + 3665u * x_31 * W,   |ysum_31| <= T + x_31 * |wsum_31|;
// the same two cases as above leave
//   wsum_31 >= 0:  T - dx * A >= 500u * t' + 254u * x_31 * wsum_31 + 4090u * x_31 * W,
//   wsum_31 < 0:   T - dx * A >= 500u * t' + 252u * x_31 * |wsum_31| + 4090u * x_31 * W.
constexpr float ROUND_END_W = 0x1p-12f;                   // 4096u
constexpr float ROUND_AT = 1.0f + 0x1p-16f;               // 1 + 256u
constexpr float ROUND_DX = 0x1p-14f;                      // 1024u
// A wavefront's scans are tested by rounds until the first of them comes close to its close, about half of a row where 64 ... 256 of
// them share a wavefront (the first closes at 0.50 ... 0.57 of a row, the mean at 0.80): a round is 363 vector instructions
// instead of 467.  us without / with: 4096 rows of 784 to 800 neurons 260 / 243, 25 088 segments of 1152 to 128 350 / 335, 6272 of 2304 to 256
// 396 / 374, 65 536 of 576 to 64 (staged) 222 / 211; from 400 inputs on: 131 072 segments of 288 to 32 164 / 173, 32 768 of 288 to 64 64.7 / 67.1,
// 2048 rows of 300 to 800 61.9 / 62.4, since a wavefront fills its pipeline a second time when it goes over to chunks.  16W * 32 / I is about
// the slack of a round next to a threshold of one; beyond 0.6 of it rounds end early (576 inputs with deviation 3.87 / sqrt(I): at 0.15 of a row).
constexpr float ROUNDS_UP_TO = 0.6f;
constexpr int ROUNDS_FROM = 400;
// Few wavefronts (LONE): 53 instructions a chunk instead of 64, 37 of them vector and LDS ones instead of 51, with the decision once per turn of
// the entries' ring, whose requests and weights go on into the chunks behind.  A wavefront fetches a second loop of some 3 KB of code for it, so only the rows of slices of
// eight columns are long enough: 2560 inputs and more, or from here on layers of at most eight neurons (us of the layer without / with: 49 segments of
// 4608 to 512 95 / 86, 49 of 2560 to 512 60 / 55, 200 of 3000 to 300 87 / 80, 300 of 1280 to 8 35 / 33, 1000 of 1280 to 8 36.4 / 34.9, 600 of 1400 to 5 38 / 36,
// 3000 of 2300 to 8 86 / 82; of the scan, deviation 3.87 / sqrt(I), 49 of 4608 to 512 109 / 102, 100 of 4096 to 256 87 / 80, 200 of 3000 to 300
// 136 / 134; sixteen columns, 16 of 2048 to 512 33.9 / 35.0, 100 of 2400 to 64 38.6 / 40.4, 128 of 1521 to 500 32.1 / 33.0).
constexpr int LONE_ROUNDS_FROM = 1280;

// The test of a chunk for one scan of every lane: wb, yb are the sums behind it.  Lanes in the mask `open`
// that pass take them over; open lanes that fail keep the sums from before the chunk, take the chunk's
// first index as kcur and leave `open`.  The arithmetic does not depend on EXEC or branches (lanes that
// are not open compute along and discard), so the compiler is free to interleave it with the LDS traffic
// of the next chunk; the decision works on lane masks in scalar registers.
// x7e = FILTER_AT * x[7], dx = x[7] - x[0] + FILTER_DX * x[7], thr = FILTER_END_W * W * x[7] (+ dx * 4W where the smallest weight
// sum is bounded), low: the smallest weight sum or zero, or its bound + 4W.
__device__ __forceinline__ void filter_test(float& wsum, float& ysum, int& kcur, uint64_t& open, int k, float wb, float yb,
                                            float x7e, float thr, float dx, float low) {
    const float bound = __fmaf_rn(dx, low, __fmaf_rn(-x7e, wb, yb));
    uint64_t stop;
    // (two statements: the first has scalar results only, so the masks stay uniform values for the compiler
    // also where no branch depends on them)
    asm("v_cmp_gt_f32_e32 vcc, %[m], %[thr]\n"                       // pass: false for NaN on either side
        "s_andn2_b64 %[stop], %[open], vcc\n"
        "s_and_b64 %[open], %[open], vcc\n"
        : [open] "+s"(open), [stop] "=&s"(stop)
        : [m] "v"(bound), [thr] "v"(thr)
        : "vcc", "scc");
    asm("v_cndmask_b32_e64 %[ws], %[ws], %[wb], %[open]\n"
        "v_cndmask_b32_e64 %[ys], %[ys], %[yb], %[open]\n"
        "v_cndmask_b32_e64 %[kf], %[kf], %[vk], %[stop]\n"
        : [ws] "+v"(wsum), [ys] "+v"(ysum), [kf] "+v"(kcur)
        : [open] "s"(open), [stop] "s"(stop), [wb] "v"(wb), [yb] "v"(yb), [vk] "v"(k));
}

// Whether a scan that has consumed k > 0 inputs, with a positive weight sum ws and not fired, is certain never to
// fire on the inputs [k, n) of its row.  Called by the whole wavefront with uniform
// arguments; wcol is the scan's column of the slice.  depth = ysum - x*ws behind the last input consumed.
// While the weight sum stays positive, ysum - x*wsum only falls, up to the roundings of the two sums, and the
// reference's `fired` test is false as long as it is negative.  The running weight sums are formed here in
// another order (64 inputs at a time by a wavefront scan), so they and the depth have to keep a margin.  With
// m = n - k, M the largest and T the sum of absolute values of the weights seen, u = 2^-24:
//   the reference's weight sums differ from the true ones by at most m*u*M', M' their largest absolute value, and
//   those formed here by at most u*(6T + (m/64 + 1)*M');
//   every step moves ysum - x*wsum by at most u*(|ysum| + x*|wsum|) more than it should, and
//   |ysum| <= |depth| + 2*x_last*M'.
// (Factors rounded up generously: the margins are of the order of 1e-3.)
template <int COLS>
__device__ bool never_fires(const float* __restrict__ xs, const int32_t* __restrict__ pr, const float* __restrict__ wcol, int k,
                            int n, float ws, float ys, int lane) {
    const float depth = __fmaf_rn(-xs[k - 1], ws, ys);
    constexpr int BATCH = 4;                                        // wavefronts of inputs whose rows are requested together
    float carry = ws, low = ws, high = ws, total = 0.0f;
    for (int base = k; base < n; base += BATCH * kWave) {
        float wt[BATCH];
        int row[BATCH];
#pragma unroll
        for (int b = 0; b < BATCH; ++b) row[b] = base + b * kWave + lane < n ? pr[base + b * kWave + lane] : -1;
#pragma unroll
        for (int b = 0; b < BATCH; ++b) wt[b] = row[b] >= 0 ? wcol[row[b] * COLS] : 0.0f;
#pragma unroll
        for (int b = 0; b < BATCH; ++b) {
            float s = wt[b];
            total += fabsf(s);
#pragma unroll
            for (int d = 1; d < kWave; d <<= 1) {
                const float up = __shfl_up(s, d, kWave);
                s += lane >= d ? up : 0.0f;
            }
            s += carry;
            low = fminf(low, s);
            high = fmaxf(high, s);
            carry = __shfl(s, kWave - 1, kWave);
        }
    }
#pragma unroll
    for (int d = kWave / 2; d > 0; d >>= 1) {
        low = fminf(low, __shfl_xor(low, d, kWave));
        high = fmaxf(high, __shfl_xor(high, d, kWave));
        total += __shfl_xor(total, d, kWave);
    }
    const float u = 0x1p-24f * 1.1f, m = (float)(n - k + 64), x_last = xs[n - 1];
    const float low_margin = u * (1.02f * m * high + 8.0f * total);
    const float depth_margin = u * m * (3.0f * x_last * high + fabsf(depth)) * 1.1f;
    return low > low_margin && depth < -depth_margin && total < INFINITY;
}

// Largest of the threads' `m` over the workgroup, the same value in every thread.  `red` is room for
// one float per wavefront; the call contains the workgroup barrier that also publishes whatever the
// threads wrote to LDS before it.
__device__ __forceinline__ float block_max(float m, float* __restrict__ red) {
#pragma unroll
    for (int d = kWave / 2; d > 0; d >>= 1) m = fmaxf(m, __shfl_xor(m, d, kWave));
    if (threadIdx.x % kWave == 0) red[threadIdx.x / kWave] = m;
    __syncthreads();
    const int waves = blockDim.x / kWave;
    float r = red[0];
    for (int v = 1; v < waves; ++v) r = fmaxf(r, red[v]);
    return r;
}

// Value of `v` in lane 4*(lane/4) + q: a quad broadcast, which the hardware applies as an operand
// modifier (DPP) of the move or of the VOP2 instruction that consumes it.
template <int Q>
__device__ __forceinline__ float quad_broadcast(float v) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), Q * 0x55, 0xf, 0xf, true));
}

// LDS addresses of the four weight rows whose (shifted) indices lanes 2*HALF and 2*HALF + 1 of the quad
// hold, two each: adds that take the broadcast as an operand modifier.  (The two idle cycles are what a
// DPP read of a register written by the instruction before it needs.)
template <int HALF>
__device__ __forceinline__ void quad_row_addresses(int even, int odd, unsigned base, unsigned (&a)[4]) {
    if constexpr (HALF == 0)
        asm("s_nop 1\n"
            "v_add_u32_dpp %[a0], %[e], %[base] quad_perm:[0,0,0,0] row_mask:0xf bank_mask:0xf bound_ctrl:1\n"
            "v_add_u32_dpp %[a1], %[o], %[base] quad_perm:[0,0,0,0] row_mask:0xf bank_mask:0xf bound_ctrl:1\n"
            "v_add_u32_dpp %[a2], %[e], %[base] quad_perm:[1,1,1,1] row_mask:0xf bank_mask:0xf bound_ctrl:1\n"
            "v_add_u32_dpp %[a3], %[o], %[base] quad_perm:[1,1,1,1] row_mask:0xf bank_mask:0xf bound_ctrl:1\n"
            : [a0] "=&v"(a[0]), [a1] "=&v"(a[1]), [a2] "=&v"(a[2]), [a3] "=&v"(a[3])
            : [e] "v"(even), [o] "v"(odd), [base] "v"(base));
    else
        asm("s_nop 1\n"
            "v_add_u32_dpp %[a0], %[e], %[base] quad_perm:[2,2,2,2] row_mask:0xf bank_mask:0xf bound_ctrl:1\n"
            "v_add_u32_dpp %[a1], %[o], %[base] quad_perm:[2,2,2,2] row_mask:0xf bank_mask:0xf bound_ctrl:1\n"
            "v_add_u32_dpp %[a2], %[e], %[base] quad_perm:[3,3,3,3] row_mask:0xf bank_mask:0xf bound_ctrl:1\n"
            "v_add_u32_dpp %[a3], %[o], %[base] quad_perm:[3,3,3,3] row_mask:0xf bank_mask:0xf bound_ctrl:1\n"
            : [a0] "=&v"(a[0]), [a1] "=&v"(a[1]), [a2] "=&v"(a[2]), [a3] "=&v"(a[3])
            : [e] "v"(even), [o] "v"(odd), [base] "v"(base));
}

// The pieces of the fast loop for few wavefronts.  Every instruction costs such a wavefront about 4.3 clocks, whatever it is and
// whatever it depends on, except that a lane mask that goes from the vector to the scalar side and back in consecutive
// instructions costs 16 more.  So broadcasts are operands (DPP) and not moves, and the decision on a chunk is taken in the
// middle of the next one.  (What lanes read from others -- xe, xo, even, odd and the test's nx, dx, thr -- passes through a
// volatile statement with two wait states behind the last write, which a DPP read needs.)
//
// DPP control "lane N of the row of sixteen" or "lane N of the quad".
#define SNNTC_BCAST_ROW "row_newbcast:%[n] row_mask:0xf bank_mask:0xf bound_ctrl:1\n"
#define SNNTC_BCAST_ROW1 "row_newbcast:%[n1] row_mask:0xf bank_mask:0xf bound_ctrl:1\n"
#define SNNTC_BCAST_AT "row_newbcast:%[m] row_mask:0xf bank_mask:0xf bound_ctrl:1\n"
#define SNNTC_BCAST_AT1 "row_newbcast:%[m1] row_mask:0xf bank_mask:0xf bound_ctrl:1\n"
#define SNNTC_BCAST_QUAD "quad_perm:[%[n],%[n],%[n],%[n]] row_mask:0xf bank_mask:0xf bound_ctrl:1\n"
#define SNNTC_BCAST_QUAD1 "quad_perm:[%[n1],%[n1],%[n1],%[n1]] row_mask:0xf bank_mask:0xf bound_ctrl:1\n"
#define SNNTC_BCAST_QAT "quad_perm:[%[m],%[m],%[m],%[m]] row_mask:0xf bank_mask:0xf bound_ctrl:1\n"
#define SNNTC_BCAST_QAT1 "quad_perm:[%[m1],%[m1],%[m1],%[m1]] row_mask:0xf bank_mask:0xf bound_ctrl:1\n"

// Four inputs of a scan: s[0..3] the weight sums behind them, ys the other sum; the times are those that lanes N and N + 1 hold.
#define SNNTC_HALF(B, B1)                                                                                              \
    "v_add_f32_e32 %[s0], %[ws], %[w0]\n" "v_fmac_f32_dpp %[ys], %[xe], %[w0] " B                                      \
    "v_add_f32_e32 %[s1], %[s0], %[w1]\n" "v_fmac_f32_dpp %[ys], %[xo], %[w1] " B                                      \
    "v_add_f32_e32 %[s2], %[s1], %[w2]\n" "v_fmac_f32_dpp %[ys], %[xe], %[w2] " B1                                     \
    "v_add_f32_e32 %[s3], %[s2], %[w3]\n" "v_fmac_f32_dpp %[ys], %[xo], %[w3] " B1
template <bool BY_ROW, int N>
__device__ __forceinline__ void accumulate_half(float ws, float (&s)[4], float& ys, float xe, float xo, const float (&w)[4]) {
#define SNNTC_HALF_OPERANDS                                                                                            \
    : [s0] "=&v"(s[0]), [s1] "=&v"(s[1]), [s2] "=&v"(s[2]), [s3] "=&v"(s[3]), [ys] "+v"(ys)                            \
    : [ws] "v"(ws), [xe] "v"(xe), [xo] "v"(xo), [w0] "v"(w[0]), [w1] "v"(w[1]), [w2] "v"(w[2]), [w3] "v"(w[3]),        \
      [n] "n"(N), [n1] "n"(N + 1)
    if constexpr (BY_ROW) asm(SNNTC_HALF(SNNTC_BCAST_ROW, SNNTC_BCAST_ROW1) SNNTC_HALF_OPERANDS);
    else asm(SNNTC_HALF(SNNTC_BCAST_QUAD, SNNTC_BCAST_QUAD1) SNNTC_HALF_OPERANDS);
}
// LDS addresses of the four weight rows whose shifted indices lanes M and M + 1 hold.
#define SNNTC_ADDRESSES(B, B1)                                                                                         \
    "v_add_u32_dpp %[a0], %[e], %[base] " B "v_add_u32_dpp %[a1], %[o], %[base] " B                                    \
    "v_add_u32_dpp %[a2], %[e], %[base] " B1 "v_add_u32_dpp %[a3], %[o], %[base] " B1
template <bool BY_ROW, int M>
__device__ __forceinline__ void weight_addresses(unsigned (&a)[4], unsigned even, unsigned odd, unsigned base) {
#define SNNTC_ADDRESS_OPERANDS                                                                                         \
    : [a0] "=&v"(a[0]), [a1] "=&v"(a[1]), [a2] "=&v"(a[2]), [a3] "=&v"(a[3])                                           \
    : [e] "v"(even), [o] "v"(odd), [base] "v"(base), [m] "n"(M), [m1] "n"(M + 1)
    if constexpr (BY_ROW) asm(SNNTC_ADDRESSES(SNNTC_BCAST_AT, SNNTC_BCAST_AT1) SNNTC_ADDRESS_OPERANDS);
    else asm(SNNTC_ADDRESSES(SNNTC_BCAST_QAT, SNNTC_BCAST_QAT1) SNNTC_ADDRESS_OPERANDS);
}
// Whether a chunk passes (see filter_test): ysum - thr - x7e * wsum + dx * low > 0.  (Taking thr off first adds
// u * (|ysum| + thr) to the roundings, which the margins above leave room for.)  The operands of chunk P are those of lane 4 * P
// of the row (BY_ROW) or the lane's own.
// (BY_ROW: one statement, since between two the compiler puts a wait state; its vector is v127, the last that a wavefront of a
// workgroup of 16 has, because with a vector among its results the mask would count as divergent.  3136 and 6272 patches of 576 to
// 64 neurons 26.7 -> 26.7 and 41.4 -> 40.0 us, 128 rows of 512 to 1000 19.3 -> 18.6.)
template <bool BY_ROW, int P>
__device__ __forceinline__ uint64_t chunk_passes(float wb, float yb, float nx, float dx, float thr, float low) {
    uint64_t pass;
    if constexpr (BY_ROW) {
        asm("v_subrev_f32_dpp v127, %[thr], %[yb] " SNNTC_BCAST_ROW "v_fmac_f32_dpp v127, %[nx], %[wb] " SNNTC_BCAST_ROW
            "v_fmac_f32_dpp v127, %[dx], %[low] " SNNTC_BCAST_ROW "v_cmp_lt_f32_e64 %[pass], 0, v127\n"              // false for NaN
            : [pass] "=s"(pass) : [thr] "v"(thr), [yb] "v"(yb), [nx] "v"(nx), [wb] "v"(wb), [dx] "v"(dx), [low] "v"(low), [n] "n"(4 * P)
            : "v127");
    } else {
        const float t = __fmaf_rn(dx, low, __fmaf_rn(nx, wb, yb - thr));
        asm("v_cmp_lt_f32_e64 %[pass], 0, %[t]" : [pass] "=s"(pass) : [t] "v"(t));
    }
    return pass;
}

typedef __attribute__((address_space(3))) const float lds_cfloat;

// f(integral_constant<int, 0>), f(<1>), ... f(<N-1>) until one returns false; true if none did.  The
// phase number reaches f as a type, so ring slots and buffers stay compile-time register choices.
template <class F, int... PH>
__device__ __forceinline__ bool for_each_phase_impl(F&& f, std::integer_sequence<int, PH...>) {
    return (f(std::integral_constant<int, PH>{}) && ...);
}
template <int N, class F>
__device__ __forceinline__ bool for_each_phase(F&& f) {
    return for_each_phase_impl(f, std::make_integer_sequence<int, N>{});
}

// The lane's CH columns of an output row, `left` of which exist; one wide store where rows keep the alignment.
template <int CH>
__device__ __forceinline__ void store_columns(float* __restrict__ p, const float (&v)[CH], int left, int pitch) {
    if constexpr (CH == 4) {
        if ((pitch & 3) == 0 && (reinterpret_cast<uintptr_t>(p) & 15) == 0) {
            if (left > 0) *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]);
            return;
        }
    }
#pragma unroll
    for (int c = 0; c < CH; ++c)
        if (c < left) p[c] = v[c];
}

__device__ __forceinline__ uint64_t ballot(bool b) { return __builtin_amdgcn_ballot_w64(b); }
// Whether the lane's bit is set in a lane mask.
__device__ __forceinline__ bool in_mask(uint64_t m) { return __builtin_amdgcn_inverse_ballot_w64(m); }

// Value v of lane N of the lane's row of sixteen, in every lane of the row.
template <int N>
__device__ __forceinline__ float row_broadcast(float v) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x150 + N, 0xf, 0xf, true));
}
// LDS addresses of the four weight rows whose shifted indices lanes N and N + 1 of the row of sixteen hold.
template <int N>
__device__ __forceinline__ void row_row_addresses(int even, int odd, unsigned base, unsigned (&a)[4]) {
    asm("s_nop 1\n"
        "v_add_u32_dpp %[a0], %[e], %[base] row_newbcast:%[n0] row_mask:0xf bank_mask:0xf bound_ctrl:1\n"
        "v_add_u32_dpp %[a1], %[o], %[base] row_newbcast:%[n0] row_mask:0xf bank_mask:0xf bound_ctrl:1\n"
        "v_add_u32_dpp %[a2], %[e], %[base] row_newbcast:%[n1] row_mask:0xf bank_mask:0xf bound_ctrl:1\n"
        "v_add_u32_dpp %[a3], %[o], %[base] row_newbcast:%[n1] row_mask:0xf bank_mask:0xf bound_ctrl:1\n"
        : [a0] "=&v"(a[0]), [a1] "=&v"(a[1]), [a2] "=&v"(a[2]), [a3] "=&v"(a[3])
        : [e] "v"(even), [o] "v"(odd), [base] "v"(base), [n0] "n"(N), [n1] "n"(N + 1));
}

template <int COLS, int CH, bool LONE, bool WANT_K, bool ROUNDS = false, bool STAGED = false>
__global__ void __launch_bounds__(LDS_SCAN_THREADS)
scan_filter_kernel(const float* __restrict__ sorted, const int32_t* __restrict__ perm,
                   const int32_t* __restrict__ n_real, const float* __restrict__ w, float* __restrict__ y_out,
                   float* __restrict__ rcp_out, int32_t* __restrict__ k_out, int S, int I, int stride, int J,
                   int n_slices, int n_groups, int waves, NeuronParams np, TimeCopy copy) {
    extern __shared__ __align__(16) float wl[];                          // [I][COLS], then block_max's room, which the rows' staging reuses
    constexpr int LANES = COLS / CH;                       // lanes per segment
    constexpr int SEGS = kWave / LANES;                    // segments per wavefront
    static_assert(LANES % 4 == 0, "the four lanes of a quad belong to one segment");
    // How a segment's (x, row) entries reach its lanes (see the fast loop): through rows of sixteen lanes where
    // a segment has at least that many, else through quads
    constexpr bool BY_ROW = LANES % 16 == 0;
    constexpr int ROUND = 4;                               // chunks per round of the fast loop
    const int block = xcd_contiguous(blockIdx.x, gridDim.x);
    const int slice = block / n_groups;
    const int group = block - slice * n_groups;
    const int j0 = slice * COLS;
    // the slice, and the largest |w| in it (the threads' shares of the copy, then the workgroup's)
    const float w_max = block_max(fill_weight_slice<COLS>(wl, w, I, J, j0), wl + I * COLS);
    if constexpr (STAGED) __syncthreads();                  // (the room of the maximum is the rows' staging next)
    const float end_w = FILTER_END_W * w_max;               // margin of the fast loop
    const float w4 = 4.0f * 1.00001f * w_max;               // 4W of its bound on the weight sums
    const float end_w_round = ROUND_END_W * w_max;
    const bool by_rounds = __builtin_amdgcn_readfirstlane(w_max * 512.0f <= ROUNDS_UP_TO * np.theta * (float)I);
    const bool single = (S + SEGS - 1) / SEGS <= n_groups * waves;      // a wavefront has one item
    const bool tight = __builtin_amdgcn_readfirstlane(w_max > (single ? TIGHT_FROM_SINGLE : TIGHT_FROM) * np.theta);

    constexpr int NONE = 0x7fffffff;
    constexpr int ROW_SHIFT = COLS == 64 ? 8 : COLS == 32 ? 7 : COLS == 16 ? 6 : 5;      // a weight row is COLS * 4 bytes
    static_assert(COLS == 64 || COLS == 32 || COLS == 16 || COLS == 8, "slice width");

    auto scan_items = [&](auto tight_c) {                   // the rest of the kernel, in both forms
    constexpr bool TIGHT = decltype(tight_c)::value;
    const int lane = threadIdx.x % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int sub = lane / LANES, cg = lane - sub * LANES;
    const int j = j0 + CH * cg;                            // first of the lane's columns
    const float* __restrict__ wcol = wl + CH * cg;
    const unsigned wbase = (unsigned)(uintptr_t)(lds_cfloat*)wcol;          // LDS byte address of the lane's columns
    // `waves` wavefronts of the workgroup work on items; the others have only helped to copy the slice.  A group takes
    // neighbouring items where they fill its SIMDs evenly.  Otherwise (several turns, or one that fills 13 of 16 wavefronts or
    // fewer) they are dealt out one by one, so that no group has a wavefront more per SIMD than it must (1536 rows of 784 -> 800
    // 154 -> 122 us, 200 704 patches of 147 to 64 neurons 243 -> 232, 392 of 4608 to 512 200 -> 166).
    const int n_items = (S + SEGS - 1) / SEGS;
    const bool deal = n_items > n_groups * waves || (waves == 16 && n_items <= n_groups * 13);
    for (int item = deal ? wave * n_groups + group : group * waves + wave; wave < waves && item * SEGS < S; item += n_groups * waves) {
        const int seg_raw = item * SEGS + sub;
        const int seg = seg_raw < S ? seg_raw : S - 1;      // idle lanes shadow a valid segment
        const float* __restrict__ xs = sorted + (size_t)seg * stride;
        const int32_t* __restrict__ pr = perm + (size_t)seg * stride;
        const int seg0 = __builtin_amdgcn_readfirstlane(item * SEGS);
        const int n_segs = S - seg0 < SEGS ? S - seg0 : SEGS;
        const RowSource rows_of_item = make_row_source(sorted + (size_t)seg0 * stride, perm + (size_t)seg0 * stride,
                                                       n_segs * stride * (int)sizeof(float));
        const int lane_bytes = ((seg - seg0) * stride + 2 * (lane & (BY_ROW ? 15 : 3))) * (int)sizeof(float);
        const int n_seg = n_real[seg];
        const float first_x = xs[0];
        // The (x, row) stream of a segment is the same for all its lanes.  If every lane fetched the eight
        // entries of a chunk itself, a wavefront would move four kilobytes per chunk through the vector
        // memory path, which then bounds the kernel.  Instead a lane fetches two entries of both arrays with
        // two 8-byte buffer loads that need no address arithmetic, and a value reaches the other lanes as a DPP
        // broadcast: free for the row offsets, which enter the LDS address through an add that takes the
        // broadcast as an operand modifier, one move per input time (shared by the lane's CH scans).  Sixteen
        // lanes of one segment hold a whole round of four chunks, so a round takes one pair of loads; a quad
        // holds one chunk, and every chunk takes one.  (Requests past the end of a row return the next row of
        // the item, past the last one zeros: the buffer descriptor ends with the item.  Nothing uses them.)
        //
        // held: rows: block b holds the round b rounds ahead of the current one; quads: a ring of chunks.
        // The first entries are requested here, next to the two loads above and before anything waits for
        // them: practically every item starts its first pass at input 0.
        static_assert(!STAGED || (LANES == 16 && ROUND * CHUNK == 2 * LANES), "a block is a round");
        constexpr int BLOCKS = STAGED ? 1 : BY_ROW ? (LONE ? 3 : 2) : LONE ? 2 * ROUND : ROUND;
        constexpr int PHASES = BY_ROW ? ROUND * BLOCKS : BLOCKS;     // chunks held (the loop for one and two neurons per lane)
        constexpr int BLOCK_INPUTS = BY_ROW ? ROUND * CHUNK : CHUNK;
        u32x2 rx[BLOCKS], rp[BLOCKS];
        auto request = [&](int b, int k) {
            rx[b] = __builtin_amdgcn_raw_buffer_load_b64(rows_of_item.xs, lane_bytes, k * (int)sizeof(float), 0);
            rp[b] = __builtin_amdgcn_raw_buffer_load_b64(rows_of_item.pr, lane_bytes, k * (int)sizeof(float), 0);
        };
        // (no further than that: short rows would fetch the rows behind them)
        const int last_block = stride - CHUNK;
        auto request_first = [&](int k) {
#pragma unroll
            for (int b = 0; b < BLOCKS - (LONE || STAGED ? 0 : 1); ++b) request(b, LONE || STAGED ? min(k + b * BLOCK_INPUTS, last_block) : k + b * BLOCK_INPUTS);
        };
        request_first(0);
        const int n_full = n_seg & ~(CHUNK - 1);
        int n_full_max = 0, n_full_min = NONE;              // of the longest and the shortest of the wavefront's rows
#pragma unroll
        for (int q = 0; q < SEGS; ++q) {
            n_full_max = max(n_full_max, __builtin_amdgcn_readlane(n_full, q * LANES));
            n_full_min = min(n_full_min, __builtin_amdgcn_readlane(n_full, q * LANES));
        }

        // Per scan: the running sums, the number of inputs they hold (kcur), and where it stands, as lane masks (in
        // scalar registers: per-lane flags cost four-neuron lanes the registers the fast loop needs)
        //   armed    waits to run the fast loop from kcur (no reference test can close before kcur)
        //   step     has to be stepped through from kcur
        //   fin      done: sums, fired state and count are final
        //   fired    the fired state that goes with the sums
        float wsum[CH], ysum[CH];
        int kcur[CH];
        uint64_t armed[CH], step[CH], fin[CH], fired[CH], any_armed = 0, any_odd = 0;
        float wb[CH];
        if (np.bias) {
#pragma unroll
            for (int c = 0; c < CH; ++c) wb[c] = j + c < J ? w[(size_t)I * J + j + c] : 0.0f;
        }
#pragma unroll
        for (int c = 0; c < CH; ++c) {
            const bool live = seg_raw < S && j + c < J;
            bool fired0 = false;
            wsum[c] = -np.theta; ysum[c] = 0.0f;
            if (np.bias) {
                wsum[c] += wb[c];
                ysum[c] = np.biasvolt * wb[c];
                const float ya0 = wsum[c] < 0.0f ? -ysum[c] : ysum[c];
                fired0 = ya0 > fabsf(wsum[c]) * np.biasvolt;
            }
            kcur[c] = 0;
            // The fast loop takes scans whose fired state is what their sums imply between tests that
            // pass with a margin: fired exactly when the weight sum is positive, and whose remaining
            // inputs are not negative (its bounds assume x >= 0; rows are ascending).  Any other start (a
            // neuron that fired on its bias alone, a row that begins below zero) is stepped through
            // from the first input on.
            const bool plain = fired0 == (wsum[c] > 0.0f) && !fired0 && first_x >= 0.0f;
            fired[c] = ballot(fired0);
            fin[c] = ballot(!live);
            armed[c] = ballot(live && n_full > 0 && plain);
            step[c] = ballot(live && n_full > 0 && !plain);
            any_armed |= armed[c];
            any_odd |= step[c];
        }
        int kmin = any_armed != 0 ? 0 : NONE;               // every armed scan starts at input 0

        // The loop of the full chip, in pieces.
        //
        // The weights of a chunk are read in two halves of four inputs.  Per half, with h the half
        // being consumed: read the weights of half h + NH - 1, then run half h; NH = 2 keeps
        // four-neuron lanes within the registers of a 16-wavefront workgroup, the others read
        // a whole chunk ahead.  H counts halves from the start of the round.
        constexpr int NH = CH == 4 || STAGED ? 2 : 4;
        float wv[NH][CH][4];                        // [half buffer][scan][step]
        // STAGED: the round's entries in quarters of a chunk, [quarter][segment][4], times and then row indices.  LDS serves a
        // wavefront's requests in order: a round is written once all reads of the one before have been issued, and nothing has to wait.
        // Per half, its times are read one half ahead and its row indices two.
        constexpr int QUARTERS = BLOCK_INPUTS / 4;
        constexpr int STAGE_ROWS = FILTER_STAGE_BYTES / 8;
        float4 xh[2];
        int4 half_rows;
        float* const stage = wl + I * COLS + wave * (FILTER_STAGE_BYTES / 4);
        float* const stage_in = stage + ((cg >> 1) * SEGS + sub) * 4 + (cg & 1) * 2;
        float* const stage_out = stage + sub * 4;
        auto stage_x = [&] {
            *reinterpret_cast<float2*>(stage_in) = make_float2(__uint_as_float(rx[0].x), __uint_as_float(rx[0].y));
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        };
        auto stage_rows = [&] {
            *reinterpret_cast<int2*>(stage_in + STAGE_ROWS) = make_int2((int)rp[0].x, (int)rp[0].y);
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        };
        auto read_x = [&](int h) { xh[h % 2] = *reinterpret_cast<const float4*>(stage_out + h % QUARTERS * SEGS * 4); };
        auto read_rows = [&](int h) { half_rows = *reinterpret_cast<const int4*>(stage_out + STAGE_ROWS + h % QUARTERS * SEGS * 4); };
        auto read_weights = [&](int buf, const unsigned (&at)[4]) {
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                float wr[CH];
                read_columns<CH>(reinterpret_cast<lds_cfloat*>((uintptr_t)at[u]), wr);
#pragma unroll
                for (int c = 0; c < CH; ++c) wv[buf][c][u] = wr[c];
            }
        };
        auto weights = [&](auto h_c) {
            constexpr int H = decltype(h_c)::value, P = H / 2, HH = H % 2;
            unsigned at[4];
            if constexpr (STAGED) {
                const int r[4] = {half_rows.x, half_rows.y, half_rows.z, half_rows.w};
#pragma unroll
                for (int u = 0; u < 4; ++u) at[u] = ((unsigned)r[u] << ROW_SHIFT) + wbase;
            } else if constexpr (BY_ROW) {
                constexpr int b = P / ROUND;
                row_row_addresses<(P % ROUND) * 4 + HH * 2>((int)rp[b].x << ROW_SHIFT, (int)rp[b].y << ROW_SHIFT, wbase, at);
            } else {
                constexpr int b = P % ROUND;
                quad_row_addresses<HH>((int)rp[b].x << ROW_SHIFT, (int)rp[b].y << ROW_SHIFT, wbase, at);
            }
            read_weights(H % NH, at);
        };
        auto times = [&](auto h_c, float (&x)[4]) {
            constexpr int H = decltype(h_c)::value, P = H / 2, HH = H % 2;
            if constexpr (STAGED) {
                const float4 v = xh[H % 2];
                x[0] = v.x; x[1] = v.y; x[2] = v.z; x[3] = v.w;
            } else if constexpr (BY_ROW) {
                constexpr int N = P * 4 + HH * 2;
                const float xe = __uint_as_float(rx[0].x), xo = __uint_as_float(rx[0].y);
                x[0] = row_broadcast<N>(xe); x[1] = row_broadcast<N>(xo);
                x[2] = row_broadcast<N + 1>(xe); x[3] = row_broadcast<N + 1>(xo);
            } else {
                const float xe = __uint_as_float(rx[P].x), xo = __uint_as_float(rx[P].y);
                x[0] = quad_broadcast<2 * HH>(xe); x[1] = quad_broadcast<2 * HH>(xo);
                x[2] = quad_broadcast<2 * HH + 1>(xe); x[3] = quad_broadcast<2 * HH + 1>(xo);
            }
        };
        // The first weights, and what the loop expects under way, for a pass that starts at input k (its first entries are in rx, rp).
        auto start_weights = [&](int k) {
            if constexpr (STAGED) {
                stage_rows();
                stage_x();
                request(0, min(k + BLOCK_INPUTS, last_block));
                read_rows(0);
                weights(std::integral_constant<int, 0>{});
                read_rows(1);
                read_x(0);
            } else {
                weights(std::integral_constant<int, 0>{});
                if constexpr (NH == 4) {
                    weights(std::integral_constant<int, 1>{});
                    weights(std::integral_constant<int, 2>{});
                }
            }
        };
        // One chunk: wb / yb are the scans' sums behind its inputs.  The requests stay ahead of the
        // arithmetic: what a half consumes was requested a half or more ago, and what it requests has the
        // whole half to arrive.
        float yb[CH], low[CH], x0, x7;
        auto chunk = [&](auto ph_c, int k, auto by_round_c) {
            constexpr int ph = decltype(ph_c)::value;
            constexpr bool BY_ROUND = decltype(by_round_c)::value;
            if constexpr (!BY_ROW && !STAGED) request((ph + ROUND - 1) % ROUND, k + (ROUND - 1) * CHUNK);
            auto half = [&](auto half_c) {
                constexpr int hh = decltype(half_c)::value, H = 2 * ph + hh;
                weights(std::integral_constant<int, H + NH - 1>{});
                if constexpr (STAGED) {
                    if constexpr ((H + 2) % QUARTERS == 0) stage_rows();
                    read_rows(H + 2);
                    if constexpr ((H + 1) % QUARTERS == 0) {
                        stage_x();
                        request(0, min(k - ph * CHUNK + 2 * BLOCK_INPUTS, last_block));
                    }
                    read_x(H + 1);
                }
                __builtin_amdgcn_sched_barrier(0);
                float x[4];
                times(std::integral_constant<int, H>{}, x);
                if (hh == 0) x0 = x[0];
                else x7 = x[3];
#pragma unroll
                for (int u = 0; u < 4; ++u)
#pragma unroll
                    for (int c = 0; c < CH; ++c) {
                        const float wc = wv[H % NH][c][u];
                        const bool start = hh == 0 && u == 0 && (ph == 0 || !BY_ROUND);
                        const float before = wb[c];
                        wb[c] = (start ? wsum[c] : wb[c]) + wc;
                        yb[c] = __fmaf_rn(x[u], wc, start ? ysum[c] : yb[c]);
                        if (TIGHT && !BY_ROUND && u % 2 == 1) low[c] = fminf(fminf(hh == 0 && u == 1 ? 0.0f : low[c], before), wb[c]);
                    }
            };
            half(std::integral_constant<int, 0>{});
            half(std::integral_constant<int, 1>{});
        };
        // rows: the next round's block moves up, the one after it is requested
        auto next_round = [&] {
            if constexpr (BY_ROW && !STAGED) {
#pragma unroll
                for (int b = 0; b + 1 < BLOCKS; ++b) { rx[b] = rx[b + 1]; rp[b] = rp[b + 1]; }
            }
        };
        auto start_round = [&](int k0) {
            if constexpr (BY_ROW && !STAGED) request(BLOCKS - 1, k0 + (BLOCKS - 1) * BLOCK_INPUTS);
        };
        // By rounds of four chunks with one test, until the first scan of the wavefront comes close: all scans take a round over
        // together.  (Lanes without a scan compute along.)
        if constexpr (ROUNDS && !LONE) {
            if (by_rounds && any_odd == 0 && n_full_min >= ROUND * CHUNK) {
                start_weights(0);
                int k0 = 0;
                bool more = true;
                while (more && k0 + ROUND * CHUNK <= n_full_min) {
                    rotate_wave_priority(k0 / (ROUND * CHUNK) + (wave >> 2));
                    start_round(k0);
                    float x_first;
                    for_each_phase<ROUND>([&](auto ph_c) {
                        chunk(ph_c, k0 + decltype(ph_c)::value * CHUNK, std::true_type{});
                        if (decltype(ph_c)::value == 0) x_first = x0;
                        return true;
                    });
                    const float dx = __fmaf_rn(x7, ROUND_DX, x7 - x_first), x7e = x7 * ROUND_AT;
                    const float thr = __fmaf_rn(dx, 4.0f * w4, x7 * end_w_round);
                    float at_end[CH], lowest[CH];
                    uint64_t soon = 0;                      // not even with the fall that a round like this one brings
#pragma unroll
                    for (int c = 0; c < CH; ++c) {
                        at_end[c] = __fmaf_rn(-x7e, wb[c], yb[c]);
                        lowest[c] = fminf(fminf(wsum[c], wb[c]), 4.0f * w4);
                        soon |= armed[c] & ~ballot(__fmaf_rn(dx, lowest[c] - fabsf(wb[c]), at_end[c]) > thr);
                    }
                    more = soon == 0;
                    if (!more) {
                        uint64_t fails = 0;
#pragma unroll
                        for (int c = 0; c < CH; ++c) fails |= armed[c] & ~ballot(__fmaf_rn(dx, lowest[c], at_end[c]) > thr);
                        if (fails != 0) break;              // (the round again, chunk by chunk)
                    }
#pragma unroll
                    for (int c = 0; c < CH; ++c) { wsum[c] = wb[c]; ysum[c] = yb[c]; }
                    next_round();
                    k0 += ROUND * CHUNK;
                }
                kmin = k0;
#pragma unroll
                for (int c = 0; c < CH; ++c) kcur[c] = k0;
                request_first(kmin);
            }
        }

        bool first_pass = true;                             // (LONE: every armed scan takes part and starts at input 0)
        // Passes: the fast loop for the armed scans that are furthest behind, then the scans it left behind
        // step by step.  A scan that does not close there is armed again.
        // Practically every item takes one pass and a second look without work.
        for (;;) {
            uint64_t ran[CH];                               // the scans that take part in this pass's fast loop
#pragma unroll
            for (int c = 0; c < CH; ++c) ran[c] = armed[c] & ballot(kcur[c] == kmin);
            if (kmin != NONE) {
                uint64_t open[CH];                          // lanes whose scan still runs in it
#pragma unroll
                for (int c = 0; c < CH; ++c) {
                    open[c] = ran[c];
                    armed[c] &= ~ran[c];
                    if (!LONE) kcur[c] = in_mask(ran[c]) ? n_full : kcur[c];       // unless the scan stops earlier
                }
                if constexpr (LONE) {
                    // Half h (four inputs) is worked on while the weights of the next three are on their way.
                    constexpr int NH = 4;
                    float wv[NH][CH][4];                    // [half buffer][scan][input]
                    float run_w[CH], run_y[CH], end_w_of[CH], end_y_of[CH];
                    uint64_t pass[CH];
                    unsigned passed[CH];                    // chunks
                    u32x2 at[BLOCKS];                       // LDS offsets of the rows of the entries held
                    float nx, dx, thr;                      // the test's operands
                    auto shifted = [&](const u32x2& r) { return u32x2{r.x << ROW_SHIFT, r.y << ROW_SHIFT}; };
                    // They are those of the lane's quad in block b (rows) or in ring slot b (quads), from input k on.  Behind the end of a
                    // row nothing passes.
                    const int last_at = n_full - (BY_ROW ? (lane & 12) * (CHUNK / 4) : 0);
                    auto test_operands = [&](int b, int k) {
                        const float x0 = quad_broadcast<0>(__uint_as_float(rx[b].x)), x7 = quad_broadcast<3>(__uint_as_float(rx[b].y));
                        dx = __fmaf_rn(x7, FILTER_DX, x7 - x0);
                        nx = -x7 * FILTER_AT;
                        thr = TIGHT ? x7 * end_w : __fmaf_rn(dx, w4, x7 * end_w);
                        if (SEGS > 1) thr = k < last_at ? thr : INFINITY;
                    };
#pragma unroll
                    for (int c = 0; c < CH; ++c) { run_w[c] = wsum[c]; run_y[c] = ysum[c]; }
                    // (the first chunk decides on one that moves nothing)
#pragma unroll
                    for (int c = 0; c < CH; ++c) { end_w_of[c] = wsum[c]; end_y_of[c] = ysum[c]; pass[c] = ~0ull; passed[c] = ~0u; }
                    auto weights = [&](auto h_c) {
                        constexpr int H = decltype(h_c)::value, P = H / 2, HH = H % 2;
                        constexpr int B = (BY_ROW ? P / ROUND : P) % BLOCKS, M = BY_ROW ? (P % ROUND) * 4 + HH * 2 : HH * 2;
                        unsigned a[4];
                        weight_addresses<BY_ROW, M>(a, at[B].x, at[B].y, wbase);
#pragma unroll
                        for (int u = 0; u < 4; ++u) {
                            float wr[CH];
                            read_columns<CH>(reinterpret_cast<lds_cfloat*>((uintptr_t)a[u]), wr);
#pragma unroll
                            for (int c = 0; c < CH; ++c) wv[H % NH][c][u] = wr[c];
                        }
                    };
                    // The chunk tested last: scans that passed take its sums over.
                    auto decide = [&] {
#pragma unroll
                        for (int c = 0; c < CH; ++c) {
                            open[c] &= pass[c];
                            asm("v_cndmask_b32_e64 %[ws], %[ws], %[wb], %[open]\n"
                                "v_cndmask_b32_e64 %[ys], %[ys], %[yb], %[open]\n"
                                "v_addc_co_u32_e64 %[k], vcc, 0, %[k], %[open]\n"
                                : [ws] "+v"(wsum[c]), [ys] "+v"(ysum[c]), [k] "+v"(passed[c])
                                : [open] "s"(open[c]), [wb] "v"(end_w_of[c]), [yb] "v"(end_y_of[c]) : "vcc");
                        }
                    };
                    // BY_ROUND: tested with the other chunks of its round, behind the last of them.
                    static_assert(!ROUNDS || !BY_ROW, "eight-column slices alone have rows long enough");
                    float round_start[CH], x_first;
                    uint64_t soon = 0, fails = 0;
                    auto chunk = [&](auto ph_c, int k, auto by_round_c) {
                        constexpr int ph = decltype(ph_c)::value, R = BY_ROW ? ph / ROUND : ph;
                        constexpr bool BY_ROUND = decltype(by_round_c)::value;
                        // The next entry (block of four chunks, chunk) whose weights will be read, and the test's operands
                        if constexpr (!BY_ROW || ph % ROUND == 0) {
                            constexpr int B = BY_ROW ? (R + 1) % BLOCKS : (ph + 2) % BLOCKS;
                            at[B] = shifted(rp[B]);
                            if constexpr (BY_ROUND) {
                                asm volatile("s_nop 1" : "+v"(rx[R].x), "+v"(rx[R].y), "+v"(at[B].x), "+v"(at[B].y));
                            } else {
                                test_operands(R, k);
                                asm volatile("s_nop 1" : "+v"(rx[R].x), "+v"(rx[R].y), "+v"(at[B].x), "+v"(at[B].y), "+v"(nx), "+v"(dx), "+v"(thr));
                            }
                        }
                        if constexpr (BY_ROUND && ph % ROUND == 0) {
                            x_first = quad_broadcast<0>(__uint_as_float(rx[R].x));
#pragma unroll
                            for (int c = 0; c < CH; ++c) round_start[c] = run_w[c];
                        }
                        float start[CH], low[CH];
                        auto half = [&](auto half_c) {
                            constexpr int hh = decltype(half_c)::value, H = 2 * ph + hh, N = BY_ROW ? (ph % ROUND) * 4 + hh * 2 : 2 * hh;
                            weights(std::integral_constant<int, H + NH - 1>{});
                            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                            for (int c = 0; c < CH; ++c) {
                                float sums[4];
                                if (hh == 0) start[c] = run_w[c];
                                accumulate_half<BY_ROW, N>(run_w[c], sums, run_y[c], __uint_as_float(rx[R].x), __uint_as_float(rx[R].y), wv[H % NH][c]);
                                run_w[c] = sums[3];
                                if (TIGHT && !BY_ROUND)
                                    low[c] = fminf(fminf(fminf(fminf(hh == 0 ? 0.0f : low[c], sums[0]), sums[1]), sums[2]), sums[3]);
                            }
                            __builtin_amdgcn_sched_barrier(0);
                        };
                        half(std::integral_constant<int, 0>{});
                        if constexpr (!BY_ROUND) decide();
                        half(std::integral_constant<int, 1>{});
                        if constexpr (BY_ROUND && ph % ROUND == ROUND - 1) {
                            const float x7 = quad_broadcast<3>(__uint_as_float(rx[R].y));
                            const float dx = __fmaf_rn(x7, ROUND_DX, x7 - x_first), x7e = x7 * ROUND_AT;
                            const float thr = __fmaf_rn(dx, 4.0f * w4, x7 * end_w_round);
#pragma unroll
                            for (int c = 0; c < CH; ++c) {
                                const float at_end = __fmaf_rn(-x7e, run_w[c], run_y[c]), lowest = fminf(fminf(round_start[c], run_w[c]), 4.0f * w4);
                                fails |= ran[c] & ~ballot(__fmaf_rn(dx, lowest, at_end) > thr);
                                // not even with the fall that the rounds up to the next decision bring
                                if constexpr (ph == PHASES - 1)
                                    soon |= ran[c] & ~ballot(__fmaf_rn(dx, __fmaf_rn(-(float)(PHASES / ROUND), fabsf(run_w[c]), lowest), at_end) > thr);
                            }
                        }
#pragma unroll
                        for (int c = 0; c < (BY_ROUND ? 0 : CH); ++c) {
                            if (!TIGHT) low[c] = fminf(fminf(start[c], run_w[c]), w4);
                            pass[c] = chunk_passes<BY_ROW, BY_ROW ? ph % ROUND : 0>(run_w[c], run_y[c], nx, dx, thr, low[c]);
                            end_w_of[c] = run_w[c];
                            end_y_of[c] = run_y[c];
                        }
                        if constexpr (!BY_ROW) request(ph, min(k + BLOCKS * CHUNK, last_block));
                        else if constexpr (ph % ROUND == ROUND - 1) request(R, min(k - (ROUND - 1) * CHUNK + BLOCKS * BLOCK_INPUTS, last_block));
                    };
                    auto first_weights = [&] {
                        at[0] = shifted(rp[0]);
                        asm volatile("s_nop 1" : "+v"(at[0].x), "+v"(at[0].y));
                        if constexpr (!BY_ROW) {
                            at[1] = shifted(rp[1]);
                            asm volatile("s_nop 1" : "+v"(at[1].x), "+v"(at[1].y));
                        }
                        weights(std::integral_constant<int, 0>{});
                        weights(std::integral_constant<int, 1>{});
                        weights(std::integral_constant<int, 2>{});
                    };
                    first_weights();
                    int k0 = kmin;
                    bool more = true;
                    const bool rotate = waves > 4;          // (more than a wavefront per SIMD)
                    if constexpr (ROUNDS) if (by_rounds && first_pass && any_odd == 0) {
                        while (soon == 0 && k0 + PHASES * CHUNK <= n_full_min) {
                            if (rotate) rotate_wave_priority(k0 / (PHASES * CHUNK) + (wave >> 2));
                            for_each_phase<PHASES>([&](auto ph_c) {
                                chunk(ph_c, k0 + decltype(ph_c)::value * CHUNK, std::true_type{});
                                return true;
                            });
                            if (fails != 0) break;          // (its rounds again, chunk by chunk)
#pragma unroll
                            for (int c = 0; c < CH; ++c) { wsum[c] = run_w[c]; ysum[c] = run_y[c]; }
                            k0 += PHASES * CHUNK;
                        }
#pragma unroll
                        for (int c = 0; c < CH; ++c) { end_w_of[c] = wsum[c]; end_y_of[c] = ysum[c]; passed[c] = k0 / CHUNK - 1; }
                        if (fails != 0) {
                            request_first(k0);
#pragma unroll
                            for (int c = 0; c < CH; ++c) { run_w[c] = wsum[c]; run_y[c] = ysum[c]; }
                            first_weights();
                        }
                    }
                    first_pass = false;
                    // Whole rounds as long as the longest row has one left, without an exit inside (behind an exit between a request
                    // and its use the compiler would move the request to the use), then its last chunks one by one.
                    for (; k0 + PHASES * CHUNK <= n_full_max && more; k0 += PHASES * CHUNK) {
                        if (rotate) rotate_wave_priority(k0 / (PHASES * CHUNK) + (wave >> 2));
                        for_each_phase<PHASES>([&](auto ph_c) {
                            chunk(ph_c, k0 + decltype(ph_c)::value * CHUNK, std::false_type{});
                            return true;
                        });
                        uint64_t any = 0;
#pragma unroll
                        for (int c = 0; c < CH; ++c) any |= open[c];
                        more = any != 0;
                    }
                    if (more)
                        for_each_phase<PHASES>([&](auto ph_c) {
                            const int k = k0 + decltype(ph_c)::value * CHUNK;
                            if (k >= n_full_max) return false;
                            chunk(ph_c, k, std::false_type{});
                            return true;
                        });
                    decide();
#pragma unroll
                    for (int c = 0; c < CH; ++c) kcur[c] = in_mask(ran[c]) ? kmin + (int)passed[c] * CHUNK : kcur[c];
                } else {
                start_weights(kmin);
                auto test = [&](int k) {
                    const float dx = __fmaf_rn(x7, FILTER_DX, x7 - x0), x7e = x7 * FILTER_AT;
                    const float thr = TIGHT ? x7 * end_w : __fmaf_rn(dx, w4, x7 * end_w);
#pragma unroll
                    for (int c = 0; c < CH; ++c)
                        filter_test(wsum[c], ysum[c], kcur[c], open[c], k, wb[c], yb[c], x7e, thr, dx,
                                    TIGHT ? low[c] : fminf(fminf(wsum[c], wb[c]), w4));
                };
                // Whole rounds as long as the longest row has one left, without an exit inside the round: behind an
                // exit test between a request and its use, several chunks later, the compiler would move the
                // request right in front of the use, and the wavefront would wait for the whole round trip.
                // Scans whose row has ended are masked.  The last chunks of the longest row follow one by one.
                auto inside = [&](int k) {
                    const uint64_t in = __builtin_amdgcn_ballot_w64(k < n_full);
                    uint64_t any = 0;
#pragma unroll
                    for (int c = 0; c < CH; ++c) {
                        open[c] &= in;
                        any |= open[c];
                    }
                    return any != 0;
                };
                int k0 = kmin;
                bool more = true;
                for (; k0 + ROUND * CHUNK <= n_full_max && more; k0 += ROUND * CHUNK) {
                    rotate_wave_priority(k0 / (ROUND * CHUNK) + (wave >> 2));
                    start_round(k0);
                    for_each_phase<ROUND>([&](auto ph_c) {
                        const int k = k0 + decltype(ph_c)::value * CHUNK;
                        inside(k);
                        chunk(ph_c, k, std::false_type{});
                        test(k);
                        return true;
                    });
                    next_round();
                    more = inside(k0 + ROUND * CHUNK);
                }
                if (more)
                    for_each_phase<ROUND>([&](auto ph_c) {
                        const int k = k0 + decltype(ph_c)::value * CHUNK;
                        if (!inside(k)) return false;
                        chunk(ph_c, k, std::false_type{});
                        test(k);
                        return true;
                    });
                }
#pragma unroll
                for (int c = 0; c < CH; ++c) {
                    fired[c] = (fired[c] & ~ran[c]) | (ballot(wsum[c] > 0.0f) & ran[c]);
                    step[c] |= ran[c] & ballot(kcur[c] < n_full);
                }
            }

            // Stopped scans, evaluated with the reference's tests: every lane fetches its own eight inputs
            // (positions are multiples of eight inside the full chunks of the row).  A scan that closes is
            // finished.  One that does not is stepped on for two more chunks -- the fast test fails early where
            // the weight sum is small, and starting the fast loop for a chunk or two costs more -- and goes back
            // to the fast loop then, if its fired state is the plain one; otherwise (fired on a negative weight
            // sum, say) it keeps stepping here.
            //   sure: the scan is in the plain state with ysum - x*wsum well above zero (close_chunk_vector)
            uint64_t sure[CH], any_step = 0;
#pragma unroll
            for (int c = 0; c < CH; ++c) {
                sure[c] = ran[c];
                any_step |= step[c];
            }
            for (int round = 0; any_step != 0;) {
                uint64_t stuck[CH];
                // (the entries of all the lane's scans are requested before the first is worked on: one memory
                // round trip per round, not CH)
                Chunk pc[CH];
#pragma unroll
                for (int c = 0; c < CH; ++c) {
                    stuck[c] = 0;
                    load_chunk_flat(pc[c], xs, pr, in_mask(step[c]) ? kcur[c] : 0);
                }
                for_each_phase<CH>([&](auto c_c) {
                    constexpr int c = decltype(c_c)::value;
                    const uint64_t need = step[c];
                    if (need == 0) return true;
                    float pw[CHUNK];
#pragma unroll
                    for (int u = 0; u < CHUNK; ++u) pw[u] = wcol[pc[c].p[u] * COLS + c];
                    const float w0 = wsum[c], y0 = ysum[c], x7 = pc[c].x[CHUNK - 1];
                    const int k_start = kcur[c];
                    float x_exit;
                    const float slack = __fmaf_rn(FILTER_END_Y, fabsf(y0), __fmaf_rn(x7 * FILTER_END_XW, fabsf(w0), x7 * end_w));
                    const uint64_t exited = close_chunk_vector<WANT_K>(wsum[c], ysum[c], kcur[c], x_exit, need & sure[c], pc[c].x, pw, slack);
                    uint64_t positive = ballot(wsum[c] > 0.0f), now_fired = positive;
                    uint64_t closed = exited & positive & ballot(ysum[c] <= x_exit * wsum[c]);
                    const uint64_t redo = need & (~sure[c] | (exited & ~closed));
                    if (!WANT_K) kcur[c] = in_mask(need & ~closed) ? k_start + CHUNK : k_start;
                    if (redo != 0) {
                        const bool mine = in_mask(redo);
                        wsum[c] = mine ? w0 : wsum[c];
                        ysum[c] = mine ? y0 : ysum[c];
                        const bool fired0 = in_mask((sure[c] & ballot(w0 > 0.0f)) | (~sure[c] & fired[c]));
                        float ya = wsum[c] < 0.0f ? -ysum[c] : ysum[c];
                        float yg = fired0 ? ya : INFINITY;
                        uint64_t unused = 0;
                        int kc = k_start;
                        scan_chunk_vector<true>(wsum[c], ysum[c], ya, yg, kc, unused, redo, pc[c].x, pw);
                        kcur[c] = mine ? kc : kcur[c];
                        const uint64_t gone = redo & ballot(kc != k_start + CHUNK);            // closed before its last input
                        closed |= gone;
                        positive = ballot(wsum[c] > 0.0f);
                        now_fired = (now_fired & ~redo) | (redo & (gone | ballot(yg < INFINITY)));
                        sure[c] &= ~redo;
                    }
                    const uint64_t ahead = ballot(x7 >= 0.0f);                  // the inputs behind this chunk are not negative
                    const uint64_t more = need & ~closed & ballot(kcur[c] + CHUNK <= n_full);
                    const uint64_t back = round >= 2 ? more & ahead & ~(now_fired ^ positive) : 0;
                    fired[c] = (fired[c] & ~need) | (now_fired & need);
                    fin[c] |= need & closed;
                    armed[c] |= back;
                    step[c] = more & ~back;
                    stuck[c] = step[c] & ~now_fired & positive & ahead;
                    return true;
                });
                ++round;
                // A scan that missed its close by a rounding is left with a positive weight sum and not fired
                // (ysum - x*wsum < 0) -- one in about 1e5.  It cannot fire, let alone close, while the weight
                // sum stays positive, and would walk on here to the end of its row, a chunk per round, in
                // a wavefront that is alone by then.  In rounds 1, 2, 4, 8, ... the wavefront looks
                // ahead for it (never_fires): if the weight sum stays positive to the end, the scan is done.
                // (256 -> 256 channels on 14x14, 32 images, 2304 inputs: 536 -> 500 us.)
                if ((round & (round - 1)) == 0) {
                    for (;;) {
                        uint64_t lanes = 0;
                        int c_now = 0, k = 0;
                        float ws = 0.0f, ys = 0.0f;
                        for_each_phase<CH>([&](auto c_c) {
                            constexpr int c = decltype(c_c)::value;
                            if (stuck[c] == 0) return true;
                            lanes = stuck[c];
                            c_now = c; k = kcur[c]; ws = wsum[c]; ys = ysum[c];
                            stuck[c] &= stuck[c] - 1;
                            return false;
                        });
                        if (lanes == 0) break;
                        const int src = __builtin_ctzll(lanes);
                        const size_t row0 = (size_t)__builtin_amdgcn_readlane(seg, src) * stride;
                        const bool never = never_fires<COLS>(
                            sorted + row0, perm + row0, wl + CH * (src % LANES) + c_now, __builtin_amdgcn_readlane(k, src),
                            __builtin_amdgcn_readlane(n_seg, src), __int_as_float(__builtin_amdgcn_readlane(__float_as_int(ws), src)),
                            __int_as_float(__builtin_amdgcn_readlane(__float_as_int(ys), src)), lane);
                        const uint64_t bit = ballot(never) != 0 ? lanes & -lanes : 0;             // (a uniform value)
                        for_each_phase<CH>([&](auto c_c) {
                            constexpr int c = decltype(c_c)::value;
                            fin[c] |= c == c_now ? bit : 0;
                            step[c] &= ~(c == c_now ? bit : 0);
                            return true;
                        });
                    }
                }
                any_step = 0;
#pragma unroll
                for (int c = 0; c < CH; ++c) any_step |= step[c];
            }
            any_armed = 0;
#pragma unroll
            for (int c = 0; c < CH; ++c) any_armed |= armed[c];
            if (any_armed == 0) break;
            kmin = NONE;
#pragma unroll
            for (int c = 0; c < CH; ++c) kmin = in_mask(armed[c]) ? min(kmin, kcur[c]) : kmin;
#pragma unroll
            for (int d = kWave / 2; d > 0; d >>= 1) kmin = min(kmin, __shfl_xor(kmin, d, kWave));
            kmin = __builtin_amdgcn_readfirstlane(kmin);
            request_first(kmin);
        }

        // Whatever is left of a row -- fewer than eight inputs behind the full chunks -- step by step, then
        // the output.  (Rows are padded beyond their length, so the eight entries from n_full on can always be
        // read.)
        const uint64_t leftover = ballot(n_full < n_seg);
        uint64_t any_left = 0;
#pragma unroll
        for (int c = 0; c < CH; ++c) any_left |= ~fin[c] & leftover;
        if (any_left != 0) {
            Chunk tail;
            load_chunk_flat(tail, xs, pr, n_full < n_seg ? n_full : 0);
            for_each_phase<CH>([&](auto c_c) {
                constexpr int c = decltype(c_c)::value;
                const uint64_t start = ~fin[c] & leftover;
                uint64_t run = start;
                if (run == 0) return true;
                float tw[CHUNK - 1];
#pragma unroll
                for (int u = 0; u < CHUNK - 1; ++u) tw[u] = wcol[tail.p[u] * COLS + c];
                float ya = wsum[c] < 0.0f ? -ysum[c] : ysum[c];
                float yg = in_mask(fired[c]) ? ya : INFINITY;
                uint64_t closed = 0;
                for_each_phase<CHUNK - 1>([&](auto u_c) {
                    constexpr int u = decltype(u_c)::value;
                    if (u > 0) run &= ballot(n_full + u < n_seg);
                    if (run == 0) return false;
                    scan_step_vector(wsum[c], ysum[c], ya, yg, kcur[c], run, tail.x[u], tw[u]);
                    const uint64_t gone = run & ballot(kcur[c] == n_full + u);                 // did not consume the input
                    closed |= gone;
                    run &= ~gone;
                    return true;
                });
                fired[c] = (fired[c] & ~start) | (start & (closed | ballot(yg < INFINITY)));
                return true;
            });
        }
        float y[CH], r[CH];
#pragma unroll
        for (int c = 0; c < CH; ++c) {
            y[c] = np.max_time; r[c] = 0.0f;
            if (in_mask(fired[c])) {
                r[c] = 1.0f / wsum[c];
                y[c] = ysum[c] * r[c];
                if (y[c] >= np.max_time) { y[c] = np.max_time; r[c] = 0.0f; }
            }
        }
        if (seg_raw < S) {
            const size_t o = (size_t)seg * J + j;
            store_columns<CH>(y_out + o, y, J - j, J);
            store_columns<CH>(rcp_out + o, r, J - j, J);
            if (copy.dst) store_columns<CH>(copy.dst + time_copy_pixel(copy, seg) * J + j, y, J - j, J);
            if (WANT_K) {
#pragma unroll
                for (int c = 0; c < CH; ++c)
                    if (j + c < J) k_out[o + c] = (in_mask(fired[c]) && r[c] != 0.0f) ? kcur[c] : -1;
            }
        }
    }
    };
    // (Values computed before the branch would be kept for both forms and cost the loops scalar registers: 1 % of the time.)
    asm volatile("" : "+s"(n_groups), "+s"(waves), "+s"(S), "+s"(stride), "+s"(J));
    if (tight) scan_items(std::true_type{});
    else scan_items(std::false_type{});
}

__global__ void __launch_bounds__(256)
unpad_rows_kernel(const float* __restrict__ sorted, const int32_t* __restrict__ perm,
                  float* __restrict__ sorted_out, int32_t* __restrict__ perm_out, int64_t n, int I, int stride) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
    const int64_t row = t / I;
    const int col = (int)(t - row * I);
    const size_t src = (size_t)row * stride + col;
    if (sorted_out) sorted_out[t] = sorted[src];
    if (perm_out) perm_out[t] = perm[src];
}

}  // namespace

namespace {
// How many of them a launch of S segments of I inputs uses: the form with the smallest estimated time.  A SIMD
// works on its wavefronts four at a time; the time of a chunk with w of them at work and the fixed share of an
// item (first requests, evaluation of the closing chunks, leftover inputs, output) in chunks are measured
// (in 10 ns and chunks; 784 -> 800 at 64 ... 2048 rows, 27- to 4608-input patches of 1 ... 32 images).  More neurons per lane
// cost less per neuron where wavefronts abound, fewer where a SIMD gets one or two wavefronts of long rows.  us with one / two /
// four neurons per lane: 784 -> 800 at 128 rows 24.3 / 28.5 / 47.8, 384 rows 44.3 / 44.0 / 55.4, 768 rows 77 / 69 / 71, 2048 rows
// 198 / 170 / 147; 49 patches of 4608 to 512 neurons 90 / 152; 200 704 patches of 147 to 64 neurons 349 / 307 / 221;
// 25 000 rows of 5 to 379 neurons 67 / 55 / 53.
template <int COLS>
int filter_neurons(int64_t S, int64_t I, int n_slices, int cus) {
    constexpr bool full = COLS == 64;
    // (up to 4, 8, 12 and 16 wavefronts, then per 16; 64 columns: one neuron for thirteen to sixteen wavefronts of rows of middling length:
    // 1024 rows of 256 to 130 / 250 neurons 20.9 / 21.4 against 25.5 / 25.2 us, of 39 to 130 12.1 against 11.6, of 576 36.1 against 34.0)
    const int wide[3][5] = {{14, 19, 22, full && I >= 64 && I < 360 ? 29 : 32, 32},
                            {20, 29, full ? 34 : 35, full ? 51 : 53, 53}, {38, COLS == 32 ? 54 : 52, 62, 77, 77}};
    static const int narrow[2][5] = {{14, 19, 22, 32, 32}, {25, 33, 46, 58, 58}};                 // eight-column slices
    static const int fixed_chunks[3] = {6, 7, 9};
    // A single slice of 8 or 16 columns: rows come from HBM once, and quads hold too few bytes in flight for that (262 144
    // patches of 144 to 16 neurons 134 / 147 / 174 us).
    if (n_slices == 1 && COLS <= 16) return 1;
    int best = 1;
    int64_t best_time = INT64_MAX;
    for (int k = 0, ch = 1; ch <= FILTER_MAX_CH<COLS>; ++k, ch *= 2) {
        const int64_t segs = kWave / COLS * ch;
        const int64_t groups = n_slices < cus ? cus / n_slices : 1;                               // workgroups per slice
        const int64_t per_group = ((S + segs - 1) / segs + groups - 1) / groups;                  // items of the fullest
        const int* chunk_time = COLS == 8 ? narrow[k % 2] : wide[k];
        const int64_t t = (per_group <= 16 ? 16 * chunk_time[(per_group + 3) / 4 - 1] : per_group * chunk_time[4]) * (I / CHUNK + fixed_chunks[k]);
        if (t < best_time) { best_time = t; best = ch; }
    }
    return best;
}
// Which loop a launch with less than the most neurons per lane takes.  One neuron: short rows stay with the loop of the full chip --
// below a block of four chunks the other one's set-up is all it adds (512 rows of 8 / 27 to 64 neurons 6.6 against 6.8 us, 200 of 8
// to 1000 8.2 against 8.5); eight-column slices below 128 inputs, since it requests eight chunks ahead there, which such rows do not
// have (401 408 rows of 75 to 8 neurons 90 against 100).  Two neurons and 64 columns: nine to sixteen wavefronts hide what the
// lone loop saves (1536 rows of 150 to 130 neurons 18.2 against 19.8 us, 400 to 800 17.2 against 18.4; of 576 42.7 and 41.3), fewer do not (1024 of
// 576 to 130 7 % slower), nor do turns (333 of 39 to 1500 14 % slower, 700 of 576 to 800 11 %).
template <int COLS>
constexpr bool filter_lone(int ch, int64_t per_group, int64_t I) {
    if (ch == 1) return I >= (COLS == 8 ? 128 : 4 * CHUNK);
    return ch < FILTER_MAX_CH<COLS> && (COLS != 64 || per_group <= 8 || per_group > 16);
}
constexpr size_t FILTER_WIDE_COPY_BYTES = 48 * 1024;        // slices from here on are copied by 16 wavefronts

// The instantiation for ch neurons per lane.
template <int COLS, bool WANT_K>
decltype(&scan_filter_kernel<COLS, 1, true, WANT_K>) filter_kernel(int ch, bool lone, bool rounds, bool staged) {
    constexpr bool LONG_ROWS = COLS == 8, STAGES = FILTER_STAGES<COLS>;
    constexpr int MOST = FILTER_MAX_CH<COLS>;
    if (ch == 1 && lone) return rounds ? scan_filter_kernel<COLS, 1, true, WANT_K, LONG_ROWS> : scan_filter_kernel<COLS, 1, true, WANT_K>;
    if (ch == 1) return scan_filter_kernel<COLS, 1, false, WANT_K>;
    if (ch == MOST && staged)
        return rounds ? scan_filter_kernel<COLS, MOST, false, WANT_K, true, STAGES> : scan_filter_kernel<COLS, MOST, false, WANT_K, false, STAGES>;
    if (ch == MOST) return rounds ? scan_filter_kernel<COLS, MOST, false, WANT_K, true> : scan_filter_kernel<COLS, MOST, false, WANT_K>;
    if constexpr (COLS == 64) {
        if (!lone) return scan_filter_kernel<COLS, 2, false, WANT_K>;
    }
    return scan_filter_kernel<COLS, COLS == 8 ? 1 : 2, true, WANT_K>;
}

template <int COLS>
int raise_scan_lds_limits() {
    for (int ch = 1; ch <= FILTER_MAX_CH<COLS>; ch *= 2)
        for (int form = 0; form < 8; ++form) {
            const bool lone = form & 1, rounds = form & 2, staged = form & 4;
            if (lone && ch == 4) continue;
            for (const void* k : {reinterpret_cast<const void*>(filter_kernel<COLS, true>(ch, lone, rounds, staged)),
                                  reinterpret_cast<const void*>(filter_kernel<COLS, false>(ch, lone, rounds, staged))})
                SNNTC_HIP_CHECK(hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, LDS_SCAN_BYTES));
        }
    constexpr bool SORTS = split_sorts(COLS);
    const void* split[] = {reinterpret_cast<const void*>(scan_lds_split_kernel<COLS, 0, true>),
                           reinterpret_cast<const void*>(scan_lds_split_kernel<COLS, 0, false>),
                           reinterpret_cast<const void*>(scan_lds_split_kernel<COLS, SORTS ? 512 : 0, false>),
                           reinterpret_cast<const void*>(scan_lds_split_kernel<COLS, SORTS ? 1024 : 0, false>)};
    for (const void* k : split)
        SNNTC_HIP_CHECK(hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize,
                                            LDS_SCAN_BYTES - SPLIT_STATIC_LDS));
    return SNNTC_OK;
}
}  // namespace

// One-time set-up of the scan on device `dev` (which must be the current device): the CU count and
// the dynamic-LDS limit of EVERY instantiation, so that no later launch, whatever its shape, has
// to call hipFuncSetAttribute (which is not allowed while a stream is being captured).
int scan_prepare_device(int dev, int* cu_count_out) {
    static std::atomic<int> cu_count[kMaxDevices];
    if (dev < 0 || dev >= kMaxDevices) return fail(SNNTC_ERR_UNSUPPORTED, "scan: device index %d not supported", dev);
    int cus = cu_count[dev].load(std::memory_order_acquire);
    if (cus == 0) {
        hipDeviceProp_t prop;
        SNNTC_HIP_CHECK(hipGetDeviceProperties(&prop, dev));
        int rc = raise_scan_lds_limits<64>();
        if (!rc) rc = raise_scan_lds_limits<32>();
        if (!rc) rc = raise_scan_lds_limits<16>();
        if (!rc) rc = raise_scan_lds_limits<8>();
        if (rc) return rc;
        cus = prop.multiProcessorCount > 0 ? prop.multiProcessorCount : 256;
        cu_count[dev].store(cus, std::memory_order_release);
    }
    if (cu_count_out) *cu_count_out = cus;
    return SNNTC_OK;
}

namespace {
std::atomic<int> g_wait_polls{SPLIT_SPIN_LIMIT};
}

void set_scan_wait_polls(int polls) { g_wait_polls.store(polls < 0 ? SPLIT_SPIN_LIMIT : polls, std::memory_order_relaxed); }

int read_scan_giveups(int64_t* count, hipStream_t stream) {
    unsigned int v = 0;
    SNNTC_HIP_CHECK(hipMemcpyFromSymbolAsync(&v, HIP_SYMBOL(g_scan_giveups), sizeof(v), 0, hipMemcpyDeviceToHost, stream));
    SNNTC_HIP_CHECK(hipStreamSynchronize(stream));
    *count = (int64_t)v;
    return SNNTC_OK;
}

constexpr int split_segs(int cols) { return split_lanes(cols) / cols; }
// Whether a launch with slices of `cols` columns goes to scan_lds_split_kernel.
static bool takes_split(int cols, int64_t S, int64_t I, int64_t stride, int64_t J, const NeuronParams& np, int cus) {
    const int64_t items = (S + split_segs(cols) - 1) / split_segs(cols) * ((J + cols - 1) / cols);
    return items <= (int64_t)cus && I >= 2 * CHUNK * SPLIT_WAVES &&
           split_lds_bytes(split_lanes(cols), split_segs(cols), (int)stride) + SPLIT_STATIC_LDS <= (size_t)LDS_SCAN_BYTES &&
           // the gather addresses W by 24-bit multiplies and a 32-bit byte offset
           I + np.bias < (1 << 24) && J < (1 << 22) && (I + np.bias) * J * 4 < 0x7fffffffLL;
}

// Widest column slice (8..64) whose I rows fit in LDS (the bias row is read from memory); 0: none does.  (The split kernel's items are 32 lanes: where such
// slices are few enough for it they are taken: 512 -> 1000 of one row 4.2 + 13 -> 11.8 us with the order.)
static int slice_columns(int64_t S, int64_t I, int64_t stride, int64_t J, const NeuronParams& np, int cus) {
    const size_t rows = (size_t)I;
    int cols = 64;
    while (cols > 8 && (rows * cols * sizeof(float) > (size_t)LDS_SCAN_TARGET || cols / 2 >= J)) cols >>= 1;
    if (rows * cols * sizeof(float) > (size_t)LDS_SCAN_TARGET) return 0;
    return cols == 64 && takes_split(32, S, I, stride, J, np, cus) ? 32 : cols;
}

bool scan_sorts_rows(int64_t S, int64_t I, int64_t stride, int64_t J, const NeuronParams& np) {
    if (S <= 0 || J <= 0 || I > SPLIT_SORT_MAX) return false;
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess || scan_prepare_device(dev, &cus) != SNNTC_OK) return false;
    const int cols = slice_columns(S, I, stride, J, np, cus);
    return cols != 0 && split_sorts(cols) && takes_split(cols, S, I, stride, J, np, cus);
}

// Rows of less than a chunk, few enough that a wavefront per 64 neurons that reads its weights from memory is through sooner than
// a workgroup that copies a slice for them and sets the filter's loop up for nothing.  us, slices / memory: 4000 rows of 1 to
// 61 / 261 neurons 8.0 / 13.3 -> 6.3 / 10.1, 17 472 rows of 1 / 2 / 3 / 5 to 61 12.8 / 13.1 / 13.7 / 14.4 -> 9.8 / 11.0 / 12.2 / 14.0,
// of 1 to 261 27.9 -> 25.8; on the other side 17 472 of 2 / 5 to 128 14.5 / 17.0 -> 16.0 / 21.2, of 1 to 16 7.8 -> 8.8, where a wavefront
// of the other kernel holds several rows.
static bool takes_stream(int64_t S, int64_t I, int64_t J) {
    const int64_t waves = S * ((J + kWave - 1) / kWave);
    return I < CHUNK && (J > kWave / 2 ? waves * I <= (I == 1 ? 98304 : 53248) : waves <= 4096);
}

template <int COLS>
int launch_scan_lds(const float* sorted, const int32_t* perm, const int32_t* n_real, const float* w, float* y,
                    float* rcp, int32_t* causal_k, int64_t S, int64_t I, int64_t stride, int64_t J,
                    const NeuronParams& np_in, const TimeCopy& copy, size_t lds_bytes, int cus, hipStream_t stream) {
    NeuronParams np = np_in;
    np.wait_polls = g_wait_polls.load(std::memory_order_relaxed);
    const int n_slices = (int)((J + COLS - 1) / COLS);
    // Fewer items than CUs: a whole workgroup per item, its wavefronts sharing the item's tests.
    const int64_t split_items = (S + split_segs(COLS) - 1) / split_segs(COLS);
    const size_t split_lds = split_lds_bytes(split_lanes(COLS), split_segs(COLS), (int)stride);
    const bool split = takes_split(COLS, S, I, stride, J, np, cus);
    if (split) {
        const int64_t n_groups = split_items < cus / n_slices ? split_items : cus / n_slices;
        constexpr bool SORTS = split_sorts(COLS);
        auto kern = causal_k ? scan_lds_split_kernel<COLS, 0, true> : scan_lds_split_kernel<COLS, 0, false>;
        if (!perm) kern = I <= 512 ? scan_lds_split_kernel<COLS, SORTS ? 512 : 0, false> : scan_lds_split_kernel<COLS, SORTS ? 1024 : 0, false>;
        {
            KernelTimerScope timer_("scan", stream);
            hipLaunchKernelGGL(kern, dim3((unsigned)(n_slices * n_groups)), dim3(SPLIT_THREADS), split_lds, stream, sorted, perm,
                               n_real, w, y, rcp, causal_k, (int)S, (int)I, (int)stride, (int)J, n_slices, (int)n_groups, np,
                               copy);
        }
        SNNTC_HIP_CHECK(hipGetLastError());
        return SNNTC_OK;
    }

    const int ch = filter_neurons<COLS>(S, I, n_slices, cus);
    const int segs = kWave / COLS * ch;                     // segments per wavefront
    const int64_t items = (S + segs - 1) / segs;
    // One workgroup per CU (its 16 wavefronts take all registers; small slices let two of up to eight share a CU),
    // and as many of them as there are items for: a CU that holds few wavefronts of its own copies the slice
    // with a full workgroup all the same.  (Wavefronts by the items of a group: by those of the chip, a slice count that does not divide
    // it left a few items for a second turn, 512 rows of 333 to 1500 neurons 57.0 -> 49.4 us, 4096 to 130 58.7 -> 52.7.)
    const int64_t per_cu = (items * n_slices + cus - 1) / cus;
    const bool shared = per_cu <= 8 && (lds_bytes + FILTER_RED_BYTES) * 2 <= (size_t)LDS_SCAN_BYTES;
    const int64_t capacity = (int64_t)cus * (shared ? 2 : 1);
    int64_t n_groups = capacity / n_slices;
    if (n_groups < 1) n_groups = 1;
    const int64_t per_wg = (items + n_groups - 1) / n_groups;
    const int waves = (int)(per_wg >= 16 ? 16 : (per_wg + 3) / 4 * 4);
    const int64_t max_groups = (items + waves - 1) / waves;
    if (n_groups > max_groups) n_groups = max_groups;
    const int threads = lds_bytes > FILTER_WIDE_COPY_BYTES && !shared ? LDS_SCAN_THREADS : waves * kWave;
    const bool lone = filter_lone<COLS>(ch, (items + std::max(cus / n_slices, 1) - 1) / std::max(cus / n_slices, 1), I);
    const bool rounds = I >= (lone ? LONE_ROUNDS_FROM : ROUNDS_FROM);
    // Staged where the row entries of all its wavefronts fit beside the slice, broadcasts elsewhere: fewer wavefronts lose more than the
    // broadcasts cost.  us of the layer, its order included, fewer staged wavefronts (eight up to 608 inputs, four up to 624, then two
    // neurons per lane) / broadcasts: 65 536 segments of 600, 616 and 638 to 64 neurons 446 / 415, 643 / 417, 553 / 452, 4096 of 620 to 800 408 / 210,
    // 1024 of 600 to 800 78 / 71.
    const size_t staged_lds = lds_bytes + (size_t)waves * FILTER_STAGE_BYTES;
    const bool staged = FILTER_STAGES<COLS> && ch == FILTER_MAX_CH<COLS> && staged_lds * (shared ? 2 : 1) <= (size_t)LDS_SCAN_BYTES;
    auto kern = causal_k ? filter_kernel<COLS, true>(ch, lone, rounds, staged) : filter_kernel<COLS, false>(ch, lone, rounds, staged);
    {
        KernelTimerScope timer_("scan", stream);
        hipLaunchKernelGGL(kern, dim3((unsigned)(n_slices * n_groups)), dim3((unsigned)threads), staged ? staged_lds : lds_bytes + FILTER_RED_BYTES, stream,
                           sorted, perm, n_real, w, y, rcp, causal_k, (int)S, (int)I, (int)stride, (int)J, n_slices, (int)n_groups,
                           waves, np, copy);
    }
    SNNTC_HIP_CHECK(hipGetLastError());
    return SNNTC_OK;
}

int launch_scan(const float* sorted, const int32_t* perm, const int32_t* n_real, const float* w, float* y,
                float* rcp, int32_t* causal_k, int64_t S, int64_t I, int64_t stride, int64_t J,
                const NeuronParams& np, const TimeCopy& copy, hipStream_t stream) {
    if (S <= 0 || J <= 0) return SNNTC_OK;
    int dev = 0, cus = 0;
    SNNTC_HIP_CHECK(hipGetDevice(&dev));
    const int prep = scan_prepare_device(dev, &cus);
    if (prep) return prep;
    const int cols = slice_columns(S, I, stride, J, np, cus);            // none: W is streamed from memory
    const size_t lds_bytes = (size_t)I * cols * sizeof(float);
    if (cols && !takes_stream(S, I, J)) {
        switch (cols) {
            case 64: return launch_scan_lds<64>(sorted, perm, n_real, w, y, rcp, causal_k, S, I, stride, J, np, copy, lds_bytes, cus, stream);
            case 32: return launch_scan_lds<32>(sorted, perm, n_real, w, y, rcp, causal_k, S, I, stride, J, np, copy, lds_bytes, cus, stream);
            case 16: return launch_scan_lds<16>(sorted, perm, n_real, w, y, rcp, causal_k, S, I, stride, J, np, copy, lds_bytes, cus, stream);
            default: return launch_scan_lds<8>(sorted, perm, n_real, w, y, rcp, causal_k, S, I, stride, J, np, copy, lds_bytes, cus, stream);
        }
    }
    const int j_blocks = (int)((J + kWave - 1) / kWave);
    const int64_t n_items = S * j_blocks;
    const int waves_per_block = 4;
    const int64_t blocks = (n_items + waves_per_block - 1) / waves_per_block;
    if (blocks > 0x7fffffffLL) return fail(SNNTC_ERR_TOO_LARGE, "scan: grid too large");
    dim3 grid((unsigned)blocks), block(waves_per_block * kWave);
    {
        KernelTimerScope timer_("scan_stream", stream);
        if (causal_k)
            hipLaunchKernelGGL(scan_kernel<true>, grid, block, 0, stream, sorted, perm, n_real, w, y, rcp,
                               causal_k, n_items, (int)I, (int)stride, (int)J, j_blocks, np, copy);
        else
            hipLaunchKernelGGL(scan_kernel<false>, grid, block, 0, stream, sorted, perm, n_real, w, y, rcp,
                               causal_k, n_items, (int)I, (int)stride, (int)J, j_blocks, np, copy);
    }
    SNNTC_HIP_CHECK(hipGetLastError());
    return SNNTC_OK;
}

int launch_unpad_rows(const float* sorted, const int32_t* perm, float* sorted_out, int32_t* perm_out,
                      int64_t S, int64_t I, int64_t stride, hipStream_t stream) {
    const int64_t n = S * I;
    if (n <= 0 || (!sorted_out && !perm_out)) return SNNTC_OK;
    {
        KernelTimerScope timer_("unpad_rows", stream);
        hipLaunchKernelGGL(unpad_rows_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream, sorted,
                           perm, sorted_out, perm_out, n, (int)I, (int)stride);
    }
    SNNTC_HIP_CHECK(hipGetLastError());
    return SNNTC_OK;
}

}  // namespace snntc
