// Backward kernels of the dense and conv SNN-TC layers.
//
// Contract (snntc/snnfcgrad_kernels.cu.cc:60,118-120,159-173; snntc/snncvgrad_kernels.cu.cc:71,143,
// 190-204), with up = grad[:S] * oldout[S:], MAXc = MAX_SPIKE_TIME - 0.1:
//   dX[s,i] = sum_j [x_si <= y_sj and y_sj <= MAXc] up_sj * W[i,j]
//   dW[i,j] = sum_s [x_si <= MAXc and y_sj <= MAXc and x_si <= y_sj] (x_si - y_sj) * up_sj
//   dW[I,j] = the same with x = biasvolt (bias row)
// For the conv layer s runs over output pixels and x_si is gathered from the padded image; dX is
// accumulated in gather form (every input pixel sums over the output pixels whose window covers
// it), so no atomics are needed and the result does not depend on scheduling.
//
// The validity test on y is folded into one array prepared once per call,
//   upm = valid ? up : 0,
// so that a term of an output that takes no part vanishes whatever its mask says (the kernels read y
// itself, under the parameter name ym); the weight-gradient mask is folded into arithmetic: for x <= y the term (x-y) is <= 0 and
// for x > y it is > 0, hence [x <= y](x - y) == min(x - y, 0).
#include <algorithm>
#include <atomic>

#include "snntc_common.h"

namespace snntc {
namespace {

// First launch of a backward pass.  The elementwise pass over the layer's outputs,
//   upm = valid ? grad * rcp : 0   (valid: y <= MAX - 0.1),
// and the regrouped weights the channel-lane dX of conv layers reads do not depend on each other: one launch does both, the
// first prep_blocks workgroups the former, the rest the latter.
//   w[(tap, c), kc] -> wt[tap][kc / 4][c][kc % 4], one 16-byte piece per thread (cols = Kc, a multiple of 4; chan = C)
__global__ void __launch_bounds__(256)
backward_prologue_kernel(const float* __restrict__ grad, const float* __restrict__ y,
                         const float* __restrict__ rcp, float* __restrict__ upm, int64_t n, float max_cmp,
                         int prep_blocks, int vec4, const float* __restrict__ w,
                         float* __restrict__ wt, int rows, int cols, int chan, float* __restrict__ zeros,
                         int n_zeros) {
    if (blockIdx.x == 0 && (int)threadIdx.x < n_zeros) zeros[threadIdx.x] = 0.0f;    // the dParams output
    if ((int)blockIdx.x < prep_blocks) {
        const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
        if (vec4) {                                      // n a multiple of 4, the arrays 16-byte aligned
            if (4 * t >= n) return;
            const float4 yv = reinterpret_cast<const float4*>(y)[t], gv = reinterpret_cast<const float4*>(grad)[t];
            const float4 rv = reinterpret_cast<const float4*>(rcp)[t];
            float4 u;
            u.x = yv.x <= max_cmp ? gv.x * rv.x : 0.0f;
            u.y = yv.y <= max_cmp ? gv.y * rv.y : 0.0f;
            u.z = yv.z <= max_cmp ? gv.z * rv.z : 0.0f;
            u.w = yv.w <= max_cmp ? gv.w * rv.w : 0.0f;
            reinterpret_cast<float4*>(upm)[t] = u;
            return;
        }
        if (t >= n) return;
        const float yv = y[t];
        const bool valid = yv <= max_cmp;
        upm[t] = valid ? grad[t] * rcp[t] : 0.0f;
        return;
    }
    const int blk = (int)blockIdx.x - prep_blocks;
    const int k4 = cols / 4;
    const int64_t t = (int64_t)blk * blockDim.x + threadIdx.x;    // over (tap, c, kc / 4), kc / 4 fastest
    if (t >= (int64_t)rows * k4) return;
    const int64_t row = t / k4;                                   // tap * C + c
    const int q = (int)(t - row * k4);
    const int64_t tap = row / chan;
    const int c = (int)(row - tap * chan);
    reinterpret_cast<float4*>(wt)[(tap * k4 + q) * chan + c] = reinterpret_cast<const float4*>(w)[t];
}

__global__ void __launch_bounds__(256) fill_zero_kernel(float* __restrict__ p, int64_t n) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t < n) p[t] = 0.0f;
}

// Source offset of weight row e relative to the segment base (dense: the column; conv: kh/kw/c).
__device__ __forceinline__ int row_offset(const SegmentSource& src, int e) {
    if (!src.conv) return e;
    const int span = src.Kw * src.C;
    const int kh = e / span;
    return kh * src.W * src.C + (e - kh * span);
}

// Base of segment s inside the source tensor.
__device__ __forceinline__ const float* segment_base(const SegmentSource& src, int s) {
    if (!src.conv) return src.base + (size_t)s * src.I;
    const int per_img = src.Nh * src.Nw;
    const int a = s / per_img, r2 = s - a * per_img;
    const int nh = r2 / src.Nw, nw = r2 - nh * src.Nw;
    return src.base + ((size_t)(a * src.H + nh * src.Sh) * src.W + (size_t)nw * src.Sw) * src.C;
}

// The wavefront's own LDS traffic in program order: what it has written so far is what it reads from here on.
__device__ __forceinline__ void wave_lds_order() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// ---------------------------------------------------------------------------------------------
// Dense dX.  A wavefront owns a tile of 16 samples x 32 inputs, a lane 2 x 4 of it, and walks over outputs j, 16 at a time:
// y, up and W of its rows come in 16-byte pieces, a chunk ahead, go to a piece of LDS of the wavefront's own, transposed, and
// come back as three reads per output, one output ahead, for 24 vector instructions.  SPLIT wavefronts share a tile's outputs
// and are added in order through LDS; with SPLIT 1 the four wavefronts of a workgroup have tiles of their own.
// What bounds it: the compare, multiply-add and select of a term (3.3 clocks each at 4096 samples).  Before, one input and
// four samples per lane, a transposed copy of W streamed past scalar y / up: four samples per weight read, and lines of the
// scalar cache fetched four times over.  us: 333 x 1521 -> 777 60 -> 46, 4096 x 784 -> 800 519 -> 239, 256 x 784 -> 800 31 ->
// 25, 128 x 784 -> 800 20 -> 16, 16 200 patches x 500 -> 50 46 -> 27, and the copy, some 2.  (4 x 4 per lane: 228 at 4096 samples, 61
// at 333.)
// ---------------------------------------------------------------------------------------------
constexpr int DX_A = 2, DX_S = 8 * DX_A, DX_I = 32, DX_JC = 16, DX_PITCH = 36;         // (pitch: the transposing writes of the pieces spread over the banks)
constexpr int dx_threads(int split) { return (split == 1 ? 4 : split) * kWave; }     // (single-wavefront tiles of a joint launch: eight wavefronts)
constexpr int dx_lds_bytes(int split) { return dx_threads(split) / kWave * 3 * DX_JC * DX_PITCH * 4; }

// Upstream values of a backward pass: the prologue's, or (RAW) formed where they are staged, which saves small batches a launch.
struct Upstream {
    const float* up;                                       // upm, or grad
    const float* rcp;
    float max_cmp;
};
template <bool RAW, class V>
__device__ __forceinline__ V upstream_value(V up, V rcp, V y, float max_cmp) {
    if constexpr (!RAW) return up;
    else if constexpr (sizeof(V) == sizeof(float)) return y <= max_cmp ? up * rcp : 0.0f;
    else {
        V u;
#pragma unroll
        for (int q = 0; q < (int)(sizeof(V) / sizeof(float)); ++q) u[q] = y[q] <= max_cmp ? up[q] * rcp[q] : 0.0f;
        return u;
    }
}

// PATCHES: the "samples" are the implicit patches of a conv layer (src.conv) and the
// result is the gradient per patch element, dx[S, P], which cv_col2im_kernel then folds back onto the image.
template <int SPLIT, bool PATCHES, bool RAW>
__device__ __forceinline__ void
fc_grad_input_tile(const SegmentSource& src, const float* __restrict__ w, const Upstream& upstream, const float* __restrict__ ym,
                   float* __restrict__ dx, int B, int I, int J, int tiles_i, int n_tiles, int block_index, int blocks, float* dx_lds) {
    constexpr int A = DX_A, TS = DX_S, LANES = DX_JC / 4, ROWS = kWave / LANES, S_PASSES = TS / ROWS, I_PASSES = DX_I / ROWS;
    static_assert(S_PASSES * ROWS == TS && I_PASSES * ROWS == DX_I, "whole passes");
    const int lane = threadIdx.x % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int block = xcd_contiguous(block_index, blocks);
    const int tile_raw = SPLIT == 1 ? block * (int)(blockDim.x / kWave) + wave : block;
    const int tile = min(tile_raw, n_tiles - 1);
    const int ts = tile / tiles_i, s0 = ts * TS, i0 = (tile - ts * tiles_i) * DX_I;
    const int sg = lane / 8, ig = lane % 8;

    float xr[A][4], acc[A][4];
#pragma unroll
    for (int a = 0; a < A; ++a) {
        const int s = min(s0 + sg * A + a, B - 1);
        const float* xs = PATCHES ? segment_base(src, s) : src.base + (size_t)s * I;
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            const int i = min(i0 + ig * 4 + b, I - 1);
            xr[a][b] = xs[PATCHES ? row_offset(src, i) : i];
            acc[a][b] = 0.0f;
        }
    }
    // A sample's sums must not depend on the batch it is in, so the order of its additions depends on J alone: chunk c of the
    // outputs belongs to part c % 16, a part's chunks are added in turn, parts p and p + 8, the pairs p and p + 4, ... in a
    // tree -- which a wavefront with parts v, v + 8 (, v + 4, v + 12) begins.  Fewer than 64 outputs are one part.
    constexpr int PARTS = SPLIT == 1 ? 1 : 16 / SPLIT, STEP = SPLIT == 1 ? 1 : 16;
    const int chunks = (J + DX_JC - 1) / DX_JC;
    auto part = [&](int k) { return SPLIT == 1 ? 0 : wave + (k & 1) * 8 + (k >> 1) * 4; };
    auto next_chunk = [&](int k, int c) {                   // behind chunk c of the k-th part; chunks if there is none
        if (c + STEP < chunks) return c + STEP;
        int next = chunks;
#pragma unroll
        for (int m = PARTS - 1; m > 0; --m)
            if (m > k && part(m) < chunks) next = part(m);
        return next;
    };
    const int pr = lane / LANES, pj = lane % LANES * 4;     // the lane's piece: row pr (+ ROWS per pass), outputs pj ... + 3
    typedef float f4 __attribute__((ext_vector_type(4)));
    typedef float fa __attribute__((ext_vector_type(A)));
    f4 yv[S_PASSES], uv[S_PASSES], rv[S_PASSES], wv[I_PASSES];
    const float* __restrict__ upm = upstream.up;
    const float* __restrict__ rcp = upstream.rcp;
    typedef float f4_any __attribute__((ext_vector_type(4), aligned(4)));             // (four floats need no more alignment than one)
    auto piece = [&](const float* row, int j, bool whole) {
        f4 v;
        if (whole) {
            v = *reinterpret_cast<const f4_any*>(row + j);
        } else {
#pragma unroll
            for (int q = 0; q < 4; ++q) v[q] = row[min(j + q, J - 1)];
        }
        return v;
    };
    auto request = [&](int j0) {
        const bool whole = j0 + DX_JC <= J;
#pragma unroll
        for (int t = 0; t < S_PASSES; ++t) {
            const size_t row = (size_t)min(s0 + t * ROWS + pr, B - 1) * J;
            yv[t] = piece(ym + row, j0 + pj, whole);
            uv[t] = piece(upm + row, j0 + pj, whole);
            if constexpr (RAW) rv[t] = piece(rcp + row, j0 + pj, whole);
        }
#pragma unroll
        for (int t = 0; t < I_PASSES; ++t) wv[t] = piece(w + (size_t)min(i0 + t * ROWS + pr, I - 1) * J, j0 + pj, whole);
    };
    float* ys = dx_lds + wave * 3 * DX_JC * DX_PITCH;       // [output][sample | sample | input]
    float* us = ys + DX_JC * DX_PITCH;
    float* ws = us + DX_JC * DX_PITCH;
    float total[A][4], pair[A][4];
    if (part(0) < chunks) request(part(0) * DX_JC);
#pragma unroll
    for (int k = 0; k < PARTS; ++k) {
        for (int c = part(k); c < chunks; c += STEP) {
            const int j0 = c * DX_JC;
#pragma unroll
            for (int t = 0; t < S_PASSES; ++t) uv[t] = upstream_value<RAW>(uv[t], rv[t], yv[t], upstream.max_cmp);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const bool in = j0 + pj + q < J;                // outputs past the end take no part
#pragma unroll
                for (int t = 0; t < S_PASSES; ++t) {
                    ys[(pj + q) * DX_PITCH + t * ROWS + pr] = in ? yv[t][q] : -INFINITY;
                    us[(pj + q) * DX_PITCH + t * ROWS + pr] = in ? uv[t][q] : 0.0f;
                }
#pragma unroll
                for (int t = 0; t < I_PASSES; ++t) ws[(pj + q) * DX_PITCH + t * ROWS + pr] = wv[t][q];
            }
            const int next = next_chunk(k, c);
            if (next < chunks) request(next * DX_JC);
            wave_lds_order();
            fa y[2], u[2];
            f4 wj[2];
            auto fetch = [&](int b, int j) {
                y[b] = *reinterpret_cast<const fa*>(ys + j * DX_PITCH + sg * A);
                u[b] = *reinterpret_cast<const fa*>(us + j * DX_PITCH + sg * A);
                wj[b] = *reinterpret_cast<const f4*>(ws + j * DX_PITCH + ig * 4);
            };
            fetch(0, 0);
#pragma unroll
            for (int j = 0; j < DX_JC; ++j) {
                const int b2 = j & 1;
                if (j + 1 < DX_JC) fetch(b2 ^ 1, j + 1);
                __builtin_amdgcn_sched_barrier(0);
                // acc += up * w where x <= y; the others are skipped, as in the reference (snnfcgrad_kernels.cu.cc:60), not
                // added as zeros
#pragma unroll
                for (int a = 0; a < A; ++a)
#pragma unroll
                    for (int b = 0; b < 4; ++b)
                        acc[a][b] = xr[a][b] <= y[b2][a] ? __fmaf_rn(u[b2][a], wj[b2][b], acc[a][b]) : acc[a][b];
            }
            wave_lds_order();
        }
#pragma unroll
        for (int a = 0; a < A; ++a)
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                if (k == 0) total[a][b] = acc[a][b];
                else if (k == 1) total[a][b] += acc[a][b];
                else if (k == 2) pair[a][b] = acc[a][b];
                else total[a][b] += pair[a][b] + acc[a][b];
                acc[a][b] = 0.0f;
            }
    }
    if constexpr (SPLIT == 1) {
        if (tile_raw >= n_tiles) return;
#pragma unroll
        for (int a = 0; a < A; ++a)
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                const int s = s0 + sg * A + a, i = i0 + ig * 4 + b;
                if (s < B && i < I) dx[(size_t)s * I + i] = total[a][b];
            }
    } else {
        __syncthreads();
        float* red = dx_lds + wave * TS * DX_I;             // [wave][sample][input]
#pragma unroll
        for (int a = 0; a < A; ++a)
            *reinterpret_cast<f4*>(red + (sg * A + a) * DX_I + ig * 4) = f4{total[a][0], total[a][1], total[a][2], total[a][3]};
        __syncthreads();
        for (int e = threadIdx.x; e < TS * DX_I; e += dx_threads(SPLIT)) {
            const int s = s0 + e / DX_I, i = i0 + e % DX_I;
            float sum[SPLIT];
#pragma unroll
            for (int v = 0; v < SPLIT; ++v) sum[v] = dx_lds[v * TS * DX_I + e];
#pragma unroll
            for (int h = SPLIT / 2; h > 0; h /= 2)
#pragma unroll
                for (int v = 0; v < h; ++v) sum[v] += sum[v + h];
            if (s < B && i < I) dx[(size_t)s * I + i] = sum[0];
        }
    }
}

template <int SPLIT, bool PATCHES>
__global__ void __launch_bounds__(dx_threads(SPLIT), 4)
fc_grad_input_kernel(const SegmentSource src, const float* __restrict__ w, const float* __restrict__ upm,
                     const float* __restrict__ ym, float* __restrict__ dx, int B, int I, int J, int tiles_i, int n_tiles) {
    extern __shared__ __align__(16) float dx_lds[];
    fc_grad_input_tile<SPLIT, PATCHES, false>(src, w, Upstream{upm, nullptr, 0.0f}, ym, dx, B, I, J, tiles_i, n_tiles, blockIdx.x,
                                              gridDim.x, dx_lds);
}

// ---------------------------------------------------------------------------------------------
// dW for implicit conv patches.  Lanes run across outputs j (y/up rows are read
// coalesced); each thread carries RI consecutive weight rows whose x values are wave-uniform.
// The segment range is cut into gridDim.z slices; a slice is further split over the four
// wavefronts of the block.  With more than one slice the per-slice sums go to `partial` and are
// added in slice order by reduce_partials_kernel.
// ---------------------------------------------------------------------------------------------
constexpr int DW_RI = 8;
constexpr int DW_UNROLL = 4;

__global__ void __launch_bounds__(256)
grad_weight_kernel(SegmentSource src, const float* __restrict__ upm, const float* __restrict__ ym,
                   float* __restrict__ dst, int S, int J, int rows, int seg_per_slice,
                   float biasvolt, float neg_s, float post) {
    __shared__ float red[3][DW_RI][kWave];
    const int lane = threadIdx.x % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int j = blockIdx.x * kWave + lane;
    const unsigned jc = (unsigned)min(j, J - 1);
    const int i0 = blockIdx.y * DW_RI;
    const int I = src.I;

    const int s_begin = blockIdx.z * seg_per_slice;
    const int s_end = min(S, s_begin + seg_per_slice);
    const int per_wave = (s_end - s_begin + 3) / 4;
    const int s_lo = s_begin + wave * per_wave;
    const int s_hi = min(s_end, s_lo + per_wave);

    float acc[DW_RI];
#pragma unroll
    for (int r = 0; r < DW_RI; ++r) acc[r] = 0.0f;
    const float* __restrict__ ycol = ym + jc;
    const float* __restrict__ ucol = upm + jc;

    // The RI weight rows of this block are contiguous in the source (always for dense rows, for
    // patches when the rows share one (kh, kw)): their x values come as one scalar fetch.
    const bool contiguous = i0 + DW_RI <= I && (!src.conv || (i0 % src.C) + DW_RI <= src.C);
    if (contiguous) {
        const int off0 = row_offset(src, i0);
        int s = s_lo;
        for (; s + DW_UNROLL <= s_hi; s += DW_UNROLL) {
            float yv[DW_UNROLL], uv[DW_UNROLL];
            const float* xb[DW_UNROLL];
#pragma unroll
            for (int u = 0; u < DW_UNROLL; ++u) {
                yv[u] = ycol[(size_t)(s + u) * J] * -neg_s;
                uv[u] = ucol[(size_t)(s + u) * J];
                xb[u] = segment_base(src, s + u) + off0;
            }
#pragma unroll
            for (int u = 0; u < DW_UNROLL; ++u) {
#pragma unroll
                for (int r = 0; r < DW_RI; ++r)
                    acc[r] = __fmaf_rn(scaled_lead(xb[u][r], neg_s, yv[u]), uv[u], acc[r]);
            }
        }
        for (; s < s_hi; ++s) {
            const float yv = ycol[(size_t)s * J] * -neg_s, uv = ucol[(size_t)s * J];
            const float* xb = segment_base(src, s) + off0;
#pragma unroll
            for (int r = 0; r < DW_RI; ++r) acc[r] = __fmaf_rn(scaled_lead(xb[r], neg_s, yv), uv, acc[r]);
        }
    } else {
        int off[DW_RI];
        bool is_bias[DW_RI];
#pragma unroll
        for (int r = 0; r < DW_RI; ++r) {
            const int i = min(i0 + r, rows - 1);
            is_bias[r] = i >= I;
            off[r] = row_offset(src, min(i, I - 1));
        }
        for (int s = s_lo; s < s_hi; ++s) {
            const float yv = ycol[(size_t)s * J] * -neg_s, uv = ucol[(size_t)s * J];
            const float* xb = segment_base(src, s);
#pragma unroll
            for (int r = 0; r < DW_RI; ++r) {
                const float xv = is_bias[r] ? biasvolt : xb[off[r]];
                acc[r] = __fmaf_rn(scaled_lead(xv, neg_s, yv), uv, acc[r]);
            }
        }
    }
    if (wave > 0) {
#pragma unroll
        for (int r = 0; r < DW_RI; ++r) red[wave - 1][r][lane] = acc[r];
    }
    __syncthreads();
    if (wave == 0 && j < J) {
        float* out = dst + (size_t)blockIdx.z * rows * J;
#pragma unroll
        for (int r = 0; r < DW_RI; ++r) {
            if (i0 + r < rows)
                out[(size_t)(i0 + r) * J + j] =
                    (((acc[r] + red[0][r][lane]) + red[1][r][lane]) + red[2][r][lane]) * post;
        }
    }
}

// ---------------------------------------------------------------------------------------------
// dW of a dense layer.  A workgroup owns 64 weight rows x 64 outputs, its wavefronts take the slice's samples eight at a
// time in turn, a lane 8 x 8 of the tile: a sample's 64 inputs, output times and upstream values are three coalesced loads, a
// batch ahead, go to a piece of LDS of the wavefront's own and come back as six 16-byte reads for 128 vector instructions.
// Rows past the inputs read biasvolt, so the bias row needs no code of its own.  The wavefronts' sums are added in a tree
// through LDS.  FOLDS: and begun anew every `fold` turns (a batch per wavefront each), so that no chain of additions is long.
// What bounds it: the addition and the multiply-add of a term (3.3 clocks each at 4096 samples).  Before, eight rows and one
// output per lane: two LDS reads of 8 clocks and 512 bytes of y / up per 16 instructions.  us: 4096 x 784 -> 800 254 -> 158,
// 1024 rows 69 -> 47 (both + 6 for adding up slices), 333 x 1521 -> 777 48 -> 40, 128 x 784 -> 800 15 -> 13.  (The times are scaled as they
// are staged: a sum of two registers issues faster than a multiply-add of three, 225 us.)
// ---------------------------------------------------------------------------------------------
constexpr int DWD_T = 64, DWD_BATCH = 4, DWD_TURN = 8 * DWD_BATCH;       // (a turn: samples that eight wavefronts take together)

// staging: [wave][sample][x 64 | y 64 | up 64]; sums: [wave][row 32][output 64], half a tile at a time
constexpr int DWD_STAGE = DWD_BATCH * 3 * DWD_T, DWD_SUMS = DWD_T / 2 * DWD_T;
constexpr int dwd_lds_floats(int waves) { return waves * (DWD_STAGE > DWD_SUMS ? DWD_STAGE : DWD_SUMS); }

template <int WAVES, bool RAW, bool FOLDS>
__device__ __forceinline__ void
grad_weight_dense_tile(const float* __restrict__ x, const Upstream& upstream, const float* __restrict__ ym, float* __restrict__ dst,
                       int S, int I, int J, int rows, int seg_per_slice, int fold, float biasvolt, float neg_s, float post, int bx, int by,
                       int bz, float* lds) {
    constexpr int STAGE = DWD_STAGE, SUMS = DWD_SUMS, MINE = SUMS / (WAVES * kWave);
    typedef float f4 __attribute__((ext_vector_type(4)));
    const int lane = threadIdx.x % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int j0 = bx * DWD_T, i0 = by * DWD_T;
    const int s_begin = bz * seg_per_slice, s_end = min(S, s_begin + seg_per_slice);
    const int rg = lane / 8, cg = lane % 8;

    const bool is_input = i0 + lane < I;
    const float* __restrict__ xcol = x + min(i0 + lane, I - 1);
    const int jc = min(j0 + lane, J - 1);
    const float* __restrict__ ycol = ym + jc;
    const float* __restrict__ ucol = upstream.up + jc;
    const float* __restrict__ rcol = RAW ? upstream.rcp + jc : nullptr;
    float* stage = lds + wave * STAGE;

    float acc[8][8];
#pragma unroll
    for (int r = 0; r < 8; ++r)
#pragma unroll
        for (int c = 0; c < 8; ++c) acc[r][c] = 0.0f;
    float xv[DWD_BATCH], yv[DWD_BATCH], uv[DWD_BATCH], rv[DWD_BATCH];
    auto request = [&](int sb) {
#pragma unroll
        for (int q = 0; q < DWD_BATCH; ++q) {
            const int s = min(sb + q, s_end - 1);
            xv[q] = xcol[(size_t)s * I];
            yv[q] = ycol[(size_t)s * J];
            uv[q] = ucol[(size_t)s * J];
            rv[q] = 0.0f;
            if constexpr (RAW) rv[q] = rcol[(size_t)s * J];
        }
    };
    float total[FOLDS ? 2 * MINE : 1];                      // of the thread's elements of a tile
    // Adds up the wavefronts' sums, half a tile at a time: f(half, n, sum) for the thread's n-th element of it.
    auto add_up = [&](auto&& f) __attribute__((always_inline)) {
#pragma unroll
        for (int half = 0; half < 2; ++half) {
            __syncthreads();                                // (the staging, or the first half, has been read)
            float* mine = lds + wave * SUMS;
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int h = 0; h < 2; ++h)
                    *reinterpret_cast<f4*>(mine + (rg * 4 + r) * DWD_T + cg * 8 + 4 * h) =
                        f4{acc[4 * half + r][4 * h], acc[4 * half + r][4 * h + 1], acc[4 * half + r][4 * h + 2], acc[4 * half + r][4 * h + 3]};
            __syncthreads();
#pragma unroll
            for (int n = 0; n < MINE; ++n) {
                float sum[WAVES];
#pragma unroll
                for (int v = 0; v < WAVES; ++v) sum[v] = lds[v * SUMS + n * WAVES * kWave + threadIdx.x];
#pragma unroll
                for (int h = WAVES / 2; h > 0; h /= 2)
#pragma unroll
                    for (int v = 0; v < h; ++v) sum[v] += sum[v + h];
                f(half, n, sum[0]);
            }
        }
    };
    if constexpr (FOLDS)
#pragma unroll
        for (int n = 0; n < 2 * MINE; ++n) total[n] = 0.0f;
    int sb = s_begin + wave * DWD_BATCH, fold_at = s_begin + fold * WAVES * DWD_BATCH;
    if (sb < s_end) request(sb);
    for (; sb < s_end; sb += WAVES * DWD_BATCH) {
        if constexpr (FOLDS)
            if (sb - wave * DWD_BATCH == fold_at && fold_at + (WAVES - 1) * DWD_BATCH < s_end) {      // (all wavefronts or none: each has a batch in this turn)
                add_up([&](int half, int n, float sum) __attribute__((always_inline)) { total[half * MINE + n] += sum; });
#pragma unroll
                for (int r = 0; r < 8; ++r)
#pragma unroll
                    for (int c = 0; c < 8; ++c) acc[r][c] = 0.0f;
                fold_at += fold * WAVES * DWD_BATCH;
                __syncthreads();
            }
#pragma unroll
        for (int q = 0; q < DWD_BATCH; ++q) {
            stage[q * 3 * DWD_T + lane] = (is_input ? xv[q] : biasvolt) * neg_s;
            stage[q * 3 * DWD_T + DWD_T + lane] = yv[q] * -neg_s;
            stage[q * 3 * DWD_T + 2 * DWD_T + lane] = sb + q < s_end ? upstream_value<RAW>(uv[q], rv[q], yv[q], upstream.max_cmp) : 0.0f;       // samples past the end weigh nothing
        }
        if (sb + WAVES * DWD_BATCH < s_end) request(sb + WAVES * DWD_BATCH);
        wave_lds_order();
#pragma unroll 2
        for (int q = 0; q < DWD_BATCH; ++q) {
            const float* at = stage + q * 3 * DWD_T;
            float xr[8], yr[8], ur[8];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const f4 a = *reinterpret_cast<const f4*>(at + rg * 8 + 4 * h);
                const f4 b = *reinterpret_cast<const f4*>(at + DWD_T + cg * 8 + 4 * h);
                const f4 c = *reinterpret_cast<const f4*>(at + 2 * DWD_T + cg * 8 + 4 * h);
#pragma unroll
                for (int e = 0; e < 4; ++e) { xr[4 * h + e] = a[e]; yr[4 * h + e] = b[e]; ur[4 * h + e] = c[e]; }
            }
#pragma unroll
            for (int r = 0; r < 8; ++r)
#pragma unroll
                for (int c = 0; c < 8; ++c)
                    acc[r][c] = __fmaf_rn(__builtin_amdgcn_fmed3f(xr[r] + yr[c], 0.0f, 1.0f), ur[c], acc[r][c]);
        }
        wave_lds_order();
    }
    float* out = dst + (size_t)bz * rows * J;
    add_up([&](int half, int n, float sum) __attribute__((always_inline)) {
        const int e = n * WAVES * kWave + threadIdx.x;
        const int tr = e / DWD_T, i = i0 + tr / 4 * 8 + 4 * half + tr % 4, j = j0 + e % DWD_T;
        if constexpr (FOLDS) sum = total[half * MINE + n] + sum;
        if (i < rows && j < J) out[(size_t)i * J + j] = sum * post;
    });
}

template <int WAVES>
__global__ void __launch_bounds__(WAVES * kWave, 4)
grad_weight_dense_kernel(const float* __restrict__ x, const float* __restrict__ upm, const float* __restrict__ ym,
                         float* __restrict__ dst, int S, int I, int J, int rows, int seg_per_slice, float biasvolt,
                         float neg_s, float post) {
    __shared__ __align__(16) float lds[dwd_lds_floats(WAVES)];
    grad_weight_dense_tile<WAVES, false, false>(x, Upstream{upm, nullptr, 0.0f}, ym, dst, S, I, J, rows, seg_per_slice, 0, biasvolt, neg_s, post,
                                                blockIdx.x, blockIdx.y, blockIdx.z, lds);
}

// The whole backward pass of a dense layer on a small batch in one launch: dX tiles of eight wavefronts (below 64 outputs, SPLIT 1, eight
// tiles of one) and dW tiles, which both form the upstream values as they stage them.  Each part alone leaves the chip half empty and waits
// for its first loads.  us, prologue, dX and dW (and the sum of its slices) / together, 784 -> 800: 1 row 18.5 / 14.0, 64 rows 22 / 16, 128
// 27 / 19.5, 256 41.5 / 35, 400 57 / 49; 128 rows of 2048 -> 512 35 / 30, of 128 -> 128 16.5 / 10.6, of 784 -> 100 26.4 / 12.6, of 500 -> 50 29.5 / 12.8.
template <int SPLIT, bool FOLDS>
__global__ void __launch_bounds__(8 * kWave, 4)
fc_backward_kernel(const float* __restrict__ x, const float* __restrict__ w, const float* __restrict__ grad, const float* __restrict__ y,
                   const float* __restrict__ rcp, float* __restrict__ dx, float* __restrict__ dw, float* __restrict__ zeros, int n_zeros,
                   int B, int I, int J, int rows, int tiles_i, int dx_tiles, int dx_blocks, int dx_first, int dw_cols, int fold, float max_cmp, float biasvolt, float neg_s,
                   float post) {
    constexpr int FLOATS = dwd_lds_floats(8) > dx_lds_bytes(8) / 4 ? dwd_lds_floats(8) : dx_lds_bytes(8) / 4;
    __shared__ __align__(16) float lds[FLOATS];
    const Upstream upstream{grad, rcp, max_cmp};
    if (blockIdx.x == 0 && (int)threadIdx.x < n_zeros) zeros[threadIdx.x] = 0.0f;          // the dParams output
    const int dx_block = (int)blockIdx.x - dx_first;
    if (dx_block >= 0 && dx_block < dx_blocks) {
        SegmentSource src{};
        src.base = x; src.conv = 0; src.I = I;
        fc_grad_input_tile<SPLIT, false, true>(src, w, upstream, y, dx, B, I, J, tiles_i, dx_tiles, dx_block, dx_blocks, lds);
    } else {
        const int tile = dx_block < 0 ? (int)blockIdx.x : dx_block - dx_blocks, by = tile / dw_cols;
        grad_weight_dense_tile<8, true, FOLDS>(x, upstream, y, dw, B, I, J, rows, B, fold, biasvolt, neg_s, post, tile - by * dw_cols, by, 0, lds);
    }
}

// ---------------------------------------------------------------------------------------------
// Whole backward pass of a dense layer with few outputs (a classifier head: J <= 16) in one launch:
// the masked upstream values, dX and dW.  A wavefront covers 16 weight rows i (the bias row is one
// more row, with x = biasvolt and no dX) times four groups of JL adjacent columns: lane = (group,
// row).  A block takes up to NARROW_SAMPLES samples, whose scaled output times and upstream values
// it first puts into LDS; each of its wavefronts then walks every NARROW_WAVES-th sample.  dX[b, i]
// is complete after a sample -- the four column groups are added in the order (0 + 1) + (2 + 3) --
// and is stored at once; the dW sums of a lane run over the samples and are added across the
// wavefronts in wavefront order at the end.  Both inputs of the comparison x <= y are scaled by
// the same power of two, which does not change its outcome.  With more than one block of samples
// the dW sums go to `dst` as slices for reduce_partials_kernel.
// ---------------------------------------------------------------------------------------------
constexpr int NARROW_GROUPS = 4;
constexpr int NARROW_ROWS = kWave / NARROW_GROUPS;     // weight rows per block
constexpr int NARROW_JMAX = 4 * NARROW_GROUPS;
constexpr int NARROW_WAVES = 16;
constexpr int NARROW_SAMPLES = 256;

template <int JL>
__global__ void __launch_bounds__(NARROW_WAVES * kWave)
fc_backward_narrow_kernel(const float* __restrict__ x, const float* __restrict__ w,
                          const float* __restrict__ grad, const float* __restrict__ y,
                          const float* __restrict__ rcp, float* __restrict__ dx, float* __restrict__ dst,
                          int B, int I, int J, int rows, float max_cmp, float biasvolt, float neg_s, float post,
                          float* __restrict__ zeros, int n_zeros) {
    constexpr int JP = JL * NARROW_GROUPS;
    if (blockIdx.x == 0 && blockIdx.y == 0 && (int)threadIdx.x < n_zeros) zeros[threadIdx.x] = 0.0f;   // dParams
    // one more row than samples: (-inf, 0), which adds nothing, for the turns of a wavefront past
    // the block's last sample
    __shared__ float ys[NARROW_SAMPLES + 1][JP];           // scaled output time, -inf where masked out
    __shared__ float us[NARROW_SAMPLES + 1][JP];           // grad * 1/wsum, 0 where masked out
    __shared__ float red[NARROW_WAVES - 1][JL][kWave];
    const int lane = threadIdx.x % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int group = lane / NARROW_ROWS;
    const int i = blockIdx.x * NARROW_ROWS + lane % NARROW_ROWS;
    const int j0 = group * JL;                             // first column of the lane
    const int b0 = blockIdx.y * NARROW_SAMPLES;
    const int n_s = min(NARROW_SAMPLES, B - b0);

    for (int e = threadIdx.x; e < n_s * JP; e += NARROW_WAVES * kWave) {
        const int bl = e / JP, j = e - bl * JP;
        float yv = -INFINITY, uv = 0.0f;
        if (j < J) {
            const size_t t = (size_t)(b0 + bl) * J + j;
            const float yt = y[t];
            if (yt <= max_cmp) { yv = yt * -neg_s; uv = grad[t] * rcp[t]; }
        }
        ys[bl][j] = yv;
        us[bl][j] = uv;
    }
    if (threadIdx.x < JP) {
        ys[NARROW_SAMPLES][threadIdx.x] = -INFINITY;
        us[NARROW_SAMPLES][threadIdx.x] = 0.0f;
    }

    const bool is_input = i < I;
    const unsigned ic = (unsigned)min(i, I - 1);
    // the lane's input of every sample its wavefront takes, requested before anything waits
    constexpr int PER_WAVE = NARROW_SAMPLES / NARROW_WAVES;
    const float* __restrict__ xcol = x + (size_t)b0 * I + ic;
    float xs[PER_WAVE];
#pragma unroll
    for (int q = 0; q < PER_WAVE; ++q) {
        const int bl = min(wave + q * NARROW_WAVES, n_s - 1);
        xs[q] = is_input ? xcol[(size_t)bl * I] : biasvolt;
    }
    float wr[JL], acc[JL];
#pragma unroll
    for (int c = 0; c < JL; ++c) {
        wr[c] = (dx && is_input && j0 + c < J) ? w[(size_t)ic * J + j0 + c] : 0.0f;
        acc[c] = 0.0f;
    }
    __syncthreads();

    // four samples at a time, without branches, so that their LDS reads and lane exchanges overlap
    constexpr int BATCH = 4;
    static_assert(PER_WAVE % BATCH == 0, "samples per wavefront must be a multiple of the batch");
#pragma unroll
    for (int q0 = 0; q0 < PER_WAVE; q0 += BATCH) {
        float dxa[BATCH];
#pragma unroll
        for (int u = 0; u < BATCH; ++u) {
            const int bl = wave + (q0 + u) * NARROW_WAVES;
            const int row = bl < n_s ? bl : NARROW_SAMPLES;
            const float xq = xs[q0 + u] * -neg_s;
            dxa[u] = 0.0f;
#pragma unroll
            for (int c = 0; c < JL; ++c) {
                const float yv = ys[row][j0 + c], uv = us[row][j0 + c];
                acc[c] = __fmaf_rn(__builtin_amdgcn_fmed3f(yv - xq, 0.0f, 1.0f), uv, acc[c]);
                dxa[u] = __fmaf_rn(uv, xq <= yv ? wr[c] : 0.0f, dxa[u]);
            }
        }
        if (dx) {                                           // block-uniform
#pragma unroll
            for (int u = 0; u < BATCH; ++u) dxa[u] += __shfl_xor(dxa[u], NARROW_ROWS, kWave);      // (0 + 1), (2 + 3)
#pragma unroll
            for (int u = 0; u < BATCH; ++u) dxa[u] += __shfl_xor(dxa[u], 2 * NARROW_ROWS, kWave);
#pragma unroll
            for (int u = 0; u < BATCH; ++u) {
                const int bl = wave + (q0 + u) * NARROW_WAVES;
                if (group == 0 && is_input && bl < n_s) dx[(size_t)(b0 + bl) * I + i] = dxa[u];
            }
        }
    }

    if (!dst) return;
    if (wave > 0) {
#pragma unroll
        for (int c = 0; c < JL; ++c) red[wave - 1][c][lane] = acc[c];
    }
    __syncthreads();
    if (wave == 0 && i < rows) {
        float* out = dst + (size_t)blockIdx.y * rows * J + (size_t)i * J + j0;
#pragma unroll
        for (int c = 0; c < JL; ++c) {
            if (j0 + c < J) {
                float sum = acc[c];
#pragma unroll
                for (int v = 0; v < NARROW_WAVES - 1; ++v) sum += red[v][c][lane];
                out[c] = sum * post;
            }
        }
    }
}

// A block adds up 32 elements: its eight groups of 32 threads each take a contiguous eighth of the
// slices (two chains per thread keep loads in flight) and the eight sums are added in group order.
// The order of additions depends only on nsplit, never on timing.
constexpr int RED_ELEMS = 32, RED_GROUPS = 8;

__global__ void __launch_bounds__(RED_ELEMS * RED_GROUPS)
reduce_partials_kernel(const float* __restrict__ partial, float* __restrict__ out, int64_t n, int nsplit) {
    __shared__ float part[RED_GROUPS][RED_ELEMS];
    const int e = threadIdx.x % RED_ELEMS, g = threadIdx.x / RED_ELEMS;
    const int64_t t = (int64_t)blockIdx.x * RED_ELEMS + e;
    const int per = (nsplit + RED_GROUPS - 1) / RED_GROUPS;
    const int z_lo = g * per, z_hi = min(nsplit, z_lo + per);
    float a0 = 0.0f, a1 = 0.0f;
    if (t < n) {
        int z = z_lo;
        for (; z + 2 <= z_hi; z += 2) {
            a0 += partial[(size_t)z * n + t];
            a1 += partial[(size_t)(z + 1) * n + t];
        }
        if (z < z_hi) a0 += partial[(size_t)z * n + t];
    }
    part[g][e] = a0 + a1;
    __syncthreads();
    if (g == 0 && t < n) {
        float sum = part[0][e];
#pragma unroll
        for (int k = 1; k < RED_GROUPS; ++k) sum += part[k][e];
        out[t] = sum;
    }
}

// Up to eight slices of whole float4s: an element is added up by one thread, four at a time, in the same order (a slice is a group of
// its own there).  Wide layers have few slices of many elements: 4 of 2.4 M 27 -> 14 us, 3 of 1 M 67 -> 59 with the launch before it.  With too few
// for the chip a thread's chain of slices takes longer than the sums of eight groups: the line lies at about 25 600 elements for each
// slice (3 of 69 and 114 K 12.6 -> 12.4 and 13.7 -> 13.4, 5 of 98 and 175 K 14.7 -> 14.9 and 16.8 -> 16.0, 8 of 60 and 119 K 13.4 -> 14.5 and 21.7 -> 23.0).
constexpr int64_t RED_FEW_FROM = 25600;
__global__ void __launch_bounds__(256)
reduce_few_kernel(const float4* __restrict__ partial, float4* __restrict__ out, int64_t n4, int nsplit) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n4) return;
    float4 sum = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll
    for (int z = 0; z < RED_GROUPS; ++z) {
        if (z >= nsplit) break;
        const float4 v = partial[(size_t)z * n4 + t];
        sum.x += v.x; sum.y += v.y; sum.z += v.z; sum.w += v.w;
    }
    out[t] = sum;
}

// ---------------------------------------------------------------------------------------------
// Conv dX for layers the channel-lane kernel does not take (output channels not a multiple of 16, or fewer
// than 32 input channels under a kernel that is not three columns wide): the
// gradient per patch element, dxp[S, P], comes from the dense kernel above run over the implicit
// patches; here every element of the padded image adds up the patch elements that alias it, in
// (kh, kw) order.  Gather form: no atomics, fixed summation order.
// ---------------------------------------------------------------------------------------------
__global__ void __launch_bounds__(256)
cv_col2im_kernel(const float* __restrict__ dxp, float* __restrict__ dx, CropGeom crop, int64_t n, int H, int W, int C,
                 int Kh, int Kw, int Sh, int Sw, int Nh, int Nw) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
    const int c = (int)(t % C);
    const int64_t pix = t / C;
    const int wx = (int)(pix % W);
    const int64_t rowi = pix / W;
    const int h = (int)(rowi % H);
    const int a = (int)(rowi / H);
    const int oh = h - crop.top, ow = wx - crop.left;         // only the caller's window is stored
    if (oh < 0 || oh >= crop.h || ow < 0 || ow >= crop.w) return;
    const int P = Kh * Kw * C;
    float acc = 0.0f;
    for (int kh = 0; kh < Kh; ++kh) {
        const int hh = h - kh;
        if (hh < 0 || hh % Sh != 0 || hh / Sh >= Nh) continue;
        for (int kw = 0; kw < Kw; ++kw) {
            const int ww = wx - kw;
            if (ww < 0 || ww % Sw != 0 || ww / Sw >= Nw) continue;
            const size_t s = (size_t)(a * Nh + hh / Sh) * Nw + ww / Sw;
            acc += dxp[s * P + (kh * Kw + kw) * C + c];
        }
    }
    dx[(((size_t)a * crop.h + oh) * crop.w + ow) * C + c] = acc;
}

int blocks_for(int64_t n, int block) { return (int)((n + block - 1) / block); }

}  // namespace

int launch_backward_prologue(const float* grad, const float* y, const float* rcp, float* upm, int64_t n,
                             const NeuronParams& np, const float* w, float* wt, int64_t rows,
                             int64_t cols, int64_t chan, float* zeros, int n_zeros, hipStream_t stream) {
    if (!zeros) n_zeros = 0;
    const bool vec4 = n % 4 == 0 && (((uintptr_t)grad | (uintptr_t)y | (uintptr_t)rcp | (uintptr_t)upm) & 15) == 0;
    const int64_t prep_blocks = vec4 ? (n / 4 + 255) / 256 : (n + 255) / 256;
    const int64_t copy_blocks = wt ? (rows * (cols / 4) + 255) / 256 : 0;
    if (prep_blocks + copy_blocks <= 0) return n_zeros > 0 ? launch_fill_zero(zeros, n_zeros, stream) : SNNTC_OK;
    if (prep_blocks + copy_blocks > 0x7fffffffLL) return fail(SNNTC_ERR_TOO_LARGE, "backward: grid too large");
    {
        KernelTimerScope timer_("prep_upstream", stream);
        hipLaunchKernelGGL(backward_prologue_kernel, dim3((unsigned)(prep_blocks + copy_blocks)), dim3(256), 0, stream,
                           grad, y, rcp, upm, n, np.max_cmp, (int)prep_blocks, vec4 ? 1 : 0, w, wt, (int)rows, (int)cols,
                           (int)chan, zeros, n_zeros);
    }
    SNNTC_HIP_CHECK(hipGetLastError());
    return SNNTC_OK;
}

int launch_fill_zero(float* p, int64_t n, hipStream_t stream) {
    if (n <= 0) return SNNTC_OK;
    { KernelTimerScope timer_("fill_zero", stream);
    hipLaunchKernelGGL(fill_zero_kernel, dim3(blocks_for(n, 256)), dim3(256), 0, stream, p, n);
    }
    SNNTC_HIP_CHECK(hipGetLastError());
    return SNNTC_OK;
}

namespace {
// Wavefronts per tile.  Many tiles: four, which leave a CU's several workgroups to fill its SIMDs; fewer: more, so that every
// SIMD has two or so (us with 4 / 8 / 16 at 800 outputs: 200 tiles 27 / 21 / 19, 400: 30 / 28.5 / 34, 800: 47 / 49 / 63); not
// below 16 outputs each, and a single one for fewer than 64 outputs (16 200 x 500 -> 50: 26 against 32).
int dx_split(int64_t tiles, int64_t J) {
    if (J < 64) return 1;
    int split = tiles >= 640 ? 4 : tiles >= 256 ? 8 : 16;
    while (split > 4 && J < DX_JC * split) split /= 2;
    return split;
}

template <bool PATCHES>
int launch_dx(const char* name, const SegmentSource& src, const float* w, const float* upm, const float* ym, float* dx, int64_t B,
              int64_t I, int64_t J, hipStream_t stream) {
    const int rc = grad_prepare_device();
    if (rc) return rc;
    const int64_t tiles_i = (I + DX_I - 1) / DX_I, tiles = (B + DX_S - 1) / DX_S * tiles_i;
    const int split = dx_split(tiles, J);
    const int64_t blocks = split == 1 ? (tiles + 3) / 4 : tiles;
    if (blocks > 0x1fffffffLL) return fail(SNNTC_ERR_TOO_LARGE, "backward: %lld x %lld input gradients are too many", (long long)B, (long long)I);
    {
        KernelTimerScope timer_(name, stream);
        auto kern = split == 1 ? fc_grad_input_kernel<1, PATCHES> : split == 4 ? fc_grad_input_kernel<4, PATCHES>
                  : split == 8 ? fc_grad_input_kernel<8, PATCHES> : fc_grad_input_kernel<16, PATCHES>;
        hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(dx_threads(split)), dx_lds_bytes(split), stream, src, w, upm, ym, dx, (int)B, (int)I, (int)J,
                           (int)tiles_i, (int)tiles);
    }
    SNNTC_HIP_CHECK(hipGetLastError());
    return SNNTC_OK;
}
}  // namespace

// The dynamic-LDS limits of the current device, once.
int grad_prepare_device() {
    static std::atomic<bool> ready[kMaxDevices];
    int dev = 0;
    SNNTC_HIP_CHECK(hipGetDevice(&dev));
    if (dev < 0 || dev >= kMaxDevices) return fail(SNNTC_ERR_UNSUPPORTED, "backward: device index %d not supported", dev);
    if (ready[dev].load(std::memory_order_acquire)) return SNNTC_OK;
    for (const void* k : {reinterpret_cast<const void*>(fc_grad_input_kernel<16, false>), reinterpret_cast<const void*>(fc_grad_input_kernel<16, true>)})
        SNNTC_HIP_CHECK(hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, dx_lds_bytes(16)));
    ready[dev].store(true, std::memory_order_release);
    return SNNTC_OK;
}

int launch_fc_grad_input(const float* x, const float* w, const float* upm, const float* ym, float* dx,
                         int64_t B, int64_t I, int64_t J, hipStream_t stream) {
    if (B <= 0 || I <= 0) return SNNTC_OK;
    if (J <= 0) return launch_fill_zero(dx, B * I, stream);
    SegmentSource src{};
    src.base = x; src.conv = 0; src.I = (int)I;
    return launch_dx<false>("fc_grad_input", src, w, upm, ym, dx, B, I, J, stream);
}

// Number of slices the segment range is cut into for dW: none when the (row-block x column-block)
// grid alone fills the chip; otherwise up to ~1536 blocks (six per CU, all resident at once), at
// least 64 segments per slice, at most 256 slices.  Within the upper half of that range the count
// is the one whose blocks spread most evenly over the 256 CUs: the launch lasts as long as the CU
// with the most blocks, ceil(blocks / 256) of them, each 1/n of a column of work.
int weight_grad_splits(int64_t S, int64_t base_blocks) {
    if (base_blocks >= 1024) return 1;
    if (base_blocks < 1) base_blocks = 1;
    int64_t want = (1536 + base_blocks - 1) / base_blocks;
    int64_t cap = S / 64;
    if (want > cap) want = cap;
    if (want > 256) want = 256;
    if (want < 1) want = 1;
    int64_t best = want;
    double best_cost = 1e30;
    for (int64_t n = want; n >= 1 && 2 * n >= want; --n) {
        const double cost = (double)((base_blocks * n + 255) / 256) / (double)n;
        if (cost < best_cost * 0.995) { best_cost = cost; best = n; }
    }
    return (int)best;
}

int grad_weight_blocks(int64_t rows, int64_t J) {
    return (int)(((J + kWave - 1) / kWave) * ((rows + DW_RI - 1) / DW_RI));
}

// Slices of a dense layer's samples.  A CU needs about 100 clocks per sample for a tile of 64 x 64; the launch lasts as long as
// the CU with the most of them, and adding up slices costs another launch (about 5 us and the slices' traffic).  With few tiles
// the slices go on until every CU has a workgroup, in steps of a sixteenth: at 16 slices 65 536 x 64 -> 64 left seven CUs in eight
// idle (189 us; 34 with 128 slices, 20 000 x 100 -> 100 62 -> 24, 4096 x 64 -> 64 18 -> 10).
int grad_weight_dense_splits(int64_t S, int64_t I, int64_t J) {
    const int64_t tiles = ((J + DWD_T - 1) / DWD_T) * ((I + 1 + DWD_T - 1) / DWD_T);
    const int64_t most = std::min(std::max((int64_t)16, 256 / std::max((int64_t)1, tiles)), std::max((int64_t)1, S / 64));
    int best = 1;
    double best_time = 1e30;
    for (int64_t n = 1; n <= most; n = n < most ? std::min(most, n + 1 + n / 16) : n + 1) {
        const double time = (double)((tiles * n + 255) / 256) * 100.0 * (double)((S + n - 1) / n) +
                            (n > 1 ? 12000.0 + 8.0 * n * (double)(I + 1) * (double)J / 1500.0 : 0.0);
        if (time < best_time * 0.97) { best_time = time; best = (int)n; }
    }
    return best;
}

// dW, or every partial-sum slice of it, when nsplit > 1 (dst = slices).
int launch_grad_weight_rows(const SegmentSource& src, const float* upm, const float* ym, float* dst,
                            int nsplit, int64_t S, int64_t J, const NeuronParams& np,
                            hipStream_t stream) {
    const int64_t rows = (int64_t)src.I + np.bias;
    if (rows <= 0 || J <= 0 || S <= 0) return SNNTC_OK;
    if (nsplit < 1) nsplit = 1;
    const int seg_per_slice = (int)((S + nsplit - 1) / nsplit);
    const int rows_per_block = src.conv ? DW_RI : DWD_T;
    dim3 grid((unsigned)((J + kWave - 1) / kWave), (unsigned)((rows + rows_per_block - 1) / rows_per_block), (unsigned)nsplit);
    if (grid.y > 65535u) return fail(SNNTC_ERR_TOO_LARGE, "weight gradient: too many weight rows");
    {
        KernelTimerScope timer_("grad_weight", stream);
        const LeadScale ls = lead_scale(np.max_time);
        if (src.conv) {
            hipLaunchKernelGGL(grad_weight_kernel, grid, dim3(256), 0, stream, src, upm, ym, dst, (int)S, (int)J,
                               (int)rows, seg_per_slice, np.biasvolt, ls.neg_s, ls.post);
        } else {
            // eight wavefronts per tile where there are too few tiles to give every SIMD two otherwise
            const bool wide = (int64_t)grid.x * grid.y * grid.z < 512;
            auto kern = wide ? grad_weight_dense_kernel<8> : grad_weight_dense_kernel<4>;
            hipLaunchKernelGGL(kern, grid, dim3((wide ? 8 : 4) * kWave), 0, stream, src.base, upm, ym, dst, (int)S,
                               (int)src.I, (int)J, (int)rows, seg_per_slice, np.biasvolt, ls.neg_s, ls.post);
        }
    }
    SNNTC_HIP_CHECK(hipGetLastError());
    return SNNTC_OK;
}

int launch_reduce_partials(const float* partial, float* dw, int64_t n, int nsplit, hipStream_t stream) {
    if (n <= 0 || nsplit <= 1) return SNNTC_OK;
    {
        KernelTimerScope timer_("reduce_partials", stream);
        const bool few = nsplit <= RED_GROUPS && n >= RED_FEW_FROM * nsplit && n % 4 == 0 &&
                         ((reinterpret_cast<uintptr_t>(partial) | reinterpret_cast<uintptr_t>(dw)) & 15) == 0;
        if (few)
            hipLaunchKernelGGL(reduce_few_kernel, dim3(blocks_for(n / 4, 256)), dim3(256), 0, stream,
                               reinterpret_cast<const float4*>(partial), reinterpret_cast<float4*>(dw), n / 4, nsplit);
        else hipLaunchKernelGGL(reduce_partials_kernel, dim3(blocks_for(n, RED_ELEMS)), dim3(RED_ELEMS * RED_GROUPS), 0,
                           stream, partial, dw, n, nsplit);
    }
    SNNTC_HIP_CHECK(hipGetLastError());
    return SNNTC_OK;
}

// Workgroups of a joint launch: dX tiles (below 64 outputs, eight of them) and dW tiles.
struct JointGrid { int64_t dx_tiles, dx_blocks, dw_blocks; };
static JointGrid joint_grid(int64_t B, int64_t I, int64_t rows, int64_t J, bool dx) {
    JointGrid g{};
    g.dx_tiles = dx ? (B + DX_S - 1) / DX_S * ((I + DX_I - 1) / DX_I) : 0;
    g.dx_blocks = J < 64 ? (g.dx_tiles + 7) / 8 : g.dx_tiles;
    g.dw_blocks = (J + DWD_T - 1) / DWD_T * ((rows + DWD_T - 1) / DWD_T);
    return g;
}

// dX and dW of a dense layer in one launch (dX == NULL: dW alone).  `slices`: what the samples would be cut into for dW alone.
// The parts of a launch with more workgroups fill the chip by themselves, with tiles of their own (us, apart / together: 200 x 2048 ->
// 512, 1096 workgroups, 61 / 42; 333 x 1521 -> 777, 1320, 87 / 73; 400 x 3000 -> 512, 2726, 116 / 99; 512 x 3000 -> 512, 3384, 140 / 126; 300 x
// 4096 -> 1000, 3472, 211 / 214; 400 x 10 000 -> 200, 8453, 171 / 179).
// Where dW alone would be cut into slices, a tile goes over all samples here and folds its sums (joint_folds): less than the launches that
// slices need where tiles are many, or samples few (us, slices / together: 512 -> 512, 72 tiles, 270, 333, 448 rows 30 / 23, 31 / 26, 33.5 / 31,
// 480 37 / 34 but 300 -> 300, 25 tiles, 270 and 333 rows 20.6 / 22, 21 / 27; 500 -> 50, eight tiles, 200, 240, 256 rows 21 / 16.5, 21 / 18,
// 20 / 20; 128 -> 128, six tiles, 200 rows 16.1 / 16.4), and not for dW alone (256 x 300 -> 300 13 / 20, 512 -> 512 17 / 19).
constexpr int64_t JOINT_FEW_ROWS = 240;
bool fc_backward_joint_supported(int64_t B, int64_t I, int64_t J, bool dx, int slices) {
    const JointGrid g = joint_grid(B, I, I + 1, J, dx);
    if (g.dx_blocks + g.dw_blocks > 3072) return false;
    return slices == 1 || (dx && B <= 448 && (g.dw_blocks >= 64 || (g.dw_blocks >= 8 && B <= JOINT_FEW_ROWS)));
}
// How often a tile's sums are folded: as often as there would be slices, which keeps its error against 64 bits at or below that of the slices (rms, in
// units of the terms' absolute sum and 1e-9, slices / one chain per wavefront / folded: 256 x 512 -> 512 8.8 / 10.3 / 8.2, 333 rows 8.1 / 10.1 / 7.6,
// 448 7.4 / 9.7 / 7.0, 448 x 333 -> 1000 8.0 / 9.7 / 7.7).  Up to 240 rows half as often does that, since a tree adds its wavefronts and slices add
// theirs one after the other (230 x 300 -> 300 9.1 / 10.5 / 8.9).  A fold costs about 1.3 us.
static int joint_folds(int64_t B, int slices) { return slices == 1 ? 1 : B <= JOINT_FEW_ROWS ? slices / 2 + 1 : slices; }

int launch_fc_backward_joint(const float* x, const float* w, const float* grad, const float* y, const float* rcp, float* dx, float* dw,
                             float* zeros, int n_zeros, int64_t B, int64_t I, int64_t J, int slices, const NeuronParams& np, hipStream_t stream) {
    const int turns = (int)((B + DWD_TURN - 1) / DWD_TURN), folds = joint_folds(B, slices);
    const int64_t rows = I + np.bias;
    const JointGrid g = joint_grid(B, I, rows, J, dx != nullptr);
    // The longer tiles come first, so that the shorter ones fill the end: dW takes 8192 terms a sample, dX 512 an output, of which it
    // does a third as many a clock.  (us, dX / dW first: 256 x 784 -> 800 38 / 33, 400 rows 59 / 49, 300 x 1000 -> 200 30 / 25; 256 x 300 -> 2048
    // 38 / 46, 32 x 3000 -> 512 15.3 / 20.7.)  Where all workgroups, of which a CU holds two, are there at once, only much longer ones
    // (364 x 407 -> 812 35 / 31, 253 x 720 -> 557 25 / 23, 128 x 1000 -> 130 13 / 11, but 333 x 512 -> 1000 33 / 34, 121 x 1032 -> 717 23 / 22.5).  Over
    // 230 shapes of 48 to 740 rows the other order was never more than 4 % ahead, but for one case: dX tiles that are a little more than the
    // first turn, and dW tiles behind them with a CU each (dX first 0 to 7 % ahead in 20 of 27: 333 x 784 -> 800 43 / 45, 586 x 460 -> 1412 68 / 74).
    const int64_t behind = g.dx_blocks + g.dw_blocks - 512;
    const bool just_over = behind >= 128 && behind <= 256 && g.dx_blocks > 512 && g.dx_blocks <= 600;
    const bool dw_first = behind <= 0 ? 8 * B > 3 * J : 4 * B > J && !just_over;
    const LeadScale ls = lead_scale(np.max_time);
    {
        KernelTimerScope timer_("fc_backward", stream);
        auto kern = J < 64 ? (folds > 1 ? fc_backward_kernel<1, true> : fc_backward_kernel<1, false>)
                           : (folds > 1 ? fc_backward_kernel<8, true> : fc_backward_kernel<8, false>);
        hipLaunchKernelGGL(kern, dim3((unsigned)(g.dx_blocks + g.dw_blocks)), dim3(8 * kWave), 0, stream, x, w, grad, y, rcp, dx, dw, zeros,
                           zeros ? n_zeros : 0, (int)B, (int)I, (int)J, (int)rows, (int)((I + DX_I - 1) / DX_I), (int)g.dx_tiles, (int)g.dx_blocks,
                           (int)(dw_first ? g.dw_blocks : 0), (int)((J + DWD_T - 1) / DWD_T), (turns + folds - 1) / folds, np.max_cmp, np.biasvolt, ls.neg_s, ls.post);
    }
    SNNTC_HIP_CHECK(hipGetLastError());
    return SNNTC_OK;
}

bool fc_backward_narrow_supported(int64_t J) { return J >= 1 && J <= NARROW_JMAX; }

int fc_backward_narrow_splits(int64_t B) { return (int)((B + NARROW_SAMPLES - 1) / NARROW_SAMPLES); }

// dx and/or dw may be NULL.  With more than one block of samples `partial` takes the dW slices.
int launch_fc_backward_narrow(const float* x, const float* w, const float* grad, const float* y, const float* rcp,
                              float* dx, float* dw, float* partial, float* zeros, int n_zeros, int64_t B, int64_t I,
                              int64_t J, const NeuronParams& np, hipStream_t stream) {
    if (!zeros) n_zeros = 0;
    const int64_t rows = I + np.bias;
    const int nsplit = fc_backward_narrow_splits(B);
    // without dW only the input rows are needed; the bias row has no dX
    const int64_t lanes = dw ? rows : I;
    dim3 grid((unsigned)((lanes + NARROW_ROWS - 1) / NARROW_ROWS), (unsigned)nsplit);
    if (grid.y > 65535u) return fail(SNNTC_ERR_TOO_LARGE, "dense backward: batch %lld too large", (long long)B);
    float* dst = dw ? (nsplit > 1 ? partial : dw) : nullptr;
    {
        KernelTimerScope timer_("fc_backward_narrow", stream);
        const LeadScale ls = lead_scale(np.max_time);
        const int jl = (int)((J + NARROW_GROUPS - 1) / NARROW_GROUPS);      // columns per lane
        auto kern = jl == 1 ? fc_backward_narrow_kernel<1> : jl == 2 ? fc_backward_narrow_kernel<2>
                  : jl == 3 ? fc_backward_narrow_kernel<3> : fc_backward_narrow_kernel<4>;
        hipLaunchKernelGGL(kern, grid, dim3(NARROW_WAVES * kWave), 0, stream, x, w, grad, y, rcp, dx, dst, (int)B,
                           (int)I, (int)J, (int)rows, np.max_cmp, np.biasvolt, ls.neg_s, ls.post, zeros, n_zeros);
    }
    SNNTC_HIP_CHECK(hipGetLastError());
    if (!dw) return SNNTC_OK;
    return launch_reduce_partials(partial, dw, rows * J, nsplit, stream);
}

// dxp: scratch of S * P floats (gradient per patch element)
int launch_cv_grad_input(const SegmentSource& src, const float* w, const float* upm, const float* ym, float* dxp,
                         float* dx, const CropGeom& crop, const ConvGeom& g, hipStream_t stream) {
    const int64_t n = g.B * g.H * g.W * g.C;
    if (n <= 0) return SNNTC_OK;
    if (g.Kc <= 0 || g.S <= 0) return launch_fill_zero(dx, g.B * crop.h * crop.w * g.C, stream);
    const int rc = launch_dx<true>("cv_grad_input", src, w, upm, ym, dxp, g.S, g.P, g.Kc, stream);
    if (rc) return rc;
    { KernelTimerScope timer_("cv_col2im", stream);
    hipLaunchKernelGGL(cv_col2im_kernel, dim3(blocks_for(n, 256)), dim3(256), 0, stream, dxp, dx, crop, n, (int)g.H,
                       (int)g.W, (int)g.C, (int)g.Kh, (int)g.Kw, (int)g.Sh, (int)g.Sw, (int)g.Nh, (int)g.Nw);
    }
    SNNTC_HIP_CHECK(hipGetLastError());
    return SNNTC_OK;
}

}  // namespace snntc
