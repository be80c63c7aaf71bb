// Glue of the example training recipe (snntc-mnist.py:55-96): input encoding, cross-entropy against
// integer labels with the count of correct samples, and the weight-constraint cost
//     K * sum_l mean_j max(0, 1 - sum_i w_ij) + K2 * sum_l mean(w^2)
// with its gradient.  As separate framework ops these are about eighty launches of 2-7 us and twice that
// in host time, several times what the layers of a small network cost; here they are five.
#include "snntc_common.h"

namespace snntc {
namespace {

// z = exp(1 - image).  Bound by memory; four values per thread where the arrays allow 16-byte accesses.
__global__ void __launch_bounds__(256) encode_time_kernel(const float* __restrict__ image, float* __restrict__ z, long long n,
                                                          int vec) {
    const long long e = ((long long)blockIdx.x * 256 + threadIdx.x) * 4;
    if (e >= n) return;
    if (vec && e + 4 <= n) {
        float4 v = *reinterpret_cast<const float4*>(image + e);
        v.x = expf(1.0f - v.x); v.y = expf(1.0f - v.y); v.z = expf(1.0f - v.z); v.w = expf(1.0f - v.w);
        *reinterpret_cast<float4*>(z + e) = v;
        return;
    }
    for (long long k = e; k < n && k < e + 4; ++k) z[k] = expf(1.0f - image[k]);
}

// One wavefront per sample: loss against label b, gradient of the batch mean, and whether the earliest
// output (the lowest index of equal ones, a NaN before everything) is the label.  A label outside [0, J)
// leaves NaN in the loss and the gradient.
__global__ void __launch_bounds__(256)
label_loss_kernel(const float* __restrict__ times, const long long* __restrict__ labels, float* __restrict__ sample_loss,
                  float* __restrict__ dtimes, int* __restrict__ correct, int B, int J, float inv_b) {
    const int lane = threadIdx.x % kWave;
    const int b = blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave;
    if (b >= B) return;
    const float* __restrict__ t = times + (size_t)b * J;
    const long long label = labels[b];
    const bool known = label >= 0 && label < J;
    float first = INFINITY;
    int arg = 0x7fffffff;
    for (int j = lane; j < J; j += kWave) {
        const float v = isnan(t[j]) ? -INFINITY : t[j];
        if (v < first || arg == 0x7fffffff) { first = v; arg = j; }
    }
#pragma unroll
    for (int d = kWave / 2; d > 0; d >>= 1) {
        const float v = __shfl_xor(first, d, kWave);
        const int a = __shfl_xor(arg, d, kWave);
        if (v < first || (v == first && a < arg)) { first = v; arg = a; }
    }
    float se = 0.0f;
    for (int j = lane; j < J; j += kWave) se += expf(first - t[j]);
#pragma unroll
    for (int d = kWave / 2; d > 0; d >>= 1) se += __shfl_xor(se, d, kWave);
    if (lane == 0) {
        sample_loss[b] = known ? logf(se) - (first - t[label]) : NAN;
        correct[b] = known && arg == (int)label;
    }
    if (!dtimes) return;
    float* __restrict__ g = dtimes + (size_t)b * J;
    const float scale = 1.0f / se;
    for (int j = lane; j < J; j += kWave)
        g[j] = known ? ((j == (int)label ? 1.0f : 0.0f) - expf(first - t[j]) * scale) * inv_b : NAN;
}

// The weight tensors are cut into tiles of 64 rows x 64 columns; a block owns one.  The sums kernel
// leaves every tile's column sums and sum of squares; a column's sum is then the sum over its row
// tiles, at most a few dozen values, which whoever needs it adds up in order.  Both kernels read (and
// the gradient kernel rewrites) each weight once; a small network's layers make some tens of blocks, so
// what bounds them there is one trip to memory.
constexpr int kTile = 64;
constexpr int kMaxTensors = 24;

struct WeightTable {
    const float* w[kMaxTensors];
    float* grad[kMaxTensors];            // NULL: this tensor gets no gradient
    float* col_sums[kMaxTensors];        // [row tiles][cols]
    float* squares[kMaxTensors];         // [row tiles * column tiles]
    int rows[kMaxTensors], cols[kMaxTensors], row_tiles[kMaxTensors], col_tiles[kMaxTensors];
    int first_block[kMaxTensors + 1];
    int count;
};

struct Tile { int t, r, c; };
__device__ __forceinline__ Tile own_tile(const WeightTable& tab) {
    int t = 0;
    while (t + 1 < tab.count && (int)blockIdx.x >= tab.first_block[t + 1]) ++t;          // uniform
    const int k = blockIdx.x - tab.first_block[t];
    return Tile{t, k / tab.col_tiles[t], k % tab.col_tiles[t]};
}

__global__ void __launch_bounds__(256) weight_cost_sums_kernel(WeightTable tab) {
    __shared__ float part[4][kTile], sq[4];
    const Tile at = own_tile(tab);
    const int rows = tab.rows[at.t], cols = tab.cols[at.t];
    const int lane = threadIdx.x % kTile, group = threadIdx.x / kTile;
    const int j = at.c * kTile + lane, r0 = at.r * kTile;
    const float* __restrict__ w = tab.w[at.t];
    float s = 0.0f, q = 0.0f;
    if (j < cols) {
#pragma unroll 8
        for (int r = r0 + group; r < min(rows, r0 + kTile); r += 4) {
            const float v = w[(size_t)r * cols + j];
            s += v;
            q = fmaf(v, v, q);
        }
    }
    part[group][lane] = s;
#pragma unroll
    for (int d = kWave / 2; d > 0; d >>= 1) q += __shfl_xor(q, d, kWave);
    if (lane == 0) sq[group] = q;
    __syncthreads();
    if (group == 0 && j < cols)
        tab.col_sums[at.t][(size_t)at.r * cols + j] = (part[0][lane] + part[1][lane]) + (part[2][lane] + part[3][lane]);
    if (threadIdx.x == 0) tab.squares[at.t][at.r * tab.col_tiles[at.t] + at.c] = (sq[0] + sq[1]) + (sq[2] + sq[3]);
}

// grad (+)= upstream * (-K / J where the column sum lies below 1, plus 2 K2 w / n)
template <bool ACCUMULATE>
__global__ void __launch_bounds__(256) weight_cost_grad_kernel(WeightTable tab, float k, float k2, const float* __restrict__ upstream) {
    __shared__ float part[4][kTile];
    const Tile at = own_tile(tab);
    float* __restrict__ grad = tab.grad[at.t];
    if (!grad) return;                                                                   // block-uniform
    const int rows = tab.rows[at.t], cols = tab.cols[at.t];
    const int lane = threadIdx.x % kTile, group = threadIdx.x / kTile;
    const int j = at.c * kTile + lane, r0 = at.r * kTile;
    float s = 0.0f;
    if (j < cols) {
#pragma unroll 4
        for (int r = group; r < tab.row_tiles[at.t]; r += 4) s += tab.col_sums[at.t][(size_t)r * cols + j];
    }
    part[group][lane] = s;
    __syncthreads();
    if (j >= cols) return;
    s = (part[0][lane] + part[1][lane]) + (part[2][lane] + part[3][lane]);
    const float up = upstream ? *upstream : 1.0f;
    const float low = 1.0f - s >= 0.0f ? -up * k / (float)cols : 0.0f;
    const float sq = up * k2 * 2.0f / ((float)rows * (float)cols);
    const float* __restrict__ w = tab.w[at.t];
#pragma unroll 8
    for (int r = r0 + group; r < min(rows, r0 + kTile); r += 4) {
        const size_t e = (size_t)r * cols + j;
        const float g = fmaf(sq, w[e], low);
        grad[e] = ACCUMULATE ? grad[e] + g : g;
    }
}

constexpr int kTotalThreads = 1024;
__device__ __forceinline__ float block_sum(float v, float* buf) {
#pragma unroll
    for (int d = kWave / 2; d > 0; d >>= 1) v += __shfl_xor(v, d, kWave);
    __syncthreads();
    if (threadIdx.x % kWave == 0) buf[threadIdx.x / kWave] = v;
    __syncthreads();
    float s = 0.0f;
    for (int i = 0; i < kTotalThreads / kWave; ++i) s += buf[i];
    return s;
}

// One workgroup: total (+)= mean(sample_loss) + cost of the table's tensors, and the number of correct samples.
__global__ void __launch_bounds__(kTotalThreads)
recipe_total_kernel(WeightTable tab, float k, float k2, const float* __restrict__ sample_loss, const int* __restrict__ correct, int B,
                    float* __restrict__ total, long long* __restrict__ n_correct, int accumulate) {
    __shared__ float buf[kTotalThreads / kWave];
    float loss = 0.0f, hits = 0.0f;
    if (sample_loss) {
        for (int b = threadIdx.x; b < B; b += kTotalThreads) {
            loss += sample_loss[b];
            if (correct) hits += (float)correct[b];                       // exact: a thread counts far below 2^24
        }
        loss = block_sum(loss, buf) / (float)B;
        // wavefront sums of counts are added as integers: the total may exceed what fp32 counts exactly
#pragma unroll
        for (int d = kWave / 2; d > 0; d >>= 1) hits += __shfl_xor(hits, d, kWave);
        __syncthreads();
        if (threadIdx.x % kWave == 0) buf[threadIdx.x / kWave] = hits;
        __syncthreads();
        if (threadIdx.x == 0 && n_correct) {
            long long c = 0;
            for (int i = 0; i < kTotalThreads / kWave; ++i) c += (long long)buf[i];
            *n_correct = c;
        }
    }
    float wsc = 0.0f, l2 = 0.0f;
    for (int t = 0; t < tab.count; ++t) {
        float low = 0.0f, q = 0.0f;
        for (int j = threadIdx.x; j < tab.cols[t]; j += kTotalThreads) {
            float s = 0.0f;
#pragma unroll 8
            for (int r = 0; r < tab.row_tiles[t]; ++r) s += tab.col_sums[t][(size_t)r * tab.cols[t] + j];
            low += fmaxf(1.0f - s, 0.0f);
        }
        for (int i = threadIdx.x; i < tab.row_tiles[t] * tab.col_tiles[t]; i += kTotalThreads) q += tab.squares[t][i];
        wsc += low / (float)tab.cols[t];
        l2 += q / ((float)tab.rows[t] * (float)tab.cols[t]);
    }
    const float cost = block_sum(k * wsc + k2 * l2, buf);
    if (threadIdx.x == 0) *total = (accumulate ? *total : 0.0f) + loss + cost;
}

// Fills the table with as many of the tensors from index `t` on as it holds; `ws` is the scratch of tensor `t` on.
int64_t fill_table(WeightTable* tab, const float* const* w, float* const* grad, const int64_t* rows, const int64_t* cols, int count,
                   int* t, float** ws) {
    int64_t blocks = 0;
    tab->count = 0;
    for (; *t < count && tab->count < kMaxTensors; ++*t) {
        const int i = tab->count++;
        const int64_t rt = (rows[*t] + kTile - 1) / kTile, ct = (cols[*t] + kTile - 1) / kTile;
        tab->w[i] = w ? w[*t] : nullptr;
        tab->grad[i] = grad ? grad[*t] : nullptr;
        tab->rows[i] = (int)rows[*t]; tab->cols[i] = (int)cols[*t];
        tab->row_tiles[i] = (int)rt; tab->col_tiles[i] = (int)ct;
        tab->col_sums[i] = *ws; *ws += rt * cols[*t];
        tab->squares[i] = *ws; *ws += rt * ct;
        tab->first_block[i] = (int)blocks;
        blocks += rt * ct;
    }
    tab->first_block[tab->count] = (int)blocks;
    return blocks;
}

}  // namespace

int launch_encode_time(const float* image, float* z, int64_t n, hipStream_t stream) {
    if (n <= 0) return SNNTC_OK;
    const int64_t blocks = (n + 1023) / 1024;
    if (blocks > 0x7fffffffLL) return fail(SNNTC_ERR_TOO_LARGE, "encode: too many elements");
    const int vec = (((uintptr_t)image | (uintptr_t)z) & 15) == 0;
    {
        KernelTimerScope timer_("encode_time", stream);
        hipLaunchKernelGGL(encode_time_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, image, z, (long long)n, vec);
    }
    SNNTC_HIP_CHECK(hipGetLastError());
    return SNNTC_OK;
}

int launch_label_loss(const float* times, const int64_t* labels, float* sample_loss, float* dtimes, int32_t* correct, int64_t B,
                      int64_t J, hipStream_t stream) {
    if (B <= 0 || J <= 0) return SNNTC_OK;
    const int64_t blocks = (B + 3) / 4;
    {
        KernelTimerScope timer_("label_loss", stream);
        hipLaunchKernelGGL(label_loss_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, times,
                           reinterpret_cast<const long long*>(labels), sample_loss, dtimes, correct, (int)B, (int)J, 1.0f / (float)B);
    }
    SNNTC_HIP_CHECK(hipGetLastError());
    return SNNTC_OK;
}

size_t weight_cost_workspace_floats(const int64_t* rows, const int64_t* cols, int count) {
    size_t n = 0;
    for (int t = 0; t < count; ++t) {
        const size_t rt = (rows[t] + kTile - 1) / kTile, ct = (cols[t] + kTile - 1) / kTile;
        n += rt * cols[t] + rt * ct;
    }
    return n;
}

int launch_weight_cost_sums(const float* const* w, const int64_t* rows, const int64_t* cols, int count, float* ws, hipStream_t stream) {
    for (int t = 0; t < count;) {
        WeightTable tab;
        const int64_t blocks = fill_table(&tab, w, nullptr, rows, cols, count, &t, &ws);
        {
            KernelTimerScope timer_("weight_cost_sums", stream);
            hipLaunchKernelGGL(weight_cost_sums_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, tab);
        }
        SNNTC_HIP_CHECK(hipGetLastError());
    }
    return SNNTC_OK;
}

int launch_weight_cost_grad(const float* const* w, float* const* grad, const int64_t* rows, const int64_t* cols, int count, float k,
                            float k2, const float* upstream, bool accumulate, float* ws, hipStream_t stream) {
    for (int t = 0; t < count;) {
        WeightTable tab;
        const int64_t blocks = fill_table(&tab, w, grad, rows, cols, count, &t, &ws);
        {
            KernelTimerScope timer_("weight_cost_grad", stream);
            if (accumulate)
                hipLaunchKernelGGL((weight_cost_grad_kernel<true>), dim3((unsigned)blocks), dim3(256), 0, stream, tab, k, k2, upstream);
            else
                hipLaunchKernelGGL((weight_cost_grad_kernel<false>), dim3((unsigned)blocks), dim3(256), 0, stream, tab, k, k2, upstream);
        }
        SNNTC_HIP_CHECK(hipGetLastError());
    }
    return SNNTC_OK;
}

int launch_recipe_total(const int64_t* rows, const int64_t* cols, int count, float k, float k2, const float* sample_loss,
                        const int32_t* correct, int64_t B, float* total, int64_t* n_correct, float* ws, hipStream_t stream) {
    int t = 0;
    bool more = false;
    do {
        WeightTable tab;
        fill_table(&tab, nullptr, nullptr, rows, cols, count, &t, &ws);
        {
            KernelTimerScope timer_("recipe_total", stream);
            hipLaunchKernelGGL(recipe_total_kernel, dim3(1), dim3(kTotalThreads), 0, stream, tab, k, k2, more ? nullptr : sample_loss,
                               correct, (int)B, total, reinterpret_cast<long long*>(n_correct), more ? 1 : 0);
        }
        SNNTC_HIP_CHECK(hipGetLastError());
        more = true;
    } while (t < count);
    return SNNTC_OK;
}

}  // namespace snntc
