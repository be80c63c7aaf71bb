// Loss of the reference's example networks: mean categorical cross-entropy of a one-hot label
// against softmax(-t), t = output spike times (SNN_TC_Modules.py:286-288) -- the earliest output
// spike is the predicted class.  One kernel produces the per-sample loss and the gradient of the
// batch mean with respect to the spike times; as separate framework ops this is a dozen launches
// of a few microseconds each, a visible share of a small network's training step.
#include "snntc_common.h"

namespace snntc {
namespace {

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
    for (int d = kWave / 2; d > 0; d >>= 1) v = fmaxf(v, __shfl_xor(v, d, kWave));
    return v;
}
__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
    for (int d = kWave / 2; d > 0; d >>= 1) v += __shfl_xor(v, d, kWave);
    return v;
}

// One wavefront per sample.  With l = -t, p = softmax(l), T = sum_j label_j:
//   loss_b = -sum_j label_j * (l_j - logsumexp(l)),   d(mean loss)/dt_j = (label_j - p_j * T) / B
template <int BATCH>
__global__ void __launch_bounds__(256)
softmax_time_loss_kernel(const float* __restrict__ times, const float* __restrict__ label,
                         float* __restrict__ sample_loss, float* __restrict__ dtimes, int B, int J, float inv_b) {
    const int lane = threadIdx.x % kWave;
    const int b = blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave;
    if (b >= B) return;
    const float* __restrict__ t = times + (size_t)b * J;
    const float* __restrict__ y = label + (size_t)b * J;
    // BATCH values of a lane are requested together (1000 classes: three trips to memory instead of 48, 17.8 -> 7.3 us).  Requests past the
    // end repeat the last value and cost as much as others.  2048 rows, us with batches of 1 / 8 / 16: 65 classes 6.1 / 6.2 / 7.0, 128
    // 6.2 / 6.2 / 7.1, 256 6.6 / 6.5 / 7.6, 512 8.6 / 7.0 / 8.3, 700 10.3 / 9.1 / 8.9, 1000 15.8 / 10.1 / 9.8.
    auto values = [&](const float* p, int j0, float (&v)[BATCH]) {
#pragma unroll
        for (int i = 0; i < BATCH; ++i) v[i] = p[min(j0 + i * kWave + lane, J - 1)];
    };
    auto there = [&](int j0, int i) { return j0 + i * kWave + lane < J; };
    float m = -INFINITY, tv[BATCH], yv[BATCH];
    for (int j0 = 0; j0 < J; j0 += BATCH * kWave) {
        values(t, j0, tv);
#pragma unroll
        for (int i = 0; i < BATCH; ++i)
            if (there(j0, i)) m = fmaxf(m, -tv[i]);
    }
    m = wave_max(m);
    float se = 0.0f, dot = 0.0f, tot = 0.0f;
    for (int j0 = 0; j0 < J; j0 += BATCH * kWave) {
        values(t, j0, tv);
        values(y, j0, yv);
#pragma unroll
        for (int i = 0; i < BATCH; ++i)
            if (there(j0, i)) {
                const float l = -tv[i] - m;
                se += expf(l);
                dot += yv[i] * l;
                tot += yv[i];
            }
    }
    se = wave_sum(se); dot = wave_sum(dot); tot = wave_sum(tot);
    const float lse = logf(se);
    if (lane == 0 && sample_loss) sample_loss[b] = tot * lse - dot;      // -sum_j y_j (l_j - lse)
    if (dtimes) {
        float* __restrict__ g = dtimes + (size_t)b * J;
        const float scale = tot / se;
        for (int j0 = 0; j0 < J; j0 += BATCH * kWave) {
            values(t, j0, tv);
            values(y, j0, yv);
#pragma unroll
            for (int i = 0; i < BATCH; ++i)
                if (there(j0, i)) g[j0 + i * kWave + lane] = (yv[i] - expf(-tv[i] - m) * scale) * inv_b;
        }
    }
}

}  // namespace

int launch_softmax_time_loss(const float* times, const float* label, float* sample_loss, float* dtimes,
                             int64_t B, int64_t J, hipStream_t stream) {
    if (B <= 0 || J <= 0) return SNNTC_OK;
    const int waves_per_block = 4;
    const int64_t blocks = (B + waves_per_block - 1) / waves_per_block;
    if (blocks > 0x7fffffffLL) return fail(SNNTC_ERR_TOO_LARGE, "loss: too many samples");
    {
        KernelTimerScope timer_("softmax_time_loss", stream);
        auto kern = J <= kWave ? softmax_time_loss_kernel<1> : J <= 8 * kWave ? softmax_time_loss_kernel<8> : softmax_time_loss_kernel<16>;
        hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(256), 0, stream, times, label, sample_loss, dtimes, (int)B, (int)J,
                           1.0f / (float)B);
    }
    SNNTC_HIP_CHECK(hipGetLastError());
    return SNNTC_OK;
}

}  // namespace snntc
