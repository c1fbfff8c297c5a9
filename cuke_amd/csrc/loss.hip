// Margin-ranking loss over (positive, shared-negative) score pairs and its gradient.
// Not part of the reference (it has no loss); defined as
//   L = mean_{b,k} max(0, margin - sign * (pos[b] - neg[b][k])).
#include <mutex>

#include "common.hpp"
#include "loss_total.hpp"

namespace kge {

constexpr int kLossWaves = 4;

// Bound by its two passes over the [B, N] scores (read, gradient written), 128 bits per lane from four scores a row on.
// A workgroup strides over the rows and leaves ONE partial loss: with one per row the single workgroup that adds them
// up walked 16384 to 30000 doubles, 18 to 30 us; over at most kLossBlocks partials it is 2 us, which a training step gives to
// the last launch of its backward pass (kge_margin_loss_parts).

template <int V, bool RAG>
__global__ __launch_bounds__(kLossWaves *kWave) void margin_rows_kernel(
    const float *pos, const float *neg, int64_t B, int64_t N, float margin, float sign, float inv,
    float *dpos, float *dneg, double *block_loss)
{
    __shared__ double s_part[kLossWaves];
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x >> 6;
    double total = 0.0;
    for (int64_t b = (int64_t)blockIdx.x * kLossWaves + wave; b < B; b += (int64_t)gridDim.x * kLossWaves) {
        const float p = pos[b];
        float sum = 0.0f;
        int cnt = 0;
        for (int64_t k0 = lane * V; k0 < N; k0 += kWave * V) {
            const int64_t k = RAG && k0 > N - V ? N - V : k0;  // the row's last piece ends with it
            const int skip = RAG ? (int)(k0 - k) : 0;
            const Vec<V> s = Vec<V>::load(neg + b * N + k);
            Vec<V> g;
#pragma unroll
            for (int e = 0; e < V; ++e) {
                const float v = margin - sign * (p - s.v[e]);
                const bool on = v > 0.0f;
                const bool count = on && e >= skip;
                sum += count ? v : 0.0f;
                cnt += count ? 1 : 0;
                g.v[e] = on ? sign * inv : 0.0f;
            }
            if (dneg) g.store_from(dneg + b * N + k, skip);
        }
        sum = wave_sum(sum);
        cnt = wave_sum_i(cnt);
        total += (double)sum;
        if (lane == 0 && dpos) dpos[b] = -sign * inv * (float)cnt;
    }
    if (lane == 0) s_part[wave] = total;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0.0;
        for (int w = 0; w < kLossWaves; ++w) t += s_part[w];
        block_loss[blockIdx.x] = t;
    }
}

__global__ __launch_bounds__(256) void margin_total_kernel(kge_loss_total total)
{
    __shared__ double s[256];
    loss_total_block(total, s);
}

// Scratch of kge_margin_loss_static: the partial losses, at most one double per positive.  Every
// GPU the library runs on holds its own copy of this array (512 KiB) until the process ends.
constexpr int64_t kStaticLossRows = KGE_MARGIN_LOSS_STATIC_MAX_BATCH;
static __device__ __align__(256) double scratch[kStaticLossRows];

constexpr int kMaxDevices = 64;
static std::mutex g_scratch_mutex;
static double *g_scratch_ptr[kMaxDevices];  // device address of `scratch` on each device, once looked up

// Device address of `scratch` on the current device (the array's name is only a host-side handle).
static int static_scratch(double **out)
{
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return KGE_ELAUNCH;
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (!g_scratch_ptr[dev]) {
        void *p = nullptr;
        if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) return KGE_ELAUNCH;
        g_scratch_ptr[dev] = static_cast<double *>(p);
    }
    *out = g_scratch_ptr[dev];
    return KGE_OK;
}

}  // namespace kge

using namespace kge;

extern "C" {

size_t kge_margin_loss_workspace(int64_t batch, int64_t n_neg)
{
    (void)n_neg;
    return batch > 0 ? sizeof(double) * (size_t)batch : 0;
}

// The row kernel, and what is left to add up behind it.
static int launch_rows(const float *pos, const float *neg, int64_t batch, int64_t n_neg, float margin, float sign, float *loss, float *dpos,
                       float *dneg, void *workspace, size_t workspace_bytes, kge_loss_total *total, hipStream_t st)
{
    if (batch < 0 || n_neg < 0 || !loss) return KGE_EINVAL;
    if (batch > 0 && n_neg > 0 && (!pos || !neg)) return KGE_EINVAL;
    if (batch > 0 && (!workspace || workspace_bytes < sizeof(double) * (size_t)batch)) return KGE_EWORKSPACE;
    const double count = (double)batch * (double)n_neg;
    const float inv = count > 0 ? (float)(1.0 / count) : 0.0f;
    double *rows = static_cast<double *>(workspace);
    const int64_t want = ceil_div(batch, kLossWaves);
    const int blocks = (int)(want < kLossBlocks ? want : kLossBlocks);  // (one partial each: never more than the workspace's `batch`)
    if (batch > 0) {
        const dim3 grid((unsigned)blocks), block(kLossWaves * kWave);
        const auto kernel = n_neg % 4 == 0 ? margin_rows_kernel<4, false> : (quad_row(n_neg) ? margin_rows_kernel<4, true> : margin_rows_kernel<1, false>);
        hipLaunchKernelGGL(kernel, grid, block, 0, st, pos, neg, batch, n_neg, margin, sign, inv, dpos, dneg, rows);
    }
    *total = kge_loss_total{rows, blocks, count > 0 ? 1.0 / count : 0.0, loss};
    return KGE_OK;
}

int kge_margin_loss(const float *pos, const float *neg, int64_t batch, int64_t n_neg, float margin,
                    float sign, float *loss, float *dpos, float *dneg, void *workspace,
                    size_t workspace_bytes, void *stream)
{
    kge_loss_total total;
    hipStream_t st = as_stream(stream);
    if (const int rc = launch_rows(pos, neg, batch, n_neg, margin, sign, loss, dpos, dneg, workspace, workspace_bytes, &total, st)) return rc;
    hipLaunchKernelGGL(margin_total_kernel, dim3(1), dim3(256), 0, st, total);
    KGE_CHECK_LAUNCH();
    return KGE_OK;
}

int kge_margin_loss_parts(const float *pos, const float *neg, int64_t batch, int64_t n_neg, float margin,
                          float sign, float *loss, float *dpos, float *dneg, void *workspace,
                          size_t workspace_bytes, kge_loss_total *total, void *stream)
{
    if (!total || batch < 1) return KGE_EINVAL;
    if (const int rc = launch_rows(pos, neg, batch, n_neg, margin, sign, loss, dpos, dneg, workspace, workspace_bytes, total, as_stream(stream))) return rc;
    KGE_CHECK_LAUNCH();
    return KGE_OK;
}

int kge_margin_loss_static(const float *pos, const float *neg, int64_t batch, int64_t n_neg, float margin,
                           float sign, float *loss, float *dpos, float *dneg, void *stream)
{
    if (batch > kStaticLossRows) return KGE_EWORKSPACE;  // more rows than the built-in scratch holds
    double *rows = nullptr;
    const int rc = static_scratch(&rows);
    if (rc) return rc;
    // every slot the total kernel reads is written by the row kernel of the same call first,
    // so nothing left behind by an earlier call needs clearing
    return kge_margin_loss(pos, neg, batch, n_neg, margin, sign, loss, dpos, dneg, rows,
                           sizeof(double) * (size_t)kStaticLossRows, stream);
}

}  // extern "C"
