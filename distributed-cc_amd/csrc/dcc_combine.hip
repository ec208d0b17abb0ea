// Linear combinations of many tensors and dot products of many vectors, one launch each.
//
// The lower-order part of an iteration is some 60 contractions and 50 copies, sums, transposes, divisions and
// dot products of a few hundred to a few hundred thousand elements; each as its own launch costs 5 to 8 us
// whatever its size, which was two thirds of an iteration at nocc=5, nvir=8.  A combination job is
//     dst = [sum_t coef_t sum_{s < count_t} src_t[s cstride_t + strided]  (+ beta dst)] / D
// over up to four indices, optionally added to a second array; the jobs of one launch are independent, a
// workgroup takes 1024 consecutive elements of one job, found by binary search over the jobs' first
// workgroups.  Terms are added in their order, so results do not depend on timing.
#include "dcc_common.h"

namespace {

constexpr int kThreads = 256;
constexpr int kPer = 4;         // elements per thread
constexpr int kDotBlocks = 64;  // partial sums per dot product

__global__ __launch_bounds__(kThreads) void combine_kernel(const dcc_combine_job *__restrict__ jobs,
                                                           const dcc_combine_term *__restrict__ terms, int njobs) {
    int lo = 0, hi = njobs - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) / 2;
        if (jobs[mid].begin <= (int64_t)blockIdx.x) lo = mid;
        else hi = mid - 1;
    }
    const dcc_combine_job &j = jobs[lo];
    const uint32_t e1 = (uint32_t)j.shape[1], e2 = (uint32_t)j.shape[2], e3 = (uint32_t)j.shape[3];
    const uint32_t total = (uint32_t)(j.shape[0] * j.shape[1] * j.shape[2] * j.shape[3]);   // < 2^31
    const uint32_t t0 = (uint32_t)((int64_t)blockIdx.x - j.begin) * (kThreads * kPer) + threadIdx.x;
    uint32_t x[kPer][4];
    double v[kPer];
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
        const uint32_t t = min(t0 + u * kThreads, total - 1);   // repeated, not stored
        const uint32_t a = t / e3, b = a / e2;
        x[u][3] = t - a * e3;
        x[u][2] = a - b * e2;
        x[u][0] = b / e1;
        x[u][1] = b - x[u][0] * e1;
        v[u] = 0.0;
    }
    auto off = [&](const int64_t *s, int u) {
        return x[u][0] * s[0] + x[u][1] * s[1] + x[u][2] * s[2] + x[u][3] * s[3];
    };
    int64_t d[kPer];
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
        d[u] = off(j.dst_stride, u);
        if (j.beta != 0.0)
            v[u] = j.beta * (j.dst_f32 ? (double)static_cast<const float *>(j.dst)[d[u]]
                                       : static_cast<const double *>(j.dst)[d[u]]);
    }
    for (int64_t n = 0; n < j.nterm; ++n) {
        const dcc_combine_term &q = terms[j.term0 + n];
        int64_t o[kPer];
#pragma unroll
        for (int u = 0; u < kPer; ++u) o[u] = off(q.stride, u);
        for (int64_t s = 0; s < q.count; ++s)
#pragma unroll
            for (int u = 0; u < kPer; ++u) {
                const int64_t at = s * q.cstride + o[u];
                v[u] += q.coef * (q.f32 ? (double)static_cast<const float *>(q.src)[at]
                                        : static_cast<const double *>(q.src)[at]);
            }
    }
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
        const uint32_t t = t0 + u * kThreads;
        if (t >= total) continue;
        if (j.rank == 1) v[u] /= j.eia[t];
        else if (j.rank == 2) v[u] /= j.eia[x[u][0] * e2 + x[u][2]] + j.eia[x[u][1] * e2 + x[u][3]];
        if (j.dst_f32) static_cast<float *>(j.dst)[d[u]] = (float)v[u];
        else static_cast<double *>(j.dst)[d[u]] = v[u];
        if (j.acc != nullptr) j.acc[t] += v[u];
    }
}

__device__ __forceinline__ double block_sum(double a) {
    __shared__ double red[kThreads / 64];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) a += __shfl_down(a, off, 64);
    if (threadIdx.x % 64 == 0) red[threadIdx.x / 64] = a;
    __syncthreads();
    double s = 0.0;
    for (int w = 0; w < (int)blockDim.x / 64; ++w) s += red[w];
    return s;
}

__global__ __launch_bounds__(kThreads) void dots_kernel(const dcc_dot_job *__restrict__ jobs,
                                                        double *__restrict__ partials) {
    const dcc_dot_job &j = jobs[blockIdx.y];
    double a = 0.0;
    for (int64_t t = blockIdx.x * kThreads + threadIdx.x; t < j.n; t += kDotBlocks * kThreads) {
        double y = j.y[t];
        if (j.u != nullptr) {   // y[i,j,a,b] + u[i,a] u[j,b]
            const uint32_t nv = (uint32_t)j.nv, q = (uint32_t)t / nv, b = (uint32_t)t - q * nv, q2 = q / nv;
            const uint32_t aa = q - q2 * nv, i = q2 / (uint32_t)j.no, jj = q2 - i * (uint32_t)j.no;
            y += j.u[i * nv + aa] * j.u[jj * nv + b];
        }
        a += j.x[t] * y;
    }
    const double s = block_sum(a);
    if (threadIdx.x == 0) partials[blockIdx.y * kDotBlocks + blockIdx.x] = s;
}

__global__ __launch_bounds__(kDotBlocks) void dots_final_kernel(const dcc_dot_job *__restrict__ jobs,
                                                                const double *__restrict__ partials) {
    const double s = block_sum(partials[blockIdx.x * kDotBlocks + threadIdx.x]);
    if (threadIdx.x == 0) *jobs[blockIdx.x].out = s;
}

}  // namespace

extern "C" {

int dcc_combine(const dcc_combine_job *jobs, const dcc_combine_term *terms, int64_t njobs, int64_t nworkgroups,
                dcc_stream_t stream) {
    DCC_CHECK(njobs >= 0 && nworkgroups >= 0, "negative argument");
    DCC_CHECK(njobs < ((int64_t)1 << 30) && nworkgroups < ((int64_t)1 << 31), "too many jobs");
    if (njobs == 0 || nworkgroups == 0) return 0;
    DCC_CHECK(jobs != nullptr && terms != nullptr, "null pointer");
    hipLaunchKernelGGL(combine_kernel, dim3((unsigned)nworkgroups), dim3(kThreads), 0, dcc::as_stream(stream), jobs,
                       terms, (int)njobs);
    DCC_LAUNCH_CHECK();
    return 0;
}

int64_t dcc_dots_partials(void) { return kDotBlocks; }

int dcc_dots_f64(const dcc_dot_job *jobs, int64_t njobs, double *partials, dcc_stream_t stream) {
    DCC_CHECK(njobs >= 0 && njobs < 65536, "bad job count");
    if (njobs == 0) return 0;
    DCC_CHECK(jobs != nullptr && partials != nullptr, "null pointer");
    hipLaunchKernelGGL(dots_kernel, dim3(kDotBlocks, (unsigned)njobs), dim3(kThreads), 0, dcc::as_stream(stream), jobs,
                       partials);
    DCC_LAUNCH_CHECK();
    hipLaunchKernelGGL(dots_final_kernel, dim3((unsigned)njobs), dim3(kDotBlocks), 0, dcc::as_stream(stream), jobs,
                       partials);
    DCC_LAUNCH_CHECK();
    return 0;
}

}  // extern "C"
