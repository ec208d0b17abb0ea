// One DIIS step on device vectors (distr_cc/diis.py:105-145) in two passes over the history.
//
// Every kernel here is HBM-bound; the step is priced by how often a vector is read.  The push reads x, the
// previous iterate and the other error vectors once (2 + nd - 1 reads, 2 writes) for the new error and all
// its dot products; the combination reads the nd history vectors and the previous iterate once (nd + 1
// reads, 2 writes) for the new iterate and the norm of its change.  Separate copies, updates and dot
// products read and wrote 8 nd + 17 vectors: at 14.5 million elements and nd = 6 the step took 1.39 ms, and
// takes 0.48 ms this way (2.1 GB, 4.3 TB/s: the rate of a plain copy).
// A workgroup sums its partials in a fixed order and a second kernel sums the workgroups', so results do not
// depend on timing.
#include "dcc_common.h"

#include <type_traits>

namespace {

constexpr int kMax = 8;        // vectors per launch
constexpr int kBlocks = 1024;  // partial sums per dot product
constexpr int kThreads = 256;

struct Vectors {
    const double *v[kMax];
    double c[kMax];
};

typedef double d2 __attribute__((ext_vector_type(2)));

// Sums of M values over the workgroup into partials[m * kBlocks + block].
template <int M>
__device__ __forceinline__ void block_sums(const double *acc, double *__restrict__ partials) {
    __shared__ double red[M][kThreads / 64];
    const int lane = threadIdx.x % 64, w = threadIdx.x / 64;
#pragma unroll
    for (int m = 0; m < M; ++m) {
        double a = acc[m];
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) a += __shfl_down(a, off, 64);
        if (lane == 0) red[m][w] = a;
    }
    __syncthreads();
    if (threadIdx.x < M) {
        double a = 0.0;
#pragma unroll
        for (int q = 0; q < kThreads / 64; ++q) a += red[threadIdx.x][q];
        partials[threadIdx.x * kBlocks + blockIdx.x] = a;
    }
}

// f(E, i) over pairs of elements (16-byte accesses) where the buffers are aligned, over single ones elsewhere.
template <bool PAIRS, typename F> __device__ __forceinline__ void for_elements(int64_t n, F &&f) {
    const int64_t stride = (int64_t)gridDim.x * kThreads, t = (int64_t)blockIdx.x * kThreads + threadIdx.x;
    if constexpr (PAIRS) {
        for (int64_t i = t; i < n / 2; i += stride) f(d2{}, i);
        if (n % 2 && t == 0) f(double{}, n - 1);
    } else {
        for (int64_t i = t; i < n; i += stride) f(double{}, i);
    }
}

template <typename E> __device__ __forceinline__ E at(const double *p, int64_t i) {
    return reinterpret_cast<const E *>(p)[i];
}
__device__ __forceinline__ double dot(double a, double b) { return a * b; }
__device__ __forceinline__ double dot(d2 a, d2 b) { return a[0] * b[0] + a[1] * b[1]; }

// PUSH: xs = x, es = x - xprev.  partials of es . h.v[m] for m < M; `self` (>= 0): that vector is es itself.
template <int M, bool PUSH, bool PAIRS>
__global__ __launch_bounds__(kThreads) void push_kernel(const double *__restrict__ x, const double *__restrict__ xprev,
                                                        double *__restrict__ xs, double *es, Vectors h, int self,
                                                        int64_t n, double *__restrict__ partials) {
    double acc[M] = {};
    for_elements<PAIRS>(n, [&](auto tag, int64_t i) {
        typedef decltype(tag) E;
        E e, o[M];
#pragma unroll
        for (int m = 0; m < M; ++m)
            if (m != self) o[m] = at<E>(h.v[m], i);
        if constexpr (PUSH) {
            const E v = at<E>(x, i);
            e = v - at<E>(xprev, i);
            reinterpret_cast<E *>(xs)[i] = v;
            reinterpret_cast<E *>(es)[i] = e;
        } else {
            e = at<E>(es, i);
        }
#pragma unroll
        for (int m = 0; m < M; ++m) acc[m] += dot(e, m == self ? e : o[m]);
    });
    block_sums<M>(acc, partials);
}

// out (+)= sum_m h.c[m] h.v[m]; LAST: partials of |out - xprev|^2, then xprev = out.
template <int M, bool FIRST, bool LAST, bool PAIRS>
__global__ __launch_bounds__(kThreads) void combine_kernel(double *__restrict__ out, double *__restrict__ xprev,
                                                           Vectors h, int64_t n, double *__restrict__ partials) {
    double acc[1] = {0.0};
    for_elements<PAIRS>(n, [&](auto tag, int64_t i) {
        typedef decltype(tag) E;
        E s = FIRST ? E{} : at<E>(out, i);
#pragma unroll
        for (int m = 0; m < M; ++m) s += h.c[m] * at<E>(h.v[m], i);
        reinterpret_cast<E *>(out)[i] = s;
        if constexpr (LAST) {
            const E d = s - at<E>(xprev, i);
            acc[0] += dot(d, d);
            reinterpret_cast<E *>(xprev)[i] = s;
        }
    });
    if constexpr (LAST) block_sums<1>(acc, partials);
}

__global__ __launch_bounds__(kThreads) void sums_kernel(const double *__restrict__ partials, double *__restrict__ out) {
    double a[1] = {0.0};
    for (int i = threadIdx.x; i < kBlocks; i += kThreads) a[0] += partials[blockIdx.x * kBlocks + i];
    __shared__ double red[kThreads / 64];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) a[0] += __shfl_down(a[0], off, 64);
    if (threadIdx.x % 64 == 0) red[threadIdx.x / 64] = a[0];
    __syncthreads();
    if (threadIdx.x == 0) {
        double s = 0.0;
        for (int q = 0; q < kThreads / 64; ++q) s += red[q];
        out[blockIdx.x] = s;
    }
}

// f(integral_constant<int, m>) for 1 <= m <= kMax
template <int M = 1, typename F> void with_count(int m, F &&f) {
    if constexpr (M < kMax)
        if (m > M) return with_count<M + 1>(m, f);
    f(std::integral_constant<int, M>{});
}

bool aligned(const double *p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; }

}  // namespace

extern "C" {

int64_t dcc_diis_partials(void) { return kMax * kBlocks; }

int dcc_diis_push_f64(const double *x, const double *xprev, double *xs, const double *const *errors, int64_t nvec,
                      int64_t head, int64_t n, double *partials, double *out, dcc_stream_t stream) {
    DCC_CHECK(n >= 0 && nvec >= 1 && head >= 0 && head < nvec, "bad extents");
    DCC_CHECK(errors && partials && out, "null pointer");
    DCC_CHECK(n == 0 || (x && xprev && xs), "null pointer");
    hipStream_t s = dcc::as_stream(stream);
    double *es = const_cast<double *>(errors[head]);
    bool pairs = aligned(x) && aligned(xprev) && aligned(xs);
    for (int64_t i = 0; i < nvec; ++i) {
        DCC_CHECK(errors[i] != nullptr || n == 0, "null pointer");
        pairs = pairs && aligned(errors[i]);
    }
    for (int64_t v0 = 0; v0 < nvec; v0 += kMax) {
        const int m = (int)(nvec - v0 < kMax ? nvec - v0 : kMax);
        Vectors h{};
        for (int i = 0; i < m; ++i) h.v[i] = errors[v0 + i];
        const int self = head >= v0 && head < v0 + m ? (int)(head - v0) : -1;
        with_count(m, [&](auto mc) {
            constexpr int M = decltype(mc)::value;
            auto k = v0 == 0 ? (pairs ? push_kernel<M, true, true> : push_kernel<M, true, false>)
                             : (pairs ? push_kernel<M, false, true> : push_kernel<M, false, false>);
            hipLaunchKernelGGL(k, dim3(kBlocks), dim3(kThreads), 0, s, x, xprev, xs, es, h, self, n, partials);
        });
        DCC_LAUNCH_CHECK();
        hipLaunchKernelGGL(sums_kernel, dim3(m), dim3(kThreads), 0, s, partials, out + v0);
        DCC_LAUNCH_CHECK();
    }
    return 0;
}

int dcc_diis_combine_f64(double *xnew, double *xprev, const double *const *vectors, const double *coef, int64_t nvec,
                         int64_t n, double *partials, double *out, dcc_stream_t stream) {
    DCC_CHECK(n >= 0 && nvec >= 1, "bad extents");
    DCC_CHECK(vectors && coef && partials && out, "null pointer");
    DCC_CHECK(n == 0 || (xnew && xprev), "null pointer");
    hipStream_t s = dcc::as_stream(stream);
    bool pairs = aligned(xnew) && aligned(xprev);
    for (int64_t i = 0; i < nvec; ++i) {
        DCC_CHECK(vectors[i] != nullptr || n == 0, "null pointer");
        pairs = pairs && aligned(vectors[i]);
    }
    for (int64_t v0 = 0; v0 < nvec; v0 += kMax) {
        const int m = (int)(nvec - v0 < kMax ? nvec - v0 : kMax);
        Vectors h{};
        for (int i = 0; i < m; ++i) {
            h.v[i] = vectors[v0 + i];
            h.c[i] = coef[v0 + i];
        }
        const bool first = v0 == 0, last = v0 + kMax >= nvec;
        with_count(m, [&](auto mc) {
            constexpr int M = decltype(mc)::value;
            auto pick = [&](auto p) {
                constexpr bool P = decltype(p)::value;
                return first ? (last ? combine_kernel<M, true, true, P> : combine_kernel<M, true, false, P>)
                             : (last ? combine_kernel<M, false, true, P> : combine_kernel<M, false, false, P>);
            };
            auto k = pairs ? pick(std::true_type{}) : pick(std::false_type{});
            hipLaunchKernelGGL(k, dim3(kBlocks), dim3(kThreads), 0, s, xnew, xprev, h, n, partials);
        });
        DCC_LAUNCH_CHECK();
    }
    hipLaunchKernelGGL(sums_kernel, dim3(1), dim3(kThreads), 0, s, partials, out);
    DCC_LAUNCH_CHECK();
    return 0;
}

}  // extern "C"
