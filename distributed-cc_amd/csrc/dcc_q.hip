// Kernels of the (Q)/[Q] energy (distr_cc/rccsdt_q.py:943-1177).
#include "dcc_common.h"

namespace {

// out[a,b,c,i,j,k] (a,b,c < vpad) = T[ijk][abc] for a,b,c < nvir, 0 in the padding.
// T3 is the canonical i<=j<=k block array; the ordered (i,j,k) maps onto its
// canonical block with the simultaneous permutation of (a,b,c).
__global__ void t3_to_abc_kernel(const double *__restrict__ t3, int no, int nv, int vp, double *__restrict__ out) {
    const int64_t o = no, v = nv, p = vp;
    const int64_t total = p * p * p * o * o * o;
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= total) return;
    const int k = (int)(t % o), j = (int)((t / o) % o), i = (int)((t / (o * o)) % o);
    const int64_t abc = t / (o * o * o);
    const int c = (int)(abc % p), b = (int)((abc / p) % p), a = (int)(abc / (p * p));
    double val = 0.0;
    if (a < nv && b < nv && c < nv) {
        // sort (i,j,k) carrying (a,b,c) along
        int oi[3] = {i, j, k}, vi[3] = {a, b, c};
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int u = 0; u < 2 - s; ++u)
                if (oi[u] > oi[u + 1]) {
                    int x = oi[u]; oi[u] = oi[u + 1]; oi[u + 1] = x;
                    x = vi[u]; vi[u] = vi[u + 1]; vi[u + 1] = x;
                }
        const int64_t n = no;
        const int64_t ci = oi[0], cj = oi[1], ck = oi[2];
        const int64_t ni = n - ci;
        const int64_t lin = (n * (n + 1) * (n + 2) - ni * (ni + 1) * (ni + 2)) / 6 +
                            (cj - ci) * (2 * n - cj - ci + 1) / 2 + (ck - cj);
        val = t3[lin * v * v * v + ((int64_t)vi[0] * v + vi[1]) * v + vi[2]];
    }
    out[t] = val;
}

// Canonical index of a sorted triple x <= y <= z of n values, lexicographic (distribute_t3.py:51-60,
// the same closed form for occupied and virtual triples).
__device__ __forceinline__ int64_t tri_lin(int64_t n, int64_t x, int64_t y, int64_t z) {
    const int64_t m = n - x;
    return (n * (n + 1) * (n + 2) - m * (m + 1) * (m + 2)) / 6 + (y - x) * (2 * n - y - x + 1) / 2 + (z - y);
}

// Inverse of tri_lin (x <= y <= z < n) by counting.
__device__ __forceinline__ void tri_decode(int64_t n, int64_t lin, int &x, int &y, int &z) {
    x = 0;
    while (x + 1 < n && tri_lin(n, x + 1, x + 1, x + 1) <= lin) ++x;
    y = x;
    while (y + 1 < n && tri_lin(n, x, y + 1, y + 1) <= lin) ++y;
    z = (int)(lin - tri_lin(n, x, y, y)) + y;
}

// Sort three keys ascending, carrying three values along (ties keep their order).
__device__ __forceinline__ void sort3_carry(int k[3], int w[3]) {
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int u = 0; u < 2 - s; ++u)
            if (k[u] > k[u + 1]) {
                int t = k[u]; k[u] = k[u + 1]; k[u + 1] = t;
                t = w[u]; w[u] = w[u + 1]; w[u + 1] = t;
            }
}

// IJK -> ABC: out[lin(a,b,c), i, j, k] = T[ijk][abc] for a <= b <= c and every ordered (i,j,k), from the
// canonical i <= j <= k blocks.  One workgroup per virtual triple; threads run over (i,j,k), so every
// output row of o^3 values is written contiguously.
__global__ __launch_bounds__(256) void t3_tri_to_abc_packed_kernel(const double *__restrict__ t3, int no, int nv,
                                                                   double *__restrict__ out) {
    __shared__ int sabc[3];
    const int64_t lin = blockIdx.x;
    if (threadIdx.x == 0) tri_decode(nv, lin, sabc[0], sabc[1], sabc[2]);
    __syncthreads();
    const int64_t o = no, v = nv, o3 = o * o * o;
    for (int64_t t = threadIdx.x; t < o3; t += blockDim.x) {
        int occ[3] = {(int)(t / (o * o)), (int)((t / o) % o), (int)(t % o)};
        int vir[3] = {sabc[0], sabc[1], sabc[2]};
        sort3_carry(occ, vir);
        out[lin * o3 + t] = t3[tri_lin(o, occ[0], occ[1], occ[2]) * v * v * v + ((int64_t)vir[0] * v + vir[1]) * v +
                               vir[2]];
    }
}

// ABC -> dense: out[a,b,c,i,j,k] (a,b,c < vpad) = T_{ijk}^{abc} for a,b,c < nvir (0 in the padding) from
// the ABC array t3_abc[lin(a<=b<=c), i, j, k]; (a,b,c) is sorted carrying (i,j,k) along.  One workgroup
// per (a,b,c) of the dense output.
__global__ __launch_bounds__(256) void t3_abc_packed_to_dense_kernel(const double *__restrict__ t3_abc, int no,
                                                                     int nv, int vp, double *__restrict__ out) {
    const int64_t abc = blockIdx.x;
    const int a = (int)(abc / ((int64_t)vp * vp)), b = (int)((abc / vp) % vp), c = (int)(abc % vp);
    const int64_t o = no, o3 = o * o * o;
    double *dst = out + abc * o3;
    if (a >= nv || b >= nv || c >= nv) {
        for (int64_t t = threadIdx.x; t < o3; t += blockDim.x) dst[t] = 0.0;
        return;
    }
    int key[3] = {a, b, c}, pos[3] = {0, 1, 2};
    sort3_carry(key, pos);
    const double *src = t3_abc + tri_lin(nv, key[0], key[1], key[2]) * o3;
    for (int64_t t = threadIdx.x; t < o3; t += blockDim.x) {
        const int y[3] = {(int)(t / (o * o)), (int)((t / o) % o), (int)(t % o)};
        dst[t] = src[((int64_t)y[pos[0]] * o + y[pos[1]]) * o + y[pos[2]]];
    }
}

// factor of the restricted a<=b<=c<=d sum (distr_cc/rccsdt_q.py:410-428)
__device__ __forceinline__ double q_factor(int a, int b, int c, int d) {
    if (a < b && b < c && c < d) return 24.0;
    if ((a == b && b < c && c < d) || (a < b && b == c && c < d) || (a < b && b < c && c == d)) return 12.0;
    if (a == b && b < c && c == d) return 6.0;
    return 0.0;
}

constexpr int kQThreads = 256;
constexpr int kQMaxO4 = 6561;  // nocc <= 9: two o^4 FP64 buffers in LDS

// Task block start letters and the (a,b,c,d) of workgroup blockIdx.x of a chunk of tasks.
struct QQuad {
    int a, b, c, d;
};

__device__ __forceinline__ QQuad q_quad(const int *__restrict__ tasks, int bs) {
    const int bs4 = bs * bs * bs * bs;
    const int64_t task = blockIdx.x / bs4;
    const int e = (int)(blockIdx.x % bs4);
    const int ia = e / (bs * bs * bs), ib = (e / (bs * bs)) % bs, ic = (e / bs) % bs, id = e % bs;
    return {tasks[4 * task] + ia, tasks[4 * task + 1] + ib, tasks[4 * task + 2] + ic, tasks[4 * task + 3] + id};
}

// z4_sq[i,j,k,l] of (a,b,c,d) from <ab|ij> and t2, both (vp, vp, o, o) (rccsdt_q.py:1143-1150).
__device__ __forceinline__ double q_zsq(const double *__restrict__ vvoo, const double *__restrict__ t2, int64_t v,
                                        int o, const QQuad &q, int i, int j, int k, int l) {
    auto VV = [&](int p, int r, int s, int u) { return vvoo[((p * v + r) * o + s) * o + u]; };
    auto T2 = [&](int p, int r, int s, int u) { return t2[((p * v + r) * o + s) * o + u]; };
    const int a = q.a, b = q.b, c = q.c, d = q.d;
    return VV(a, b, i, j) * T2(c, d, k, l) + VV(a, c, i, k) * T2(b, d, j, l) + VV(a, d, i, l) * T2(b, c, j, k) +
           VV(b, c, j, k) * T2(a, d, i, l) + VV(b, d, j, l) * T2(a, c, i, k) + VV(c, d, k, l) * T2(a, b, i, j);
}

// Workgroup sums of (paren, bracket) into partials[2 * wg + {0, 1}].
__device__ __forceinline__ void q_store_partials(double paren, double bracket, double *__restrict__ partials,
                                                 int64_t wg) {
    __shared__ double red[2][kQThreads / 64];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        paren += __shfl_down(paren, off, 64);
        bracket += __shfl_down(bracket, off, 64);
    }
    const int lane = threadIdx.x % 64, wave = threadIdx.x / 64;
    if (lane == 0) {
        red[0][wave] = paren;
        red[1][wave] = bracket;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        double p = 0.0, q = 0.0;
        for (int w = 0; w < kQThreads / 64; ++w) {
            p += red[0][w];
            q += red[1][w];
        }
        partials[2 * wg] = p;
        partials[2 * wg + 1] = q;
    }
}

// One workgroup per (task, a, b, c, d): t4 = P4_444[(t4 + z4_p) / D] * factor on
// the o^4 occupied block, then partial sums <t4, z4_p> and <t4, z4_sq> with
// z4_sq built on the fly from <ab|ij> (vvoo) and t2 (vvoo layout).  nocc <= 9:
// both intermediates of P4_444 live in LDS.
__global__ __launch_bounds__(kQThreads) void q_finalize_kernel(
    const double *__restrict__ t4, const double *__restrict__ z4, const int *__restrict__ tasks, int bs, int no,
    int nv, int vp, const double *__restrict__ e_occ, const double *__restrict__ e_vir,
    const double *__restrict__ vvoo, const double *__restrict__ t2, double *__restrict__ partials) {
    extern __shared__ double lds[];
    const int o = no, o2 = o * o, o3 = o2 * o, o4 = o3 * o;
    double *b0 = lds, *b1 = lds + o4;
    const QQuad q = q_quad(tasks, bs);
    double paren = 0.0, bracket = 0.0;
    const double fac = (q.a < nv && q.b < nv && q.c < nv && q.d < nv) ? q_factor(q.a, q.b, q.c, q.d) : 0.0;
    if (fac != 0.0) {  // uniform over the workgroup
        const int64_t base = blockIdx.x * (int64_t)o4;
        const double ev = e_vir[q.a] + e_vir[q.b] + e_vir[q.c] + e_vir[q.d];
        for (int x = threadIdx.x; x < o4; x += kQThreads) {
            const int i = x / o3, j = (x / o2) % o, k = (x / o) % o, l = x % o;
            const double den = e_occ[i] + e_occ[j] + e_occ[k] + e_occ[l] - ev;
            const double num = t4[base + x] + z4[base + x];
            b0[x] = fabs(den) > 1e-15 ? num / den : 0.0;
        }
        __syncthreads();
        // (2 - P_ab - P_ac - P_ad) on the occupied positions
        for (int x = threadIdx.x; x < o4; x += kQThreads) {
            const int i = x / o3, j = (x / o2) % o, k = (x / o) % o, l = x % o;
            b1[x] = 2.0 * b0[x] - b0[((j * o + i) * o + k) * o + l] - b0[((k * o + j) * o + i) * o + l] -
                    b0[((l * o + j) * o + k) * o + i];
        }
        __syncthreads();
        // (2 - P_bc - P_bd)
        for (int x = threadIdx.x; x < o4; x += kQThreads) {
            const int i = x / o3, j = (x / o2) % o, k = (x / o) % o, l = x % o;
            b0[x] = 2.0 * b1[x] - b1[((i * o + k) * o + j) * o + l] - b1[((i * o + l) * o + k) * o + j];
        }
        __syncthreads();
        for (int x = threadIdx.x; x < o4; x += kQThreads) {
            const int i = x / o3, j = (x / o2) % o, k = (x / o) % o, l = x % o;
            // (2 - P_cd), then the factor
            const double t = fac * (2.0 * b0[x] - b0[((i * o + j) * o + l) * o + k]);
            paren += t * z4[base + x];
            bracket += t * q_zsq(vvoo, t2, vp, o, q, i, j, k, l);
        }
    }
    q_store_partials(paren, bracket, partials, blockIdx.x);
}

// The same update for any nocc, with one o^4 intermediate per workgroup in the global workspace ws
// (o^4 doubles at ws + blockIdx.x * o^4).  The denominator is invariant under permutations of
// (i,j,k,l), so b1 = (2 - P_ab - P_ac - P_ad)(t4 + z4) / D is formed in one pass from t4 and z4 at
// the four positions; (2 - P_cd)(2 - P_bc - P_bd) b1 expands to
//   4 b1[ijkl] - 2 b1[ikjl] - 2 b1[ilkj] - 2 b1[ijlk] + b1[iljk] + b1[iklj].
__global__ __launch_bounds__(kQThreads) void q_finalize_ws_kernel(
    const double *__restrict__ t4, const double *__restrict__ z4, const int *__restrict__ tasks, int bs, int no,
    int nv, int vp, const double *__restrict__ e_occ, const double *__restrict__ e_vir,
    const double *__restrict__ vvoo, const double *__restrict__ t2, double *__restrict__ ws,
    double *__restrict__ partials) {
    const int64_t o = no, o2 = o * o, o3 = o2 * o, o4 = o3 * o;
    const QQuad q = q_quad(tasks, bs);
    double paren = 0.0, bracket = 0.0;
    const double fac = (q.a < nv && q.b < nv && q.c < nv && q.d < nv) ? q_factor(q.a, q.b, q.c, q.d) : 0.0;
    if (fac != 0.0) {  // uniform over the workgroup
        const int64_t base = blockIdx.x * o4;
        const double *s4 = t4 + base, *z = z4 + base;
        double *b1 = ws + base;
        const double ev = e_vir[q.a] + e_vir[q.b] + e_vir[q.c] + e_vir[q.d];
        auto S = [&](int64_t y) { return s4[y] + z[y]; };
        for (int64_t x = threadIdx.x; x < o4; x += kQThreads) {
            const int64_t i = x / o3, j = (x / o2) % o, k = (x / o) % o, l = x % o;
            const double den = e_occ[i] + e_occ[j] + e_occ[k] + e_occ[l] - ev;
            const double num = 2.0 * S(x) - S(((j * o + i) * o + k) * o + l) - S(((k * o + j) * o + i) * o + l) -
                               S(((l * o + j) * o + k) * o + i);
            b1[x] = fabs(den) > 1e-15 ? num / den : 0.0;
        }
        __syncthreads();
        for (int64_t x = threadIdx.x; x < o4; x += kQThreads) {
            const int64_t i = x / o3, j = (x / o2) % o, k = (x / o) % o, l = x % o;
            const double t = fac * (4.0 * b1[x] - 2.0 * b1[((i * o + k) * o + j) * o + l] -
                                    2.0 * b1[((i * o + l) * o + k) * o + j] - 2.0 * b1[((i * o + j) * o + l) * o + k] +
                                    b1[((i * o + l) * o + j) * o + k] + b1[((i * o + k) * o + l) * o + j]);
            paren += t * z[x];
            bracket += t * q_zsq(vvoo, t2, vp, (int)o, q, (int)i, (int)j, (int)k, (int)l);
        }
    }
    q_store_partials(paren, bracket, partials, blockIdx.x);
}

// ---------------------------------------------------------------------------------------------
// Fused (Q) quadruple: one workgroup forms z4 and t4 of one (a,b,c,d) in LDS and finishes it there.
//
// The 24 z4 and 24 t4 terms of rccsdt_q.py:1014-1129 are two kinds of product over the o^4 block:
//   pair terms, (p,q) one of the six virtual pairs, r < s the other two, x,y,z,n occupied indices that
//     sit in the slots of p, q, r, s:
//       z4[x,y,z,n] += sum_e T[p,q,e,x,y,z] V[r,s,e,n]    and the same with r and s (and z, n) swapped
//       t4[x,y,z,n] -= sum_m Wo[p,q,m,x,y,z] t2[r,s,m,n]  (likewise)
//     Both share the left operand, so they are one product of o^3 rows by 2 o columns.
//   square terms, per partition of the four into rows {y,z} and columns {x,s}:
//       t4 += Wv[x,y,z,e,Y,Z] t2[e,s,X,S],  z4 -= T[x,y,z,m,Y,Z] vooo[s,m,S,X]
//     for (x,s), (s,x) and with the roles of rows and columns exchanged: four terms of one o^2 x o^2
//     product accumulated before they are added.  (T[x,y,z,..] with x in any order: T is symmetric.)
// Products run on v_mfma_f64_16x16x4 with both operands read straight from L2 (rows of T, Wo, Wv and t2
// are contiguous, 128-byte pieces); every element of the o^4 block is added by one lane per barrier
// interval, so the sums have a fixed order.  z4 and t4 never reach HBM: written and read back by 48
// batched GEMMs and a finalize pass they were 811 GB at nocc=8, nvir=40 and bound the evaluation: a whole
// (Q) call at nocc=8, nvir=38 takes 53 ms this way against 312 ms, at nocc=5, nvir=19 1.2 ms against 5.9 ms.
// The kernel is 41.5 ms of that at nocc=8, 0.64 ms at nocc=5.  Two workgroups fit a CU at nocc=8, so latency
// bounds it: loads several MFMA steps ahead and the deal over the XCDs took it there from 46.1 and 0.80 ms.
// (One loop over all terms that also keeps the next term's first loads in flight over the barriers was
// slower, 50.4 and 0.88 ms: its operands and LDS strides are then no constants of the code.)
// The block is stored with odd strides so that lanes running over any occupied index hit distinct banks.
struct QQuadArgs {
    const double *T, *vvvo, *vooo, *t2, *Wv, *Wo, *vvoo, *e_occ, *e_vir;
    const int *tasks, *slots;   // slots: per task the 12 Wv slots of its ordered block triples, or null
    int bs, nv, vp;
    int64_t total;   // quadruples: tasks * bs^4
    double *partials;
};

typedef double qd4 __attribute__((ext_vector_type(4)));

template <int O> struct QBlk {
    static constexpr int O2 = O * O, O3 = O2 * O, O4 = O3 * O;
    static constexpr int S1 = O | 1, S2 = (O * S1) | 1, S3 = (O * S2) | 1, SZ = O * S3;
    static constexpr int RF3 = (O3 + 15) / 16;              // row fragments of a pair term
    static constexpr int CF3 = (2 * O + 15) / 16;           // column fragments of a pair term
    static constexpr int RB = CF3 == 1 ? (RF3 + 3) / 4 : 4;  // row fragments per wave and pass (registers)
    static constexpr int RF2 = (O2 + 15) / 16, NF2 = RF2 * RF2, TF2 = (NF2 + 3) / 4;
    // MFMA steps per stage of loads: a stage is in flight while the previous one is multiplied, and an L2 load
    // takes as long as some 20 MFMAs of a wave, so the fewer products a step has the more steps go together
    static constexpr int KU3 = RB > 4 || CF3 > 1 ? 2 : RB > 2 ? 3 : 2, KU2 = TF2 > 4 ? 1 : TF2 == 3 ? 4 : TF2 > 1 ? 5 : 2;
    // with four row fragments a wave's fragments w, w + 4, .. share their rows
    static constexpr int NA2 = RF2 == 4 ? 1 : TF2;
    static constexpr int WAVES = O == 9 ? 1 : O >= 6 ? 2 : 5;   // resident per SIMD (LDS: two at O = 8, one at 9)
    __device__ static int pos(int slot) { return slot == 0 ? S3 : slot == 1 ? S2 : slot == 2 ? S1 : 1; }
    // LDS position of the linear element x of the o^4 block
    __device__ static int at(int x) { return x / O3 * S3 + x / O2 % O * S2 + x / O % O * S1 + x % O; }
};

// dst[x,y,z,n] (+)= sign * sum_k A[k][x,y,z] B1[k][n] and dst[x,y,n,z] (+)= sign * sum_k A[k][x,y,z] B2[k][n]
// with A of O^3 columns per k and B of O per k; sx..sn: LDS strides of the slots of x, y, z, n.
template <int O>
__device__ __forceinline__ void q_pair_term(const double *__restrict__ A, const double *__restrict__ B1,
                                            const double *__restrict__ B2, int K, double sign, double *dst, int sx,
                                            int sy, int sz, int sn) {
    typedef QBlk<O> G;
    const int lane = threadIdx.x % 64, w = threadIdx.x / 64, lr = lane % 16, lk = lane / 16;
    const double *bp[G::CF3];
    bool bok[G::CF3];
#pragma unroll
    for (int c = 0; c < G::CF3; ++c) {
        const int col = lr + 16 * c;
        bok[c] = col < 2 * O;
        bp[c] = !bok[c] ? B1 : col < O ? B1 + col : B2 + (col - O);
    }
    for (int g = 0; g < G::RF3; g += 4 * G::RB) {
        const double *ap[G::RB];
#pragma unroll
        for (int r = 0; r < G::RB; ++r) ap[r] = A + min((g + w + 4 * r) * 16 + lr, G::O3 - 1);
        qd4 acc[G::RB][G::CF3];
#pragma unroll
        for (int r = 0; r < G::RB; ++r)
#pragma unroll
            for (int c = 0; c < G::CF3; ++c) acc[r][c] = qd4{0, 0, 0, 0};
        // k of this lane in steps of 4; beyond K the last k is read and multiplied by zero
        double a[2][G::KU3][G::RB], b[2][G::KU3][G::CF3];
        auto load = [&](int s, int k0) {
#pragma unroll
            for (int q = 0; q < G::KU3; ++q) {
                if (k0 + 4 * q >= K) break;   // uniform
                const int k = k0 + 4 * q + lk, kk = min(k, K - 1);
#pragma unroll
                for (int r = 0; r < G::RB; ++r) a[s][q][r] = ap[r][(int64_t)kk * G::O3];
#pragma unroll
                for (int c = 0; c < G::CF3; ++c) {
                    const double x = bp[c][kk * O];
                    b[s][q][c] = k < K && bok[c] ? x : 0.0;
                }
            }
        };
        auto mul = [&](int s, int k0) {
#pragma unroll
            for (int q = 0; q < G::KU3; ++q) {
                if (k0 + 4 * q >= K) break;
#pragma unroll
                for (int r = 0; r < G::RB; ++r)
#pragma unroll
                    for (int c = 0; c < G::CF3; ++c)
                        acc[r][c] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[s][q][r], b[s][q][c], acc[r][c], 0, 0, 0);
            }
        };
        constexpr int KS = 4 * G::KU3;
        load(0, 0);
        for (int k0 = 0; k0 < K; k0 += 2 * KS) {
            load(1, k0 + KS);
            mul(0, k0);
            load(0, k0 + 2 * KS);
            mul(1, k0 + KS);
        }
        // the two terms of a column group touch the same elements: one barrier interval each
#pragma unroll
        for (int t = 0; t < 2; ++t) {
#pragma unroll
            for (int c = 0; c < G::CF3; ++c) {
                const int col = lr + 16 * c, n = t ? col - O : col;
                if (n < 0 || n >= O) continue;
#pragma unroll
                for (int r = 0; r < G::RB; ++r)
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const int row = (g + w + 4 * r) * 16 + lk + 4 * q;
                        if (row >= G::O3) continue;
                        const int x = row / G::O2, y = row / O % O, z = row % O;
                        double *d = dst + x * sx + y * sy + (t ? z * sn + n * sz : z * sz + n * sn);
                        *d += sign * acc[r][c][q];
                    }
            }
            __syncthreads();
        }
    }
}

// acc += sum_k A[k ka + row] B[k kb + col] over K for this wave's fragments of an O^2 x O^2 product;
// TR / TC: the row / column pair (u,v) is stored as [v][u] in its operand.
template <int O, bool TR, bool TC>
__device__ __forceinline__ void q_square_acc(const double *__restrict__ A, int64_t ka, const double *__restrict__ B,
                                             int64_t kb, int K, qd4 *acc) {
    typedef QBlk<O> G;
    const int lane = threadIdx.x % 64, w = threadIdx.x / 64, lr = lane % 16, lk = lane / 16;
    int ar[G::NA2], bc[G::TF2];
#pragma unroll
    for (int t = 0; t < G::TF2; ++t) {
        const int f = min(w + 4 * t, G::NF2 - 1);
        const int row = min(f % G::RF2 * 16 + lr, G::O2 - 1), col = min(f / G::RF2 * 16 + lr, G::O2 - 1);
        if (t < G::NA2) ar[t] = TR ? row % O * O + row / O : row;
        bc[t] = TC ? col % O * O + col / O : col;
    }
    double a[2][G::KU2][G::NA2], b[2][G::KU2][G::TF2];
    auto load = [&](int s, int k0) {
#pragma unroll
        for (int q = 0; q < G::KU2; ++q) {
            if (k0 + 4 * q >= K) break;   // uniform
            const int k = k0 + 4 * q + lk, kk = min(k, K - 1);
            const double *ak = A + kk * ka, *bk = B + kk * kb;
#pragma unroll
            for (int t = 0; t < G::TF2; ++t) {
                if (t < G::NA2) a[s][q][t] = ak[ar[t]];
                const double x = bk[bc[t]];
                b[s][q][t] = k < K ? x : 0.0;
            }
        }
    };
    auto mul = [&](int s, int k0) {
#pragma unroll
        for (int q = 0; q < G::KU2; ++q) {
            if (k0 + 4 * q >= K) break;
#pragma unroll
            for (int t = 0; t < G::TF2; ++t)
                acc[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[s][q][G::NA2 == 1 ? 0 : t], b[s][q][t], acc[t],
                                                                0, 0, 0);
        }
    };
    constexpr int KS = 4 * G::KU2;
    load(0, 0);
    for (int k0 = 0; k0 < K; k0 += 2 * KS) {
        load(1, k0 + KS);
        mul(0, k0);
        load(0, k0 + 2 * KS);
        mul(1, k0 + KS);
    }
}

// dst += sign * acc, rows (y,z) and columns (x,s) with the LDS strides of their slots
template <int O>
__device__ __forceinline__ void q_square_add(const qd4 *acc, double sign, double *dst, int sy, int sz, int sx, int ss) {
    typedef QBlk<O> G;
    const int lane = threadIdx.x % 64, w = threadIdx.x / 64, lr = lane % 16, lk = lane / 16;
#pragma unroll
    for (int t = 0; t < G::TF2; ++t) {
        const int f = w + 4 * t;
        const int col = f / G::RF2 * 16 + lr;
        if (f >= G::NF2 || col >= G::O2) continue;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int row = f % G::RF2 * 16 + lk + 4 * q;
            if (row < G::O2) dst[row / O * sy + row % O * sz + col / O * sx + col % O * ss] += sign * acc[t][q];
        }
    }
}

template <int O>
__global__ __launch_bounds__(kQThreads) __attribute__((amdgpu_waves_per_eu(QBlk<O>::WAVES)))
void q_quad_kernel(const QQuadArgs p) {
    typedef QBlk<O> G;
    extern __shared__ double lds[];
    double *Z = lds, *S = lds + G::SZ;
    // 256 consecutive quadruples run on one XCD (they share T[a,b], T[a,c], T[b,c] slices in its L2), and such
    // units are dealt round robin: the early tasks have many (a,b,c,d) without weight, and an eighth of the
    // list each left XCDs idle a third of the time.
    const int bs = p.bs, bs3 = bs * bs * bs, bs4 = bs3 * bs;
    const uint32_t unit = blockIdx.x / 8 / 256 * 8 + blockIdx.x % 8;
    const int64_t wg = (int64_t)unit * 256 + blockIdx.x / 8 % 256;
    if (wg >= p.total) return;
    const int64_t task = wg / (uint32_t)bs4;
    const int e0 = (int)(wg - task * bs4);
    const int in[4] = {e0 / bs3, e0 / (bs * bs) % bs, e0 / bs % bs, e0 % bs};   // index within each block
    int v[4];                                                                   // a, b, c, d
#pragma unroll
    for (int u = 0; u < 4; ++u) v[u] = p.tasks[4 * task + u] + in[u];
    const double fac = v[0] < p.nv && v[1] < p.nv && v[2] < p.nv && v[3] < p.nv ? q_factor(v[0], v[1], v[2], v[3]) : 0.0;
    if (fac == 0.0) {   // uniform over the workgroup
        if (threadIdx.x == 0) {
            p.partials[2 * wg] = 0.0;
            p.partials[2 * wg + 1] = 0.0;
        }
        return;
    }
    const int64_t vp = p.vp;
    const int K = p.nv;
    for (int x = threadIdx.x; x < 2 * G::SZ; x += kQThreads) lds[x] = 0.0;
    __syncthreads();
    // ---- pair terms: (p,q) over the six pairs, r < s the others ----
#pragma unroll
    for (int u = 0; u < 6; ++u) {
        constexpr int PP[6] = {0, 0, 0, 1, 1, 2}, QQ[6] = {1, 2, 3, 2, 3, 3};
        constexpr int RR[6] = {2, 1, 1, 0, 0, 0}, SS[6] = {3, 3, 2, 3, 2, 1};
        const int P = PP[u], Q = QQ[u], R = RR[u], X = SS[u];
        const int64_t pq = v[P] * vp + v[Q], rs = v[R] * vp + v[X], sr = v[X] * vp + v[R];
        const double *A = p.T + pq * vp * G::O3, *Ao = p.Wo + pq * O * G::O3;
        const double *B1 = p.vvvo + rs * vp * O, *B2 = p.vvvo + sr * vp * O;
        const double *C1 = p.t2 + rs * G::O2, *C2 = p.t2 + sr * G::O2;
        const int sx = G::pos(P), sy = G::pos(Q), sz = G::pos(R), sn = G::pos(X);
        q_pair_term<O>(A, B1, B2, K, 1.0, Z, sx, sy, sz, sn);
        q_pair_term<O>(Ao, C1, C2, O, -1.0, S, sx, sy, sz, sn);
    }
    // ---- square terms: columns (a, s), rows the other two ----
    auto wv = [&](int x, int y, int z) {   // Wv[v[x], v[y], v[z]]
        if (p.slots == nullptr) return p.Wv + ((v[x] * vp + v[y]) * vp + v[z]) * vp * G::O2;
        // slot of the ordered block triple: x, and the position of the letter left out among the other three
        const int left = 6 - x - y - z;
        const int64_t slot = p.slots[12 * task + 3 * x + (left > x ? left - 1 : left)];
        return p.Wv + (slot * bs3 + (in[x] * bs + in[y]) * bs + in[z]) * vp * G::O2;
    };
    auto tm = [&](int x, int y, int z) { return p.T + ((v[x] * vp + v[y]) * vp + v[z]) * G::O3; };
    auto t2 = [&](int s) { return p.t2 + v[s] * (int64_t)G::O2; };
    auto vo = [&](int s) { return p.vooo + v[s] * (int64_t)G::O3; };
#pragma unroll
    for (int s = 1; s < 4; ++s) {
        const int y = s == 1 ? 2 : 1, z = s == 3 ? 2 : 3;
        qd4 acc[G::TF2];
#pragma unroll
        for (int t = 0; t < G::TF2; ++t) acc[t] = qd4{0, 0, 0, 0};
        const int64_t kt = vp * G::O2;
        q_square_acc<O, false, false>(wv(0, y, z), G::O2, t2(s), kt, K, acc);
        q_square_acc<O, false, true>(wv(s, y, z), G::O2, t2(0), kt, K, acc);
        q_square_acc<O, false, false>(t2(z), kt, wv(y, 0, s), G::O2, K, acc);
        q_square_acc<O, true, false>(t2(y), kt, wv(z, 0, s), G::O2, K, acc);
        q_square_add<O>(acc, 1.0, S, G::pos(y), G::pos(z), G::pos(0), G::pos(s));
#pragma unroll
        for (int t = 0; t < G::TF2; ++t) acc[t] = qd4{0, 0, 0, 0};
        q_square_acc<O, false, true>(tm(0, y, z), G::O2, vo(s), G::O2, O, acc);
        q_square_acc<O, false, false>(tm(s, y, z), G::O2, vo(0), G::O2, O, acc);
        q_square_acc<O, true, false>(vo(z), G::O2, tm(y, 0, s), G::O2, O, acc);
        q_square_acc<O, false, false>(vo(y), G::O2, tm(z, 0, s), G::O2, O, acc);
        q_square_add<O>(acc, -1.0, Z, G::pos(y), G::pos(z), G::pos(0), G::pos(s));
        __syncthreads();
    }
    // ---- P4_444 of (t4 + z4) / D times the factor (see q_finalize_ws_kernel for the expanded form) ----
    constexpr int NX = (G::O4 + kQThreads - 1) / kQThreads;
    double val[NX];
    const double ev = p.e_vir[v[0]] + p.e_vir[v[1]] + p.e_vir[v[2]] + p.e_vir[v[3]];
#pragma unroll
    for (int n = 0; n < NX; ++n) {
        const int x = threadIdx.x + n * kQThreads;
        if (x < G::O4) S[G::at(x)] += Z[G::at(x)];
    }
    __syncthreads();
    auto ix = [](int i, int j, int k, int l) { return i * G::S3 + j * G::S2 + k * G::S1 + l; };
#pragma unroll
    for (int n = 0; n < NX; ++n) {
        const int x = threadIdx.x + n * kQThreads;
        if (x >= G::O4) continue;
        const int i = x / G::O3, j = x / G::O2 % O, k = x / O % O, l = x % O;
        const double den = p.e_occ[i] + p.e_occ[j] + p.e_occ[k] + p.e_occ[l] - ev;
        const double num = 2.0 * S[ix(i, j, k, l)] - S[ix(j, i, k, l)] - S[ix(k, j, i, l)] - S[ix(l, j, k, i)];
        val[n] = fabs(den) > 1e-15 ? num / den : 0.0;
    }
    __syncthreads();
#pragma unroll
    for (int n = 0; n < NX; ++n) {
        const int x = threadIdx.x + n * kQThreads;
        if (x < G::O4) S[G::at(x)] = val[n];
    }
    __syncthreads();
    double paren = 0.0, bracket = 0.0;
#pragma unroll
    for (int n = 0; n < NX; ++n) {
        const int x = threadIdx.x + n * kQThreads;
        if (x >= G::O4) continue;
        const int i = x / G::O3, j = x / G::O2 % O, k = x / O % O, l = x % O;
        val[n] = fac * (4.0 * S[ix(i, j, k, l)] - 2.0 * S[ix(i, k, j, l)] - 2.0 * S[ix(i, l, k, j)] -
                        2.0 * S[ix(i, j, l, k)] + S[ix(i, l, j, k)] + S[ix(i, k, l, j)]);
        paren += val[n] * Z[ix(i, j, k, l)];
    }
    __syncthreads();
    // <ab|ij> and t2 of the six pairs, in the space of z4
    for (int x = threadIdx.x; x < 12 * G::O2; x += kQThreads) {
        const int m = x / G::O2, u = m % 6, y = x % G::O2;
        const int a = u < 3 ? 0 : u < 5 ? 1 : 2, b = u < 3 ? u + 1 : u < 5 ? u - 1 : 3;
        Z[x] = (m < 6 ? p.vvoo : p.t2)[(v[a] * vp + v[b]) * G::O2 + y];
    }
    __syncthreads();
#pragma unroll
    for (int n = 0; n < NX; ++n) {
        const int x = threadIdx.x + n * kQThreads;
        if (x >= G::O4) continue;
        const int i = x / G::O3, j = x / G::O2 % O, k = x / O % O, l = x % O;
        auto VV = [&](int u, int s, int t) { return Z[u * G::O2 + s * O + t]; };
        auto T2 = [&](int u, int s, int t) { return Z[(6 + u) * G::O2 + s * O + t]; };
        bracket += val[n] * (VV(0, i, j) * T2(5, k, l) + VV(1, i, k) * T2(4, j, l) + VV(2, i, l) * T2(3, j, k) +
                             VV(3, j, k) * T2(2, i, l) + VV(4, j, l) * T2(1, i, k) + VV(5, k, l) * T2(0, i, j));
    }
    q_store_partials(paren, bracket, p.partials, wg);
}

template <int O> int q_quads_launch(const QQuadArgs &a, int64_t grid, hipStream_t s) {
    // the two blocks; at the end 12 o^2 matrix elements take their place (more than the blocks at small o)
    constexpr size_t bytes = sizeof(double) * (2 * QBlk<O>::SZ > 12 * O * O ? 2 * QBlk<O>::SZ : 12 * O * O);
    hipLaunchKernelGGL(q_quad_kernel<O>, dim3((unsigned)grid), dim3(kQThreads), bytes, s, a);
    DCC_LAUNCH_CHECK();
    return 0;
}

}  // namespace

extern "C" {

int dcc_t3_to_abc_f64(const double *t3_tri, int64_t nocc, int64_t nvir, int64_t vpad, double *out,
                      dcc_stream_t stream) {
    DCC_CHECK(nocc >= 0 && nvir >= 0 && vpad >= nvir, "bad extents");
    const int64_t total = vpad * vpad * vpad * nocc * nocc * nocc;
    if (total == 0) return 0;
    DCC_CHECK(t3_tri != nullptr && out != nullptr, "null pointer");
    DCC_CHECK((total + 255) / 256 < ((int64_t)1 << 31), "grid too large");
    hipLaunchKernelGGL(t3_to_abc_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0,
                       dcc::as_stream(stream), t3_tri, (int)nocc, (int)nvir, (int)vpad, out);
    DCC_LAUNCH_CHECK();
    return 0;
}

int dcc_t3_tri_to_abc_packed_f64(const double *t3_tri, int64_t nocc, int64_t nvir, double *t3_abc,
                                 dcc_stream_t stream) {
    DCC_CHECK(nocc >= 0 && nvir >= 0, "bad extents");
    const int64_t nabc = nvir * (nvir + 1) * (nvir + 2) / 6;
    if (nabc == 0 || nocc == 0) return 0;
    DCC_CHECK(t3_tri != nullptr && t3_abc != nullptr, "null pointer");
    DCC_CHECK(nabc < ((int64_t)1 << 31), "grid too large");
    hipLaunchKernelGGL(t3_tri_to_abc_packed_kernel, dim3((unsigned)nabc), dim3(256), 0, dcc::as_stream(stream),
                       t3_tri, (int)nocc, (int)nvir, t3_abc);
    DCC_LAUNCH_CHECK();
    return 0;
}

int dcc_t3_abc_packed_to_dense_f64(const double *t3_abc, int64_t nocc, int64_t nvir, int64_t vpad, double *out,
                                   dcc_stream_t stream) {
    DCC_CHECK(nocc >= 0 && nvir >= 0 && vpad >= nvir, "bad extents");
    const int64_t n = vpad * vpad * vpad;
    if (n == 0 || nocc == 0) return 0;
    DCC_CHECK(t3_abc != nullptr && out != nullptr, "null pointer");
    DCC_CHECK(n < ((int64_t)1 << 31), "grid too large");
    hipLaunchKernelGGL(t3_abc_packed_to_dense_kernel, dim3((unsigned)n), dim3(256), 0, dcc::as_stream(stream),
                       t3_abc, (int)nocc, (int)nvir, (int)vpad, out);
    DCC_LAUNCH_CHECK();
    return 0;
}

int dcc_q_finalize_f64(const double *t4, const double *z4, const int32_t *tasks, int64_t ntask, int64_t blksize,
                       int64_t nocc, int64_t nvir, int64_t vpad, const double *e_occ, const double *e_vir,
                       const double *vvoo, const double *t2, double *ws, double *partials, dcc_stream_t stream) {
    DCC_CHECK(ntask >= 0 && blksize > 0 && nocc > 0 && nvir > 0 && vpad >= nvir, "bad extents");
    const int64_t o4 = nocc * nocc * nocc * nocc;
    DCC_CHECK(ws != nullptr || o4 <= kQMaxO4, "nocc > 9 needs the workspace ws (ntask * blksize^4 * nocc^4 doubles)");
    const int64_t nwg = ntask * blksize * blksize * blksize * blksize;
    if (nwg == 0) return 0;
    DCC_CHECK(t4 && z4 && tasks && e_occ && e_vir && vvoo && t2 && partials, "null pointer");
    DCC_CHECK(nwg < ((int64_t)1 << 31), "grid too large");
    if (ws == nullptr) {
        hipLaunchKernelGGL(q_finalize_kernel, dim3((unsigned)nwg), dim3(kQThreads), (size_t)(2 * o4 * sizeof(double)),
                           dcc::as_stream(stream), t4, z4, tasks, (int)blksize, (int)nocc, (int)nvir, (int)vpad,
                           e_occ, e_vir, vvoo, t2, partials);
    } else {
        hipLaunchKernelGGL(q_finalize_ws_kernel, dim3((unsigned)nwg), dim3(kQThreads), 0, dcc::as_stream(stream), t4,
                           z4, tasks, (int)blksize, (int)nocc, (int)nvir, (int)vpad, e_occ, e_vir, vvoo, t2, ws,
                           partials);
    }
    DCC_LAUNCH_CHECK();
    return 0;
}

int dcc_q_quads_f64(const double *T, const double *vvvo, const double *vooo, const double *vvoo, const double *t2,
                    const double *Wv, const double *Wo, const int32_t *slots, const int32_t *tasks, int64_t ntask,
                    int64_t blksize, int64_t nocc, int64_t nvir, int64_t vpad, const double *e_occ,
                    const double *e_vir, double *partials, dcc_stream_t stream) {
    DCC_CHECK(ntask >= 0 && blksize > 0 && nocc > 0 && nvir > 0 && vpad >= nvir, "bad extents");
    DCC_CHECK(nocc <= 9, "nocc > 9: the o^4 blocks exceed LDS, use dcc_q_finalize_f64 with a workspace");
    const int64_t nwg = ntask * blksize * blksize * blksize * blksize;
    if (nwg == 0) return 0;
    DCC_CHECK(T && vvvo && vooo && vvoo && t2 && Wv && Wo && tasks && e_occ && e_vir && partials, "null pointer");
    const QQuadArgs a{T,     vvvo,  vooo,  t2,           Wv,        Wo,        vvoo,  e_occ,
                      e_vir, tasks, slots, (int)blksize, (int)nvir, (int)vpad, nwg, partials};
    hipStream_t s = dcc::as_stream(stream);
    const int64_t grid = (nwg + 2047) / 2048 * 2048;   // units of 256 on each of the eight XCDs
    DCC_CHECK(grid * kQThreads < ((int64_t)1 << 32), "grid too large");
    switch (nocc) {
        case 1: return q_quads_launch<1>(a, grid, s);
        case 2: return q_quads_launch<2>(a, grid, s);
        case 3: return q_quads_launch<3>(a, grid, s);
        case 4: return q_quads_launch<4>(a, grid, s);
        case 5: return q_quads_launch<5>(a, grid, s);
        case 6: return q_quads_launch<6>(a, grid, s);
        case 7: return q_quads_launch<7>(a, grid, s);
        case 8: return q_quads_launch<8>(a, grid, s);
        default: return q_quads_launch<9>(a, grid, s);
    }
}

}  // extern "C"
