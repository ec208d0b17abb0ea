// Output tiles of the batched gather-GEMM for problems that leave the 64x64..128x128 tiles of
// dcc_gemm_tile.h idle: few or narrow outputs, short of one full tile per CU, against a K of hundreds
// to tens of thousands (r1, F_oo, F_vv, W_oooo, the singles/doubles intermediates and their adjoints).
//
// What bounds those is latency along a serial K loop: a 64x64 tile steps K by 16 behind one barrier, 1.2
// to 1.5 us per step when nothing else runs on the CU, whatever M and N are.  Here a workgroup's waves
// split K instead: a tile is (16 FX) x (16 FY), wave w multiplies every W-th block of 16 k values straight
// from global memory into registers (no LDS, no barrier, the next stage's loads in flight), and the W
// partial tiles are added in LDS in wave order at the end, so results do not depend on timing.
// A lane holds 4 consecutive k of its row (the k order inside a block is the same for both operands), so a
// K-contiguous operand is read as element pairs and a row-contiguous one as whole lines of 16 rows.
// With one wave (short K, nothing to split) the k order is the staged tiles' (4 consecutive k per MFMA),
// and with it every bit of the result.
// Rows of the tile walk X, columns (consecutive lanes) walk Y; the host makes Y the operand that carries
// the contiguous index of C.
#pragma once

#include "dcc_gemm_tile.h"

namespace dcc_gemm {

enum : int {
    kSkinnyPairX = 1,   // X / Y: k, k + 1 from an even k are adjacent and aligned (pair loads)
    kSkinnyPairY = 2,
    kSkinnyStepX = 4,   // X / Y: the k of a lane's group have a constant stride in memory
    kSkinnyStepY = 8,
    kSkinnySwap = 16,   // X is operand B (rows n), Y is operand A (columns m)
};

template <typename T>
struct SkinnyArgs {
    int N, K;
    double alpha, beta;
    const T *X, *Y;
    T *C;
    dcc_idxmap xm, ym, cx, cy;
    KMap xk, yk;
    const dcc_batch *batches;
    int tiles_x, tiles_y;
    int64_t total_tiles;
    int flags;
};

template <typename T, int FX, int FY, int W> struct SkinnySmem {
    static constexpr int v = W * FX * FY * 256;
};

// K blocks of 16 per stage: two where a tile has a single fragment per operand, so that a stage keeps
// enough loads in flight
template <int FX, int FY> struct SkinnyKB {
    static constexpr int v = FX * FY == 1 ? 2 : 1;
};

template <typename T, int FX, int FY, int W>
__device__ __forceinline__ void skinny_tile(const SkinnyArgs<T> &p, int64_t batch, int tx, int ty, T *smem) {
    typedef Mfma<T> MF;
    typedef typename MF::acc_t acc_t;
    constexpr int KB = SkinnyKB<FX, FY>::v;
    const int tid = threadIdx.x, lane = tid % 64, lr = lane % 16, lk = lane / 16;
    const int w = __builtin_amdgcn_readfirstlane(tid / 64);
    const dcc_batch bt = p.batches[batch];
    const bool swap = p.flags & kSkinnySwap;
    const int64_t xb = swap ? 0 : bt.m_begin, xe = swap ? p.N : bt.m_end;
    const int64_t yb = swap ? bt.m_begin : 0, ye = swap ? bt.m_end : p.N;
    const int64_t x0 = xb + (int64_t)tx * 16 * FX, y0 = yb + (int64_t)ty * 16 * FY;
    if (x0 >= xe || y0 >= ye) return;   // uniform
    // rows past the end repeat the last one: their products are never stored
    const T *xp[FX], *yp[FY];
#pragma unroll
    for (int f = 0; f < FX; ++f) {
        const int64_t x = x0 + 16 * f + lr < xe ? x0 + 16 * f + lr : xe - 1;
        xp[f] = p.X + (swap ? bt.b_off : bt.a_off) + map_off(p.xm, (uint32_t)x, batch);
    }
#pragma unroll
    for (int f = 0; f < FY; ++f) {
        const int64_t y = y0 + 16 * f + lr < ye ? y0 + 16 * f + lr : ye - 1;
        yp[f] = p.Y + (swap ? bt.a_off : bt.b_off) + map_off(p.ym, (uint32_t)y, batch);
    }
    // batch offsets may be odd: checked here for the pair loads
    const bool vx = (p.flags & kSkinnyPairX) && ((swap ? bt.b_off : bt.a_off) & 1) == 0;
    const bool vy = (p.flags & kSkinnyPairY) && ((swap ? bt.a_off : bt.b_off) & 1) == 0;
    const bool sx = p.flags & kSkinnyStepX, sy = p.flags & kSkinnyStepY;

    // this thread's elements of C, their old values loaded while the products run
    constexpr int NE = (FX * FY * 256 + W * 64 - 1) / (W * 64);
    T *c[NE];
    T old[NE];
#pragma unroll
    for (int n = 0; n < NE; ++n) {
        const int e = tid + n * W * 64, f = e / 256, r = e / 64 % 4, el = e % 64;
        const int64_t x = x0 + f / FY * 16 + MF::row(el / 16, r), y = y0 + f % FY * 16 + el % 16;
        c[n] = e < FX * FY * 256 && x < xe && y < ye
                   ? p.C + bt.c_off + map_off(p.cx, (uint32_t)x, batch) + map_off(p.cy, (uint32_t)y, batch)
                   : nullptr;
        old[n] = p.beta != 0.0 && c[n] != nullptr ? *c[n] : T(0);
    }

    typedef T T2 __attribute__((ext_vector_type(2)));
    // 4 values of every fragment: at k .. k+3, or with one wave k, k+4, k+8, k+12.  Beyond K offset 0 is read;
    // mul zeroes those values (a select here would wait for the load, and the stage ahead would not be ahead:
    // a cycle at nocc=8, nvir=38 took 4.84 ms that way and takes 4.73 ms)
    constexpr int KS = W == 1 ? 4 : 1;
    auto load = [&](auto &reg, const T *const *ptr, const KMap &km, dcc::KIter &it, uint32_t k, bool vec, bool step,
                    auto nf) {
        constexpr int NF = decltype(nf)::value;
        if (W > 1 && vec) {   // K is even: a pair is inside or outside as a whole
#pragma unroll
            for (int h = 0; h < 4; h += 2) {
                const bool ok = k + h < (uint32_t)p.K;
                const int64_t o = !ok ? 0 : h == 0 ? it.off : step ? it.off + 2 * km.s2 : koff(km, k + 2);
#pragma unroll
                for (int f = 0; f < NF; ++f) {
                    const T2 v = *reinterpret_cast<const T2 *>(ptr[f] + o);
                    reg[f][h] = v[0];
                    reg[f][h + 1] = v[1];
                }
            }
        } else {
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const bool ok = k + KS * s < (uint32_t)p.K;
                const int64_t o = !ok ? 0 : s == 0 ? it.off : step ? it.off + KS * s * km.s2 : koff(km, k + KS * s);
#pragma unroll
                for (int f = 0; f < NF; ++f) reg[f][s] = ptr[f][o];
            }
        }
        dcc::kstep(km, it);
    };
    acc_t acc[FX][FY];
#pragma unroll
    for (int i = 0; i < FX; ++i)
#pragma unroll
        for (int j = 0; j < FY; ++j) acc[i][j] = acc_t{0, 0, 0, 0};
    T xr[2][KB][FX][4], yr[2][KB][FY][4];
    uint32_t k = W == 1 ? lk : 16 * w + 4 * lk;
    dcc::KIter xi = dcc::kiter(p.xk, k), yi = dcc::kiter(p.yk, k);
    auto stage = [&](int s) {
#pragma unroll
        for (int b = 0; b < KB; ++b) {
            load(xr[s][b], xp, p.xk, xi, k, vx, sx, std::integral_constant<int, FX>{});
            load(yr[s][b], yp, p.yk, yi, k, vy, sy, std::integral_constant<int, FY>{});
            k += 16 * W;
        }
    };
    // block 0 of the stage is the wave's block kb of 16 * W k values
    auto mul = [&](int s, int kb) {
#pragma unroll
        for (int b = 0; b < KB; ++b) {
            const uint32_t first = 16u * (uint32_t)(w + W * (kb + b));   // of this block
            if (first + 16 > (uint32_t)p.K) {   // uniform
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const bool ok = first + (uint32_t)(W == 1 ? lk + 4 * e : 4 * lk + e) < (uint32_t)p.K;
#pragma unroll
                    for (int i = 0; i < FX; ++i) xr[s][b][i][e] = ok ? xr[s][b][i][e] : T(0);
#pragma unroll
                    for (int j = 0; j < FY; ++j) yr[s][b][j][e] = ok ? yr[s][b][j][e] : T(0);
                }
            }
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int i = 0; i < FX; ++i)
#pragma unroll
                    for (int j = 0; j < FY; ++j) acc[i][j] = MF::step(xr[s][b][i][e], yr[s][b][j][e], acc[i][j]);
        }
    };
    const int nblk = (p.K + 15) / 16;
    const int mine = nblk > w ? (nblk - w + W - 1) / W : 0;   // blocks of this wave
    if (mine > 0) {
        stage(0);
        for (int b = 0; b < mine; b += 2 * KB) {
            stage(1);
            mul(0, b);
            stage(0);
            mul(1, b + KB);
        }
    }
    // partial tiles: [wave][fragment][r][lane]
#pragma unroll
    for (int i = 0; i < FX; ++i)
#pragma unroll
        for (int j = 0; j < FY; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) smem[((w * FX * FY + i * FY + j) * 4 + r) * 64 + lane] = acc[i][j][r];
    __syncthreads();
#pragma unroll
    for (int n = 0; n < NE; ++n) {
        if (c[n] == nullptr) continue;
        const int e = tid + n * W * 64;
        T sum = smem[e];
#pragma unroll
        for (int q = 1; q < W; ++q) sum += smem[q * FX * FY * 256 + e];
        double v = p.alpha * (double)sum;
        if (p.beta != 0.0) v += p.beta * (double)old[n];
        *c[n] = (T)v;
    }
}

// Whether the k of a lane's group stay in the innermost level of the map.
inline bool k_groups_step(const dcc_idxmap &k, int64_t K, int w) {
    return k.e2 % (w == 1 ? 16 : 4) == 0 || k.e2 >= K;
}

// Whether k, k + 1 from an even k are adjacent in memory and aligned as a pair in every row.
inline bool k_pairs(const void *base, const dcc_idxmap &rows, const dcc_idxmap &k, int64_t K, size_t esize) {
    if (reinterpret_cast<uintptr_t>(base) % (2 * esize) != 0 || rows.table != nullptr || K % 2 != 0) return false;
    if (k.s2 != 1 || (k.e2 < K && (k.e2 % 2 != 0 || k.s0 % 2 != 0 || k.s1 % 2 != 0))) return false;
    return rows.s0 % 2 == 0 && rows.s1 % 2 == 0 && rows.s2 % 2 == 0;
}

inline int skinny_flags(const void *X, const dcc_idxmap &xm, const dcc_idxmap &xk, const void *Y, const dcc_idxmap &ym,
                        const dcc_idxmap &yk, int64_t K, bool swap, size_t esize, int w) {
    return (swap ? kSkinnySwap : 0) | (k_groups_step(xk, K, w) ? kSkinnyStepX : 0) |
           (k_groups_step(yk, K, w) ? kSkinnyStepY : 0) | (k_pairs(X, xm, xk, K, esize) ? kSkinnyPairX : 0) |
           (k_pairs(Y, ym, yk, K, esize) ? kSkinnyPairY : 0);
}

constexpr int64_t kSkinnyBase = 64;   // numbers of tiles: shapes below, skinny variants from here

// The variants: fragments of X and Y per tile and waves that split K.
struct SkinnyVariant {
    int fx, fy, w;
};
constexpr int kSkinnyVariants = 10;
constexpr SkinnyVariant kSkinny[kSkinnyVariants] = {{1, 1, 4}, {1, 1, 8}, {1, 1, 16}, {1, 2, 4}, {2, 1, 4},
                                                    {1, 4, 2}, {1, 4, 4}, {4, 1, 2},  {4, 1, 4}, {1, 1, 1}};

// Sizes of a launch (one problem, or the sums over a group of them), for the choice of a variant.
struct SkinnySize {
    int64_t t64 = 0, t16 = 0;        // tiles of 64 x 64 and of 16 x 16
    int64_t rx = 0, ry = 0, K = 0;   // longest row and column extents and K
    void add(int64_t x, int64_t y, int64_t k, int64_t nbatch) {
        t64 += nbatch * ((x + 63) / 64) * ((y + 63) / 64);
        t16 += nbatch * ((x + 15) / 16) * ((y + 15) / 16);
        rx = x > rx ? x : rx;
        ry = y > ry ? y : ry;
        K = k > K ? k : K;
    }
};

// Variant of a launch, or -1 where the 64 x 64 .. 128 x 128 tiles are the better ones.  Measured in FP64:
//   * one side of at most 16 against a long one (at least 64): the tile is 64 long on that side, so the wide
//     operand is read once at 16 products per element (t3 -> r1 at nocc=10, nvir=90 1.22 ms against 2.89,
//     t3 -> r2 E_ooov 1.10 against 2.07); two waves per tile for a short K.
//   * at most half a 64 x 64 tile per CU: 16 x 16 tiles with the more waves the longer K and the fewer tiles
//     (5 x 5 x 1805: 24 us against 164; 240 x 240 x 240: 11 us against 32; 36 x 36 x 1600: 20 against 106),
//     16 x 32 tiles from 512 16 x 16 tiles on (1600 x 240 x 240: 17 us against 32).
//   * K up to 64 there: one wave per 16 x 16 tile (240 x 240 x 36: 10 us against 23).
//   * above that the staged tiles win (900 x 900 x 900, 225 tiles: 73 us against 80).
// `only`: a variant in any case (groups of many small problems).
inline int skinny_variant(const SkinnySize &z, bool only = false) {
    const int64_t lo = z.rx < z.ry ? z.rx : z.ry, hi = z.rx < z.ry ? z.ry : z.rx;
    if (lo <= 16 && hi >= 64 && z.K > 64 && (z.t64 > 64 || z.t16 > 512))
        return (z.ry >= z.rx ? 5 : 7) + (z.K > 128 ? 1 : 0);
    if (z.t64 > 128 && !only) return -1;
    if (z.K <= 64) return 9;
    if (z.t16 > 512) return z.ry >= z.rx ? 3 : 4;
    if (z.t16 > 128) return z.K >= 384 ? 1 : 0;
    return z.K >= 768 ? 2 : z.K >= 384 ? 1 : 0;
}

// f(std::integral_constant<int, FX>, <FY>, <W>) of variant v.
template <typename F> int skinny_dispatch(int v, F &&f) {
    using std::integral_constant;
    typedef integral_constant<int, 1> I1;
    typedef integral_constant<int, 2> I2;
    typedef integral_constant<int, 4> I4;
    switch (v) {
        case 0: return f(I1{}, I1{}, I4{});
        case 1: return f(I1{}, I1{}, integral_constant<int, 8>{});
        case 2: return f(I1{}, I1{}, integral_constant<int, 16>{});
        case 3: return f(I1{}, I2{}, I4{});
        case 4: return f(I2{}, I1{}, I4{});
        case 5: return f(I1{}, I4{}, I2{});
        case 6: return f(I1{}, I4{}, I4{});
        case 7: return f(I4{}, I1{}, I2{});
        case 8: return f(I4{}, I1{}, I4{});
        default: return f(I1{}, I1{}, I1{});
    }
}

}  // namespace dcc_gemm
