// cullst stages on the GPU (Cullst/cullSTData.c, cullStats.c,
// cullSmooth.c, cullIslands.c).
//
// cullSTData culls in place in raster order, so a cell's decision sees the
// decisions already taken for earlier cells of the same pass.  The GPU
// solves that recurrence exactly as a fixpoint: every iteration re-decides
// all cells in parallel, earlier cells taking their decision from the
// previous iteration; the sequential result is the unique fixpoint and is
// reached when an iteration changes nothing (a dependency chain of length
// k is settled after k iterations).  A single-workgroup wavefront kernel
// (cell (i, j) runs at step i*(bR/2+1) + j) finishes the pass if the
// fixpoint has not settled after kMaxIter iterations.
#include <math.h>
#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <mutex>
#include <string>
#include <vector>

#include "st_ctx.h"

// The cull arithmetic mirrors the reference operation by operation; no FMA
// contraction anywhere in this file.
#pragma clang fp contract(off)

namespace {

constexpr float kNoData = -2.0e9f;
constexpr int kMaxIter = 48;
constexpr int kCullCount = 8, kCullSlots = 8;  // words of CullDev::counters that count the culled cells
constexpr int kAhead = 3;  // fixpoint iterations launched before their change counts are read
// Box sides of the median test (k_cull_iter's tile with its halo: 67 KB of LDS
// at 45).
constexpr int kMaxBox = 45;

__device__ inline bool valid2(float r, float a)
{
    return r > (float)(1 - ST_LARGEINT) && a > (float)(1 - ST_LARGEINT);
}

struct CullDev {
    int nR, nA;
    float *offR, *offA, *corr;
    uint8_t *type;
    const uint8_t *mask;
    float *offRS, *offAS, *sigmaR, *sigmaA;
    float *R0, *A0;       // state at the start of a cullSTData pass
    uint8_t *cPrev, *cNew; // cull decisions of the pass
    int *counters;        // [2] max root, [3] good cells, [4] cells with data, [5 ..] changes per iteration, [8 ..] culled cells
    int *parent, *root, *bbox;   // islands
};

// Pre-pass of cullSTData (cullSTData.c:34-68).
__global__ void k_cull_prepass(CullDev D, float corrThresh, int singleMT)
{
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= D.nR * D.nA)
        return;
    if (D.corr[c] < corrThresh) {
        D.offR[c] = kNoData;
        D.offA[c] = kNoData;
        D.type[c] = 0;
    }
    if (D.mask) {
        const unsigned char mv = (unsigned char)D.mask[c] & 4;
        if (mv > 0 && D.type[c] > 2) {
            D.offR[c] = kNoData;
            D.offA[c] = kNoData;
            D.type[c] = 0;
        }
        if (singleMT > 0 && D.type[c] != singleMT) {
            D.offR[c] = kNoData;
            D.offA[c] = kNoData;
            D.type[c] = 0;
        }
    }
    D.R0[c] = D.offR[c];
    D.A0[c] = D.offA[c];
    D.cPrev[c] = 0;
}

// Start of a cullLSData pass (cullLSData.c:37-58): the pass state, and the
// counts of good cells ([3]) and cells with data ([4]).
__global__ void k_cull_ls_begin(CullDev D, const uint8_t *type, uint8_t noDataToUse)
{
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    const bool in = c < D.nR * D.nA;
    bool good = false, data = false;
    if (in) {
        D.R0[c] = D.offR[c];
        D.A0[c] = D.offA[c];
        D.cPrev[c] = 0;
        good = valid2(D.offR[c], D.offA[c]);
        data = (type[c] & noDataToUse) == 0;
    }
    const unsigned long long g = __ballot(good), d = __ballot(data);
    if ((threadIdx.x & 63) == 0) {
        if (g)
            atomicAdd(&D.counters[3], __popcll(g));
        if (d)
            atomicAdd(&D.counters[4], __popcll(d));
    }
}

// Landsat variant of the median test (cullLSData.c:66-121): the box's
// good points all carrying the slow-velocity bit switch the limits to
// 40 m/yr over deltaT in pixels (at least 0.2), and a cell whose Y is not
// above NODATA + 1 is culled.
struct LsArg {
    const uint8_t *type;
    uint8_t slow;
    double noData1;  // NODATA + 1
    double deltaT, dx, dy;
};

// Largest float not above m: d > m exactly when d > float_floor(m), for float d.
__device__ inline float float_floor(double m)
{
    const float f = (float)m;
    return (double)f > m ? nextafterf(f, -INFINITY) : f;
}

// The median test of cullSTData.c:73-122 without the median.  With n box
// values the reference takes the k-th smallest m (k = n / 2, at least 1) and
// culls the cell x when fl(x - m) leaves [-max, max].  fl(x - u) does not rise
// with u, so the values u with fl(x - u) > max are the smallest ones: m is
// among them exactly when there are at least k; and those with fl(x - u) <
// -max are the largest: m is among them when there are at least n - k + 1.
// Counting replaces the selection, and ties, infinities and a NaN x decide as
// there (a comparison with NaN is false).
struct MedianCount {
    int n = 0, loR = 0, hiR = 0, loA = 0, hiA = 0;

    // v: a box value pair, NaN when it takes no part
    __device__ inline void add(float xR, float xA, float2 v, float maxR, float maxA)
    {
        const float dR = xR - v.x, dA = xA - v.y;
        n += v.x == v.x;
        loR += dR > maxR;
        hiR += dR < -maxR;
        loA += dA > maxA;
        hiA += dA < -maxA;
    }
    __device__ inline bool off() const
    {
        const int k = n / 2 > 0 ? n / 2 : 1, m = n - k + 1;
        return loR >= k || hiR >= m || loA >= k || hiA >= m;
    }
};

// The slow-velocity limits of the Landsat variant, range then azimuth.
__device__ inline float2 ls_slow_limits(const LsArg &L)
{
    const double m = 40.0 / 365. * L.deltaT;
    double mX = m, mY = m;
    mX /= L.dx;
    mY /= L.dy;
    mX = mX > 0.2 ? mX : 0.2;
    mY = mY > 0.2 ? mY : 0.2;
    return make_float2(float_floor(mX), float_floor(mY));
}

// The pair (r, a) of cell q, NaN when invalid or already culled.
__device__ inline float2 box_value(const CullDev &D, int q, bool culled)
{
    const float r = D.R0[q], a = D.A0[q];
    const float nan = __int_as_float(0x7fc00000);
    return !culled && valid2(r, a) ? make_float2(r, a) : make_float2(nan, nan);
}

__device__ inline int wave_sum(int v)
{
    for (int o = 32; o > 0; o >>= 1)
        v += __shfl_xor(v, o);
    return v;
}

// Median test of one cell by one wavefront, lanes over the box; LS selects
// the Landsat limits (cullLSData.c); maxA / maxR are then maxY / maxX.
template <bool LS>
__device__ inline bool cull_decide(const CullDev &D, int c, int bR, int bA, int nGood, float maxA, float maxR,
                                   const uint8_t *earlier, const LsArg &L)
{
    const int lane = threadIdx.x & 63;
    const int i = c / D.nR, j = c - (c / D.nR) * D.nR;
    const int i1 = imax(0, i - bA / 2), i2 = imin(D.nA - 1, i + bA / 2);
    const int j1 = imax(0, j - bR / 2), j2 = imin(D.nR - 1, j + bR / 2);
    const int bw = j2 - j1 + 1, cnt = bw * (i2 - i1 + 1);
    auto value = [&](int s, int &q) {
        q = (i1 + s / bw) * D.nR + j1 + s % bw;
        return box_value(D, q, q < c && earlier[q]);
    };
    if constexpr (LS) {
        bool fast = false;
        for (int s = lane; s < cnt; s += 64) {
            int q;
            const float2 v = value(s, q);
            fast |= v.x == v.x && !(L.type[q] & L.slow);
        }
        if (!__ballot(fast)) {
            const float2 m = ls_slow_limits(L);
            maxR = m.x;
            maxA = m.y;
        }
    }
    const float xR = D.R0[c], xA = D.A0[c];
    MedianCount M;
    for (int s = lane; s < cnt; s += 64) {
        int q;
        M.add(xR, xA, value(s, q), maxR, maxA);
    }
    M.n = wave_sum(M.n);
    M.loR = wave_sum(M.loR);
    M.hiR = wave_sum(M.hiR);
    M.loA = wave_sum(M.loA);
    M.hiA = wave_sum(M.hiA);
    if (M.n <= nGood)
        return true;
    if constexpr (LS) {
        if (!((double)xA > L.noData1))
            return true;
    }
    return M.off();
}

// One fixpoint iteration, a thread per cell: the tile of box values with its
// halo in LDS twice, as they stand (E: culled cells of the previous iteration
// out) and before any cull (N); a cell reads E for the cells before it in
// raster order and N from itself on.  Bound: VALU, about 12 instructions per
// box value (box 9 on 821 x 571 cells: 45 us per iteration; 1.13 ms with one
// wave per cell ranking the box by counting).
constexpr int kTileR = 32, kTileA = 8;  // 256 threads
constexpr size_t cull_tile_bytes(int bR, int bA, bool ls)
{
    return (size_t)(kTileR + bR / 2 * 2) * (kTileA + bA / 2 * 2) * (2 * sizeof(float2) + (ls ? 1 : 0));
}
template <bool LS>
__global__ void __launch_bounds__(256) k_cull_iter(CullDev D, int bR, int bA, int nGood, float maxA, float maxR,
                                                   LsArg L, int slot)
{
    extern __shared__ float2 cull_lds[];
    const int hR = bR / 2, hA = bA / 2, tw = kTileR + 2 * hR, cells = tw * (kTileA + 2 * hA);
    float2 *E = cull_lds, *N = cull_lds + cells;
    uint8_t *fastB = (uint8_t *)(cull_lds + 2 * cells);
    const int nbx = (D.nR + kTileR - 1) / kTileR, t = threadIdx.x;
    const int i0 = (int)blockIdx.x / nbx * kTileA, j0 = (int)blockIdx.x % nbx * kTileR;
    for (int e = t; e < cells; e += 256) {
        const int ii = i0 - hA + e / tw, jj = j0 - hR + e % tw;
        const float nan = __int_as_float(0x7fc00000);
        float2 n = make_float2(nan, nan), v = n;
        bool fast = false;
        if (ii >= 0 && ii < D.nA && jj >= 0 && jj < D.nR) {
            const int q = ii * D.nR + jj;
            n = box_value(D, q, false);
            v = D.cPrev[q] ? v : n;
            if constexpr (LS)
                fast = !(L.type[q] & L.slow);
        }
        N[e] = n;
        E[e] = v;
        if constexpr (LS)
            fastB[e] = fast;
    }
    __syncthreads();
    const int ti = t / kTileR, tj = t % kTileR, i = i0 + ti, j = j0 + tj;
    bool changed = false;
    if (i < D.nA && j < D.nR) {
        const int c = i * D.nR + j, bw = 2 * hR + 1, at = ti * tw + tj;
        if constexpr (LS) {
            bool fast = false;
            for (int a = 0; a <= 2 * hA; a++)
                for (int r = 0; r < bw; r++) {
                    const int e = at + a * tw + r;
                    const float x = (a < hA || (a == hA && r < hR) ? E[e] : N[e]).x;
                    fast |= x == x && fastB[e];
                }
            if (!fast) {
                const float2 m = ls_slow_limits(L);
                maxR = m.x;
                maxA = m.y;
            }
        }
        const float xR = D.R0[c], xA = D.A0[c];
        MedianCount M;
        for (int a = 0; a < hA; a++)
#pragma unroll 3
            for (int r = 0; r < bw; r++)
                M.add(xR, xA, E[at + a * tw + r], maxR, maxA);
        for (int r = 0; r < hR; r++)
            M.add(xR, xA, E[at + hA * tw + r], maxR, maxA);
        for (int r = hR; r < bw; r++)
            M.add(xR, xA, N[at + hA * tw + r], maxR, maxA);
        for (int a = hA + 1; a <= 2 * hA; a++)
#pragma unroll 3
            for (int r = 0; r < bw; r++)
                M.add(xR, xA, N[at + a * tw + r], maxR, maxA);
        bool cull = M.n <= nGood || M.off();
        if constexpr (LS)
            cull = cull || !((double)xA > L.noData1);
        D.cNew[c] = cull ? 1 : 0;
        changed = (D.cPrev[c] != 0) != cull;
    }
    const unsigned long long m = __ballot(changed);
    if (m && (t & 63) == 0)
        atomicAdd(&D.counters[slot], __popcll(m));
}

// Exact sequential order for the leftover case: one workgroup sweeps the
// wavefront steps, one wave per cell of a step.
template <bool LS>
__global__ void __launch_bounds__(1024) k_cull_wavefront(CullDev D, int bR, int bA, int nGood, float maxA, float maxR,
                                                         LsArg L)
{
    const int w = threadIdx.x >> 6, nw = blockDim.x >> 6;
    const int s = bR / 2 + 1;
    const int steps = (D.nA - 1) * s + D.nR;
    for (int T = 0; T < steps; T++) {
        // cells with i*s + j == T
        const int iLo = imax(0, (T - (D.nR - 1) + s - 1) / s), iHi = imin(D.nA - 1, T / s);
        for (int i = iLo + w; i <= iHi; i += nw) {
            const int j = T - i * s;
            const int c = i * D.nR + j;
            const bool cull = cull_decide<LS>(D, c, bR, bA, nGood, maxA, maxR, D.cNew, L);
            if ((threadIdx.x & 63) == 0)
                D.cNew[c] = cull ? 1 : 0;
        }
        __syncthreads();
    }
}

__global__ void k_cull_apply(CullDev D)
{
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    const bool in = c < D.nR * D.nA, cull = in && D.cNew[c];
    if (in) {
        D.offR[c] = cull ? kNoData : D.R0[c];
        D.offA[c] = cull ? kNoData : D.A0[c];
    }
    const unsigned long long m = __ballot(cull);
    __shared__ int part[4];
    if ((threadIdx.x & 63) == 0)
        part[threadIdx.x >> 6] = __popcll(m);
    __syncthreads();
    // spread over kCullSlots words: one word takes some 12 ns per atomic, and
    // a whole scene has thousands of workgroups
    if (threadIdx.x == 0) {
        const int k = part[0] + part[1] + part[2] + part[3];
        if (k)
            atomicAdd(&D.counters[kCullCount + blockIdx.x % kCullSlots], k);
    }
}

// The plane fit of cullStats: least squares y ~ A x over the box's n good
// points, A's rows (c0, ii, jj), singular values below 1e-5 of the largest
// dropped (svdfit's rule).  A = B T with B's rows (1, di, dj), di = ii - i and
// dj = jj - j, and T = [c0 i j; 0 1 0; 0 0 1]; B's Gram matrix holds small
// integers, so its Cholesky factor L is exact to a rounding and A = Q (L^T T)
// with orthonormal Q: the one-sided Jacobi SVD of A's columns is that of the
// 3 x 3 matrix L^T T, and u_k . y is (L^T T v_k) . (Q^T y).  The sweeps run
// over three rows instead of the 81 of the box; they stop at column-pair
// cosines below 1e-13.
struct BoxGram {
    double l11, l21, l31, l22, l32, l33;

    __device__ inline void factor(int n, int si, int sj, int sii, int sij, int sjj)
    {
        // every numerator is an exact integer (n <= 81, |di|, |dj| <= 4)
        const double dn = (double)n;
        const double pii = (double)(n * sii - si * si), pij = (double)(n * sij - si * sj), pjj = (double)(n * sjj - sj * sj);
        l11 = sqrt(dn);
        l21 = (double)si / l11;
        l31 = (double)sj / l11;
        l22 = sqrt(pii / dn);
        l32 = pii > 0.0 ? pij / (dn * l22) : 0.0;
        l33 = pii > 0.0 ? sqrt((pii * pjj - pij * pij) / (dn * pii)) : sqrt(pjj / dn);
    }
};

// b: B^T y.
__device__ inline void lsq3(double c0, double i, double j, const BoxGram &G, const double b[3], double x[3])
{
    const double R[3][3] = {{G.l11 * c0, G.l11 * i + G.l21, G.l11 * j + G.l31}, {0.0, G.l22, G.l32}, {0.0, 0.0, G.l33}};
    const double z0 = b[0] / G.l11;
    const double z1 = G.l22 > 0.0 ? (b[1] - G.l21 * z0) / G.l22 : 0.0;
    const double z2 = G.l33 > 0.0 ? (b[2] - G.l31 * z0 - G.l32 * z1) / G.l33 : 0.0;
    double V[9] = {1, 0, 0, 0, 1, 0, 0, 0, 1};
    for (int sweep = 0; sweep < 30; sweep++) {
        double off = 0.0;
#pragma unroll
        for (int p = 0; p < 2; p++)
#pragma unroll
            for (int q = p + 1; q < 3; q++) {
                double alpha = 0, beta = 0, gamma = 0;
#pragma unroll
                for (int r = 0; r < 3; r++) {
                    const double up = R[r][0] * V[0 * 3 + p] + R[r][1] * V[1 * 3 + p] + R[r][2] * V[2 * 3 + p];
                    const double uq = R[r][0] * V[0 * 3 + q] + R[r][1] * V[1 * 3 + q] + R[r][2] * V[2 * 3 + q];
                    alpha += up * up;
                    beta += uq * uq;
                    gamma += up * uq;
                }
                if (gamma == 0.0)
                    continue;
                const double conv = fabs(gamma) / sqrt(alpha * beta);
                if (conv > off)
                    off = conv;
                if (conv < 1e-13)
                    continue;
                const double zeta = (beta - alpha) / (2.0 * gamma);
                const double t = (zeta >= 0 ? 1.0 : -1.0) / (fabs(zeta) + sqrt(1.0 + zeta * zeta));
                const double c = 1.0 / sqrt(1.0 + t * t), s = c * t;
#pragma unroll
                for (int r = 0; r < 3; r++) {
                    const double vp = V[r * 3 + p], vq = V[r * 3 + q];
                    V[r * 3 + p] = c * vp - s * vq;
                    V[r * 3 + q] = s * vp + c * vq;
                }
            }
        if (off < 1e-13)
            break;
    }
    double w2[3], uy[3], w[3], wmax = 0;
#pragma unroll
    for (int k = 0; k < 3; k++) {
        w2[k] = uy[k] = 0;
#pragma unroll
        for (int r = 0; r < 3; r++) {
            const double u = R[r][0] * V[0 * 3 + k] + R[r][1] * V[1 * 3 + k] + R[r][2] * V[2 * 3 + k];
            w2[k] += u * u;
            uy[k] += u * (r == 0 ? z0 : r == 1 ? z1 : z2);
        }
        w[k] = sqrt(w2[k]);
        if (w[k] > wmax)
            wmax = w[k];
    }
    const double thresh = 1.0e-5 * wmax;
    double coef[3];
#pragma unroll
    for (int k = 0; k < 3; k++)
        coef[k] = (w[k] < thresh || w[k] == 0.0) ? 0.0 : uy[k] / w2[k];
#pragma unroll
    for (int r = 0; r < 3; r++)
        x[r] = V[r * 3 + 0] * coef[0] + V[r * 3 + 1] * coef[1] + V[r * 3 + 2] * coef[2];
}

// cullStats (cullStats.c:19-144), a thread per cell, the 9 x 9 boxes from an
// LDS tile.  Bound: FP64 VALU (two passes over 81 box values and the 3 x 3
// sweeps).  addQuant: cullLSStats adds the quantisation variance `quant`
// before the square root (cullLSStats.c:144-146).
__global__ void __launch_bounds__(256) k_cull_stats(CullDev D, int addQuant, double quant)
{
    constexpr int b = 9, h = b / 2, tw = kTileR + 2 * h, cells = tw * (kTileA + 2 * h);
    __shared__ float2 tile[cells];  // NaN: no good value
    const int nbx = (D.nR + kTileR - 1) / kTileR, t = threadIdx.x;
    const int i0 = (int)blockIdx.x / nbx * kTileA, j0 = (int)blockIdx.x % nbx * kTileR;
    for (int e = t; e < cells; e += 256) {
        const int ii = i0 - h + e / tw, jj = j0 - h + e % tw;
        const float nan = __int_as_float(0x7fc00000);
        float2 v = make_float2(nan, nan);
        if (ii >= 0 && ii < D.nA && jj >= 0 && jj < D.nR) {
            const int q = ii * D.nR + jj;
            const float r = D.offR[q], a = D.offA[q];
            if (valid2(r, a))
                v = make_float2(r, a);
        }
        tile[e] = v;
    }
    __syncthreads();
    const int ti = t / kTileR, tj = t % kTileR, i = i0 + ti, j = j0 + tj, at = ti * tw + tj;
    if (i >= D.nA || j >= D.nR)
        return;
    const int c = i * D.nR + j;
    int n = 0, si = 0, sj = 0, sii = 0, sij = 0, sjj = 0;
    double meanA = 0.0, meanR = 0.0, bR[3] = {0, 0, 0}, bA[3] = {0, 0, 0};
    for (int di = -h; di <= h; di++)
#pragma unroll
        for (int dj = -h; dj <= h; dj++) {
            const float2 v = tile[at + (di + h) * tw + dj + h];
            if (v.x == v.x) {
                n++;
                si += di;
                sj += dj;
                sii += di * di;
                sij += di * dj;
                sjj += dj * dj;
                meanA += v.y;
                meanR += v.x;
                bR[1] += (double)di * v.x;
                bR[2] += (double)dj * v.x;
                bA[1] += (double)di * v.y;
                bA[2] += (double)dj * v.y;
            }
        }
    if (!(n > 8 && D.offR[c] > (float)(1 - ST_LARGEINT))) {
        D.sigmaA[c] = kNoData;
        D.sigmaR[c] = kNoData;
        return;
    }
    bR[0] = meanR;
    bA[0] = meanA;
    meanA /= (double)n;
    meanR /= (double)n;
    BoxGram G;
    G.factor(n, si, sj, sii, sij, sjj);
    double aR[3], aA[3];
    lsq3((double)(float)meanR, (double)i, (double)j, G, bR, aR);
    lsq3((double)(float)meanA, (double)i, (double)j, G, bA, aA);
    aR[0] *= meanR;
    aA[0] *= meanA;
    double mA = 0.0, mR = 0.0, varR = 0.0, varA = 0.0;
    for (int di = -h; di <= h; di++)
#pragma unroll
        for (int dj = -h; dj <= h; dj++) {
            const float2 v = tile[at + (di + h) * tw + dj + h];
            if (v.x == v.x) {
                const float ii = (float)(i + di), jj = (float)(j + dj);
                const float oR = (float)(v.x - (aR[0] + aR[1] * ii + aR[2] * jj));
                const float oA = (float)(v.y - (aA[0] + aA[1] * ii + aA[2] * jj));
                mA += oA;
                mR += oR;
                varA += oA * oA;
                varR += oR * oR;
            }
        }
    float sA = (float)(varA / (float)(n - 3));
    float sR = (float)(varR / (float)(n - 3));
    sA = (float)(sA - mA * mA / (float)((n - 3) * n));
    sR = (float)(sR - mR * mR / (float)((n - 3) * n));
    sA = (float)(0.00001 > sA ? 0.00001 : sA);
    sR = (float)(0.00001 > sR ? 0.00001 : sR);
    if (addQuant) {
        sR = (float)(sR + quant);
        sA = (float)(sA + quant);
    }
    D.sigmaA[c] = (float)sqrt((double)sA);
    D.sigmaR[c] = (float)sqrt((double)sR);
}

// cullSmooth (cullSmooth.c:29-103)
__device__ inline float s_weight(int m, int s)
{
    const float w2 = (float)((double)s / 2.0 - 0.01);
    return (m < -w2 || m > w2) ? 0.5f : 1.0f;
}

__global__ void k_cull_smooth(CullDev D, int sR, int sA)
{
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= D.nR * D.nA)
        return;
    const float nlooks[4] = {0.0f, 1.0f, 0.25f, 0.015f};
    const int i = c / D.nR, j = c - (c / D.nR) * D.nR;
    const int i1 = imax(0, i - sA / 2), i2 = imin(D.nA - 1, i + sA / 2);
    const int j1 = imax(0, j - sR / 2), j2 = imin(D.nR - 1, j + sR / 2);
    double ngood = 0, meanA = 0.0, meanR = 0.0;
    float nLooksEff = 0.0f;
    for (int ii = i1; ii <= i2; ii++)
        for (int jj = j1; jj <= j2; jj++) {
            const int o = ii * D.nR + jj;
            if (valid2(D.offR[o], D.offA[o])) {
                const double w = (double)(s_weight(ii - i, sA) * s_weight(jj - j, sR));
                ngood += w;
                nLooksEff = (float)(nLooksEff + w * nlooks[(int)D.type[o] & 3]);
                meanA += w * D.offA[o];
                meanR += w * D.offR[o];
            }
        }
    if (((ngood > 1) || (sA == 1) || (sR == 1)) && D.offR[c] > (float)(1 - ST_LARGEINT) &&
        D.sigmaA[c] > (float)(1 - ST_LARGEINT)) {
        nLooksEff = (float)(nLooksEff > 1. ? nLooksEff : 1.);
        D.sigmaA[c] = (float)(D.sigmaA[c] / sqrt((double)nLooksEff));
        D.sigmaR[c] = (float)(D.sigmaR[c] / sqrt((double)nLooksEff));
        D.offRS[c] = (float)(meanR / (float)ngood);
        D.offAS[c] = (float)(meanA / (float)ngood);
    } else {
        D.offRS[c] = kNoData;
        D.offAS[c] = kNoData;
    }
}

// cullLSSmooth (cullLSSmooth.c:11-73): unweighted box mean, effective
// looks = the count of good cells.
__global__ void k_cull_ls_smooth(CullDev D, int sX, int sY)
{
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= D.nR * D.nA)
        return;
    const int i = c / D.nR, j = c - (c / D.nR) * D.nR;
    const int i1 = imax(0, i - sY / 2), i2 = imin(D.nA - 1, i + sY / 2);
    const int j1 = imax(0, j - sX / 2), j2 = imin(D.nR - 1, j + sX / 2);
    unsigned ngood = 0;
    float nLooksEff = 0.0f;
    double meanY = 0.0, meanX = 0.0;
    for (int ii = i1; ii <= i2; ii++)
        for (int jj = j1; jj <= j2; jj++) {
            const int o = ii * D.nR + jj;
            if (valid2(D.offR[o], D.offA[o])) {
                ngood++;
                nLooksEff++;
                meanY += D.offA[o];
                meanX += D.offR[o];
            }
        }
    if (((ngood > 1) || (sY == 1) || (sX == 1)) && D.offR[c] > (float)(1 - ST_LARGEINT) &&
        D.sigmaA[c] > (float)(1 - ST_LARGEINT)) {
        nLooksEff = (float)(nLooksEff > 1. ? nLooksEff : 1.);
        D.sigmaA[c] = (float)(D.sigmaA[c] / sqrt((double)nLooksEff));
        D.sigmaR[c] = (float)(D.sigmaR[c] / sqrt((double)nLooksEff));
        D.offRS[c] = (float)(meanX / (float)ngood);
        D.offAS[c] = (float)(meanY / (float)ngood);
    } else {
        D.offRS[c] = kNoData;
        D.offAS[c] = kNoData;
    }
}

// cullIslands (cullIslands.c:13-198): 4-connected components of valid
// smoothed cells by atomic union-find.  Roots are the smallest member
// index, i.e. the component's first cell in raster order, which is the
// order a raster-scan labeller numbers components in; the component with
// the largest root therefore carries the last label, which the reference
// leaves alone (the loops stop at maxLabel - 1).
__device__ inline bool isl_valid(const CullDev &D, int c) { return D.offRS[c] >= (float)(-ST_LARGEINT + 1000); }

// Parent links only ever point to a smaller index, so every value a thread
// reads for par[x] is an ancestor of x, and path halving (par[x] = par[par[x]])
// may race with other finds and with the linking CAS without breaking a tree:
// it writes only to nodes that are no longer roots.  Loads and stores are
// agent-scope atomics so a retried find sees links made by other waves.
__device__ inline int uf_ld(const int *par, int x) { return __hip_atomic_load(par + x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }

__device__ inline int uf_find(int *par, int x)
{
    while (true) {
        const int p = uf_ld(par, x);
        if (p == x)
            return x;
        const int g = uf_ld(par, p);
        if (g == p)
            return p;
        __hip_atomic_store(par + x, g, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        x = g;
    }
}

__device__ inline void uf_unite(int *par, int a, int b)
{
    while (true) {
        a = uf_find(par, a);
        b = uf_find(par, b);
        if (a == b)
            return;
        if (a < b) {
            const int t = a;
            a = b;
            b = t;
        }
        if (atomicCAS(&par[a], a, b) == a)
            return;
    }
}

// Each valid cell starts linked to the first cell of its row run (within the
// 64 cells of its wave; a run that comes in from the wave before is linked on
// at the wave's first cell), and a run's first cell to the one above it when
// that is valid.
__global__ void k_isl_init(CullDev D)
{
    const int c = blockIdx.x * blockDim.x + threadIdx.x, lane = threadIdx.x & 63;
    const bool in = c < D.nR * D.nA, v = in && isl_valid(D, c);
    const bool start = v && !(c % D.nR > 0 && isl_valid(D, c - 1));
    const unsigned long long m = __ballot(start) & ((2ull << lane) - 1ull);
    if (!in)
        return;
    int p = c;
    if (start) {
        if (c >= D.nR && isl_valid(D, c - D.nR))
            p = c - D.nR;
    } else if (v) {
        p = m ? c - lane + 63 - __clzll((long long)m) : lane ? c - lane : c - 1;
    }
    D.parent[c] = p;
}

// The edges the initial links leave out: up, from a cell that is not the
// first of its run; and of those only where the run above begins, or the cell
// to the left would have made the same join.
__global__ void k_isl_merge(CullDev D)
{
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= D.nR * D.nA || c < D.nR || !isl_valid(D, c))
        return;
    const int j = c % D.nR;
    if (j > 0 && isl_valid(D, c - 1) && isl_valid(D, c - D.nR) && !isl_valid(D, c - D.nR - 1))
        uf_unite(D.parent, c, c - D.nR);
}

// Roots and bounding boxes.  Most cells of a wave share a root (one large
// component covers most of a grid), so the min/max are first reduced over
// the lanes with the same root and one lane per root issues the atomics.
__global__ void k_isl_bbox(CullDev D)
{
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    const bool v = c < D.nR * D.nA && isl_valid(D, c);
    int r = -1, i = 0, j = 0;
    if (v) {
        r = uf_find(D.parent, c);
        D.root[c] = r;
        i = c / D.nR;
        j = c - i * D.nR;
    }
    int rmax = r;
    for (int o = 32; o > 0; o >>= 1)
        rmax = max(rmax, __shfl_xor(rmax, o));
    const int lane = threadIdx.x & 63;
    // (atomics only where they would change the value: every wave of the large
    // component meets the same five words)
    if (lane == 0 && rmax > uf_ld(D.counters, 2))
        atomicMax(&D.counters[2], rmax);
    unsigned long long pending = __ballot(v);
    while (pending) {
        const int leader = __ffsll((long long)pending) - 1;
        const int rl = __shfl(r, leader);
        const bool mine = v && r == rl;
        int jmin = mine ? j : 0x7fffffff, jmax = mine ? j : -0x7fffffff;
        int imin = mine ? i : 0x7fffffff, imax = mine ? i : -0x7fffffff;
        for (int o = 32; o > 0; o >>= 1) {
            jmin = min(jmin, __shfl_xor(jmin, o));
            jmax = max(jmax, __shfl_xor(jmax, o));
            imin = min(imin, __shfl_xor(imin, o));
            imax = max(imax, __shfl_xor(imax, o));
        }
        if (lane == leader) {
            if (jmin < uf_ld(D.bbox, 4 * rl + 0))
                atomicMin(&D.bbox[4 * rl + 0], jmin);
            if (jmax > uf_ld(D.bbox, 4 * rl + 1))
                atomicMax(&D.bbox[4 * rl + 1], jmax);
            if (imin < uf_ld(D.bbox, 4 * rl + 2))
                atomicMin(&D.bbox[4 * rl + 2], imin);
            if (imax > uf_ld(D.bbox, 4 * rl + 3))
                atomicMax(&D.bbox[4 * rl + 3], imax);
        }
        pending &= ~__ballot(mine);
    }
}

__global__ void k_isl_bbox_init(CullDev D)
{
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= D.nR * D.nA)
        return;
    D.bbox[4 * c + 0] = 0x7fffffff;
    D.bbox[4 * c + 1] = -0x7fffffff;
    D.bbox[4 * c + 2] = 0x7fffffff;
    D.bbox[4 * c + 3] = -0x7fffffff;
}

__global__ void k_isl_remove(CullDev D, int thresh)
{
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= D.nR * D.nA || !isl_valid(D, c))
        return;
    const int r = D.root[c];
    if (r == D.counters[2])
        return;
    const int *bb = D.bbox + 4 * r;
    if ((bb[1] - bb[0]) <= thresh && (bb[3] - bb[2]) <= thresh) {
        D.offRS[c] = kNoData;
        if (D.offAS)
            D.offAS[c] = kNoData;
    }
}

inline unsigned nb(int n) { return (unsigned)((n + 255) / 256); }

// Fixpoint iterations before the wavefront kernel takes over;
// SPECKLE_AMD_CULL_ITERS lowers it (0 runs every pass on the wavefront
// kernel), which the tests use to cover both schedules.
int max_iterations()
{
    const char *e = getenv("SPECKLE_AMD_CULL_ITERS");
    if (!e || !*e)
        return kMaxIter;
    const int v = atoi(e);
    return v < 0 ? 0 : (v > kMaxIter ? kMaxIter : v);
}

struct CullRun {
    st_ctx *ctx;
    st_cull_params *cp;
    CullDev D{};
    int n;
    Arena *ar = nullptr;  // where the grids are carved from
    Arena fixedBuf;       // a caller-given buffer (the no-allocation entry point)

    CullRun(st_ctx *c, st_cull_params *p) : ctx(c), cp(p)
    {
        ST_REQUIRE(cp && cp->nR > 0 && cp->nA > 0 && cp->offR && cp->offA, ST_ERR_ARG, "cull grids");
        n = cp->nR * cp->nA;
        ctx->arena_reserve(cull_device_bytes((size_t)n) + (size_t)4 * 4 * n + 4 * 256);
        ar = &ctx->arena;
        alloc(cp->nR, cp->nA);
        take_mask();
    }
    // Every grid in `bytes` of device memory at `base`: allocates nothing.
    CullRun(st_ctx *c, st_cull_params *p, void *base, size_t bytes) : ctx(c), cp(p)
    {
        ST_REQUIRE(cp && cp->nR > 0 && cp->nA > 0 && cp->offR && cp->offA, ST_ERR_ARG, "cull grids");
        n = cp->nR * cp->nA;
        fixedBuf.base = (char *)base;
        fixedBuf.cap = bytes;
        ar = &fixedBuf;
        alloc(cp->nR, cp->nA);
        take_mask();
    }
    void take_mask()
    {
        if (cp->mask) {
            uint8_t *m = ar->take<uint8_t>(n);
            put(m, cp->mask, n);
            D.mask = m;
        }
    }
    // Device copies of every grid of the stages (n x 72 bytes).
    void alloc(int nR, int nA)
    {
        D.offR = ar->take<float>(n);
        D.offA = ar->take<float>(n);
        D.corr = ar->take<float>(n);
        D.type = ar->take<uint8_t>(n);
        carve(nR, nA);
    }
    // The stage grids other than offR / offA / corr / type, after what is
    // in use.
    void carve(int nR, int nA)
    {
        Arena &a = *ar;
        D.nR = nR;
        D.nA = nA;
        D.mask = nullptr;
        D.offRS = a.take<float>(n);
        D.offAS = a.take<float>(n);
        D.sigmaR = a.take<float>(n);
        D.sigmaA = a.take<float>(n);
        D.R0 = a.take<float>(n);
        D.A0 = a.take<float>(n);
        D.cPrev = a.take<uint8_t>(n);
        D.cNew = a.take<uint8_t>(n);
        D.counters = a.take<int>(16);
        D.parent = a.take<int>(n);
        D.root = a.take<int>(n);
        D.bbox = a.take<int>(4 * (size_t)n);
    }
    CullRun(st_ctx *c, int nR, int nA) : ctx(c), cp(nullptr)
    {
        n = nR * nA;
        ctx->arena_reserve(cull_device_bytes((size_t)n) + (size_t)4 * 4 * n + 4 * 256);
        ar = &ctx->arena;
        alloc(nR, nA);
    }
    // On grids already on the device (tracking outputs): no arena reset.
    CullRun(st_ctx *c, st_cull_params *p, float *dOffR, float *dOffA, float *dCorr, uint8_t *dType)
        : ctx(c), cp(p)
    {
        ST_REQUIRE(cp && cp->nR > 0 && cp->nA > 0, ST_ERR_ARG, "cull grids");
        n = cp->nR * cp->nA;
        ar = &ctx->arena;
        D.offR = dOffR;
        D.offA = dOffA;
        D.corr = dCorr;
        D.type = dType;
        carve(cp->nR, cp->nA);
        take_mask();
    }
    template <class T>
    void put(T *d, const T *h, size_t cnt)
    {
        if (h)
            ST_HIP(hipMemcpyAsync(d, h, cnt * sizeof(T), hipMemcpyHostToDevice, ctx->stream));
    }
    template <class T>
    void get(T *h, const T *d, size_t cnt)
    {
        if (h)
            ST_HIP(hipMemcpyAsync(h, d, cnt * sizeof(T), hipMemcpyDeviceToHost, ctx->stream));
    }
    // one workgroup per kTileR x kTileA cells
    dim3 tiles() const { return dim3((unsigned)((D.nR + kTileR - 1) / kTileR) * (unsigned)((D.nA + kTileA - 1) / kTileA)); }
    int counter(int k)
    {
        int v = 0;
        ST_HIP(hipMemcpyAsync(&v, D.counters + k, sizeof(int), hipMemcpyDeviceToHost, ctx->stream));
        ST_HIP(hipStreamSynchronize(ctx->stream));
        return v;
    }

    void st_data()
    {
        hipLaunchKernelGGL(k_cull_prepass, dim3(nb(n)), dim3(256), 0, ctx->stream, D, cp->corrThresh, cp->singleMT);
        cp->nCulled = median_pass<false>(cp->bR, cp->bA, cp->nGood, cp->maxA, cp->maxR, LsArg{});
    }
    // The in-place raster-order median pass on the state left in R0 / A0:
    // fixpoint iterations, the wavefront kernel if they have not settled,
    // then the culls are applied.  Returns the number of culled cells.
    template <bool LS>
    int median_pass(int bR, int bA, int nGood, float maxA, float maxR, const LsArg &L)
    {
        ST_REQUIRE(bR >= 1 && bA >= 1 && (bR / 2) * 2 + 1 <= kMaxBox && (bA / 2) * 2 + 1 <= kMaxBox,
                   ST_ERR_UNSUPPORTED, "box sizes above 45");
        hipStream_t st = ctx->stream;
        bool settled = false;
        const int maxIter = max_iterations();
        int got[kCullCount + kCullSlots - 5];  // counters 5 ..
        // kAhead iterations and the culls applied per look at the change counts:
        // a pass settles in two or three, iterations after that change nothing,
        // and applying is repeated if it had not settled
        for (int it = 0; !settled;) {
            const int ahead = std::min(kAhead, maxIter - it);
            ST_HIP(hipMemsetAsync(D.counters + 5, 0, sizeof(got), st));
            for (int k = 0; k < ahead; k++, it++) {
                hipLaunchKernelGGL(k_cull_iter<LS>, tiles(), dim3(256), cull_tile_bytes(bR, bA, LS), st, D, bR, bA, nGood,
                                   maxA, maxR, L, 5 + k);
                std::swap(D.cPrev, D.cNew);
            }
            std::swap(D.cPrev, D.cNew);  // cNew holds the last decisions
            if (ahead <= 0) {
                hipLaunchKernelGGL(k_cull_wavefront<LS>, dim3(1), dim3(1024), 0, st, D, bR, bA, nGood, maxA, maxR, L);
                settled = true;
            }
            hipLaunchKernelGGL(k_cull_apply, dim3(nb(n)), dim3(256), 0, st, D);
            ST_HIP(hipGetLastError());
            ST_HIP(hipMemcpyAsync(got, D.counters + 5, sizeof(got), hipMemcpyDeviceToHost, st));
            ST_HIP(hipStreamSynchronize(st));
            for (int k = 0; k < ahead; k++)
                settled = settled || got[k] == 0;
            if (!settled)
                std::swap(D.cPrev, D.cNew);
        }
        int culled = 0;
        for (int k = 0; k < kCullSlots; k++)
            culled += got[kCullCount - 5 + k];
        return culled;
    }
    void stats()
    {
        cp->bR = cp->bA = 9;  // cullStats.c:38-39
        hipLaunchKernelGGL(k_cull_stats, tiles(), dim3(256), 0, ctx->stream, D, 0, 0.0);
        ST_HIP(hipGetLastError());
    }
    void smooth()
    {
        ST_REQUIRE(cp->sR >= 1 && cp->sA >= 1, ST_ERR_ARG, "smoothing window");
        hipLaunchKernelGGL(k_cull_smooth, dim3(nb(n)), dim3(256), 0, ctx->stream, D, cp->sR, cp->sA);
        ST_HIP(hipGetLastError());
    }
    void islands() { islands_t(cp->islandThresh); }
    void islands_t(int thresh)
    {
        hipStream_t st = ctx->stream;
        ST_HIP(hipMemsetAsync(D.counters + 2, 0xff, sizeof(int), st));  // max root = -1
        hipLaunchKernelGGL(k_isl_init, dim3(nb(n)), dim3(256), 0, st, D);
        hipLaunchKernelGGL(k_isl_bbox_init, dim3(nb(n)), dim3(256), 0, st, D);
        hipLaunchKernelGGL(k_isl_merge, dim3(nb(n)), dim3(256), 0, st, D);
        hipLaunchKernelGGL(k_isl_bbox, dim3(nb(n)), dim3(256), 0, st, D);
        hipLaunchKernelGGL(k_isl_remove, dim3(nb(n)), dim3(256), 0, st, D, thresh);
        ST_HIP(hipGetLastError());
    }
};

}  // namespace

// Arena bytes the stage grids take beyond offR / offA / corr / type,
// including the optional mask and the 256-byte alignment of each grid.
size_t cull_device_bytes(size_t n) { return n * 56 + n + 16 * 256 + 65536; }

void st_cull_chain_device(st_ctx *c, st_cull_params *cp, float *dOffR, float *dOffA, float *dCorr, uint8_t *dType)
{
    CullRun R(c, cp, dOffR, dOffA, dCorr, dType);
    ST_REQUIRE(cp->sigmaR && cp->sigmaA && cp->offRS && cp->offAS, ST_ERR_ARG, "cull arrays");
    R.st_data();
    R.st_data();
    R.st_data();
    R.stats();
    R.smooth();
    if (cp->islandThresh > 0)
        R.islands();
    R.get(cp->sigmaR, R.D.sigmaR, R.n);
    R.get(cp->sigmaA, R.D.sigmaA, R.n);
    R.get(cp->offRS, R.D.offRS, R.n);
    R.get(cp->offAS, R.D.offAS, R.n);
}

extern "C" int st_cull_st_data(st_ctx *c, st_cull_params *cp)
{
    return st_guard(c, [&]() {
        CullRun R(c, cp);
        ST_REQUIRE(cp->corr && cp->type, ST_ERR_ARG, "corr/type");
        R.put(R.D.offR, cp->offR, R.n);
        R.put(R.D.offA, cp->offA, R.n);
        R.put(R.D.corr, cp->corr, R.n);
        R.put(R.D.type, cp->type, R.n);
        R.st_data();
        R.get(cp->offR, R.D.offR, R.n);
        R.get(cp->offA, R.D.offA, R.n);
        R.get(cp->type, R.D.type, R.n);
        ST_HIP(hipStreamSynchronize(c->stream));
    });
}

extern "C" int st_cull_stats(st_ctx *c, st_cull_params *cp)
{
    return st_guard(c, [&]() {
        CullRun R(c, cp);
        ST_REQUIRE(cp->sigmaR && cp->sigmaA, ST_ERR_ARG, "sigma outputs");
        R.put(R.D.offR, cp->offR, R.n);
        R.put(R.D.offA, cp->offA, R.n);
        R.stats();
        R.get(cp->sigmaR, R.D.sigmaR, R.n);
        R.get(cp->sigmaA, R.D.sigmaA, R.n);
        ST_HIP(hipStreamSynchronize(c->stream));
    });
}

extern "C" int st_cull_smooth(st_ctx *c, st_cull_params *cp)
{
    return st_guard(c, [&]() {
        CullRun R(c, cp);
        ST_REQUIRE(cp->sigmaR && cp->sigmaA && cp->offRS && cp->offAS && cp->type, ST_ERR_ARG, "smooth arrays");
        R.put(R.D.offR, cp->offR, R.n);
        R.put(R.D.offA, cp->offA, R.n);
        R.put(R.D.type, cp->type, R.n);
        R.put(R.D.sigmaR, cp->sigmaR, R.n);
        R.put(R.D.sigmaA, cp->sigmaA, R.n);
        R.smooth();
        R.get(cp->sigmaR, R.D.sigmaR, R.n);
        R.get(cp->sigmaA, R.D.sigmaA, R.n);
        R.get(cp->offRS, R.D.offRS, R.n);
        R.get(cp->offAS, R.D.offAS, R.n);
        ST_HIP(hipStreamSynchronize(c->stream));
    });
}

extern "C" int st_cull_islands(st_ctx *c, st_cull_params *cp)
{
    return st_guard(c, [&]() {
        CullRun R(c, cp);
        ST_REQUIRE(cp->offRS, ST_ERR_ARG, "offRS");
        R.put(R.D.offRS, cp->offRS, R.n);
        if (cp->offAS)
            R.put(R.D.offAS, cp->offAS, R.n);
        else
            R.D.offAS = nullptr;
        R.islands();
        R.get(cp->offRS, R.D.offRS, R.n);
        if (cp->offAS)
            R.get(cp->offAS, R.D.offAS, R.n);
        ST_HIP(hipStreamSynchronize(c->stream));
    });
}

namespace {

// cullst's order on host grids: upload, cullSTData x3, cullStats,
// cullSmooth, cullIslands, download.  staged: through the context's pinned
// buffer, one copy each way over the run of grids alloc() carves (copies from
// and to pageable memory go through the driver's own staging, one grid after
// another).
void cull_chain_host(st_ctx *c, st_cull_params *cp, CullRun &R, bool staged)
{
    const CullDev &D = R.D;
    const size_t f4 = (size_t)R.n * sizeof(float);
    char *const dev = (char *)D.offR;  // the first of the grids
    const size_t in = (size_t)((char *)D.type - dev) + R.n, all = (size_t)((char *)D.sigmaA - dev) + f4;
    char *stg = staged ? (char *)c->pinned_reserve(all) : nullptr;
    auto at = [&](const void *d) { return stg + ((const char *)d - dev); };
    if (staged) {
        parallel_copy({{at(D.offR), cp->offR, f4}, {at(D.offA), cp->offA, f4}, {at(D.corr), cp->corr, f4},
                       {at(D.type), cp->type, (size_t)R.n}});
        ST_HIP(hipMemcpyAsync(dev, stg, in, hipMemcpyHostToDevice, c->stream));
    } else {
        R.put(D.offR, cp->offR, R.n);
        R.put(D.offA, cp->offA, R.n);
        R.put(D.corr, cp->corr, R.n);
        R.put(D.type, cp->type, R.n);
    }
    R.st_data();
    R.st_data();
    R.st_data();
    R.stats();
    R.smooth();
    if (cp->islandThresh > 0)
        R.islands();
    if (staged) {
        ST_HIP(hipMemcpyAsync(stg, dev, all, hipMemcpyDeviceToHost, c->stream));
        ST_HIP(hipStreamSynchronize(c->stream));
        parallel_copy({{cp->offR, at(D.offR), f4}, {cp->offA, at(D.offA), f4}, {cp->type, at(D.type), (size_t)R.n},
                       {cp->sigmaR, at(D.sigmaR), f4}, {cp->sigmaA, at(D.sigmaA), f4}, {cp->offRS, at(D.offRS), f4},
                       {cp->offAS, at(D.offAS), f4}});
        return;
    }
    R.get(cp->offR, D.offR, R.n);
    R.get(cp->offA, D.offA, R.n);
    R.get(cp->type, D.type, R.n);
    R.get(cp->sigmaR, D.sigmaR, R.n);
    R.get(cp->sigmaA, D.sigmaA, R.n);
    R.get(cp->offRS, D.offRS, R.n);
    R.get(cp->offAS, D.offAS, R.n);
    ST_HIP(hipStreamSynchronize(c->stream));
}

bool cull_arrays(const st_cull_params *cp)
{
    return cp->corr && cp->type && cp->sigmaR && cp->sigmaA && cp->offRS && cp->offAS;
}

constexpr size_t kNoAllocCells = (size_t)1 << 19;  // 524 288 grid points
// the stage grids (50 B per point), the four input grids (13 B), the mask
// (1 B), with room to spare, and 256-byte alignment of each of the 18 grids
constexpr size_t kNoAllocBytes = kNoAllocCells * (56 + 1 + 13 + 1) + 18 * 256 + 4096;

}  // namespace

// ---- the entry point that allocates nothing ------------------------------
// Every grid of the chain lives in this file-scope device array.  In host
// code `scratch` is only a stand-in name: its device address on each GPU
// comes from hipGetSymbolAddress, resolved once per device (st_ctx_create
// calls cull_noalloc_init), and only that address is handed to the
// kernels and copies.
static __device__ __align__(256) unsigned char scratch[kNoAllocBytes];

namespace {

constexpr int kMaxDevices = 64;
std::mutex gScratchMu;               // guards gScratch and serialises the calls
void *gScratch[kMaxDevices] = {};    // device address of `scratch` per device

}  // namespace

void cull_noalloc_init(int device)
{
    std::lock_guard<std::mutex> lk(gScratchMu);
    ST_REQUIRE(device >= 0 && device < kMaxDevices, ST_ERR_ARG, "device index");
    if (gScratch[device])
        return;
    void *p = nullptr;
    ST_HIP(hipSetDevice(device));
    ST_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    ST_REQUIRE(p != nullptr, ST_ERR_HIP, "no device address for the cull scratch array");
    gScratch[device] = p;
}

extern "C" int st_cull_run(st_ctx *c, st_cull_params *cp)
{
    return st_guard(c, [&]() {
        CullRun R(c, cp);
        ST_REQUIRE(cull_arrays(cp), ST_ERR_ARG, "cull arrays");
        cull_chain_host(c, cp, R, true);
    });
}

extern "C" int st_cull_run_noalloc(st_ctx *c, st_cull_params *cp)
{
    return st_guard(c, [&]() {
        ST_REQUIRE(cp && cp->nR > 0 && cp->nA > 0 && cp->offR && cp->offA && cull_arrays(cp), ST_ERR_ARG,
                   "cull grids");
        ST_REQUIRE((size_t)cp->nR * cp->nA <= kNoAllocCells, ST_ERR_ARG,
                   "grid of " + std::to_string((size_t)cp->nR * cp->nA) + " points above the " +
                       std::to_string(kNoAllocCells) + " the no-allocation cull holds");
        // one call at a time per process: every context on a device shares
        // the device's array
        std::lock_guard<std::mutex> lk(gScratchMu);
        void *base = (c->device >= 0 && c->device < kMaxDevices) ? gScratch[c->device] : nullptr;
        ST_REQUIRE(base, ST_ERR_HIP, "cull scratch array not set up on this device");
        CullRun R(c, cp, base, kNoAllocBytes);
        cull_chain_host(c, cp, R, false);  // allocates nothing, pinned host memory included
    });
}

namespace {

// Cullls on the cullst machinery: X / Y in the offR / offA slots, XS / YS
// in offRS / offAS, sigmaX / sigmaY in sigmaR / sigmaA.
struct CullLSRun {
    st_cull_ls_params *cp;
    CullRun R;
    LsArg L{};

    static st_cull_ls_params *check(st_cull_ls_params *p)
    {
        ST_REQUIRE(p && p->nx > 0 && p->ny > 0 && p->X && p->Y, ST_ERR_ARG, "cull grids");
        return p;
    }
    CullLSRun(st_ctx *c, st_cull_ls_params *p) : cp(check(p)), R(c, p->nx, p->ny) {}

    void ls_data()
    {
        ST_REQUIRE(cp->dx != 0 && cp->dy != 0, ST_ERR_ARG, "pixel sizes");
        hipStream_t st = R.ctx->stream;
        ST_HIP(hipMemsetAsync(R.D.counters + 3, 0, 2 * sizeof(int), st));
        hipLaunchKernelGGL(k_cull_ls_begin, dim3(nb(R.n)), dim3(256), 0, st, R.D, R.D.type, cp->noDataToUseMask);
        ST_HIP(hipGetLastError());
        const int nGoodPts = R.counter(3), nWithData = R.counter(4);
        if (cp->nMatch < 0) {
            cp->nAttempt = nWithData;
            cp->nMatch = nGoodPts;
        }
        L.type = R.D.type;
        L.slow = cp->slowVelMask;
        L.noData1 = (double)cp->noData + 1.0;
        L.deltaT = cp->deltaT;
        L.dx = cp->dx;
        L.dy = cp->dy;
        cp->nCulled = R.median_pass<true>(cp->bR, cp->bA, cp->nGood, cp->maxY, cp->maxX, L);
    }
    void ls_stats()
    {
        ST_REQUIRE(cp->nover > 0, ST_ERR_ARG, "nover");
        cp->bR = cp->bA = 9;  // cullLSStats.c:39-40
        const double q = ((1.0 / cp->nover) * (1.0 / cp->nover)) / 12.;
        hipLaunchKernelGGL(k_cull_stats, R.tiles(), dim3(256), 0, R.ctx->stream, R.D, 1, q);
        ST_HIP(hipGetLastError());
    }
    void ls_smooth()
    {
        ST_REQUIRE(cp->sX >= 1 && cp->sY >= 1, ST_ERR_ARG, "smoothing window");
        hipLaunchKernelGGL(k_cull_ls_smooth, dim3(nb(R.n)), dim3(256), 0, R.ctx->stream, R.D, cp->sX, cp->sY);
        ST_HIP(hipGetLastError());
    }
};

}  // namespace

extern "C" int st_cull_ls_data(st_ctx *c, st_cull_ls_params *cp)
{
    return st_guard(c, [&]() {
        CullLSRun L(c, cp);
        ST_REQUIRE(cp->type, ST_ERR_ARG, "type");
        L.R.put(L.R.D.offR, cp->X, L.R.n);
        L.R.put(L.R.D.offA, cp->Y, L.R.n);
        L.R.put(L.R.D.type, cp->type, L.R.n);
        L.ls_data();
        L.R.get(cp->X, L.R.D.offR, L.R.n);
        L.R.get(cp->Y, L.R.D.offA, L.R.n);
        ST_HIP(hipStreamSynchronize(c->stream));
    });
}

extern "C" int st_cull_ls_stats(st_ctx *c, st_cull_ls_params *cp)
{
    return st_guard(c, [&]() {
        CullLSRun L(c, cp);
        ST_REQUIRE(cp->sigmaX && cp->sigmaY, ST_ERR_ARG, "sigma outputs");
        L.R.put(L.R.D.offR, cp->X, L.R.n);
        L.R.put(L.R.D.offA, cp->Y, L.R.n);
        L.ls_stats();
        L.R.get(cp->sigmaX, L.R.D.sigmaR, L.R.n);
        L.R.get(cp->sigmaY, L.R.D.sigmaA, L.R.n);
        ST_HIP(hipStreamSynchronize(c->stream));
    });
}

extern "C" int st_cull_ls_smooth(st_ctx *c, st_cull_ls_params *cp)
{
    return st_guard(c, [&]() {
        CullLSRun L(c, cp);
        ST_REQUIRE(cp->sigmaX && cp->sigmaY && cp->XS && cp->YS, ST_ERR_ARG, "smooth arrays");
        L.R.put(L.R.D.offR, cp->X, L.R.n);
        L.R.put(L.R.D.offA, cp->Y, L.R.n);
        L.R.put(L.R.D.sigmaR, cp->sigmaX, L.R.n);
        L.R.put(L.R.D.sigmaA, cp->sigmaY, L.R.n);
        L.ls_smooth();
        L.R.get(cp->sigmaX, L.R.D.sigmaR, L.R.n);
        L.R.get(cp->sigmaY, L.R.D.sigmaA, L.R.n);
        L.R.get(cp->XS, L.R.D.offRS, L.R.n);
        L.R.get(cp->YS, L.R.D.offAS, L.R.n);
        ST_HIP(hipStreamSynchronize(c->stream));
    });
}

extern "C" int st_cull_ls_islands(st_ctx *c, st_cull_ls_params *cp)
{
    return st_guard(c, [&]() {
        CullLSRun L(c, cp);
        ST_REQUIRE(cp->XS, ST_ERR_ARG, "XS");
        L.R.put(L.R.D.offRS, cp->XS, L.R.n);
        if (cp->YS)
            L.R.put(L.R.D.offAS, cp->YS, L.R.n);
        else
            L.R.D.offAS = nullptr;
        L.R.islands_t(cp->islandThresh);
        L.R.get(cp->XS, L.R.D.offRS, L.R.n);
        if (cp->YS)
            L.R.get(cp->YS, L.R.D.offAS, L.R.n);
        ST_HIP(hipStreamSynchronize(c->stream));
    });
}

extern "C" int st_cull_ls_run(st_ctx *c, st_cull_ls_params *cp)
{
    return st_guard(c, [&]() {
        CullLSRun L(c, cp);
        ST_REQUIRE(cp->type && cp->sigmaX && cp->sigmaY && cp->XS && cp->YS, ST_ERR_ARG, "cull arrays");
        L.R.put(L.R.D.offR, cp->X, L.R.n);
        L.R.put(L.R.D.offA, cp->Y, L.R.n);
        L.R.put(L.R.D.type, cp->type, L.R.n);
        cp->nMatch = -1;
        L.ls_data();
        L.ls_data();
        L.ls_data();
        L.ls_stats();
        L.ls_smooth();
        if (cp->islandThresh > 0)
            L.R.islands_t(cp->islandThresh);
        L.R.get(cp->X, L.R.D.offR, L.R.n);
        L.R.get(cp->Y, L.R.D.offA, L.R.n);
        L.R.get(cp->sigmaX, L.R.D.sigmaR, L.R.n);
        L.R.get(cp->sigmaY, L.R.D.sigmaA, L.R.n);
        L.R.get(cp->XS, L.R.D.offRS, L.R.n);
        L.R.get(cp->YS, L.R.D.offAS, L.R.n);
        ST_HIP(hipStreamSynchronize(c->stream));
    });
}
