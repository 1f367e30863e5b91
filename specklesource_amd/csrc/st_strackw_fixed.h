// strackw's passes at fixed window sizes (wRa and wAa each one of 128, 192,
// 256, 384), included by st_strackw.hip inside its anonymous namespace.  The
// same transforms as the general kernels, in the same order and with the same
// roundings (fftn), with less between them:
//   k_wf_rows    range interpolation of both windows; of the chip's only the
//                columns its detection reads                      -> T
//   k_wf_cols    azimuth interpolation, |z|^2 scale               -> U (floats)
//   k_wf_detect  boxcar, square root: search image s, chip image c, column
//                sums of s and s^2 over 32-row tiles              -> Sf, Cf
//   k_wf_zrows   forward range transforms of s + i c              -> Zs
//   k_wf_cross   forward azimuth transforms of columns l and -l of two patches,
//                their cross spectra G0 + i G1                    -> G
//   k_wf_urows   range inverse, the lag columns only              -> X
//   k_wf_lags    azimuth inverse of the lag columns: both patches'
//                correlations at the lags                         -> Gf
// followed by k_w_ncc and k_w_refine.
//
// Values stay in registers between the stages of a transform and images are
// stored as floats, of the chip only what is read; the general passes exchange
// every stage through LDS with a block barrier and move complex images.  576
// windows of 384^2, general -> here: interpolation 6.6 -> 2.3 ms, detection
// 2.04 -> 0.79, correlation transforms with the cross spectra 7.0 -> 3.0.
// k_wf_zrows, k_wf_urows and k_wf_lags run at 3.7 to 5.4 TB/s, the cross spectra
// at 3.3, the interpolation at 2.8 with LDS and VALU issue beside it.

// Geometry for window side N: M = 2 N interpolated samples, C columns (or
// slots) and R rows per workgroup.
template <int N>
struct WfGeom {
    static constexpr int M = 2 * N, VN = fftn::Plan<N>::V, LN = fftn::Plan<N>::LANES;
    static constexpr int VM = fftn::Plan<M>::V, LM = fftn::Plan<M>::LANES;
    // LDS: the twiddle table (M elements), then a region per row or column.
    // Full regions hold M + M / 8 complex elements and some: 8 more than a
    // multiple of 32, so that stores and loads of 8 columns across 8 regions meet
    // no bank twice.  Where a lane holds 24 values (a third of the lanes that 8
    // take) full regions would leave two waves per SIMD: there the kernels that
    // can exchange real and imaginary parts in turn (half regions: M + M / 8
    // floats and some, 8 more than a multiple of 64).
    static constexpr int PB = (M + M / 8 + 23) / 32 * 32 + 8;
    static constexpr bool HALF = VM == 24;
    static constexpr int PF = HALF ? (M + M / 8 + 24 + 55) / 64 * 64 + 8 : 2 * PB;  // floats
    using Ex = std::conditional_t<HALF, float, float2>;
    static constexpr int R = 256 / LM, NTHR = R * LM;
    static constexpr int C = 8, NTHC = C * LM;
    static constexpr size_t TW = M * sizeof(float2);
    static constexpr size_t LDSR = TW + (size_t)R * PF * sizeof(float), LDSC = TW + (size_t)C * PF * sizeof(float);
    static constexpr size_t LDSF = TW + (size_t)C * PB * sizeof(float2);
    static_assert(LM == 2 * LN && VM == VN, "lane groups");
    // start of lane group g's exchanges.  Full regions start 8 elements of 32
    // apart, which keeps groups of 8 lanes off each other's banks: groups of 16
    // need 16.  Half regions start 8 floats apart and need as much as the group
    // has lanes.
    template <int LANES>
    __device__ static inline float2 *full(float2 *lds, int g)
    {
        return lds + g * PB + (LANES == 16 ? (g & 1) * 8 : 0);
    }
    template <int LANES>
    __device__ static inline Ex *ex(float2 *lds, int g)
    {
        if constexpr (HALF)
            return (float *)lds + g * PF + (LANES == 32 ? (g & 1) * 24 : LANES == 16 ? (g & 3) * 8 : 0);
        else
            return full<LANES>(lds, g);
    }
    __device__ static inline float2 *region(float2 *lds, int g) { return lds + g * (PF / 2); }
    static_assert(PB >= M + M / 8 + (LM == 16 ? 8 : 0) && PF >= M + M / 8 + (HALF ? 24 : 0), "room for the shift");
};

struct WfBatch {
    float *U;    // [2][B][W_A][W_R] |z|^2 scale of the search, of the chip
    float *Sf;   // [B][W_A][W_R] search image
    float *Cf;   // [B][wA2][wR2] chip image
    float2 *G;   // [(B + 1) / 2][W_A][W_R] cross spectra of two patches
    float2 *X;   // [(B + 1) / 2][W_A][pitchX] after the range inverse, by lag
    float *Gf;   // [B][nLagA][nLagR] correlation at the lags
    int pitchX;  // nLagR rounded up to 16
};

// Columns of the chip's interpolated image that k_wf_detect reads: its inner
// region and the boxcar's reach.
__host__ __device__ inline int2 wf_chip_cols(const WPar &p)
{
    const int h = p.navgA > 1 || p.navgR > 1 ? p.navgR : 0, e0 = p.epR * WOS;
    return make_int2(imax(0, e0 - h), imin(p.W_R, e0 + p.wR2 + h));
}

// A lane's samples r + LN k of image row a.
template <int N>
__device__ inline void wf_samples(const Images &im, int img, int a, int r, bool inside, float2 (&v)[WfGeom<N>::VN])
{
    constexpr int V = WfGeom<N>::VN, LN = WfGeom<N>::LN;
    if (inside) {
        const size_t o = (size_t)a * (img ? im.nr2 : im.nr1) + r;
        const void *d = img ? im.img2 : im.img1;
        if (im.stype == ST_SAMPLE_C64) {
#pragma unroll
            for (int k = 0; k < V; k++)
                v[k] = ((const float2 *)d + o)[LN * k];
        } else {
#pragma unroll
            for (int k = 0; k < V; k++) {
                const short2 s = ((const short2 *)d + o)[LN * k];
                v[k] = make_float2((float)s.x, (float)s.y);
            }
        }
    } else {
#pragma unroll
        for (int k = 0; k < V; k++)
            v[k] = sample0(im, img, a, r + LN * k);
    }
}

template <int N>
__global__ void __launch_bounds__(WfGeom<N>::NTHR, 4) k_wf_rows(WPar p, int off, WBatch Bt, int B)
{
    using G = WfGeom<N>;
    constexpr int V = G::VN, NW = G::NTHR / 64;
    extern __shared__ float2 tw[];
    float2 *ldsf = tw + G::M;
    __shared__ double sh[NW][4];
    const int z = blockIdx.y, img = z >= B ? 1 : 0, b = z - img * B, t = threadIdx.x;
    const int4 q = Bt.pos[off + b];
    const int rr = img ? q.z : q.x, ra = img ? q.w : q.y;
    const int i0 = blockIdx.x * G::R;
    // the rows here and the next one inside the image: no tests per sample
    const int nr = img ? p.im.nr2 : p.im.nr1, na = img ? p.im.na2 : p.im.na1;
    const bool inside = rr >= 0 && rr + N <= nr && ra + i0 >= 0 && ra + i0 + G::R < na;
    double s[4] = {0, 0, 0, 0};  // sum x, sum x[i + 1] conj(x[i]) (re, im)
    float2 v[V];
    if (t < G::R * G::LN) {
        const int j = t % G::LN, i = i0 + t / G::LN;
        const bool next = i + 1 < p.wAa;
        wf_samples<N>(p.im, img, ra + i, rr + j, inside, v);
#pragma unroll
        for (int r = 0; r < V; r++) {
            s[0] += v[r].x;
            s[1] += v[r].y;
        }
        if (i == 0 || !next) {
            // this row's sum alone (the lanes of the row hold it)
            double e0 = s[0], e1 = s[1];
            for (int o = 1; o < G::LN; o <<= 1) {
                e0 += __shfl_xor(e0, o);
                e1 += __shfl_xor(e1, o);
            }
            if (j == 0) {
                double *E = Bt.dopE + 4 * z + (i == 0 ? 0 : 2);
                E[0] = e0;
                E[1] = e1;
            }
        }
        if (next) {
            float2 w[V];
            wf_samples<N>(p.im, img, ra + i + 1, rr + j, inside, w);
#pragma unroll
            for (int r = 0; r < V; r++) {
                const float2 x1 = w[r], x0 = v[r];
                s[2] += (double)x1.x * x0.x + (double)x1.y * x0.y;
                s[3] += (double)x1.y * x0.x - (double)x1.x * x0.y;
            }
        }
    }
    fftn::table<G::M>(tw);
    __syncthreads();
    if (t < G::R * G::LN) {
        const int j = t % G::LN;
        float2 *out = G::region(ldsf, t / G::LN);
        fftn::fft<N, -1, G::M>(v, j, G::template ex<G::LN>(ldsf, t / G::LN), tw);
#pragma unroll
        for (int r = 0; r < V; r++)
            out[j + G::LN * r] = v[r];
    }
    for (int o = 32; o > 0; o >>= 1)
#pragma unroll
        for (int k = 0; k < 4; k++)
            s[k] += __shfl_xor(s[k], o);
    if ((t & 63) == 0)
#pragma unroll
        for (int k = 0; k < 4; k++)
            sh[t >> 6][k] = s[k];
    __syncthreads();
    if (t < 4) {
        double a = 0;
        for (int w = 0; w < NW; w++)
            a += sh[w][t];
        Bt.dop[((size_t)z * gridDim.x + blockIdx.x) * 4 + t] = a;
    }
    const int j = t % G::LM, i = i0 + t / G::LM;
    const float2 *in = G::region(ldsf, t / G::LM);
#pragma unroll
    for (int r = 0; r < V; r++) {
        // bins 0 .. N / 2 - 1 stay, the Nyquist bin and the negative
        // frequencies move to the top, zeros between
        const int m = j + G::LM * r;
        v[r] = r < V / 4 ? in[m] : r >= V - V / 4 ? in[m - N] : make_float2(0.f, 0.f);
    }
    fft8::wave_sync();
    fftn::fft<G::M, +1, G::M>(v, j, G::template ex<G::LM>(ldsf, t / G::LM), tw);
    const int2 cols = img ? wf_chip_cols(p) : make_int2(0, p.W_R);
    float2 *T = Bt.T + ((size_t)z * p.wAa + i) * p.W_R;
#pragma unroll
    for (int r = 0; r < V; r++) {
        const int m = j + G::LM * r;
        if (m >= cols.x && m < cols.y)
            T[m] = v[r];
    }
}

// Workgroups of a patch: column blocks of the search image, then those of the
// chip's columns.
template <int N>
__global__ void __launch_bounds__(WfGeom<N>::NTHC) k_wf_cols(WPar p, WBatch Bt, WfBatch F, int B, int nb0)
{
    using G = WfGeom<N>;
    constexpr int V = G::VN, C = G::C, M = G::M, LM = G::LM, LN = G::LN;
    extern __shared__ float2 tw[];
    float2 *ldsf = tw + G::M;
    const int nbx = gridDim.x, total = nbx * gridDim.y, flat = blockIdx.y * nbx + blockIdx.x, per = total / 8;
    const int L = flat < per * 8 ? (flat % 8) * per + flat / 8 : flat;  // neighbouring column blocks on one XCD
    const int b = L / nbx, blk = L - b * nbx, img = blk >= nb0 ? 1 : 0, z = img * B + b, t = threadIdx.x;
    const int c0 = img ? (wf_chip_cols(p).x / C + blk - nb0) * C : blk * C;
    const float2 *T = Bt.T + (size_t)z * p.wAa * p.W_R + c0;
    {
        constexpr int K = N / LM;
        const unsigned at = (t / C) * p.W_R + t % C;  // beside a uniform base
        float2 u[K];
#pragma unroll
        for (int k = 0; k < K; k++)
            u[k] = (T + (size_t)(k * LM) * p.W_R)[at];
#pragma unroll
        for (int k = 0; k < K; k++)
            G::region(ldsf, t % C)[t / C + k * LM] = u[k];
    }
    fftn::table<G::M>(tw);
    __syncthreads();
    if (t < C * LN) {
        const int j = t % LN;
        float2 *io = G::region(ldsf, t / LN);
        float2 v[V];
#pragma unroll
        for (int r = 0; r < V; r++)
            v[r] = io[j + LN * r];
        fft8::wave_sync();
        fftn::fft<N, -1, G::M>(v, j, G::template ex<LN>(ldsf, t / LN), tw);
#pragma unroll
        for (int r = 0; r < V; r++)
            io[j + LN * r] = v[r];
    }
    __syncthreads();
    {
        const int j = t % LM, az = Bt.az[b];
        const float2 *in = G::region(ldsf, t / LM);
        float2 v[V];
#pragma unroll
        for (int r = 0; r < V; r++) {
            v[r] = make_float2(0.f, 0.f);
            if (r < V / 4 || r >= V - V / 4) {
                int k = j + LM * r + (r < V / 4 ? 0 : N - M) + az;  // in [0, 2 N)
                k -= k >= N ? N : 0;
                v[r] = in[k];
            }
        }
        fft8::wave_sync();
        fftn::fft<M, +1, G::M>(v, j, G::template ex<LM>(ldsf, t / LM), tw);
        float *exf = (float *)G::region(ldsf, t / LM);
#pragma unroll
        for (int r = 0; r < V; r++) {
#pragma clang fp contract(off)
            exf[j + LM * r] = (v[r].x * v[r].x + v[r].y * v[r].y) * p.scale;
        }
    }
    __syncthreads();
    float *U = F.U + (size_t)z * p.W_A * p.W_R + c0;
    const unsigned at = (t / C) * p.W_R + t % C;
#pragma unroll
    for (int k = 0; k < M / LM; k++)
        (U + (size_t)(k * LM) * p.W_R)[at] = ((const float *)G::region(ldsf, t % C))[t / C + k * LM];
}

template <int N>
__global__ void __launch_bounds__(WfGeom<N>::NTHR) k_wf_zrows(WPar p, WBatch Bt, WfBatch F)
{
    using G = WfGeom<N>;
    constexpr int V = G::VM, LM = G::LM;
    extern __shared__ float2 tw[];
    float2 *ldsf = tw + G::M;
    const int b = blockIdx.y, t = threadIdx.x, j = t % LM, y = blockIdx.x * G::R + t / LM;
    const float *S = F.Sf + ((size_t)b * p.W_A + y) * p.W_R + j;
    const int yc = y - p.epA * WOS, e0 = p.epR * WOS;
    const float *Cr = F.Cf + ((size_t)b * p.wA2 + yc) * p.wR2 - e0 + j;
    const bool in = yc >= 0 && yc < p.wA2;
    float2 v[V];
#pragma unroll
    for (int r = 0; r < V; r++) {
        const int x = j + LM * r;
        v[r] = make_float2(S[LM * r], in && x >= e0 && x < e0 + p.wR2 ? Cr[LM * r] : 0.f);
    }
    fftn::table<G::M>(tw);
    __syncthreads();
    fftn::fft<G::M, -1, G::M>(v, j, G::template ex<LM>(ldsf, t / LM), tw);
    float2 *Z = Bt.Zs + ((size_t)b * p.W_A + y) * p.W_R + j;
#pragma unroll
    for (int r = 0; r < V; r++)
        Z[LM * r] = v[r];
}

template <int N>
__global__ void __launch_bounds__(WfGeom<N>::NTHR, 4) k_wf_urows(WPar p, WfBatch F)
{
    using G = WfGeom<N>;
    constexpr int V = G::VM, M = G::M, LM = G::LM;
    extern __shared__ float2 tw[];
    float2 *ldsf = tw + G::M;
    const int q = blockIdx.y, t = threadIdx.x, j = t % LM, y = blockIdx.x * G::R + t / LM;
    const float2 *Gq = F.G + ((size_t)q * p.W_A + y) * p.W_R + j;
    float2 v[V];
#pragma unroll
    for (int r = 0; r < V; r++)
        v[r] = Gq[LM * r];
    fftn::table<G::M>(tw);
    __syncthreads();
    fftn::fft<M, +1, G::M>(v, j, G::template ex<LM>(ldsf, t / LM), tw);
    const int lagR = WOS * p.epR;
    float2 *X = F.X + ((size_t)q * p.W_A + y) * F.pitchX;
#pragma unroll
    for (int r = 0; r < V; r++) {
        const int m = j + LM * r, s = m <= lagR ? m + lagR : m - M + lagR;
        if (s >= 0 && s < p.nLagR)
            X[s] = v[r];
    }
}

// Lag columns past nLagR (the last workgroup's) hold whatever X did there;
// they stay in their own regions and are not stored.
template <int N>
__global__ void __launch_bounds__(WfGeom<N>::NTHC) k_wf_lags(WPar p, WfBatch F, int B)
{
    using G = WfGeom<N>;
    constexpr int V = G::VM, C = G::C, M = G::M, LM = G::LM;
    extern __shared__ float2 tw[];
    float2 *ldsf = tw + G::M;
    const int nbx = gridDim.x, total = nbx * gridDim.y, flat = blockIdx.y * nbx + blockIdx.x, per = total / 8;
    const int L = flat < per * 8 ? (flat % 8) * per + flat / 8 : flat;
    const int q = L / nbx, c0 = (L - q * nbx) * C, t = threadIdx.x, j = t % LM;
    const float2 *X = F.X + (size_t)q * p.W_A * F.pitchX + c0;
    float2 *ex = ldsf + (t / LM) * G::PB;
    {
        float2 u[M / LM];
        const unsigned at = (t / C) * F.pitchX + t % C;
#pragma unroll
        for (int k = 0; k < M / LM; k++)
            u[k] = (X + (size_t)(k * LM) * F.pitchX)[at];
#pragma unroll
        for (int k = 0; k < M / LM; k++)
            ldsf[(t % C) * G::PB + t / C + k * LM] = u[k];
    }
    fftn::table<G::M>(tw);
    __syncthreads();
    float2 v[V];
#pragma unroll
    for (int r = 0; r < V; r++)
        v[r] = ex[j + LM * r];
    fft8::wave_sync();
    fftn::fft<M, +1, G::M>(v, j, G::template full<LM>(ldsf, t / LM), tw);
    fft8::wave_sync();
#pragma unroll
    for (int r = 0; r < V; r++)
        ex[j + LM * r] = v[r];
    __syncthreads();
    const int lagA = WOS * p.epA, s = c0 + t % C;
    float *g0 = F.Gf + (size_t)(2 * q) * p.nLagA * p.nLagR + s, *g1 = g0 + (size_t)p.nLagA * p.nLagR;
    const bool in = s < p.nLagR, second = 2 * q + 1 < B;
#pragma unroll
    for (int k = 0; k < M / LM; k++) {
        const int n = t / C + k * LM, i = n <= lagA ? n + lagA : n - M + lagA;  // lag row of output n
        if (in && i >= 0 && i < p.nLagA) {
            const float2 x = ldsf[(t % C) * G::PB + n];
            g0[(size_t)i * p.nLagR] = x.x;
            if (second)
                g1[(size_t)i * p.nLagR] = x.y;
        }
    }
}

#pragma clang fp contract(off)
constexpr int kDetW = 64;  // columns of a k_wf_detect tile (kTile rows)

// A tile's haloed source from |z|^2 scale: rows clamped to [0, ymax], columns
// to [0, W_R - 1] (four at a time: segments start at multiples of four, as does
// W_R, so that a segment lies inside the image or beside it).
__device__ inline void wf_tile(float *d, const float *U, int W, int y0, int x0, int TH, int TW, int ymax)
{
    const int seg = TW / 4;
    for (int t = threadIdx.x; t < TH * seg; t += 256) {
        const int ty = t / seg, tx = (t - ty * seg) * 4, x = x0 + tx;
        const float *row = U + (size_t)imin(imax(y0 + ty, 0), ymax) * W;
        float4 v;
        if (x >= 0 && x < W) {
            v = *(const float4 *)(row + x);
        } else {
            const float e = row[x < 0 ? 0 : W - 1];
            v = make_float4(e, e, e, e);
        }
        *(float4 *)(d + ty * TW + tx) = v;
    }
}

// Boxcar sums of four neighbours from row[0], each in the order of the
// reference's loops.  H >= 0: both half-widths are H.
template <int H>
__device__ inline void wf_box(const float *row, int TW, int hA, int hR, float (&v)[4])
{
#pragma unroll
    for (int k = 0; k < 4; k++)
        v[k] = 0.f;
    if constexpr (H >= 0) {
#pragma unroll
        for (int m = 0; m <= 2 * H; m++) {
            float w[4 + 2 * H];
#pragma unroll
            for (int n = 0; n < 4 + 2 * H; n++)
                w[n] = row[m * TW + n];
#pragma unroll
            for (int n = 0; n <= 2 * H; n++)
#pragma unroll
                for (int k = 0; k < 4; k++)
                    v[k] += w[n + k];
        }
    } else {
        for (int m = 0; m <= 2 * hA; m++) {
            const float *r = row + m * TW;
            float w0 = r[0], w1 = r[1], w2 = r[2];
            for (int n = 0; n <= 2 * hR; n++) {
                const float w3 = r[n + 3];
                v[0] += w0;
                v[1] += w1;
                v[2] += w2;
                v[3] += w3;
                w0 = w1;
                w1 = w2;
                w2 = w3;
            }
        }
    }
}

// detectPatch from the detected images (k_w_detect's boxcar, clamps and sums):
// tiles of kTile rows by kDetW columns, four neighbouring cells per thread, the
// chip's cells in a second turn through the same LDS tile.  H: wf_box's, 0 where
// there is no boxcar.
//
// Bound: the (2 h + 1)^2 ordered sums and their LDS reads, which four
// neighbours share, then the column sums.  576 patches of 768^2, 5 x 5 boxcar:
// 0.75 ms; 1.87 with one cell per thread and one load per sample.
template <int H>
__global__ void __launch_bounds__(256) k_wf_detect(WPar p, WBatch Bt, WfBatch F, int B)
{
    extern __shared__ float4 w_det_lds4[];
    __shared__ float sv[kTile][kDetW + 1];
    float *d = (float *)w_det_lds4;
    const int b = blockIdx.z;
    const size_t NN = (size_t)p.W_A * p.W_R;
    const int hA = H >= 0 ? H : p.navgA, hR = H >= 0 ? H : p.navgR, hp = (hR + 3) / 4 * 4;
    const int y0 = blockIdx.y * kTile, x0 = blockIdx.x * kDetW;
    const int TH = kTile + 2 * hA, TW = kDetW + 2 * hp;
    wf_tile(d, F.U + b * NN, p.W_R, y0 - hA, x0 - hp, TH, TW, p.W_A - 1);
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kTile * kDetW / 1024; k++) {
        const int t = threadIdx.x + 256 * k, oy = t / (kDetW / 4), ox = (t % (kDetW / 4)) * 4;
        float v[4];
        wf_box<H>(d + oy * TW + ox + hp - hR, TW, hA, hR, v);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            v[i] = sqrtf(v[i]);
            sv[oy][ox + i] = v[i];
        }
        *(float4 *)(F.Sf + b * NN + (size_t)(y0 + oy) * p.W_R + x0 + ox) = make_float4(v[0], v[1], v[2], v[3]);
    }
    __syncthreads();
    // column sums of s and of s^2 (FP64) over the tile's rows
    if (threadIdx.x < 2 * kDetW) {
        const int c = threadIdx.x % kDetW;
        const bool sq = threadIdx.x >= kDetW;
        double a = 0.0;
        for (int oy = 0; oy < kTile; oy++) {
            const float v = sv[oy][c];
            a += sq ? v * v : v;
        }
        Bt.csum[(((size_t)b * gridDim.y + blockIdx.y) * 2 + (sq ? 1 : 0)) * p.W_R + x0 + c] = a;
    }
    const int c0 = p.epA * WOS, c1 = c0 + p.wA2;  // chip rows [c0, c1)
    const int e0 = p.epR * WOS, e1 = e0 + p.wR2;  // chip cols [e0, e1)
    if (y0 >= c1 || y0 + kTile <= c0 || x0 >= e1 || x0 + kDetW <= e0)
        return;
    // the azimuth clamp is the reference's, written with the range pad; the
    // columns that k_wf_cols left out reach no cell of the chip
    const int kmaxC = imin(p.epR * WOS + p.wA2 + p.navgA - 1, p.W_A - 1);
    wf_tile(d, F.U + ((size_t)B + b) * NN, p.W_R, y0 - hA, x0 - hp, TH, TW, kmaxC);
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kTile * kDetW / 1024; k++) {
        const int t = threadIdx.x + 256 * k, oy = t / (kDetW / 4), ox = (t % (kDetW / 4)) * 4;
        const int y = y0 + oy, x = x0 + ox;
        if (y < c0 || y >= c1 || x + 3 < e0 || x >= e1)
            continue;
        float v[4];
        wf_box<H>(d + oy * TW + ox + hp - hR, TW, hA, hR, v);
        float *c = F.Cf + ((size_t)b * p.wA2 + y - c0) * p.wR2 - e0 + x;
#pragma unroll
        for (int i = 0; i < 4; i++)
            if (x + i >= e0 && x + i < e1)
                c[i] = sqrtf(v[i]);
    }
}

inline void launch_wf_detect(const WPar &p, const WBatch &Bt, const WfBatch &F, int nb, hipStream_t st)
{
    const bool box = p.navgA > 1 || p.navgR > 1;  // detectPatch's test
    const int hA = box ? p.navgA : 0, hR = box ? p.navgR : 0;
    const size_t lds = (size_t)(kTile + 2 * hA) * (kDetW + (hR + 3) / 4 * 8) * sizeof(float);
    const dim3 g(p.W_R / kDetW, p.W_A / kTile, nb);
    if (!box)
        hipLaunchKernelGGL(k_wf_detect<0>, g, dim3(256), lds, st, p, Bt, F, nb);
    else if (hA == 2 && hR == 2)  // the trackers' own boxcar
        hipLaunchKernelGGL(k_wf_detect<2>, g, dim3(256), lds, st, p, Bt, F, nb);
    else
        hipLaunchKernelGGL(k_wf_detect<-1>, g, dim3(256), lds, st, p, Bt, F, nb);
}

// S conj(C) at a frequency from Z there (a) and at its mirror (c): k_w_cross's
// expressions.
__device__ inline float2 wf_cross(float2 a, float2 c)
{
    const float2 S = make_float2(0.5f * (a.x + c.x), 0.5f * (a.y - c.y));
    const float2 Cc = make_float2(0.5f * (a.y + c.y), 0.5f * (c.x - a.x));
    return cmulconj(S, Cc);
}

// Slot c of a workgroup: column l = c0 + c and its mirror W_R - l (W_R / 2 for
// l = 0, both their own mirrors) of patches 2 q and 2 q + 1, one lane group.
// The slot's LDS region holds one column at a time: loads and stores in whole
// segments of C columns pass through it, and so do the mirrored reads.
template <int N>
__global__ void __launch_bounds__(WfGeom<N>::NTHC, 2) k_wf_cross(WPar p, WBatch Bt, WfBatch F, int B)
{
    using G = WfGeom<N>;
    constexpr int V = G::VM, C = G::C, M = G::M, LM = G::LM;
    extern __shared__ float2 tw[];
    float2 *ldsf = tw + G::M;
    const int nbx = gridDim.x, total = nbx * gridDim.y, flat = blockIdx.y * nbx + blockIdx.x, per = total / 8;
    const int Lb = flat < per * 8 ? (flat % 8) * per + flat / 8 : flat;
    const int q = Lb / nbx, c0 = (Lb - q * nbx) * C, t = threadIdx.x, W = p.W_R, H = W / 2;
    const int j = t % LM, slot = t / LM;
    float2 *ex = ldsf + slot * G::PB, *sx = G::template full<LM>(ldsf, slot);
    const bool self = c0 + slot == 0;
    fftn::table<G::M>(tw);
    // column of load / store lane t % C on side s (0: l, 1: mirror)
    auto col = [&](int s) {
        const int l = c0 + t % C;
        return s == 0 ? l : l == 0 ? H : W - l;
    };
    auto load = [&](const float2 *Z, int s, float2(&v)[V]) {
        float2 u[M / LM];
        const unsigned at = (t / C) * W + col(s);
#pragma unroll
        for (int k = 0; k < M / LM; k++)
            u[k] = (Z + (size_t)(k * LM) * W)[at];
        __syncthreads();  // the region's last readers are done
#pragma unroll
        for (int k = 0; k < M / LM; k++)
            ldsf[(t % C) * G::PB + t / C + k * LM] = u[k];
        __syncthreads();
#pragma unroll
        for (int r = 0; r < V; r++)
            v[r] = ex[j + LM * r];
        fft8::wave_sync();
    };
    float2 g[2][V];  // G0 + i G1 of column l, of its mirror
    auto patch = [&](auto h) {
        const float2 *Z = Bt.Zs + (size_t)(2 * q + h) * p.W_A * W;
        float2 x[V], y[V];
        load(Z, 0, x);
        __builtin_amdgcn_sched_barrier(0);
        fftn::fft<M, -1, G::M>(x, j, sx, tw);
        __builtin_amdgcn_sched_barrier(0);
        load(Z, 1, y);
        __builtin_amdgcn_sched_barrier(0);
        fftn::fft<M, -1, G::M>(y, j, sx, tw);
        __builtin_amdgcn_sched_barrier(0);
        // side s: the region takes the column at -l (columns 0 and W_R / 2 are their own)
        auto side = [&](auto s) {
            float2(&m)[V] = s == 0 ? x : y;
#pragma unroll
            for (int r = 0; r < V; r++)
                ex[j + LM * r] = self == (s == 0) ? x[r] : y[r];
            fft8::wave_sync();
#pragma unroll
            for (int r = 0; r < V; r++) {
                const float2 d = wf_cross(m[r], ex[r == 0 && j == 0 ? 0 : M - j - LM * r]);
                g[s][r] = h == 0 ? d : make_float2(g[s][r].x - d.y, g[s][r].y + d.x);
            }
            fft8::wave_sync();
        };
        side(std::integral_constant<int, 0>());
        side(std::integral_constant<int, 1>());
    };
    patch(std::integral_constant<int, 0>());
    if (2 * q + 1 < B)  // the same for the whole workgroup
        patch(std::integral_constant<int, 1>());
    float2 *Gq = F.G + (size_t)q * p.W_A * W;
#pragma unroll
    for (int s = 0; s < 2; s++) {
#pragma unroll
        for (int r = 0; r < V; r++)
            ex[j + LM * r] = g[s][r];
        __syncthreads();
        const unsigned at = (t / C) * W + col(s);
#pragma unroll
        for (int k = 0; k < M / LM; k++)
            (Gq + (size_t)(k * LM) * W)[at] = ldsf[(t % C) * G::PB + t / C + k * LM];
        __syncthreads();
    }
}

#pragma clang fp contract(on)

inline bool wf_covered(const WPar &p) { return fftn::covered(p.wRa) && fftn::covered(p.wAa); }

template <class F>
void wf_size(int n, F f)
{
    switch (n) {
    case 128: f(std::integral_constant<int, 128>()); break;
    case 192: f(std::integral_constant<int, 192>()); break;
    case 256: f(std::integral_constant<int, 256>()); break;
    default: f(std::integral_constant<int, 384>()); break;
    }
}

// Rows per workgroup of k_wf_rows (its Doppler partials).
inline int wf_rows_per_block(int wRa)
{
    int r = 1;
    wf_size(wRa, [&](auto n) { r = WfGeom<decltype(n)::value>::R; });
    return r;
}
