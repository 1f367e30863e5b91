// Amplitude tries of 128 x 128 sample patches (the doubled window of 64
// samples, and 128 px windows), included by st_strack.hip inside its
// anonymous namespace.
//
// The W x W arrays of a try (W = 256: 512 KB of complex values) exceed a CU's
// LDS, so the passes of k_amp_fused run as kernels over a batch of tries with
// the arrays between them in memory:
//   k_amp_items     corners, bounds, Doppler shift
//   k_ampl_rows     patches from the image, range transforms     -> F [2B][ws][ws]
//   k_ampl_cols     azimuth transform, rotation, pad, inverse    -> T [2B][W][ws]
//   k_ampl_det      range pad and inverse of both images' rows, amplitudes,
//                   partial sums                                 -> v [B][W][W]
//   k_amp_stat      zero test and means
//   k_ampl_fwd      means removed, range transform of v1 + i v2  -> Z [B][W][W]
//   k_ampl_cross    azimuth transforms of columns l and -l, separation, F1
//                   conj(F2), azimuth inverse of l <= W / 2      -> S [B][W][W / 2 + 1 of W]
//   k_ampl_mag      range inverse, two rows per transform, |s|, coarse top two
// Same order and arithmetic as the staged kernels of other sizes (k_amp_colx
// .. k_amp_rowmag): bit-identical surfaces.  Every pass reads and writes whole
// 128-byte segments; columns go through LDS 16 at a time.
//
// Bound: HBM traffic: 4.7 MB per try (writes as counted, reads as laid out) at
// 4.0 TB/s; k_ampl_det also issues a VALU instruction on 77 % of the SIMDs'
// cycles, the others on 30 to 49 %.  6 732 doubled windows: 2.4 us per try with
// the staged kernels, 1.2 us with these.
constexpr int kAlWS = 128, kAlW = 256, kAlPitch = kAlW + kAlW / 8 + 1;
constexpr int kAlCols = 16;                   // columns of one pass (128 bytes of a row)
constexpr int kAlRows = 8;                    // rows of W per 256-thread workgroup
constexpr int kAlBlocks = kAlW / kAlRows;     // row workgroups per try (partials of the sums)
constexpr int kAlMagBlocks = kAlBlocks / 2;   // of k_ampl_mag (two rows per transform)

// Corners, bounds and Doppler shift of the tries: state 0 (out of bounds) or
// 2, az in units of ws.  DOP: the try's own estimate, left for the doubled
// window (one workgroup per try; else one thread).
template <int DOP>
__global__ void __launch_bounds__(NT) k_amp_items(KPar P, Pts S, const int *__restrict__ list, int count, int ws, int sc,
                                                   AmpBatch A)
{
    __shared__ double sh[NT / 64];
    const int it = DOP ? (int)blockIdx.x : (int)(blockIdx.x * NT + threadIdx.x);
    if (it >= count)
        return;
    const int pt = list[it];
    const int i = pt / P.nR, j = pt - (pt / P.nR) * P.nR;
    const int a1 = P.aStart + i * P.deltaA - P.wA / 2 * sc, r1 = P.rStart + j * P.deltaR - P.wR / 2 * sc;
    const int r2 = r1 + (S.r2[pt] - S.r1[pt]), a2 = a1 + (S.a2[pt] - S.a1[pt]);
    const bool ok = in_bounds(r1, a1, ws, ws, P.im.nr1, P.im.na1) && in_bounds(r2, a2, ws, ws, P.im.nr2, P.im.na2);
    int az = S.azUse[pt];
    if (DOP && ok) {
        auto get = [&](int e, float2 &x, float2 &y) {
            const int ii = e / ws, jj = e - (e / ws) * ws;
            x = load_sample(P.im.img1, P.im.stype, P.im.nr1, a1 + ii, r1 + jj);
            y = load_sample(P.im.img2, P.im.stype, P.im.nr2, a2 + ii, r2 + jj);
        };
        az = doppler_shift(get, ws, ws, ws, P.wA, sh);
        if (threadIdx.x == 0)
            S.azUse[pt] = az;
    }
    if (!DOP || threadIdx.x == 0) {
        A.state[it] = ok ? 2 : 0;
        A.az[it] = (int)((float)az * (float)ws / (float)P.wA);
    }
}

template <int STYPE>
__global__ void __launch_bounds__(256) k_ampl_rows(KPar P, Pts S, const int *__restrict__ list, int B, int sc, AmpBatch A)
{
    constexpr int WS = kAlWS, LS = WS / 8, R = 256 / LS, PB = WS + WS / 8 + 1;
    __shared__ float2 lds[R * PB];
    int z, blk;
    xcd_item_block(gridDim.x, z, blk);
    const int b = z % B, g = z / B, t = threadIdx.x, j = t % LS, row = t / LS, a = blk * R + row;
    if (A.state[b] != 2)
        return;
    const AmpItem w = amp_item(P, S, list[b], WS, sc);
    const void *img = g ? P.im.img2 : P.im.img1;
    const size_t o = (size_t)((g ? w.a2 : w.a1) + a) * (g ? P.im.nr2 : P.im.nr1) + (g ? w.r2 : w.r1) + j;
    float2 v[8];
#pragma unroll
    for (int r = 0; r < 8; r++) {
        if constexpr (STYPE == ST_SAMPLE_C64) {
            v[r] = __builtin_bit_cast(float2, ((const gu64 *)img)[o + LS * r]);
        } else {
            const unsigned q = ((const gu32 *)img)[o + LS * r];
            v[r] = make_float2((float)(short)(q & 0xffffu), (float)(short)(q >> 16));
        }
    }
    fft8::Twiddles<WS> tw;
    tw.load(j);
    fft8::fft<WS, -1>(v, j, lds + row * PB, tw);
    float2 *F = A.I + ((size_t)z * WS + a) * WS + j;
#pragma unroll
    for (int q = 0; q < 8; q++)
        F[LS * q] = v[q];
}

__global__ void __launch_bounds__(512) k_ampl_cols(int B, AmpBatch A)
{
    constexpr int WS = kAlWS, W = kAlW, LS = WS / 8, LW = W / 8, C = kAlCols, PB = kAlPitch, RP = 512 / C;
    __shared__ float2 lds[C * PB];
    int z, blk;
    xcd_item_block(gridDim.x, z, blk);
    const int b = z % B, t = threadIdx.x, c0 = blk * C;
    if (A.state[b] != 2)
        return;
    const float2 *F = A.I + (size_t)z * WS * WS + c0;
    {
        float2 u[WS / RP];
#pragma unroll
        for (int i = 0; i < WS / RP; i++)
            u[i] = F[(size_t)(t / C + i * RP) * WS + t % C];
#pragma unroll
        for (int i = 0; i < WS / RP; i++)
            lds[(t % C) * PB + t / C + i * RP] = u[i];
    }
    __syncthreads();
    if (t < C * LS) {
        const int j = t % LS;
        float2 *ex = lds + (t / LS) * PB;
        float2 v[8];
        fft8::Twiddles<WS> tw;
        tw.load(j);
#pragma unroll
        for (int r = 0; r < 8; r++)
            v[r] = ex[j + LS * r];
        fft8::wave_sync();
        fft8::fft<WS, -1>(v, j, ex, tw);
#pragma unroll
        for (int q = 0; q < 8; q++)
            ex[j + LS * q] = v[q];
    }
    __syncthreads();
    {
        const int j = t % LW, az = A.az[b];
        float2 *ex = lds + (t / LW) * PB;
        float2 v[8];
        fft8::Twiddles<W> tw;
        tw.load(j);
#pragma unroll
        for (int r = 0; r < 8; r++)
            v[r] = r < 2 || r > 5 ? ex[(j + LW * r + az) & (WS - 1)] : make_float2(0.f, 0.f);
        fft8::wave_sync();
        fft8::fft<W, +1>(v, j, ex, tw);
#pragma unroll
        for (int q = 0; q < 8; q++)
            ex[j + LW * q] = v[q];
    }
    __syncthreads();
    float2 *T = A.F + (size_t)z * W * WS + c0;
#pragma unroll
    for (int i = 0; i < W / RP; i++) {
        const int n = t / C + i * RP;
        T[(size_t)n * WS + t % C] = lds[(t % C) * PB + n];
    }
}

__global__ void __launch_bounds__(256) k_ampl_det(int B, int isf, AmpBatch A)
{
    constexpr int WS = kAlWS, W = kAlW, LW = W / 8, PB = kAlPitch;
    __shared__ float2 lds[kAlRows * PB];
    __shared__ AmpSums sh[4];
    int b, blk;
    xcd_item_block(gridDim.x, b, blk);
    if (A.state[b] != 2)
        return;
    const int t = threadIdx.x, j = t % LW, n = blk * kAlRows + t / LW;
    float2 *ex = lds + (t / LW) * PB;
    fft8::Twiddles<W> tw;
    tw.load(j);
    float2 p[2][8];
#pragma unroll
    for (int g = 0; g < 2; g++) {
        const float2 *T = A.F + (((size_t)g * B + b) * W + n) * WS + j;
#pragma unroll
        for (int r = 0; r < 8; r++)
            p[g][r] = r < 2 ? T[LW * r] : r > 5 ? T[LW * r - WS] : make_float2(0.f, 0.f);
    }
    constexpr float scale = (float)(1. / ((double)WS * WS * WS * WS * 8));
    const float thr = isf ? 1.0e-15f : 1.0e-6f;
    double sm[4] = {0, 0, 0, 0};
    float v1[8], v2[8];
    unsigned mask = 0;
    auto detect = [&](const float2 (&z)[8], float (&v)[8], double &s, double &m) {
        float x[8];
        amp_detect(z, scale, x, v);
#pragma unroll
        for (int r = 0; r < 8; r++) {
            mask |= (x[r] < thr ? 1u : 0u) << r;
            s += x[r];
            m += v[r];
        }
    };
    fft8::fft<W, +1>(p[0], j, ex, tw);
    detect(p[0], v1, sm[0], sm[2]);
    fft8::fft<W, +1>(p[1], j, ex, tw);
    detect(p[1], v2, sm[1], sm[3]);
    float2 *V = A.S + ((size_t)b * W + n) * W + j;
#pragma unroll
    for (int q = 0; q < 8; q++)
        V[LW * q] = make_float2(v1[q], v2[q]);
    amp_sums_put(sm, sh);
    amp_count_put(__popc(mask), sh);
    __syncthreads();
    if (t == 0) {
        const AmpSums s = amp_sums_get<4, 4>(sh);
        A.dpart[(size_t)b * kAlBlocks + blk] = AmpPart{s.v[0], s.v[1], s.v[2], s.v[3], s.n, 0};
    }
}

__global__ void __launch_bounds__(256) k_ampl_fwd(AmpBatch A)
{
    constexpr int W = kAlW, LW = W / 8, PB = kAlPitch;
    __shared__ float2 lds[kAlRows * PB];
    __shared__ AmpSums sh[4];
    int b, blk;
    xcd_item_block(gridDim.x, b, blk);
    if (A.state[b] != 2)
        return;
    const int t = threadIdx.x, j = t % LW, n = blk * kAlRows + t / LW;
    const double m1 = A.mean[b].x, m2 = A.mean[b].y;
    fft8::Twiddles<W> tw;
    tw.load(j);
    const float2 *V = A.S + ((size_t)b * W + n) * W + j;
    float2 x[8];
    double pw[2] = {0, 0};
#pragma unroll
    for (int r = 0; r < 8; r++)
        x[r] = V[LW * r];
#pragma unroll
    for (int r = 0; r < 8; r++) {
#pragma clang fp contract(off)
        float a = x[r].x, c = x[r].y;
        if (a > 1.0e-20)
            a = (float)(a - m1);
        c = (float)(c - m2);
        pw[0] += a * a;
        pw[1] += c * c;
        x[r] = make_float2(a, c);
    }
    fft8::fft<W, -1>(x, j, lds + (t / LW) * PB, tw);
    float2 *Z = A.F + ((size_t)b * W + n) * W + j;
#pragma unroll
    for (int q = 0; q < 8; q++)
        Z[LW * q] = x[q];
    amp_sums_put(pw, sh);
    __syncthreads();
    if (t == 0) {
        const AmpSums s = amp_sums_get<4, 2>(sh);
        A.ppart[(size_t)b * kAlBlocks + blk] = make_double2(s.v[0], s.v[1]);
    }
}

// Slot s of a workgroup: column l = c0 + s in LDS row s and its mirror W - l
// (W / 2 for l = 0) in row 16 + s, both transformed by one lane group.
constexpr size_t kAlLdsCross = (size_t)2 * kAlCols * kAlPitch * sizeof(float2);
__global__ void __launch_bounds__(512) k_ampl_cross(AmpBatch A)
{
    constexpr int W = kAlW, H = W / 2, LW = W / 8, C = kAlCols, PB = kAlPitch, RP = 512 / C;
    extern __shared__ float2 lds[];  // [2 C][PB]
    int b, blk;
    xcd_item_block(gridDim.x, b, blk);
    if (A.state[b] != 2)
        return;
    const int t = threadIdx.x, c0 = blk * C;
    const float2 *Z = A.F + (size_t)b * W * W;
    {
        const int c = t % C, l = c0 + c, lm = l == 0 ? H : W - l;
        constexpr int NP = W / RP / 2;
#pragma unroll
        for (int half = 0; half < 2; half++) {
            float2 u[NP], v[NP];
#pragma unroll
            for (int i = 0; i < NP; i++) {
                const size_t o = (size_t)(t / C + (half * NP + i) * RP) * W;
                u[i] = Z[o + l];
                v[i] = Z[o + lm];
            }
#pragma unroll
            for (int i = 0; i < NP; i++) {
                const int a = t / C + (half * NP + i) * RP;
                lds[c * PB + a] = u[i];
                lds[(C + c) * PB + a] = v[i];
            }
        }
    }
    __syncthreads();
    {
        const int j = t % LW, s = t / LW;
        float2 *X = lds + s * PB, *Y = lds + (C + s) * PB;
        const bool self = c0 + s == 0;  // columns 0 and W / 2 are their own mirrors
        fft8::Twiddles<W> tw;
        tw.load(j);
        float2 x[8], y[8];
#pragma unroll
        for (int r = 0; r < 8; r++) {
            x[r] = X[j + LW * r];
            y[r] = Y[j + LW * r];
        }
        fft8::wave_sync();
        fft8::fft<W, -1>(x, j, X, tw);
        fft8::fft<W, -1>(y, j, Y, tw);
#pragma unroll
        for (int q = 0; q < 8; q++) {
            X[j + LW * q] = x[q];
            Y[j + LW * q] = y[q];
        }
        fft8::wave_sync();
        const float2 *M = self ? X : Y;
#pragma unroll
        for (int q = 0; q < 8; q++)
            x[q] = amp_cross_sep(x[q], M[(W - j - LW * q) & (W - 1)]);
        if (self) {
#pragma unroll
            for (int q = 0; q < 8; q++)
                y[q] = amp_cross_sep(y[q], Y[(W - j - LW * q) & (W - 1)]);
        }
        fft8::wave_sync();
        fft8::fft<W, +1>(x, j, X, tw);
#pragma unroll
        for (int q = 0; q < 8; q++)
            X[j + LW * q] = x[q];
        if (self) {
            fft8::fft<W, +1>(y, j, Y, tw);
            // column W / 2, once per try
            float2 *Sb = A.S + (size_t)b * W * W + H;
#pragma unroll
            for (int q = 0; q < 8; q++)
                Sb[(size_t)(j + LW * q) * W] = y[q];
        }
    }
    __syncthreads();
    float2 *Sb = A.S + (size_t)b * W * W + c0;
#pragma unroll
    for (int i = 0; i < W / RP; i++) {
        const int n = t / C + i * RP;
        Sb[(size_t)n * W + t % C] = lds[(t % C) * PB + n];
    }
}

__global__ void __launch_bounds__(256) k_ampl_mag(AmpBatch A)
{
    constexpr int WS = kAlWS, W = kAlW, LW = W / 8, PB = kAlPitch;
    __shared__ float2 lds[kAlRows * PB];
    __shared__ Top2 sht[4];
    __shared__ int srank;
    int b, blk;
    xcd_item_block(gridDim.x, b, blk);
    Top2 *part = A.part + (size_t)b * kAlMagBlocks + blk;
    const int t = threadIdx.x, j = t % LW, n = 2 * (blk * kAlRows + t / LW);
    if (A.state[b] != 2) {
        if (t == 0)
            *part = Top2{0.0f, 0x7fffffff, 0.0f, 0.0f};
        return;
    }
    if (t == 0)
        srank = 0x7fffffff;
    fft8::Twiddles<W> tw;
    tw.load(j);
    const float2 *T = A.S + ((size_t)b * W + n) * W;
    float2 s[8];
#pragma unroll
    for (int r = 0; r < 8; r++) {
        const int m = j + LW * r, la = m <= WS ? m : W - m;
        float2 a = T[la], c = T[W + la];
        if (m > WS) {
            a.y = -a.y;
            c.y = -c.y;
        }
        s[r] = make_float2(a.x - c.y, a.y + c.x);
    }
    fft8::fft<W, +1>(s, j, lds + (t / LW) * PB, tw);
    const int I = (n + WS) & (W - 1);
    float *M = A.mag + ((size_t)b * W + I) * W;
    Top2 best{0.0f, 0x7fffffff, 0.0f, 0.0f};
#pragma unroll
    for (int q = 0; q < 8; q++) {
        const int J = (j + LW * q + WS) & (W - 1);
        s[q] = make_float2(fabsf(s[q].x), fabsf(s[q].y));
        M[J] = s[q].x;
        M[W + J] = s[q].y;
        max2_add(best, s[q].x);
        max2_add(best, s[q].y);
    }
    const float mine = best.v1;
    best = wg_max2<256>(best, sht);
    if (best.v1 > 0.0f && mine == best.v1) {
        int rk = 0x7fffffff;
#pragma unroll
        for (int q = 0; q < 8; q++) {
            const int J = (j + LW * q + WS) & (W - 1);
            if (s[q].x == best.v1)
                rk = min(rk, surf_rank<WS>(I, J));
            if (s[q].y == best.v1)
                rk = min(rk, surf_rank<WS>(I + 1, J));
        }
        atomicMin(&srank, rk);
    }
    __syncthreads();
    if (t == 0) {
        best.r1 = srank;
        *part = best;
    }
}

// The passes up to the coarse top two (A.part, A.mag) for nb tries.
inline void launch_amp_large(st_ctx *ctx, const KPar &P, const Pts &S, const int *list, int nb, int sc, const AmpBatch &A)
{
    hipStream_t st = ctx->stream;
    const bool isf = P.im.stype == ST_SAMPLE_C64;
    if (P.noComplex && sc == 1)
        hipLaunchKernelGGL(k_amp_items<1>, dim3(nb), dim3(NT), 0, st, P, S, list, nb, kAlWS, sc, A);
    else
        hipLaunchKernelGGL(k_amp_items<0>, dim3((nb + NT - 1) / NT), dim3(NT), 0, st, P, S, list, nb, kAlWS, sc, A);
    const dim3 gr(kAlWS / 16, 2 * nb);
    if (isf)
        hipLaunchKernelGGL(k_ampl_rows<ST_SAMPLE_C64>, gr, dim3(256), 0, st, P, S, list, nb, sc, A);
    else
        hipLaunchKernelGGL(k_ampl_rows<ST_SAMPLE_CI16>, gr, dim3(256), 0, st, P, S, list, nb, sc, A);
    hipLaunchKernelGGL(k_ampl_cols, dim3(kAlWS / kAlCols, 2 * nb), dim3(512), 0, st, nb, A);
    hipLaunchKernelGGL(k_ampl_det, dim3(kAlBlocks, nb), dim3(256), 0, st, nb, isf ? 1 : 0, A);
    hipLaunchKernelGGL(k_amp_stat, dim3(nb), dim3(64), 0, st, A.dpart, kAlBlocks, kAlW, kAlW, A.state, A.mean);
    hipLaunchKernelGGL(k_ampl_fwd, dim3(kAlBlocks, nb), dim3(256), 0, st, A);
    hipLaunchKernelGGL(k_ampl_cross, dim3(kAlWS / kAlCols, nb), dim3(512), kAlLdsCross, st, A);
    hipLaunchKernelGGL(k_amp_psum, dim3((nb + 127) / 128), dim3(128), 0, st, A.ppart, kAlBlocks, nb, kAlW, kAlW, A.state,
                       A.p);
    hipLaunchKernelGGL(k_ampl_mag, dim3(kAlMagBlocks, nb), dim3(256), 0, st, A);
}
