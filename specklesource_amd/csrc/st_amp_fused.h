// Fused amplitude tries for square patches of ws = 16, 32, 64 samples
// (included by st_strack.hip inside its anonymous namespace).
//
// getAmpPatches + ampMatch (speckleTrack.c:398-484, 1006-1189): both patches
// interpolated to W = 2 ws, detected, and their W x W amplitudes correlated.
// One workgroup takes one try at a time and keeps everything between the
// windows and the block around the peak in LDS and registers: the transforms
// are fft8's (eight values per lane, N / 8 lanes per row or column), in the
// order and with the arithmetic of the staged kernels (k_amp_colx ..
// k_amp_rowmag), so the surface is theirs bit for bit.
//
// LDS holds W rows of W + W / 8 elements.  A row is at once the storage of a
// row (or the values of a column while it is transformed) and the private
// exchange region of the lane group that works on it:
//   A  range transforms of the ws rows of both windows
//   B  azimuth transforms of the 2 ws columns, rotation by the Doppler shift,
//      zero pad to W, azimuth inverse
//   C  range pad and inverse of the W rows, one image after the other, from
//      the four non-zero values each lane has of both; amplitudes, zero test,
//      sums stay with the lane
//   D  means removed, range transform of v1 + i v2: the lane has the very
//      elements the transform starts from
//   E  azimuth transforms; the spectra separated from Z(k, l) and Z(-k, -l),
//      F1 conj(F2), azimuth inverse of the columns l <= W / 2 (the
//      correlation is real)
//   F  range inverse, two rows per transform, |s|, coarse top two
// The refinement and the width samples follow in k_cpx_refine.
//
// Bound: FP32 VALU issue (a VALU instruction on 83 % of the SIMDs' cycles at
// ws = 32, on 76 % at 64).  Per try, 28 665 tries at ws = 32: 34 ns (the staged
// kernels 143 ns); 9 744 at ws = 64: 164 ns (600 ns).

// Workgroup geometry for W = 2 ws: U = 2 units of eight values per lane, so
// that the half-size passes (A, B, F) occupy every lane with one.  Measured at
// ws = 32, 28 665 tries: four 4-wave workgroups per CU 35 ns per try, two
// 8-wave ones (one unit per lane) 65 ns.
template <int WS>
struct AmpGeom {
    static constexpr int W = 2 * WS, UNITS = W * W / 8, U = 2, NTH = UNITS / U;
    static constexpr int PB = W + W / 8 + 1;  // row pitch: odd, so that the rows of a column access spread over the banks
    static constexpr size_t LDS = (size_t)W * PB * sizeof(float2);
    // waves per SIMD asked of the compiler: what the LDS allows (one 16-wave
    // workgroup per CU at ws = 64, four 4-wave ones at 32, sixteen 1-wave ones
    // at 16)
    static constexpr int OCC = 4;
};

// Power |z|^2 scale and amplitude of H interpolated samples; bit-identical to
// sqrtf (short form when no value of the wave is below 2^-96).
__device__ inline void amp_detect(const float2 (&y)[8], float scale, float (&x)[8], float (&a)[8])
{
    constexpr int H = 8;
#pragma unroll
    for (int j = 0; j < H; j++) {
#pragma clang fp contract(off)
        x[j] = (y[j].x * y[j].x + y[j].y * y[j].y) * scale;
    }
    if (!sqrt_needs_full(x)) {
#pragma unroll
        for (int j = 0; j < H; j++)
            a[j] = sqrt_rn_normal(x[j]);
    } else {
#pragma unroll
        for (int j = 0; j < H; j++)
            a[j] = sqrtf(x[j]);
    }
}

// Sums of N doubles (and a count) over the workgroup: wave sums into LDS; the
// caller's barrier; then every thread adds them up in wave order.
struct AmpSums {
    double v[4];
    int n;
};

template <int N>
__device__ inline void amp_sums_put(double (&s)[N], AmpSums *sh)
{
    group_sum_last<64>(s);
    if ((threadIdx.x & 63) == 63)
#pragma unroll
        for (int k = 0; k < N; k++)
            sh[threadIdx.x >> 6].v[k] = s[k];
}

__device__ inline void amp_count_put(int n, AmpSums *sh)
{
    int c[1] = {n};
    group_sum_last<64>(c);
    if ((threadIdx.x & 63) == 63)
        sh[threadIdx.x >> 6].n = c[0];
}

template <int NW, int N>
__device__ inline AmpSums amp_sums_get(const AmpSums *sh)
{
    AmpSums r = sh[0];
#pragma unroll
    for (int w = 1; w < NW; w++) {
#pragma unroll
        for (int k = 0; k < N; k++)
            r.v[k] += sh[w].v[k];
        r.n += sh[w].n;
    }
    return r;
}

// A try's windows: getAmpPatches' corners and bounds, the same on every lane.
struct AmpItem {
    int pt, r1, a1, r2, a2, ok;
};

__device__ inline AmpItem amp_item(const KPar &P, const Pts &S, int pt, int ws, int sc)
{
    AmpItem o;
    o.pt = __builtin_amdgcn_readfirstlane(pt);
    const int i = o.pt / P.nR, j = o.pt - (o.pt / P.nR) * P.nR;
    o.a1 = P.aStart + i * P.deltaA - P.wA / 2 * sc;
    o.r1 = P.rStart + j * P.deltaR - P.wR / 2 * sc;
    o.r2 = __builtin_amdgcn_readfirstlane(o.r1 + (S.r2[o.pt] - S.r1[o.pt]));
    o.a2 = __builtin_amdgcn_readfirstlane(o.a1 + (S.a2[o.pt] - S.a1[o.pt]));
    o.ok = in_bounds(o.r1, o.a1, ws, ws, P.im.nr1, P.im.na1) && in_bounds(o.r2, o.a2, ws, ws, P.im.nr2, P.im.na2);
    return o;
}

// The result of a try that leaves before the correlation (st 0: out of
// bounds, 1: no data).
__device__ inline void amp_no_match(const AmpBatch &A, int it, int st)
{
    A.state[it] = (uint8_t)st;
    A.have[it] = 0;
    A.res[it].lmOk = 0;
    A.res[it].I = A.res[it].J = -1000;
}

// Doppler shift of a window pair, in units of ws, from both windows' lag sums
// (re, im), as estDopCarrier1 and its rounding give it: none for a sum that is
// zero or not a number.
template <int WS>
__device__ inline int amp_doppler(const double (*z)[2])
{
    const double all = z[0][0] + z[0][1] + z[1][0] + z[1][1];  // finite samples give finite sums
    return all == all ? doppler_round(z[0][0], z[0][1], z[1][0], z[1][1], WS, c_root256) : 0;
}

// The coarse peak of a try or its rejection near the border (findCPeak), and
// the cells of the block around it that k_cpx_refine reads, from M(I, J).
template <int NTH, class Surf>
__device__ inline void amp_peak_out(const AmpBatch &A, int it, const Top2 &best, int W, Surf M)
{
    PeakRes *res = &A.res[it];
    const int t = threadIdx.x, WS = W / 2;
    int I = -1000, J = -1000;
    float raw = 0.f;
    if (best.r1 != 0x7fffffff) {
        const int q = best.r1 & 3, ij = best.r1 >> 2, i0 = ij / WS, j0 = ij - (ij / WS) * WS;
        I = (q == 0 || q == 3) ? i0 : i0 + WS;
        J = (q == 0 || q == 2) ? j0 : j0 + WS;
        raw = best.v1;
    }
    const bool edge = I < NFAST / 2 || I > W - NFAST / 2 || J < NFAST / 2 || J > W - NFAST / 2;
    if (t == 0) {
        res->gap = raw > 0 ? (raw - best.v2) / raw : 0.f;
        res->snr = best.sum > 0.0f ? best.v1 * (float)(W * W) / best.sum : 0.0f;
        res->lmOk = 0;
        res->fi = res->fj = -1;
        res->fineMax = 0;
        res->fineGap = 0;
        res->I = edge ? -1000 : I;
        res->J = edge ? -1000 : J;
        res->raw = edge ? -1.f : raw;
    }
    if (!edge) {
        float *nb = A.nb + (size_t)it * kNbc;
        for (int e = t; e < kNbc; e += NTH) {
            const int ri = I - kNb / 2 + kNbMap.ri[e], ci = J - kNb / 2 + kNbMap.ci[e];
            nb[e] = (ri >= 0 && ri < W && ci >= 0 && ci < W) ? M(ri, ci) : 0.0f;
        }
    }
}

// DOP: the try estimates its own Doppler shift (-noComplex, small window)
// and leaves it for the doubled one.  Persistent over the work list in
// XCD-contiguous order (as k_cpx_fused).
template <int WS, int STYPE, int DOP>
__global__ void __launch_bounds__(AmpGeom<WS>::NTH) __attribute__((amdgpu_waves_per_eu(AmpGeom<WS>::OCC, 8)))
k_amp_fused(KPar P, Pts S, const int *__restrict__ list, int count, int sc, AmpBatch A)
{
    using G = AmpGeom<WS>;
    constexpr int W = G::W, NTH = G::NTH, NW = NTH / 64, U = G::U, PB = G::PB;
    constexpr int LW = W / 8, LS = WS / 8;  // lanes per W-point and per ws-point transform
    constexpr int UH = U / 2;               // units per lane of the half-size passes
    static_assert(UH == 1, "the Doppler sums of a window are complete after one turn");
    constexpr int SPAN = WS == 16 ? 32 : 64, NP = 2 * WS * LS / SPAN;  // partials of the Doppler sums, half per window
    constexpr bool isf = STYPE == ST_SAMPLE_C64;
    extern __shared__ float2 lds[];  // [W][PB]
    __shared__ AmpSums shs[NW], shp[NW];
    __shared__ Top2 sht[NW];
    __shared__ double stp[NP][4];  // Doppler partials: sums of the samples, of the lag products
    __shared__ int sAz, srank;
    const int Gr = gridDim.x, Q = Gr / 8;
    const int base = (Gr % 8 == 0) ? (blockIdx.x % 8) * Q + blockIdx.x / 8 : blockIdx.x;
    // the thread index behind an opaque copy, taken anew in every pass: the
    // compiler would otherwise keep the addresses of all passes in registers
    auto tid = [] {
        int x = threadIdx.x;
        asm volatile("" : "+v"(x));
        return x;
    };
    auto row = [&](int n) { return lds + n * PB; };
    fft8::Twiddles<W> twW;
    twW.load(threadIdx.x % LW);
    for (int it = base; it < count; it += Gr) {
        const int t = threadIdx.x;
        const AmpItem w = amp_item(P, S, list[it], WS, sc);
        if (!w.ok) {
            if (t == 0)
                amp_no_match(A, it, 0);
            continue;
        }
        fft8::Twiddles<WS> twS;
        twS.load(tid() % LS);
        // ---- A: unit (g, a, j): row a of window g
        {
#pragma unroll
            for (int i = 0; i < UH; i++) {
                const int u = tid() + i * NTH, j = u % LS, a = u / LS % WS, g = u / (LS * WS);
                const void *img = g ? P.im.img2 : P.im.img1;
                const int nr = g ? P.im.nr2 : P.im.nr1;
                const size_t o = (size_t)((g ? w.a2 : w.a1) + a) * nr + (g ? w.r2 : w.r1) + j;
                auto load = [&](size_t e) {
                    if constexpr (isf) {
                        return __builtin_bit_cast(float2, ((const gu64 *)img)[e]);
                    } else {
                        const unsigned v = ((const gu32 *)img)[e];
                        return make_float2((float)(short)(v & 0xffffu), (float)(short)(v >> 16));
                    }
                };
                float2 v[8];
#pragma unroll
                for (int r = 0; r < 8; r++)
                    v[r] = load(o + LS * r);
                if constexpr (DOP != 0) {
                    // The mean first, then the lag products of what is left, as
                    // doppler_shift does (one pass over the products with the mean
                    // still in them loses the mean's share of the digits).  A wave's
                    // units are of one window (ws^2 / 8 each).
                    const bool lag = a > 0;
                    const int e = u / SPAN;
                    const bool last = (t & (SPAN - 1)) == SPAN - 1;
                    float2 pv[8];
#pragma unroll
                    for (int r = 0; r < 8; r++)
                        pv[r] = lag ? load(o - nr + LS * r) : make_float2(0.f, 0.f);
                    double acc[2] = {0, 0};
#pragma unroll
                    for (int r = 0; r < 8; r++) {
                        acc[0] += v[r].x;
                        acc[1] += v[r].y;
                    }
                    group_sum_last<SPAN>(acc);
                    if (last) {
                        stp[e][0] = acc[0];
                        stp[e][1] = acc[1];
                    }
                    __syncthreads();
                    double m[2] = {0, 0};
#pragma unroll
                    for (int k = 0; k < NP / 2; k++) {
                        m[0] += stp[g * (NP / 2) + k][0];
                        m[1] += stp[g * (NP / 2) + k][1];
                    }
                    constexpr double perSample = 1.0 / ((double)WS * WS);  // a power of two: exact
                    m[0] *= perSample;
                    m[1] *= perSample;
                    acc[0] = acc[1] = 0;
                    if (lag)
#pragma unroll
                        for (int r = 0; r < 8; r++) {
                            const double ar = v[r].x - m[0], ai = v[r].y - m[1], br = pv[r].x - m[0], bi = pv[r].y - m[1];
                            acc[0] += ar * br + ai * bi;
                            acc[1] += ai * br - ar * bi;
                        }
                    group_sum_last<SPAN>(acc);
                    if (last) {
                        stp[e][2] = acc[0];
                        stp[e][3] = acc[1];
                    }
                }
                float2 *ex = row(a) + g * (WS + WS / 8);
                fft8::fft<WS, -1>(v, j, ex, twS);
#pragma unroll
                for (int q = 0; q < 8; q++)
                    ex[j + LS * q] = v[q];
            }
        }
        __syncthreads();
        if (t == 0) {
            int az = S.azUse[w.pt];
            if constexpr (DOP != 0) {
                double z[2][2] = {{0, 0}, {0, 0}};
                for (int e = 0; e < NP; e++)
                    for (int k = 0; k < 2; k++)
                        z[e / (NP / 2)][k] += stp[e][2 + k];
                az = (int)((float)amp_doppler<WS>(z) * (float)P.wA / (float)WS);
                S.azUse[w.pt] = az;
            }
            sAz = (int)((float)az * (float)WS / (float)P.wA);
            srank = 0x7fffffff;
        }
        // ---- B: unit (g, l, j): column l of window g's row spectra
        {
            float2 v[UH][8];
            {
#pragma unroll
                for (int i = 0; i < UH; i++) {
                    const int u = tid() + i * NTH, j = u % LS, c = u / LS, at = c % WS + (c / WS) * (WS + WS / 8);
#pragma unroll
                    for (int r = 0; r < 8; r++)
                        v[i][r] = row(j + LS * r)[at];
                }
            }
            __syncthreads();
            {
#pragma unroll
                for (int i = 0; i < UH; i++) {
                    const int u = tid() + i * NTH, j = u % LS, c = u / LS;
                    fft8::fft<WS, -1>(v[i], j, row(c), twS);
#pragma unroll
                    for (int q = 0; q < 8; q++)
                        row(c)[j + LS * q] = v[i][q];
                }
            }
        }
        __syncthreads();
        {
            // unit (column c, j): rotated and padded to W (elements 2 .. 5 are the pad's zeros)
            const int az = sAz;
            float2 v[U][8];
#pragma unroll
            for (int i = 0; i < U; i++) {
                const int u = tid() + i * NTH, j = u % LW, c = u / LW;
#pragma unroll
                for (int r = 0; r < 8; r++) {
                    v[i][r] = make_float2(0.f, 0.f);
                    if (r < 2 || r > 5)
                        v[i][r] = row(c)[(j + LW * r + az) & (WS - 1)];
                }
            }
            fft8::wave_sync();
#pragma unroll
            for (int i = 0; i < U; i++) {
                const int u = tid() + i * NTH;
                fft8::fft<W, +1>(v[i], u % LW, row(u / LW), twW);
            }
            __syncthreads();
#pragma unroll
            for (int i = 0; i < U; i++) {
                const int u = tid() + i * NTH, j = u % LW, c = u / LW, at = c;  // T[n][g][la] at g ws + la
#pragma unroll
                for (int q = 0; q < 8; q++)
                    row(j + LW * q)[at] = v[i][q];
            }
        }
        __syncthreads();
        // ---- C: unit (n, j): both images' row n; then D
        float v1[U][8], v2[U][8];
        double sm[4] = {0, 0, 0, 0};
        int nz = 0;
        {
            constexpr float scale = (float)(1. / ((double)WS * WS * WS * WS * 8));
            const float thr = isf ? 1.0e-15f : 1.0e-6f;
#pragma unroll
            for (int i = 0; i < U; i++) {
                const int u = tid() + i * NTH, j = u % LW;
                float2 *ex = row(u / LW);
                float2 p[2][8];
#pragma unroll
                for (int g = 0; g < 2; g++)
#pragma unroll
                    for (int r = 0; r < 8; r++)
                        p[g][r] = r < 2   ? ex[g * WS + j + LW * r]
                                  : r > 5 ? ex[g * WS + j + LW * r - WS]
                                          : make_float2(0.f, 0.f);
                fft8::wave_sync();
                unsigned mask = 0;  // cells where either image is below the threshold
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
                fft8::fft<W, +1>(p[0], j, ex, twW);
                detect(p[0], v1[i], sm[0], sm[2]);
                __builtin_amdgcn_sched_barrier(0);
                fft8::fft<W, +1>(p[1], j, ex, twW);
                detect(p[1], v2[i], sm[1], sm[3]);
                nz += __popc(mask);
            }
        }
        amp_sums_put(sm, shs);
        amp_count_put(nz, shs);
        __syncthreads();
        const AmpSums tot = amp_sums_get<NW, 4>(shs);
        constexpr double NWW = (double)W * (double)W;
        if (tot.n > 20 || tot.v[0] < 1.0e-6 || tot.v[1] < 1.0e-6) {
            if (t == 0)
                amp_no_match(A, it, 1);
            __syncthreads();
            continue;
        }
        {
            const double m1 = tot.v[2] / NWW, m2 = tot.v[3] / NWW;
            double pw[2] = {0, 0};
#pragma unroll
            for (int i = 0; i < U; i++) {
                const int u = tid() + i * NTH, j = u % LW;
                float2 *ex = row(u / LW);
                float2 x[8];
#pragma unroll
                for (int r = 0; r < 8; r++) {
#pragma clang fp contract(off)
                    float a = v1[i][r], b = v2[i][r];
                    if (a > 1.0e-20)
                        a = (float)(a - m1);
                    b = (float)(b - m2);
                    pw[0] += a * a;
                    pw[1] += b * b;
                    x[r] = make_float2(a, b);
                }
                fft8::fft<W, -1>(x, j, ex, twW);
#pragma unroll
                for (int q = 0; q < 8; q++)
                    ex[j + LW * q] = x[q];
            }
            amp_sums_put(pw, shp);
        }
        __syncthreads();
        if (t == 0) {
            const AmpSums pw = amp_sums_get<NW, 2>(shp);
            A.p[2 * it] = pw.v[0] / NWW;
            A.p[2 * it + 1] = pw.v[1] / NWW;
            A.state[it] = 2;
            A.have[it] = 1;
        }
        // ---- E: unit (l, j): column l
        {
            float2 v[U][8];
#pragma unroll
            for (int i = 0; i < U; i++) {
                const int u = tid() + i * NTH, j = u % LW, l = u / LW;
#pragma unroll
                for (int r = 0; r < 8; r++)
                    v[i][r] = row(j + LW * r)[l];
            }
            __syncthreads();
#pragma unroll
            for (int i = 0; i < U; i++) {
                const int u = tid() + i * NTH, j = u % LW, l = u / LW;
                fft8::fft<W, -1>(v[i], j, row(l), twW);
#pragma unroll
                for (int q = 0; q < 8; q++)
                    row(l)[j + LW * q] = v[i][q];
            }
            __syncthreads();
#pragma unroll
            for (int i = 0; i < U; i++) {
                const int u = tid() + i * NTH, j = u % LW, l = u / LW;
                const float2 *m = row((W - l) & (W - 1));
                if (l <= WS)
#pragma unroll
                    for (int q = 0; q < 8; q++)
                        v[i][q] = amp_cross_sep(v[i][q], m[(W - j - LW * q) & (W - 1)]);
            }
            __syncthreads();
#pragma unroll
            for (int i = 0; i < U; i++) {
                const int u = tid() + i * NTH, j = u % LW, l = u / LW;
                if (l <= WS)
                    fft8::fft<W, +1>(v[i], j, row(l), twW);
            }
            __syncthreads();
#pragma unroll
            for (int i = 0; i < U; i++) {
                const int u = tid() + i * NTH, j = u % LW, l = u / LW;
                if (l <= WS)
#pragma unroll
                    for (int q = 0; q < 8; q++)
                        row(j + LW * q)[l] = v[i][q];
            }
        }
        __syncthreads();
        // ---- F: unit (q, j): rows 2 q and 2 q + 1
        Top2 best{0.0f, 0x7fffffff, 0.0f, 0.0f};
        float2 s[UH][8];
        {
#pragma unroll
            for (int i = 0; i < UH; i++) {
                const int u = tid() + i * NTH, j = u % LW, n = 2 * (u / LW);
#pragma unroll
                for (int r = 0; r < 8; r++) {
                    const int m = j + LW * r, la = m <= WS ? m : W - m;
                    float2 a = row(n)[la], c = row(n + 1)[la];
                    if (m > WS) {
                        a.y = -a.y;
                        c.y = -c.y;
                    }
                    s[i][r] = make_float2(a.x - c.y, a.y + c.x);
                }
                fft8::wave_sync();
                fft8::fft<W, +1>(s[i], j, row(n), twW);
#pragma unroll
                for (int q = 0; q < 8; q++) {
                    s[i][q] = make_float2(fabsf(s[i][q].x), fabsf(s[i][q].y));
                    max2_add(best, s[i][q].x);
                    max2_add(best, s[i][q].y);
                }
            }
        }
        __syncthreads();  // the rows are read: the LDS takes the fftshifted surface
        float *Ms = (float *)lds;
        auto cell = [&](int u, int q, int &I, int &J) {
            I = (2 * (u / LW) + WS) & (W - 1);
            J = (u % LW + LW * q + WS) & (W - 1);
        };
        {
#pragma unroll
            for (int i = 0; i < UH; i++)
#pragma unroll
                for (int q = 0; q < 8; q++) {
                    int I, J;
                    cell(t + i * NTH, q, I, J);
                    Ms[I * W + J] = s[i][q].x;
                    Ms[(I + 1) * W + J] = s[i][q].y;
                }
        }
        const float mine = best.v1;
        best = wg_max2<NTH>(best, sht);
        if (best.v1 > 0.0f && mine == best.v1) {
            // the maximum's rank: its holders look it up among their own cells
            int rk = 0x7fffffff;
#pragma unroll 1
            for (int e = 0; e < UH * 8; e++) {
                int I, J;
                cell(t + (e >> 3) * NTH, e & 7, I, J);
                if (Ms[I * W + J] == best.v1)
                    rk = min(rk, surf_rank<WS>(I, J));
                if (Ms[(I + 1) * W + J] == best.v1)
                    rk = min(rk, surf_rank<WS>(I + 1, J));
            }
            atomicMin(&srank, rk);
        }
        __syncthreads();
        best.r1 = srank;
        amp_peak_out<NTH>(A, it, best, W, [&](int I, int J) { return Ms[I * W + J]; });
        __syncthreads();
    }
}

template <int WS, int STYPE, int DOP>
void launch_amp_fused_k(st_ctx *ctx, const KPar &P, const Pts &S, const int *list, int count, int sc, const AmpBatch &A)
{
    using G = AmpGeom<WS>;
    int perCU = 0, ncu = 0;
    ST_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&perCU, k_amp_fused<WS, STYPE, DOP>, G::NTH, G::LDS));
    ST_HIP(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, ctx->device));
    const int grid = std::max(1, std::min(count, std::max(1, perCU) * ncu));
    hipLaunchKernelGGL((k_amp_fused<WS, STYPE, DOP>), dim3(grid), dim3(G::NTH), G::LDS, ctx->stream, P, S, list, count,
                       sc, A);
    ST_HIP(hipGetLastError());
}

template <int WS>
void launch_amp_fused(st_ctx *ctx, const KPar &P, const Pts &S, const int *list, int count, int sc, const AmpBatch &A)
{
    const bool dop = P.noComplex && sc == 1;
    if (P.im.stype == ST_SAMPLE_C64)
        dop ? launch_amp_fused_k<WS, ST_SAMPLE_C64, 1>(ctx, P, S, list, count, sc, A)
            : launch_amp_fused_k<WS, ST_SAMPLE_C64, 0>(ctx, P, S, list, count, sc, A);
    else
        dop ? launch_amp_fused_k<WS, ST_SAMPLE_CI16, 1>(ctx, P, S, list, count, sc, A)
            : launch_amp_fused_k<WS, ST_SAMPLE_CI16, 0>(ctx, P, S, list, count, sc, A);
}
