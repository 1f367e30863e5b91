// Register transforms of length N = 128, 192, 256, 384, 512, 768 on
// LANES = N / V adjacent lanes of one wave, V = 8 values per lane (powers of
// two) or 24 (three times a power of two): lane j holds x[j + LANES i],
// i = 0 .. V - 1, on entry and on return.  Stages, twiddle values and product
// contractions are those of stfft::Engine's plan for N (as fft8, whose exchange
// through a private LDS region of N + N / 8 elements it shares), so the
// results are bit-identical to its LDS passes.
#pragma once

#include "st_fft8.h"

namespace fftn {

// exp(-2 pi i e / 512) and exp(-2 pi i e / 768)
extern __constant__ float2 c_tw512[512], c_tw768[768];

template <int N>
struct Plan {
    static_assert(N == 128 || N == 192 || N == 256 || N == 384 || N == 512 || N == 768, "transform length");
    static constexpr int V = N % 3 ? 8 : 24, LANES = N / V, REGION = N + N / 8;
};

inline bool covered(int n) { return n == 128 || n == 192 || n == 256 || n == 384; }

// Fills tw[e] = exp(-2 pi i e / L), e < L, by all threads of a workgroup (a
// barrier follows before its use).  The stages read their twiddles from there:
// a lane's own values come from up to 64 places of the table, which LDS serves
// several times as fast as the vector caches do.
template <int L>
__device__ inline void table(float2 *tw)
{
    for (int e = threadIdx.x; e < L; e += blockDim.x)
        tw[e] = L % 3 ? c_tw512[e * (512 / L)] : c_tw768[e * (768 / L)];
}

template <int SIGN>
__device__ inline void dft3(float2 &a, float2 &b, float2 &d)
{
#pragma clang fp contract(off)
    const float c = -0.5f, s = 0.86602540378443864676f * SIGN;
    const float2 t1 = cadd(b, d), t2 = csub(b, d);
    const float2 m = make_float2(fmaf(c, t1.x, a.x), fmaf(c, t1.y, a.y));
    a = cadd(a, t1);
    b = make_float2(fmaf(-s, t2.y, m.x), fmaf(s, t2.x, m.y));
    d = make_float2(fmaf(s, t2.y, m.x), fmaf(-s, t2.x, m.y));
}

// One stage: butterflies jj = j + LANES u, u < V / R, on elements u + (V / R) r.
template <int N, int R, int NS, int SIGN, int L, class EX>
__device__ inline void stage(float2 (&v)[Plan<N>::V], int j, EX *ex, const float2 *tw)
{
    constexpr int V = Plan<N>::V, LANES = Plan<N>::LANES, NB = V / R;
    static_assert(NB * R == V, "radix divides the lane's values");
    // opaque: no stage's addresses are computed ahead and held in registers
    asm volatile("" : "+v"(j));
#pragma unroll
    for (int u = 0; u < NB; u++) {
        const int k = (j + LANES * u) % NS;
        if constexpr (NS > 1) {
#pragma unroll
            for (int r = 1; r < R; r++)
                v[u + NB * r] = fft8::mul_tw<SIGN>(v[u + NB * r], tw[k * r * (L / (NS * R))]);
        }
        if constexpr (R == 8) {
            float2 w[8];
#pragma unroll
            for (int r = 0; r < 8; r++)
                w[r] = v[u + NB * r];
            fft8::dft8<SIGN>(w);
#pragma unroll
            for (int r = 0; r < 8; r++)
                v[u + NB * r] = w[r];
        } else if constexpr (R == 4) {
            stfft::dft4(v[u], v[u + NB], v[u + 2 * NB], v[u + 3 * NB], SIGN);
        } else {
            dft3<SIGN>(v[u], v[u + NB], v[u + 2 * NB]);
        }
    }
    if constexpr (NS * R < N && NS % LANES == 0) {
        // the next stage's inputs are the lane's own: element j + LANES i moves
        // to another i
        constexpr int S = NS / LANES;
        float2 w[V];
#pragma unroll
        for (int u = 0; u < NB; u++)
#pragma unroll
            for (int q = 0; q < R; q++)
                w[(u / S) * S * R + u % S + S * q] = v[u + NB * q];
#pragma unroll
        for (int i = 0; i < V; i++)
            v[i] = w[i];
    } else if constexpr (NS * R < N) {
        // float2 regions take both parts at once, float ones the real parts, then the imaginary
        constexpr int PARTS = sizeof(EX) == sizeof(float2) ? 1 : 2;
#pragma unroll
        for (int p = 0; p < PARTS; p++) {
#pragma unroll
            for (int u = 0; u < NB; u++) {
                const int jj = j + LANES * u, at = (jj / NS) * NS * R + jj % NS;
#pragma unroll
                for (int q = 0; q < R; q++) {
                    if constexpr (PARTS == 1)
                        ex[fft8::pad(at + q * NS)] = v[u + NB * q];
                    else
                        ex[fft8::pad(at + q * NS)] = p == 0 ? v[u + NB * q].x : v[u + NB * q].y;
                }
            }
            fft8::wave_sync();
#pragma unroll
            for (int i = 0; i < V; i++) {
                if constexpr (PARTS == 1)
                    v[i] = ex[fft8::pad(j + LANES * i)];
                else
                    (p == 0 ? v[i].x : v[i].y) = ex[fft8::pad(j + LANES * i)];
            }
            fft8::wave_sync();
        }
    }
}

// tw: table<L>, L a multiple of N.
template <int N, int SIGN, int L, class EX>
__device__ inline void fft(float2 (&v)[Plan<N>::V], int j, EX *ex, const float2 *tw)
{
    static_assert(L % N == 0, "table of twiddles");
    stage<N, 8, 1, SIGN, L>(v, j, ex, tw);
    if constexpr (N == 128) {
        stage<N, 4, 8, SIGN, L>(v, j, ex, tw);
        stage<N, 4, 32, SIGN, L>(v, j, ex, tw);
    } else if constexpr (N == 192) {
        stage<N, 8, 8, SIGN, L>(v, j, ex, tw);
        stage<N, 3, 64, SIGN, L>(v, j, ex, tw);
    } else if constexpr (N == 256) {
        stage<N, 8, 8, SIGN, L>(v, j, ex, tw);
        stage<N, 4, 64, SIGN, L>(v, j, ex, tw);
    } else if constexpr (N == 384) {
        stage<N, 4, 8, SIGN, L>(v, j, ex, tw);
        stage<N, 4, 32, SIGN, L>(v, j, ex, tw);
        stage<N, 3, 128, SIGN, L>(v, j, ex, tw);
    } else if constexpr (N == 512) {
        stage<N, 8, 8, SIGN, L>(v, j, ex, tw);
        stage<N, 8, 64, SIGN, L>(v, j, ex, tw);
    } else {
        stage<N, 8, 8, SIGN, L>(v, j, ex, tw);
        stage<N, 4, 64, SIGN, L>(v, j, ex, tw);
        stage<N, 3, 256, SIGN, L>(v, j, ex, tw);
    }
}

}  // namespace fftn
