// Register transforms of power-of-two length N = 16 .. 256 on N / 8 adjacent
// lanes, eight values per lane: lane j holds x[j + (N / 8) r], r = 0 .. 7, on
// entry and on return.  The stages are those of stfft::Engine's plan for N
// (the same radices, twiddles and butterfly code, so the values are the ones
// its LDS passes give); between two stages the values of the lane group go
// through a private LDS region of N + N / 8 elements (one pad element per
// eight, so that neither the stride-8 stores nor the unit-stride loads
// conflict).  A lane group never leaves its wave: no barrier.
//
// Eight values per lane keep a transform at some 50 registers, which leaves
// room for 4 to 8 waves per SIMD to hide the LDS round trips.
#pragma once

#include "st_fftlds.h"

namespace fft8 {

// exp(-2 pi i j / 256)
extern __constant__ float2 c_tw256[256];

// Orders the LDS accesses of one wave (the hardware keeps them in order; the
// fence keeps the compiler from moving them).
__device__ inline void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

__device__ inline int pad(int i) { return i + (i >> 3); }
template <int N>
constexpr int region()
{
    return N + N / 8;
}

// A lane's twiddles of the N-point transform, exp(-2 pi i k r / (8 ns)) or
// (4 ns) with the lane's k in each stage after the first; loaded once and
// kept in registers (the inverse takes their conjugates).
template <int N>
struct Twiddles {
    // 64, 256: radix 8 at ns = 8.  128: radix 4 at ns = 8 (three of them)
    static constexpr int N1 = N == 64 || N == 256 ? 7 : N == 128 ? 3 : 1;
    // the last radix-4 stage's pair of butterflies (none at 64)
    static constexpr int N2 = N == 64 ? 1 : 3;
    float2 t[N1], a[N2], b[N2];

    __device__ inline void load(int j)
    {
        if constexpr (N1 > 1) {
            constexpr int len = N == 128 ? 32 : 64;
#pragma unroll
            for (int r = 1; r <= N1; r++)
                t[r - 1] = get((j & 7) * r * (256 / len));
        }
        if constexpr (N2 > 1) {
#pragma unroll
            for (int r = 1; r <= 3; r++) {
                a[r - 1] = get(j * r * (256 / N));
                b[r - 1] = get((j + N / 8) * r * (256 / N));
            }
        }
    }

  private:
    // the opaque copy keeps the value in registers (the compiler would load it again at every use)
    __device__ static inline float2 get(int e)
    {
        float2 w = c_tw256[e];
        asm volatile("" : "+v"(w.x), "+v"(w.y));
        return w;
    }
};

// a w (SIGN < 0) or a conj(w), contracted as the engine's products are (the
// compiler is free to fuse either product of a sum; these are the forms it
// takes in all of the engine's stages).
template <int SIGN>
__device__ inline float2 mul_tw(float2 a, float2 w)
{
#pragma clang fp contract(off)
    if constexpr (SIGN < 0)
        return make_float2(fmaf(a.x, w.x, -(a.y * w.y)), fmaf(a.y, w.x, a.x * w.y));
    else
        return make_float2(fmaf(a.x, w.x, a.y * w.y), fmaf(a.y, w.x, -(a.x * w.y)));
}

// stfft::dft8: the 8-point transform with the products by exp(SIGN i pi / 4)
// and exp(SIGN 3 i pi / 4) contracted as there.
template <int SIGN>
__device__ inline void dft8(float2 (&v)[8])
{
#pragma clang fp contract(off)
    const float h = 0.70710678118654752440f, s = SIGN * h;
    float2 e0 = v[0], e1 = v[2], e2 = v[4], e3 = v[6];
    float2 o0 = v[1], o1 = v[3], o2 = v[5], o3 = v[7];
    stfft::dft4(e0, e1, e2, e3, SIGN);
    stfft::dft4(o0, o1, o2, o3, SIGN);
    o1 = make_float2(fmaf(-o1.y, s, o1.x * h), fmaf(o1.y, h, o1.x * s));
    o2 = stfft::mul_si(o2, SIGN);
    o3 = make_float2(fmaf(o3.x, -h, -(o3.y * s)), fmaf(o3.x, s, o3.y * -h));
    v[0] = cadd(e0, o0);
    v[4] = csub(e0, o0);
    v[1] = cadd(e1, o1);
    v[5] = csub(e1, o1);
    v[2] = cadd(e2, o2);
    v[6] = csub(e2, o2);
    v[3] = cadd(e3, o3);
    v[7] = csub(e3, o3);
}

// One radix-8 stage on the lane's eight values, t: their twiddles (nullptr:
// the first stage).
template <int SIGN>
__device__ inline void radix8(float2 (&v)[8], const float2 *t)
{
    if (t) {
#pragma unroll
        for (int r = 1; r < 8; r++)
            v[r] = mul_tw<SIGN>(v[r], t[r - 1]);
    }
    dft8<SIGN>(v);
}

// Two radix-4 butterflies: jj = j (even elements) and j + N / 8 (odd ones),
// inputs jj + (N / 4) r.
template <int SIGN>
__device__ inline void radix4x2(float2 (&v)[8], const float2 *a, const float2 *b)
{
    if (a) {
#pragma unroll
        for (int r = 1; r < 4; r++) {
            v[2 * r] = mul_tw<SIGN>(v[2 * r], a[r - 1]);
            v[2 * r + 1] = mul_tw<SIGN>(v[2 * r + 1], b[r - 1]);
        }
    }
    stfft::dft4(v[0], v[2], v[4], v[6], SIGN);
    stfft::dft4(v[1], v[3], v[5], v[7], SIGN);
}

// Reload the lane's inputs j + (N / 8) r after a stage has stored its outputs.
template <int N>
__device__ inline void reload(float2 (&v)[8], int j, const float2 *ex)
{
    wave_sync();
#pragma unroll
    for (int r = 0; r < 8; r++)
        v[r] = ex[pad(j + (N / 8) * r)];
    wave_sync();
}

template <int N, int SIGN>
__device__ inline void fft(float2 (&v)[8], int j, float2 *ex, const Twiddles<N> &tw)
{
    static_assert(N == 16 || N == 32 || N == 64 || N == 128 || N == 256, "transform length");
    if constexpr (N == 16) {  // 4 x 4
        radix4x2<SIGN>(v, nullptr, nullptr);
#pragma unroll
        for (int q = 0; q < 4; q++) {
            ex[pad(4 * j + q)] = v[2 * q];
            ex[pad(4 * (j + 2) + q)] = v[2 * q + 1];
        }
        reload<N>(v, j, ex);
        radix4x2<SIGN>(v, tw.a, tw.b);
    } else {
        radix8<SIGN>(v, nullptr);
#pragma unroll
        for (int q = 0; q < 8; q++)
            ex[pad(8 * j + q)] = v[q];
        reload<N>(v, j, ex);
        if constexpr (N == 32) {  // 8 x 4
            radix4x2<SIGN>(v, tw.a, tw.b);
        } else if constexpr (N == 64) {  // 8 x 8
            radix8<SIGN>(v, tw.t);
        } else if constexpr (N == 128) {  // 8 x 4 x 4
            radix4x2<SIGN>(v, tw.t, tw.t);
#pragma unroll
            for (int q = 0; q < 4; q++) {
                ex[pad((j >> 3) * 32 + (j & 7) + 8 * q)] = v[2 * q];
                ex[pad(((j + 16) >> 3) * 32 + (j & 7) + 8 * q)] = v[2 * q + 1];
            }
            reload<N>(v, j, ex);
            radix4x2<SIGN>(v, tw.a, tw.b);
        } else {  // 8 x 8 x 4
            radix8<SIGN>(v, tw.t);
#pragma unroll
            for (int q = 0; q < 8; q++)
                ex[pad((j >> 3) * 64 + (j & 7) + 8 * q)] = v[q];
            reload<N>(v, j, ex);
            radix4x2<SIGN>(v, tw.a, tw.b);
        }
    }
}

}  // namespace fft8
