// Device results of the short forms in st_math.h and of the Gaussian fit's sums,
// for tests/test_gpu_math.py.
// Host arrays in and out; every entry returns 0 or the HIP error.
#include <hip/hip_runtime.h>

#include "st_math.h"
#include "st_track_common.h"

using namespace sttrack;

namespace sttrack {
__constant__ double2 c_root256[256];
__constant__ double c_refR[kFine * NFAST];
__constant__ double2 c_refB[16];
}  // namespace sttrack

namespace {

enum { DIV_BY = 0, DIV_SQRT = 1 };

__global__ void k_div(int kind, const double *x, const double *n, double *q, int count)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < count)
        q[i] = kind == DIV_BY ? div_by(x[i], n[i], 1.0 / n[i]) : div_sqrt(x[i], n[i]);
}

// Floats [lo, hi) whose short root is not the rounded FP64 one (which rounds to
// the correct float: 53 bits are more than 2 * 24 + 1).
__global__ void k_sqrt(unsigned lo, unsigned hi, unsigned long long *bad)
{
    unsigned long long n = 0;
    for (unsigned u = lo + blockIdx.x * blockDim.x + threadIdx.x; u < hi; u += gridDim.x * blockDim.x) {
        const float x = __uint_as_float(u);
        n += __float_as_uint(sqrt_rn_normal(x)) != __float_as_uint((float)sqrt((double)x));
    }
    if (n)
        atomicAdd(bad, n);
}

__global__ void k_needs_full(const float *x, int *r, int waves)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i / 64 >= waves)
        return;
    const float v[2] = {x[2 * i], x[2 * i + 1]};
    r[i] = sqrt_needs_full(v);
}

#pragma clang fp contract(off)
// solve3 in its textbook form (mrqmin's gaussj: pivots by index, whole rows).
__device__ int solve3_plain(float m[3][3], float b[3])
{
    int used[3] = {0, 0, 0};
    for (int it = 0; it < 3; it++) {
        float big = 0;
        int r = -1, c = -1;
        for (int j = 0; j < 3; j++)
            for (int k = 0; k < 3; k++)
                if (!used[j] && !used[k] && fabsf(m[j][k]) >= big) {
                    big = fabsf(m[j][k]);
                    r = j;
                    c = k;
                }
        if (r < 0)
            return 0;
        used[c] = 1;
        for (int l = 0; l < 3; l++) {
            const float t = m[r][l];
            m[r][l] = m[c][l];
            m[c][l] = t;
        }
        const float t = b[r];
        b[r] = b[c];
        b[c] = t;
        if (m[c][c] == 0.0f)
            return 0;
        const float pinv = (float)(1.0 / (double)m[c][c]);
        m[c][c] = 1.0f;
        for (int l = 0; l < 3; l++)
            m[c][l] *= pinv;
        b[c] *= pinv;
        for (int q = 0; q < 3; q++) {
            if (q == c)
                continue;
            const float d = m[q][c];
            m[q][c] = 0.0f;
            for (int l = 0; l < 3; l++)
                m[q][l] -= m[c][l] * d;
            b[q] -= b[c] * d;
        }
    }
    return 1;
}

// out [2][count][4]: whether solved, and the solution where it was, of solve3
// and of solve3_plain.  in [count][12]: matrix, right-hand side.
__global__ void k_solve3(const float *in, float *out, int count)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= count)
        return;
    for (int f = 0; f < 2; f++) {
        float m[3][3], b[3], *o = out + ((size_t)f * count + i) * 4;
        for (int j = 0; j < 3; j++) {
            for (int k = 0; k < 3; k++)
                m[j][k] = in[12 * (size_t)i + 3 * j + k];
            b[j] = in[12 * (size_t)i + 9 + j];
        }
        const int ok = f ? solve3_plain(m, b) : solve3(m, b);
        o[0] = (float)ok;
        for (int j = 0; j < 3; j++)
            o[1 + j] = ok ? b[j] : 0.0f;
    }
}

// lm_coef as the reference writes it: a division for every quotient.
__device__ void lm_coef_plain(const float *x, const float *y, const float a[3], float alpha[3][3], float beta[3],
                              float *chisq)
{
    const float sg = 0.1f, sig2i = (float)(1.0 / (double)(sg * sg));
    for (int j = 0; j < 3; j++) {
        beta[j] = 0.0f;
        for (int k = 0; k < 3; k++)
            alpha[j][k] = 0.0f;
    }
    *chisq = 0.0f;
    for (int i = 0; i < NGAUSS; i++) {
        const float s = a[2], t = x[i] - a[1];
        const float arg = (float)(0.5 * (double)t * (double)t / (double)(s * s)), ex = (float)exp(-(double)arg);
        const float ymod = a[0] * ex;
        const float d[3] = {ex, ymod * t / (s * s), ymod * t * t / (s * s * s)};
        const float dy = y[i] - ymod;
        for (int l = 0; l < 3; l++) {
            const float wt = d[l] * sig2i;
            for (int m = 0; m <= l; m++)
                alpha[l][m] += wt * d[m];
            beta[l] += dy * wt;
        }
        *chisq += dy * dy * sig2i;
    }
    for (int j = 1; j < 3; j++)
        for (int k = 0; k < j; k++)
            alpha[k][j] = alpha[j][k];
}

// out [2][count][13]: alpha, beta, chisq of lm_coef and of lm_coef_plain.
__global__ void k_lm_coef(const float *y, const float *a, float *out, int count)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= count)
        return;
    float x[NGAUSS];
    for (int k = 0; k < NGAUSS; k++)
        x[k] = (float)k;
    for (int f = 0; f < 2; f++) {
        float alpha[3][3], beta[3], chisq, *o = out + ((size_t)f * count + i) * 13;
        if (f)
            lm_coef_plain(x, y + (size_t)NGAUSS * i, a + 3 * (size_t)i, alpha, beta, &chisq);
        else
            lm_coef(x, y + (size_t)NGAUSS * i, a + 3 * (size_t)i, alpha, beta, &chisq);
        for (int j = 0; j < 3; j++) {
            for (int k = 0; k < 3; k++)
                o[3 * j + k] = alpha[j][k];
            o[9 + j] = beta[j];
        }
        o[12] = chisq;
    }
}

template <class T>
struct Buf {
    T *p = nullptr;
    explicit Buf(size_t n) { (void)hipMalloc((void **)&p, n * sizeof(T)); }
    ~Buf() { (void)hipFree(p); }
};

}  // namespace

extern "C" int mc_div(int kind, const double *x, const double *n, double *q, int count)
{
    Buf<double> dx(count), dn(count), dq(count);
    if (!dx.p || !dn.p || !dq.p)
        return hipErrorOutOfMemory;
    hipError_t e = hipMemcpy(dx.p, x, count * sizeof(double), hipMemcpyHostToDevice);
    if (e == hipSuccess)
        e = hipMemcpy(dn.p, n, count * sizeof(double), hipMemcpyHostToDevice);
    if (e == hipSuccess) {
        hipLaunchKernelGGL(k_div, dim3((count + 255) / 256), dim3(256), 0, 0, kind, dx.p, dn.p, dq.p, count);
        e = hipGetLastError();
    }
    return e == hipSuccess ? hipMemcpy(q, dq.p, count * sizeof(double), hipMemcpyDeviceToHost) : e;
}

// in [count][6]: c, mean, var, s1, s2, n
__global__ void k_ncc(const double *in, double *out, int count)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < count) {
        const double *v = in + 6 * (size_t)i;
        out[i] = ncc_value(v[0], v[1], v[2], v[3], v[4], v[5], 1.0 / v[5], 1.0 / (v[5] - 1.0));
    }
}

extern "C" int mc_ncc(const double *in, double *out, int count)
{
    Buf<double> di(6 * (size_t)count), dout(count);
    if (!di.p || !dout.p)
        return hipErrorOutOfMemory;
    hipError_t e = hipMemcpy(di.p, in, 6 * sizeof(double) * count, hipMemcpyHostToDevice);
    if (e == hipSuccess) {
        hipLaunchKernelGGL(k_ncc, dim3((count + 255) / 256), dim3(256), 0, 0, di.p, dout.p, count);
        e = hipGetLastError();
    }
    return e == hipSuccess ? hipMemcpy(out, dout.p, sizeof(double) * count, hipMemcpyDeviceToHost) : e;
}

extern "C" int mc_lm_coef(const float *y, const float *a, float *out, int count)
{
    Buf<float> dy((size_t)NGAUSS * count), da(3 * (size_t)count), dout(26 * (size_t)count);
    if (!dy.p || !da.p || !dout.p)
        return hipErrorOutOfMemory;
    hipError_t e = hipMemcpy(dy.p, y, NGAUSS * sizeof(float) * count, hipMemcpyHostToDevice);
    if (e == hipSuccess)
        e = hipMemcpy(da.p, a, 3 * sizeof(float) * count, hipMemcpyHostToDevice);
    if (e == hipSuccess) {
        hipLaunchKernelGGL(k_lm_coef, dim3((count + 127) / 128), dim3(128), 0, 0, dy.p, da.p, dout.p, count);
        e = hipGetLastError();
    }
    return e == hipSuccess ? hipMemcpy(out, dout.p, 26 * sizeof(float) * count, hipMemcpyDeviceToHost) : e;
}

extern "C" int mc_solve3(const float *in, float *out, int count)
{
    Buf<float> di(12 * (size_t)count), dout(8 * (size_t)count);
    if (!di.p || !dout.p)
        return hipErrorOutOfMemory;
    hipError_t e = hipMemcpy(di.p, in, 12 * sizeof(float) * count, hipMemcpyHostToDevice);
    if (e == hipSuccess) {
        hipLaunchKernelGGL(k_solve3, dim3((count + 127) / 128), dim3(128), 0, 0, di.p, dout.p, count);
        e = hipGetLastError();
    }
    return e == hipSuccess ? hipMemcpy(out, dout.p, 8 * sizeof(float) * count, hipMemcpyDeviceToHost) : e;
}

extern "C" int mc_sqrt(unsigned lo, unsigned hi, unsigned long long *bad)
{
    Buf<unsigned long long> d(1);
    if (!d.p || lo > hi || hi > 0xff000000u)
        return hipErrorInvalidValue;
    *bad = 0;
    hipError_t e = hipMemcpy(d.p, bad, sizeof(*bad), hipMemcpyHostToDevice);
    if (e == hipSuccess) {
        hipLaunchKernelGGL(k_sqrt, dim3(4096), dim3(256), 0, 0, lo, hi, d.p);
        e = hipGetLastError();
    }
    return e == hipSuccess ? hipMemcpy(bad, d.p, sizeof(*bad), hipMemcpyDeviceToHost) : e;
}

// x [waves][64][2] -> r [waves][64]
extern "C" int mc_needs_full(const float *x, int *r, int waves)
{
    Buf<float> dx((size_t)waves * 128);
    Buf<int> dr((size_t)waves * 64);
    if (!dx.p || !dr.p)
        return hipErrorOutOfMemory;
    hipError_t e = hipMemcpy(dx.p, x, sizeof(float) * 128 * waves, hipMemcpyHostToDevice);
    if (e == hipSuccess) {
        hipLaunchKernelGGL(k_needs_full, dim3((waves + 3) / 4), dim3(256), 0, 0, dx.p, dr.p, waves);
        e = hipGetLastError();
    }
    return e == hipSuccess ? hipMemcpy(r, dr.p, sizeof(int) * 64 * waves, hipMemcpyDeviceToHost) : e;
}
