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

#pragma clang fp contract(off)
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
