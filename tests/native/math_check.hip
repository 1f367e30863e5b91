// Device results of the short forms in st_math.h, for tests/test_gpu_math.py.
// Host arrays in and out; every entry returns 0 or the HIP error.
#include <hip/hip_runtime.h>

#include "st_math.h"

using namespace sttrack;

namespace {

enum { DIV_BY = 0, DIV_SQRT = 1 };

__global__ void k_div(int kind, const double *x, const double *n, double *q, int count)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < count)
        q[i] = kind == DIV_BY ? div_by(x[i], n[i], 1.0 / n[i]) : div_sqrt(x[i], n[i]);
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
