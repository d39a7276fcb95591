// Known-answer kernel for the in-range FP64 operations of fenice_amd/csrc/fvg_device.hpp and CellQuot of k_cells, compiled
// from the same headers with the library's flags: element k of out is form(a[k], b[k]). Used by test_gpu_arith.py.
#include "../fenice_amd/csrc/fvg_kernels_impl.hpp"

using namespace fvg;

namespace {

enum { DVP = 0, DVX = 1, SQX = 2, RECIP_RHO = 3, CELL_QUOT = 4, CELL_H2 = 5, BY_CONST = 6, QUOT6 = 7, DIV = 8, SQRT = 9 };

__global__ __launch_bounds__(256) void k_arith(int form, const double* a, const double* b, long long n, double* out, int* bad) {
    const long long k = (long long)blockIdx.x * 256 + threadIdx.x;
    if (k >= n) return;
    const double x = a[k], y = b[k];
    double r = 0.0;
    int f = 0;
    switch (form) {
    case DVP: r = dvp<true>(x, y); break;
    case DVX: r = dvx<true>(x, y); break;
    case SQX: r = sqx<true>(x); break;
    case RECIP_RHO: r = recip_rho(x); break;
    case CELL_QUOT:
    case CELL_H2: {   // bad: the quotient is not used
        CellQuot q(form == CELL_QUOT ? y : 1.0);
        r = form == CELL_QUOT ? q.by_rho(x) : q.by_h2(x, y, 1.0 / y);
        f = q.bad;
        break;
    }
    case DIV: r = x / y; break;   // the compiler's
    case SQRT: r = sqrt(x); break;
    case BY_CONST: r = by_const<true>(x, y, 1.0 / y); break;
    default: r = quot6(x); break;
    }
    out[k] = r;
    bad[k] = f;
}

}   // namespace

// 0, or the HIP error
extern "C" int arith_check(int form, const double* a, const double* b, long long n, double* out, int* bad) {
    double *da = nullptr, *db = nullptr, *dout = nullptr;
    int* dbad = nullptr;
    const size_t bytes = sizeof(double) * (size_t)n;
    hipError_t e = hipMalloc(&da, bytes);
    if (e == hipSuccess) e = hipMalloc(&db, bytes);
    if (e == hipSuccess) e = hipMalloc(&dout, bytes);
    if (e == hipSuccess) e = hipMalloc(&dbad, sizeof(int) * (size_t)n);
    if (e == hipSuccess) e = hipMemcpy(da, a, bytes, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(db, b, bytes, hipMemcpyHostToDevice);
    if (e == hipSuccess) {
        hipLaunchKernelGGL(k_arith, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, nullptr, form, da, db, n, dout, dbad);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipMemcpy(out, dout, bytes, hipMemcpyDeviceToHost);
    if (e == hipSuccess) e = hipMemcpy(bad, dbad, sizeof(int) * (size_t)n, hipMemcpyDeviceToHost);
    hipFree(da);
    hipFree(db);
    hipFree(dout);
    hipFree(dbad);
    return (int)e;
}
