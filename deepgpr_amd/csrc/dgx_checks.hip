// The value checks of a solve's inputs in one pass.
//
// A workgroup reduces its share of the three material arrays, the waveforms and
// the locations to 11 numbers, each the minimum over what it saw; the host
// takes the minimum over the workgroups (a few kB). As separate reductions these
// were some 35 launches a call, most of the time of a small solve's
// preparation, and 9 passes over a large model instead of one; the pass itself is
// bound by its bytes (12 a cell).
#include <algorithm>

#include "dgx_device.h"
#include "dgx_internal.h"

namespace dgx {

namespace {

__device__ __forceinline__ bool finite(float v) { return (__float_as_uint(v) & 0x7f800000u) != 0x7f800000u; }

template <typename I>
__device__ __forceinline__ bool inside(const void* loc, long long n, const int (&shape)[3], long long first,
                                       long long step)
{
    bool ok = true;
    for (long long x = first; x < n; x += step) {
        const I v = ((const I*)loc)[x];
        const int c = (int)(x % 3);
        ok = ok && v >= 0 && v < (I)(c == 0 ? shape[0] : (c == 1 ? shape[1] : shape[2]));
    }
    return ok;
}

__global__ __launch_bounds__(256) void k_model_checks(ModelChecks m)
{
    __shared__ float part[4][kModelChecks];
    const long long first = (long long)blockIdx.x * 256 + threadIdx.x, step = (long long)gridDim.x * 256;
    const float inf = __builtin_inff();
    float v[kModelChecks] = {1.0f, 1.0f, 1.0f, 1.0f, inf, inf, inf, inf, inf, 1.0f, 1.0f};
    for (long long x = first; x < m.cells; x += step) {
        const float e = m.er[x], s = m.se[x], u = m.mr[x];
        v[0] = finite(e) ? v[0] : 0.0f;
        v[1] = finite(s) ? v[1] : 0.0f;
        v[2] = finite(u) ? v[2] : 0.0f;
        v[4] = fminf(v[4], e);
        v[5] = fminf(v[5], s);
        v[6] = fminf(v[6], u);
        v[7] = fminf(v[7], e * u);
        v[8] = fminf(v[8], -s);
    }
    for (long long x = first; x < m.nwave; x += step) v[3] = finite(m.wave[x]) ? v[3] : 0.0f;
    const bool in_src = m.src64 ? inside<long long>(m.src, m.nsrc, m.shape, first, step)
                                : inside<int>(m.src, m.nsrc, m.shape, first, step);
    const bool in_rx = m.rx64 ? inside<long long>(m.rx, m.nrx, m.shape, first, step)
                              : inside<int>(m.rx, m.nrx, m.shape, first, step);
    v[9] = in_src ? 1.0f : 0.0f;
    v[10] = in_rx ? 1.0f : 0.0f;
#pragma unroll
    for (int c = 0; c < kModelChecks; ++c) {
#pragma unroll
        for (int d = 32; d; d >>= 1) v[c] = fminf(v[c], __shfl_xor(v[c], d));
        if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6][c] = v[c];
    }
    __syncthreads();
    if (threadIdx.x < kModelChecks) {
        const int c = threadIdx.x;
        m.out[(long long)blockIdx.x * kModelChecks + c] =
            fminf(fminf(part[0][c], part[1][c]), fminf(part[2][c], part[3][c]));
    }
}

}  // namespace

void launch_model_checks(const ModelChecks& m, int blocks, hipStream_t st)
{
    hipLaunchKernelGGL(k_model_checks, dim3((unsigned)blocks), dim3(256), 0, st, m);
}

}  // namespace dgx
