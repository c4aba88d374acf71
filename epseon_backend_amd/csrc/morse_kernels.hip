// morse_kernels.hip -- gfx950 kernels of the Morse table
//   V_i = D (1 - exp(-a (r_i - r_e)))^2
// of every potential of a fit, and of its gradient with respect to D, a, r_e.
//
// The tabulated potential of the reference is
// cpp/gpu/include/epseon/gpu/task_configurator/potential_source.hpp:43-183
// (it has no gradients).
//
// As single tensor operations the table is six passes over memory and its
// gradient fifteen and five reductions: 215 and 570 us for 256 x 50,000 points.
// Here each is one pass, bound by HBM: 24 bytes a point forward (r in; V and
// r - r_e out), 53 us = 5.8 TB/s; 16 backward (dL/dV and r - r_e in), 35 + 4 us
// = 5.3 TB/s, with the exponential computed again instead of kept.  (A copy of
// 2 GiB reaches 4.9 TB/s; of these 307 and 205 MB a part comes from the
// last-level cache.)  The
// operations on a point are those of the tensor expressions in the same order
// (no contraction); only the order of the gradient's sums is this file's own.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "epseon_hip.h"
#include "records.hpp"

namespace epseon::hip {

namespace {

// A workgroup takes this many consecutive points of one potential, eight per
// lane, loaded before the first is used: 256 x 50,000 points are 6,400
// workgroups, one potential of 7,001 points is four.
constexpr int32_t kMorseLanes = 256;
constexpr int32_t kMorsePerLane = 8;
constexpr int32_t kMorseChunk = kMorseLanes * kMorsePerLane;

// Launches stay below 2^32 lanes.
constexpr int64_t kMorseMaxBlocks = int64_t(1) << 23;

__global__ void __launch_bounds__(kMorseLanes)
    morse_table_kernel(const double* __restrict__ r, const double* __restrict__ de, const double* __restrict__ a,
                       const double* __restrict__ re, const int64_t n, const uint32_t chunks, double* __restrict__ v,
                       double* __restrict__ d)
{
    const uint32_t row = blockIdx.x / chunks;
    const int64_t i0 = static_cast<int64_t>(blockIdx.x % chunks) * kMorseChunk + threadIdx.x;
    const int64_t at = row * n;
    const double dr = de[row], ar = a[row], rr = re[row];
    double x[kMorsePerLane];
#pragma unroll
    for (int32_t q = 0; q < kMorsePerLane; ++q) {
        const int64_t i = i0 + q * kMorseLanes;
        x[q] = i < n ? r[at + i] : rr;
    }
#pragma unroll
    for (int32_t q = 0; q < kMorsePerLane; ++q) {
        const int64_t i = i0 + q * kMorseLanes;
        if (i < n) {
            const double s = x[q] - rr;
            const double y = 1.0 - exp(-ar * s);
            v[at + i] = dr * y * y;
            if (d != nullptr)
                d[at + i] = s;
        }
    }
}

// Sum over the workgroup of each of three values; thread 0 gets them.
__device__ __forceinline__ void sum3(double (&s)[3], double (*part)[3])
{
#pragma unroll
    for (int32_t w = 32; w > 0; w >>= 1)
#pragma unroll
        for (int32_t c = 0; c < 3; ++c)
            s[c] += __shfl_down(s[c], w, 64);
    if (threadIdx.x % 64 == 0)
        for (int32_t c = 0; c < 3; ++c)
            part[threadIdx.x / 64][c] = s[c];
    __syncthreads();
    if (threadIdx.x == 0)
        for (int32_t c = 0; c < 3; ++c)
            s[c] = (part[0][c] + part[1][c]) + (part[2][c] + part[3][c]);
}

// Sums over one chunk of g dV/dD, g dV/da and g dV/dr_e: out[c][block].
// With one chunk per potential these are the gradients.
__global__ void __launch_bounds__(kMorseLanes)
    morse_vjp_kernel(const double* __restrict__ g, const double* __restrict__ d, const double* __restrict__ de,
                     const double* __restrict__ a, const int64_t n, const uint32_t chunks, double* __restrict__ out)
{
    __shared__ double part[kMorseLanes / 64][3];
    const uint32_t row = blockIdx.x / chunks;
    const int64_t i0 = static_cast<int64_t>(blockIdx.x % chunks) * kMorseChunk + threadIdx.x;
    const int64_t at = row * n;
    const double dr = de[row], ar = a[row];
    double gv[kMorsePerLane], dv[kMorsePerLane];
#pragma unroll
    for (int32_t q = 0; q < kMorsePerLane; ++q) {
        const int64_t i = i0 + q * kMorseLanes;
        gv[q] = i < n ? g[at + i] : 0.0;
        dv[q] = i < n ? d[at + i] : 0.0;
    }
    double s[3] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int32_t q = 0; q < kMorsePerLane; ++q) {
        // Points past the end would add 0 times a finite value, or NaN where
        // a parameter is infinite.
        if (i0 + q * kMorseLanes < n) {
            const double e = exp(-ar * dv[q]);
            const double y = 1.0 - e;
            const double gy = gv[q] * y;
            const double t = (gy * dr + gv[q] * (dr * y)) * e;
            s[0] += gy * y;
            s[1] += t * dv[q];
            s[2] -= t * ar;
        }
    }
    sum3(s, part);
    if (threadIdx.x == 0)
        for (int64_t c = 0; c < 3; ++c)
            out[c * gridDim.x + blockIdx.x] = s[c];
}

// out[c][row] = sum over the row's chunks of part[c][row * chunks + k].
__global__ void __launch_bounds__(kMorseLanes)
    morse_sum_kernel(const double* __restrict__ part, const uint32_t chunks, double* __restrict__ out)
{
    __shared__ double lds[kMorseLanes / 64][3];
    const int64_t rows = gridDim.x, row = blockIdx.x;
    double s[3] = {0.0, 0.0, 0.0};
    for (uint32_t k = threadIdx.x; k < chunks; k += kMorseLanes)
        for (int64_t c = 0; c < 3; ++c)
            s[c] += part[(c * rows + row) * chunks + k];
    sum3(s, lds);
    if (threadIdx.x == 0)
        for (int64_t c = 0; c < 3; ++c)
            out[c * rows + row] = s[c];
}

// Chunks per potential, or 0 where the sizes don't fit one launch.
int64_t morse_chunks(const int64_t rows, const int64_t points)
{
    if (rows < 1 || points < 1 || points > (int64_t(1) << 40) || rows > kMorseMaxBlocks)
        return 0;
    const int64_t chunks = (points + kMorseChunk - 1) / kMorseChunk;
    return chunks <= kMorseMaxBlocks / rows ? chunks : 0;
}

int launched(const char* what)
{
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? EPSEON_OK : hip_fail(e, what);
}

}  // namespace

}  // namespace epseon::hip

extern "C" {

int epseon_morse_chunks(int64_t rows, int64_t points)
{
    return static_cast<int>(epseon::hip::morse_chunks(rows, points));
}

int epseon_morse_table(const double* r, const double* de, const double* a, const double* re, int64_t rows,
                       int64_t points, double* v, double* d, void* stream)
{
    using namespace epseon::hip;
    const int64_t chunks = morse_chunks(rows, points);
    if (chunks == 0 || r == nullptr || de == nullptr || a == nullptr || re == nullptr || v == nullptr)
        return fail(EPSEON_ERR_INVALID, "epseon_morse_table: null pointer or sizes that no launch takes");
    hipLaunchKernelGGL(morse_table_kernel, dim3(static_cast<unsigned>(rows * chunks)), dim3(kMorseLanes), 0,
                       static_cast<hipStream_t>(stream), r, de, a, re, points, static_cast<uint32_t>(chunks), v, d);
    return launched("epseon_morse_table");
}

int epseon_morse_vjp(const double* g, const double* d, const double* de, const double* a, int64_t rows,
                     int64_t points, double* part, double* grad, void* stream)
{
    using namespace epseon::hip;
    const int64_t chunks = morse_chunks(rows, points);
    if (chunks == 0 || g == nullptr || d == nullptr || de == nullptr || a == nullptr || grad == nullptr ||
        (chunks > 1 && part == nullptr))
        return fail(EPSEON_ERR_INVALID, "epseon_morse_vjp: null pointer or sizes that no launch takes");
    const hipStream_t s = static_cast<hipStream_t>(stream);
    const uint32_t c = static_cast<uint32_t>(chunks);
    hipLaunchKernelGGL(morse_vjp_kernel, dim3(static_cast<unsigned>(rows * chunks)), dim3(kMorseLanes), 0, s, g, d, de,
                       a, points, c, chunks > 1 ? part : grad);
    if (chunks > 1)
        hipLaunchKernelGGL(morse_sum_kernel, dim3(static_cast<unsigned>(rows)), dim3(kMorseLanes), 0, s, part, c, grad);
    return launched("epseon_morse_vjp");
}

}  // extern "C"
