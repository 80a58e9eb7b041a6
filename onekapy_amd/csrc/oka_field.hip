// oka_field.hip -- the capture-probability field after the run: Pr =
// pgrid / total_weight, its optional Gaussian smoothing, and its descending
// sort for the impact curve (oneka/visualize.py:228-233, 382-385).
//
// FP64 with contraction off: the smoothing restates the separable 1-D
// correlation of scipy.ndimage.gaussian_filter(Z, sigma, mode='constant',
// cval=0.0) (visualize.py:233) in its own operation order -- for a symmetric
// kernel of radius r with weights w[0..2r] (centre w[r]), each output is
//   acc = x[0] * w[r];  then for j = r, r - 1, ..., 1:
//   acc = acc + (x[-j] + x[+j]) * w[r - j]
// with zeros outside the grid -- along axis 0 (rows), then along axis 1.
// The weights are the caller's (the host computes them as scipy does).
#include <math.h>

#include <algorithm>

#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>

#include "oka_ctx.h"
#include "oka_internal.h"

#pragma clang fp contract(off)

using namespace oka;

namespace {

constexpr int kBlock = 256;

__global__ void __launch_bounds__(kBlock) k_probability(const double *pgrid, double total, double *z,
                                                        int64_t n)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n)
        z[i] = pgrid[i] / total;   // visualize.py:230, 382
}

// One pass of the symmetric correlation along rows (axis 0: neighbours i +- j
// in column c) or columns (axis 1: neighbours c +- j in row i).
template <int kAxis>
__global__ void __launch_bounds__(kBlock) k_correlate(const double *in, double *out, int nrows,
                                                      int ncols, const double *w, int radius)
{
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (int64_t)nrows * ncols)
        return;
    const int i = (int)(idx / ncols), c = (int)(idx - (int64_t)i * ncols);
    const int pos = kAxis == 0 ? i : c, len = kAxis == 0 ? nrows : ncols;
    const int64_t step = kAxis == 0 ? ncols : 1;
    double acc = in[idx] * w[radius];
    for (int j = radius; j >= 1; --j) {
        const double lo = pos - j >= 0 ? in[idx - j * step] : 0.0;
        const double hi = pos + j < len ? in[idx + j * step] : 0.0;
        acc = acc + (lo + hi) * w[radius - j];
    }
    out[idx] = acc;
}

// Fields of whole counts 0 .. kMaxCounted (a run's pgrid with weight 1) are
// sorted by counting: a scan for the largest, a histogram, its running sum
// from the largest count down, and each output position's count by binary
// search in it.  4e6 nodes of a 10^4-realization field: 0.29 ms of kernels, of
// which the histogram's scattered atomics take 0.23 (0.81 with an atomic per
// wave for the empty and the certain nodes, which share two addresses).
constexpr int kMaxCounted = 1 << 17;
constexpr int kScanBlock = 1024;

// found[0] = 1 if some value is not such a count, found[1] = the largest that
// is; one atomic of each a workgroup.
__global__ void __launch_bounds__(kBlock) k_find_counts(const double *pgrid, int64_t n, int *found)
{
    __shared__ int s_bad, s_top;
    if (threadIdx.x == 0)
        s_bad = s_top = 0;
    __syncthreads();
    int bad = 0, top = 0;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x) {
        const double v = pgrid[i];
        if (v >= 0.0 && v <= (double)kMaxCounted && v == rint(v) && !signbit(v))
            top = max(top, (int)v);
        else
            bad = 1;
    }
    for (int off = 32; off > 0; off >>= 1) {
        bad |= __shfl_xor(bad, off);
        top = max(top, __shfl_xor(top, off));
    }
    if ((threadIdx.x & 63) == 0) {
        atomicOr(&s_bad, bad);
        atomicMax(&s_top, top);
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        if (s_bad)
            atomicOr(&found[0], 1);
        atomicMax(&found[1], s_top);
    }
}

// hist[top - v] += the counts v.  The empty and the certain nodes, most of a
// field and each one address, are added up per workgroup first.
__global__ void __launch_bounds__(kBlock) k_count_descending(const double *pgrid, int64_t n, int top,
                                                             uint32_t *hist)
{
    __shared__ uint32_t s_end[2];
    if (threadIdx.x < 2)
        s_end[threadIdx.x] = 0;
    __syncthreads();
    uint32_t none = 0, all = 0;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x) {
        const int v = (int)pgrid[i];
        if (v == 0)
            none += 1;
        else if (v == top)
            all += 1;
        else
            atomicAdd(&hist[top - v], 1u);
    }
    for (int off = 32; off > 0; off >>= 1) {
        none += __shfl_xor(none, off);
        all += __shfl_xor(all, off);
    }
    if ((threadIdx.x & 63) == 0) {
        atomicAdd(&s_end[0], all);
        atomicAdd(&s_end[1], none);
    }
    __syncthreads();
    if (threadIdx.x < 2 && s_end[threadIdx.x])
        atomicAdd(&hist[threadIdx.x == 0 ? 0 : top], s_end[threadIdx.x]);
}

// Exclusive running sum of n words in place (one workgroup).
__global__ void __launch_bounds__(kScanBlock) k_running_sum(uint32_t *h, int n)
{
    __shared__ uint32_t part[kScanBlock];
    uint32_t base = 0;
    for (int i0 = 0; i0 < n; i0 += kScanBlock) {
        const int i = i0 + (int)threadIdx.x;
        const uint32_t v = i < n ? h[i] : 0u;
        part[threadIdx.x] = v;
        __syncthreads();
        for (int off = 1; off < kScanBlock; off <<= 1) {
            const uint32_t u = (int)threadIdx.x >= off ? part[threadIdx.x - off] : 0u;
            __syncthreads();
            part[threadIdx.x] += u;
            __syncthreads();
        }
        if (i < n)
            h[i] = base + part[threadIdx.x] - v;
        base += part[kScanBlock - 1];
        __syncthreads();
    }
}

// pr[i] = count / total of the i-th node from the largest count down; first[d]
// nodes have a count above top - d.
__global__ void __launch_bounds__(kBlock) k_expand_counts(const uint32_t *first, int top,
                                                          double total, double *pr, int64_t n)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n)
        return;
    int lo = 0, hi = top;   // the last d with first[d] <= i
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (first[mid] <= (uint32_t)i)
            lo = mid;
        else
            hi = mid - 1;
    }
    pr[i] = (double)(top - lo) / total;
}

unsigned grid_for(int64_t n) { return (unsigned)((n + kBlock - 1) / kBlock); }

}  // namespace

extern "C" {

int oka_field_smooth(oka_ctx *c, int32_t nrows, int32_t ncols, const double *pgrid,
                     double total_weight, int32_t radius, const double *weights, double *out,
                     uint32_t flags)
{
    if (!c)
        return OKA_ERR_ARG;
    if (nrows < 0 || ncols < 0 || radius < 0 || (radius > 0 && !weights))
        return fail(c, OKA_ERR_ARG, "bad field or kernel sizes");
    const int64_t n = (int64_t)nrows * ncols;
    if (n == 0)
        return OKA_OK;
    if (!pgrid || !out)
        return fail(c, OKA_ERR_ARG, "pgrid/out are NULL");
    if (!(total_weight > 0.0))
        return fail(c, OKA_ERR_RANGE, "total_weight must be > 0 (an empty capture zone)");
    HIPCHK(c, hipSetDevice(c->device));
    const void *dp;
    TRY(stage_in(c, kSlotXY, pgrid, sizeof(double) * n, flags, &dp));
    void *dz;
    TRY(stage_out(c, kSlotOut, out, sizeof(double) * n, flags, false, &dz));
    hipLaunchKernelGGL(k_probability, dim3(grid_for(n)), dim3(kBlock), 0, c->stream,
                       (const double *)dp, total_weight, (double *)dz, n);
    HIPCHK(c, hipGetLastError());
    if (radius > 0) {
        const void *dw;
        TRY(stage_in(c, kSlotWells, weights, sizeof(double) * (2 * (size_t)radius + 1), 0, &dw));
        void *tmp;
        TRY(ensure(c, kSlotBitmap, sizeof(double) * n, &tmp));
        hipLaunchKernelGGL((k_correlate<0>), dim3(grid_for(n)), dim3(kBlock), 0, c->stream,
                           (const double *)dz, (double *)tmp, nrows, ncols, (const double *)dw,
                           radius);
        HIPCHK(c, hipGetLastError());
        hipLaunchKernelGGL((k_correlate<1>), dim3(grid_for(n)), dim3(kBlock), 0, c->stream,
                           (const double *)tmp, (double *)dz, nrows, ncols, (const double *)dw,
                           radius);
        HIPCHK(c, hipGetLastError());
    }
    TRY(copy_back(c, out, dz, sizeof(double) * n, flags));
    if (!(flags & OKA_ASYNC) || !(flags & OKA_PTR_DEVICE))
        HIPCHK(c, hipStreamSynchronize(c->stream));
    return OKA_OK;
}

int oka_field_sorted_probabilities(oka_ctx *c, int64_t n, const double *pgrid, double total_weight,
                                   double *pr, uint32_t flags)
{
    if (!c)
        return OKA_ERR_ARG;
    if (n < 0 || (n > 0 && (!pgrid || !pr)))
        return fail(c, OKA_ERR_ARG, "bad field");
    if (n == 0)
        return OKA_OK;
    if (n > INT32_MAX)
        return fail(c, OKA_ERR_ARG, "more than 2^31 nodes");
    if (!(total_weight > 0.0))
        return fail(c, OKA_ERR_RANGE, "total_weight must be > 0 (an empty capture zone)");
    HIPCHK(c, hipSetDevice(c->device));
    const void *dp;
    TRY(stage_in(c, kSlotXY, pgrid, sizeof(double) * n, flags, &dp));
    void *dz, *dout;
    TRY(stage_out(c, kSlotOut, pr, sizeof(double) * n, flags, false, &dout));
    // an asynchronous call (which may be under capture) cannot look first
    if (!(flags & OKA_ASYNC) || !(flags & OKA_PTR_DEVICE)) {
        void *df, *dh;
        TRY(ensure(c, kSlotEStatus, 2 * sizeof(int), &df));
        TRY(fill_u32(c, df, 2));
        const unsigned blocks = (unsigned)std::min<int64_t>(grid_for(n), (int64_t)c->num_cu * 4);
        hipLaunchKernelGGL(k_find_counts, dim3(blocks), dim3(kBlock), 0, c->stream,
                           (const double *)dp, n, (int *)df);
        HIPCHK(c, hipGetLastError());
        int found[2] = {1, 0};
        HIPCHK(c, hipMemcpyAsync(found, df, sizeof(found), hipMemcpyDeviceToHost, c->stream));
        HIPCHK(c, hipStreamSynchronize(c->stream));
        if (!found[0]) {
            const int top = found[1];
            TRY(ensure(c, kSlotMarks, sizeof(uint32_t) * ((size_t)top + 1), &dh));
            TRY(fill_u32(c, dh, (int64_t)top + 1));
            hipLaunchKernelGGL(k_count_descending, dim3(blocks), dim3(kBlock), 0, c->stream,
                               (const double *)dp, n, top, (uint32_t *)dh);
            HIPCHK(c, hipGetLastError());
            hipLaunchKernelGGL(k_running_sum, dim3(1), dim3(kScanBlock), 0, c->stream,
                               (uint32_t *)dh, top + 1);
            HIPCHK(c, hipGetLastError());
            hipLaunchKernelGGL(k_expand_counts, dim3(grid_for(n)), dim3(kBlock), 0, c->stream,
                               (const uint32_t *)dh, top, total_weight, (double *)dout, n);
            HIPCHK(c, hipGetLastError());
            TRY(copy_back(c, pr, dout, sizeof(double) * n, flags));
            HIPCHK(c, hipStreamSynchronize(c->stream));
            return OKA_OK;
        }
    }
    TRY(ensure(c, kSlotBitmap, sizeof(double) * n, &dz));
    hipLaunchKernelGGL(k_probability, dim3(grid_for(n)), dim3(kBlock), 0, c->stream,
                       (const double *)dp, total_weight, (double *)dz, n);
    HIPCHK(c, hipGetLastError());
    size_t temp = 0;
    HIPCHK(c, hipcub::DeviceRadixSort::SortKeysDescending(nullptr, temp, (const double *)dz,
                                                          (double *)dout, (int)n, 0, 64,
                                                          c->stream));
    void *dtemp;
    TRY(ensure(c, kSlotMarks, temp, &dtemp));
    HIPCHK(c, hipcub::DeviceRadixSort::SortKeysDescending(dtemp, temp, (const double *)dz,
                                                          (double *)dout, (int)n, 0, 64,
                                                          c->stream));
    TRY(copy_back(c, pr, dout, sizeof(double) * n, flags));
    if (!(flags & OKA_ASYNC) || !(flags & OKA_PTR_DEVICE))
        HIPCHK(c, hipStreamSynchronize(c->stream));
    return OKA_OK;
}

}  // extern "C"
