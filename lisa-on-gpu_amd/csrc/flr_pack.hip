// flr_pack.hip -- a packed series' per-source statistics (amplitude, power, power of the first
// differences) and its conversion to the 8-byte input formats of the mixed kernels.
//
// Bound by HBM: the statistics read each sample once, the conversion reads 16 and writes 8 bytes.
// Many short workgroups (kChunk samples of one source each) rather than a few persistent ones,
// since every workgroup's work is the same small stream; the partial sums of a source are added
// by one workgroup in a fixed order, so the results do not depend on timing. The same quantities
// from elementwise and indexed torch operations took 312 ms for one source of 2^20 samples: an
// indexed sum adds every sample of a source to one address with atomics. Statistics, conversion
// and fused launch together take 0.16 ms (the call through pyResponseTDI, MI355X).
#include "flr_internal.hpp"

#include <algorithm>

namespace flr {

constexpr int kChunk = 16 * kBlock;  // samples per workgroup

int64_t series_chunks(int64_t max_len) { return (max_len + kChunk - 1) / kChunk; }

template <typename T>
__device__ __forceinline__ double2 series_at(const T *h, int64_t i)
{
    const T v = h[i];
    return make_double2((double)v.x, (double)v.y);
}

// The larger of a and b, NaN if either is (as torch's max).
__device__ __forceinline__ double max_nan(double a, double b)
{
    return (a != a || a > b) ? a : b;
}

// One source's four statistics (the layout of flr_series_stats).
struct SeriesStats {
    double amp;   // max |h|
    double comp;  // max(|Re h|, |Im h|)
    double p;     // sum |h|^2
    double d;     // sum |h[i+1] - h[i]|^2
};

__device__ __forceinline__ void stats_join(SeriesStats &a, const SeriesStats &b)
{
    a.amp = max_nan(a.amp, b.amp);
    a.comp = max_nan(a.comp, b.comp);
    a.p += b.p;
    a.d += b.d;
}

// The workgroup's statistics in thread 0, joined in a fixed order.
__device__ __forceinline__ void stats_block(SeriesStats &a)
{
    __shared__ SeriesStats s[kBlock / 64];
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        SeriesStats b;
        b.amp = __shfl_xor(a.amp, off);
        b.comp = __shfl_xor(a.comp, off);
        b.p = __shfl_xor(a.p, off);
        b.d = __shfl_xor(a.d, off);
        stats_join(a, b);
    }
    if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = a;
    __syncthreads();
    if (threadIdx.x == 0)
        for (int w = 1; w < kBlock / 64; ++w) stats_join(a, s[w]);
    __syncthreads();  // before the next call's writes
}

// Samples [lo, hi) of source s: the whole series when there is no offset table (one source).
__device__ __forceinline__ void source_range(const int64_t *offsets, int s, int64_t max_len,
                                             int64_t &lo, int64_t &hi)
{
    lo = offsets ? offsets[s] : 0;
    hi = offsets ? offsets[s + 1] : max_len;
}

template <typename T>
__global__ __launch_bounds__(kBlock) void series_stats_kernel(const T *__restrict__ h,
                                                              const int64_t *__restrict__ offsets,
                                                              int num_sources, int64_t max_len,
                                                              SeriesStats *__restrict__ part)
{
    for (int s = blockIdx.y; s < num_sources; s += gridDim.y) {
        int64_t lo, hi;
        source_range(offsets, s, max_len, lo, hi);
        const int64_t first = lo + (int64_t)blockIdx.x * kChunk;
        if (first >= hi) continue;  // the whole workgroup
        SeriesStats a{0.0, 0.0, 0.0, 0.0};
#pragma unroll 4
        for (int r = 0; r < kChunk / kBlock; ++r) {
            const int64_t i = first + r * kBlock + threadIdx.x;
            if (i >= hi) break;
            const double2 v = series_at(h, i);
            a.amp = max_nan(a.amp, hypot(v.x, v.y));
            a.comp = max_nan(a.comp, max_nan(fabs(v.x), fabs(v.y)));
            a.p += v.x * v.x + v.y * v.y;
            if (i + 1 < hi) {
                const double2 w = series_at(h, i + 1);
                const double dx = w.x - v.x, dy = w.y - v.y;
                a.d += dx * dx + dy * dy;
            }
        }
        stats_block(a);
        if (threadIdx.x == 0) part[(int64_t)s * gridDim.x + blockIdx.x] = a;
    }
}

// One workgroup per source: the chunks' statistics (`chunks` records per source, of which the
// source's length fills the first ones).
__global__ __launch_bounds__(kBlock) void series_join_kernel(const SeriesStats *__restrict__ part,
                                                             const int64_t *__restrict__ offsets,
                                                             int num_sources, int64_t max_len,
                                                             int64_t chunks,
                                                             SeriesStats *__restrict__ stats)
{
    const int s = blockIdx.x;
    if (s >= num_sources) return;
    int64_t lo, hi;
    source_range(offsets, s, max_len, lo, hi);
    const int64_t used = (hi - lo + kChunk - 1) / kChunk;
    SeriesStats a{0.0, 0.0, 0.0, 0.0};
    for (int64_t c = threadIdx.x; c < used; c += kBlock) stats_join(a, part[s * chunks + c]);
    stats_block(a);
    if (threadIdx.x == 0) stats[s] = a;
}

// complex64 h / s with s = max |h| (Q31 false), or int32 pairs of 2^31 - 1 times h / s with
// s = max(|Re h|, |Im h|); s = 1 for a source without a positive finite-or-infinite maximum
// (zeros, NaN). One rounding of h times the reciprocal (or quotient) of the scale.
template <bool Q31>
__global__ __launch_bounds__(kBlock) void series_pack_kernel(const double2 *__restrict__ h,
                                                             const int64_t *__restrict__ offsets,
                                                             int num_sources, int64_t max_len,
                                                             const SeriesStats *__restrict__ stats,
                                                             void *__restrict__ out)
{
    for (int s = blockIdx.y; s < num_sources; s += gridDim.y) {
        int64_t lo, hi;
        source_range(offsets, s, max_len, lo, hi);
        const int64_t first = lo + (int64_t)blockIdx.x * kChunk;
        if (first >= hi) continue;
        const double top = Q31 ? stats[s].comp : stats[s].amp;
        const double sc = top > 0.0 ? top : 1.0;
        const double mul = Q31 ? 2147483647.0 / sc : 1.0 / sc;
#pragma unroll 4
        for (int r = 0; r < kChunk / kBlock; ++r) {
            const int64_t i = first + r * kBlock + threadIdx.x;
            if (i >= hi) break;
            const double2 v = h[i];
            if constexpr (Q31)
                reinterpret_cast<int2 *>(out)[i] =
                    make_int2((int)rint(v.x * mul), (int)rint(v.y * mul));
            else
                // the product by the complex number mul: a component that is not finite makes both NaN
                reinterpret_cast<float2 *>(out)[i] = make_float2(
                    (float)(v.x * mul - v.y * 0.0), (float)(v.y * mul + v.x * 0.0));
        }
    }
}

static dim3 series_grid(int64_t max_len, int num_sources)
{
    return dim3((unsigned)series_chunks(max_len), (unsigned)std::min(num_sources, 65535));
}

hipError_t launch_series_stats(const void *h, int format, const int64_t *offsets, int num_sources,
                               int64_t max_len, double *work, double *stats, hipStream_t stream)
{
    const dim3 grid = series_grid(max_len, num_sources);
    SeriesStats *part = reinterpret_cast<SeriesStats *>(work);
    switch (format) {
    case FLR_GB_COMPLEX128:
        hipLaunchKernelGGL(series_stats_kernel<double2>, grid, dim3(kBlock), 0, stream,
                           static_cast<const double2 *>(h), offsets, num_sources, max_len, part);
        break;
    case FLR_GB_COMPLEX64:
        hipLaunchKernelGGL(series_stats_kernel<float2>, grid, dim3(kBlock), 0, stream,
                           static_cast<const float2 *>(h), offsets, num_sources, max_len, part);
        break;
    default:
        hipLaunchKernelGGL(series_stats_kernel<int2>, grid, dim3(kBlock), 0, stream,
                           static_cast<const int2 *>(h), offsets, num_sources, max_len, part);
        break;
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(series_join_kernel, dim3((unsigned)num_sources), dim3(kBlock), 0, stream,
                       part, offsets, num_sources, max_len, (int64_t)grid.x,
                       reinterpret_cast<SeriesStats *>(stats));
    return hipGetLastError();
}

hipError_t launch_series_pack(const void *h, const int64_t *offsets, int num_sources,
                              int64_t max_len, const double *stats, int format, void *out,
                              hipStream_t stream)
{
    const dim3 grid = series_grid(max_len, num_sources);
    const SeriesStats *st = reinterpret_cast<const SeriesStats *>(stats);
    const double2 *src = static_cast<const double2 *>(h);
    if (format == FLR_GB_Q31)
        hipLaunchKernelGGL(series_pack_kernel<true>, grid, dim3(kBlock), 0, stream, src, offsets,
                           num_sources, max_len, st, out);
    else
        hipLaunchKernelGGL(series_pack_kernel<false>, grid, dim3(kBlock), 0, stream, src, offsets,
                           num_sources, max_len, st, out);
    return hipGetLastError();
}

}  // namespace flr
