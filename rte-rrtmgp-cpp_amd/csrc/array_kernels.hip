// Device kernels behind Array_gpu::fill and Array_gpu::subset (rte-rrtmgp-cpp_amd/include/Array.h),
// the counterparts of the reference's fill_kernel and subset_kernel (include/Array.h:296-335,
// launched at :501-511 and :583-606).  Extents and offsets are 64-bit; the element type only
// matters through its size, so one kernel per size serves every Array_gpu<T,N>.  And the strided copies
// between other libraries' tensors and Fortran-order arrays (rrtmgp_hip_copy_arrays).
#include <algorithm>
#include <cstring>

#include "common.h"

namespace rrtmgp_hip
{
constexpr int SUBSET_MAX_DIMS = 8;

template<int B> struct Word;
template<> struct Word<1> { using T = uint8_t; };
template<> struct Word<2> { using T = uint16_t; };
template<> struct Word<4> { using T = uint32_t; };
template<> struct Word<8> { using T = uint64_t; };

template<typename W>
__global__ void fill_kernel(int64_t n, W v, W* __restrict__ dst)
{
    for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += int64_t(gridDim.x) * blockDim.x)
        dst[i] = v;
}

// Subset geometry, all 0-based: source element of destination multi-index d is
//     sum_k (spread_k ? 0 : d_k + first_k) * src_stride_k,
// with first_k = start_k - offset_k - 1 (the reference's 1-based start and Array offset).
struct SubsetGeom
{
    int ndim;
    int64_t dst_dims[SUBSET_MAX_DIMS];
    int64_t src_stride[SUBSET_MAX_DIMS];
    int64_t first[SUBSET_MAX_DIMS];
    int spread[SUBSET_MAX_DIMS];
};

template<typename W>
__global__ void subset_kernel(int64_t n, SubsetGeom g, const W* __restrict__ src, W* __restrict__ dst)
{
    for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += int64_t(gridDim.x) * blockDim.x)
    {
        int64_t rem = i, s = 0;
        for (int k = 0; k < g.ndim; ++k)
        {
            const int64_t d = rem % g.dst_dims[k];
            rem /= g.dst_dims[k];
            if (!g.spread[k]) s += (d + g.first[k]) * g.src_stride[k];
        }
        dst[i] = src[s];
    }
}

inline unsigned grid_stride_blocks(int64_t n)
{
    const int64_t b = (n + 255) / 256;
    return unsigned(std::min<int64_t>(b, int64_t(device_cu_count()) * 32));
}

template<int B>
int fill_t(void* dst, int64_t n, const void* value, hipStream_t s)
{
    using W = typename Word<B>::T;
    W v;
    std::memcpy(&v, value, B);
    RRTMGP_TIMED("fill_kernel", s);
    hipLaunchKernelGGL(fill_kernel<W>, dim3(grid_stride_blocks(n)), dim3(256), 0, s, n, v, static_cast<W*>(dst));
    RRTMGP_LAUNCHED("fill_kernel");
    return RRTMGP_OK;
}

template<int B>
int subset_t(int64_t n, const SubsetGeom& g, const void* src, void* dst, hipStream_t s)
{
    using W = typename Word<B>::T;
    RRTMGP_TIMED("subset_kernel", s);
    hipLaunchKernelGGL(subset_kernel<W>, dim3(grid_stride_blocks(n)), dim3(256), 0, s, n, g,
                       static_cast<const W*>(src), static_cast<W*>(dst));
    RRTMGP_LAUNCHED("subset_kernel");
    return RRTMGP_OK;
}

// Copies of several strided 2-D arrays of float or double into arrays with the first index fastest, in one
// launch (blockIdx.y selects the array).  Latency bound at the sizes a gradient step has: one launch per array,
// with a layout pass of its own and waits on both sides, took 33 us for each of the 58 arrays of a step at
// 250 x 60 FP64; a launch of up to 16 arrays takes 8 us, and the step went from 4.0 to 3.1 ms.  Where the source
// runs along its second index, 32 x 32 tiles go through LDS, so that both sides move along their rows.
constexpr int COPY_MAX = 16;
constexpr int COPY_TILE = 32;
struct CopyItem
{
    const void* src;
    void* dst;
    int64_t n0, n1, s0, s1;          // extents, source strides in elements; dst is (n0, n1), n0 fastest
    int src_size, dst_size;          // 4 (float) or 8 (double)
};
struct CopySet { CopyItem a[COPY_MAX]; };

template<typename S, typename D>
__device__ __forceinline__ void copy_item(const CopyItem& c, D (*tile)[COPY_TILE + 1])
{
    const S* __restrict__ src = static_cast<const S*>(c.src);
    D* __restrict__ dst = static_cast<D*>(c.dst);
    const int64_t n = c.n0 * c.n1;
    if (c.s1 == 1 && c.s0 != 1 && c.n0 > 1 && c.n1 > 1)
    {
        const int64_t t0 = (c.n0 + COPY_TILE - 1) / COPY_TILE, t1 = (c.n1 + COPY_TILE - 1) / COPY_TILE;
        const int x = threadIdx.x % COPY_TILE, y = threadIdx.x / COPY_TILE;
        for (int64_t t = blockIdx.x; t < t0 * t1; t += gridDim.x)       // uniform over the work-group
        {
            const int64_t b0 = t % t0 * COPY_TILE, b1 = t / t0 * COPY_TILE;
            for (int r = y; r < COPY_TILE; r += 256 / COPY_TILE)
                if (b0 + r < c.n0 && b1 + x < c.n1) tile[r][x] = D(src[(b0 + r) * c.s0 + b1 + x]);
            __syncthreads();
            for (int r = y; r < COPY_TILE; r += 256 / COPY_TILE)
                if (b0 + x < c.n0 && b1 + r < c.n1) dst[b0 + x + c.n0 * (b1 + r)] = tile[x][r];
            __syncthreads();
        }
        return;
    }
    for (int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x; i < n; i += int64_t(gridDim.x) * 256)
        dst[i] = D(src[i % c.n0 * c.s0 + i / c.n0 * c.s1]);
}

__global__ __launch_bounds__(256)
void copy_arrays_kernel(CopySet q)
{
    __shared__ double tile[COPY_TILE][COPY_TILE + 1];
    const CopyItem& c = q.a[blockIdx.y];
    auto* td = tile;
    auto* tf = reinterpret_cast<float (*)[COPY_TILE + 1]>(&tile[0][0]);
    if (c.src_size == 4 && c.dst_size == 4) copy_item<float, float>(c, tf);
    else if (c.src_size == 4) copy_item<float, double>(c, td);
    else if (c.dst_size == 4) copy_item<double, float>(c, tf);
    else copy_item<double, double>(c, td);
}
}  // namespace rrtmgp_hip

using namespace rrtmgp_hip;

extern "C" int rrtmgp_hip_copy_arrays(int n, const rrtmgp_copy_item* items, void* stream)
{
    if (n < 0 || (n > 0 && !items)) return arg_error("copy_arrays: bad arguments");
    hipStream_t s = as_stream(stream);
    for (int k = 0; k < n;)
    {
        CopySet q{};
        int m = 0;
        int64_t most = 0;
        for (; k < n && m < COPY_MAX; ++k)
        {
            const rrtmgp_copy_item& c = items[k];
            if (c.n0 < 0 || c.n1 < 0) return arg_error("copy_arrays: negative extent");
            if ((c.src_size != 4 && c.src_size != 8) || (c.dst_size != 4 && c.dst_size != 8))
                return arg_error("copy_arrays: element sizes must be 4 or 8 bytes");
            if (c.n0 * c.n1 == 0) continue;
            if (!c.src || !c.dst) return arg_error("copy_arrays: NULL array");
            q.a[m++] = CopyItem{c.src, c.dst, c.n0, c.n1, c.s0, c.s1, c.src_size, c.dst_size};
            most = std::max(most, c.n0 * c.n1);
        }
        if (m == 0) continue;
        const unsigned bx = unsigned(std::min<int64_t>((most + 1023) / 1024, int64_t(device_cu_count()) * 8));
        RRTMGP_TIMED("copy_arrays_kernel", s);
        hipLaunchKernelGGL(copy_arrays_kernel, dim3(bx, unsigned(m)), dim3(256), 0, s, q);
        RRTMGP_LAUNCHED("copy_arrays_kernel");
    }
    return RRTMGP_OK;
}

extern "C" int rrtmgp_hip_fill(void* dst, int64_t n, int elem_size, const void* value, void* stream)
{
    if (n < 0) return arg_error("fill: negative element count");
    if (n == 0) return RRTMGP_OK;
    if (!dst || !value) return arg_error("fill: NULL pointer");
    hipStream_t s = as_stream(stream);
    switch (elem_size)
    {
        case 1: return fill_t<1>(dst, n, value, s);
        case 2: return fill_t<2>(dst, n, value, s);
        case 4: return fill_t<4>(dst, n, value, s);
        case 8: return fill_t<8>(dst, n, value, s);
        default: return arg_error("fill: element size must be 1, 2, 4 or 8 bytes");
    }
}

extern "C" int rrtmgp_hip_subset(int elem_size, int ndim, const void* src, const int64_t* src_dims,
                                 const int64_t* src_offsets, const int64_t* starts, void* dst,
                                 const int64_t* dst_dims, void* stream)
{
    if (ndim < 1 || ndim > SUBSET_MAX_DIMS) return arg_error("subset: 1 to 8 dimensions");
    if (!src_dims || !starts || !dst_dims) return arg_error("subset: NULL geometry");
    SubsetGeom g{};
    g.ndim = ndim;
    int64_t n = 1, stride = 1;
    for (int k = 0; k < ndim; ++k)
    {
        const int64_t sd = src_dims[k], dd = dst_dims[k];
        const int64_t off = src_offsets ? src_offsets[k] : 0;
        if (sd < 1 || dd < 0) return arg_error("subset: bad extents");
        g.dst_dims[k] = dd;
        g.src_stride[k] = stride;
        g.spread[k] = (sd == 1) ? 1 : 0;   // a dimension of length 1 is spread (Array.h:230-233)
        g.first[k] = starts[k] - off - 1;
        // Every read stays inside the source (the reference does not check; a fault here would be).
        if (!g.spread[k] && dd > 0 && (g.first[k] < 0 || g.first[k] + dd > sd))
            return arg_error("subset: range " + std::to_string(k + 1) + " lies outside the source array");
        n *= dd;
        stride *= sd;
    }
    if (n == 0) return RRTMGP_OK;
    if (!src || !dst) return arg_error("subset: NULL array");
    hipStream_t s = as_stream(stream);
    switch (elem_size)
    {
        case 1: return subset_t<1>(n, g, src, dst, s);
        case 2: return subset_t<2>(n, g, src, dst, s);
        case 4: return subset_t<4>(n, g, src, dst, s);
        case 8: return subset_t<8>(n, g, src, dst, s);
        default: return arg_error("subset: element size must be 1, 2, 4 or 8 bytes");
    }
}
