// Act-order weights (g_idx) whose groups are whole blocks in another order - what act-order quantizers write: every group has
// block_size elements of K, scattered. Sorting K by group turns such a node into an ordinary one over
//   B'[n, j] = B[n, order[j]],  A'[m, j] = A[m, order[j]],  order = the elements of K, group by group,
// with the scales and zero points as they are, so that the kernels for contiguous blocks serve it - of those over the repacked stream the ones with plain
// sums, which the per-element kernels have too. B' is made once for constant weights and the stream once more from it: two copies of the weights beside the caller's; A' costs one gather per call (7 KB of a 3584-element row: 2 us; one row is gathered inside the decode kernel) where the kernels that look a group up per element
// paid for it on every weight: 3584 -> 37888, one f16 row, block 128: 501 us, against 18.1 us for gather and repacked-stream kernel together.
#include <vector>

#include "common.hiph"

namespace mnb {

// One dword of B' per thread: 32 / BITS elements gathered from the same packed row; elements past K are zero.
template <int BITS>
__global__ __launch_bounds__(256) void regroup_kernel(const uint8_t* __restrict__ b, const int32_t* __restrict__ order, int64_t n, int64_t k, int64_t row_dwords,
                                                      uint32_t* __restrict__ out)
{
    constexpr int kPer = 32 / BITS, kInByte = 8 / BITS;
    const int64_t total = n * row_dwords;
    for (int64_t i = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; i < total; i += static_cast<int64_t>(gridDim.x) * blockDim.x) {
        const int64_t row = i / row_dwords, j0 = (i - row * row_dwords) * kPer;
        const uint8_t* const in = b + row * row_dwords * 4;
        uint32_t w = 0;
#pragma unroll
        for (int e = 0; e < kPer; ++e) {
            if (j0 + e >= k) break;
            const uint32_t src = static_cast<uint32_t>(order[j0 + e]);
            w |= ((in[src / kInByte] >> ((src % kInByte) * BITS)) & ((1u << BITS) - 1u)) << (e * BITS);
        }
        out[i] = w;
    }
}

// A' row by row: T is a 16- or 32-bit element; a thread writes four of them.
template <typename T>
__global__ __launch_bounds__(256) void gather_columns_kernel(const T* __restrict__ a, const int32_t* __restrict__ order, int64_t k, T* __restrict__ out)
{
    const int64_t j = (blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x) * 4;
    if (j >= k) return;
    const T* const in = a + static_cast<int64_t>(blockIdx.y) * k;
    T* const to = out + static_cast<int64_t>(blockIdx.y) * k;
    if (j + 4 <= k && (k & 3) == 0) {
        const int4 o = *reinterpret_cast<const int4*>(order + j);
        T v[4] = {in[o.x], in[o.y], in[o.z], in[o.w]};
        if constexpr (sizeof(T) == 2) *reinterpret_cast<uint2*>(to + j) = *reinterpret_cast<const uint2*>(v);
        else *reinterpret_cast<uint4*>(to + j) = *reinterpret_cast<const uint4*>(v);
    } else {
        for (int64_t e = j; e < j + 4 && e < k; ++e) to[e] = in[order[e]];
    }
}

__global__ __launch_bounds__(256) void narrow_order_kernel(const int32_t* __restrict__ order, int64_t k, uint16_t* __restrict__ order16)
{
    const int64_t i = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    if (i < k) order16[i] = static_cast<uint16_t>(order[i]);
}

}  // namespace mnb

extern "C" int rocm_launch_narrow_order(const int32_t* order, int64_t k, uint16_t* order16, rocm_stream_t stream)
{
    hipLaunchKernelGGL(mnb::narrow_order_kernel, dim3(static_cast<unsigned>((k + 255) / 256)), dim3(256), 0, static_cast<hipStream_t>(stream), order, k, order16);
    return static_cast<int>(hipGetLastError());
}

extern "C" int rocm_gidx_order(const int32_t* g_idx, int64_t k, int block_size, int32_t* order, int* regular, rocm_stream_t stream)
{
    *regular = 0;
    std::vector<int32_t> groups(static_cast<size_t>(k)), sorted(static_cast<size_t>(k));
    int e = rocm_ffi_memcpy_d2h(groups.data(), g_idx, groups.size() * sizeof(int32_t), stream);
    if (e != 0) return e;
    const int64_t kb = (k + block_size - 1) / block_size;
    std::vector<int64_t> filled(static_cast<size_t>(kb), 0);
    for (int64_t i = 0; i < k; ++i) {
        const int64_t g = groups[static_cast<size_t>(i)];
        if (g < 0 || g >= kb) return 0;
        const int64_t room = g * block_size + block_size <= k ? block_size : k - g * block_size;
        if (filled[static_cast<size_t>(g)] >= room) return 0;                  // a group of more than a block (so another has less)
        sorted[static_cast<size_t>(g * block_size + filled[static_cast<size_t>(g)]++)] = static_cast<int32_t>(i);
    }
    e = rocm_ffi_memcpy_h2d(order, sorted.data(), sorted.size() * sizeof(int32_t), stream);
    if (e == 0) *regular = 1;
    return e;
}

extern "C" int rocm_launch_regroup(const uint8_t* b, const int32_t* order, int64_t n, int64_t k, int block_size, int bits, void* out, rocm_stream_t stream)
{
    const int64_t row_dwords = (k + block_size - 1) / block_size * block_size * bits / 32;
    int64_t blocks = (n * row_dwords + 255) / 256;
    if (blocks > 65536) blocks = 65536;
    const dim3 grid(static_cast<unsigned>(blocks));
    hipStream_t s = static_cast<hipStream_t>(stream);
    uint32_t* const to = static_cast<uint32_t*>(out);
    if (bits == 2) hipLaunchKernelGGL(mnb::regroup_kernel<2>, grid, dim3(256), 0, s, b, order, n, k, row_dwords, to);
    else if (bits == 8) hipLaunchKernelGGL(mnb::regroup_kernel<8>, grid, dim3(256), 0, s, b, order, n, k, row_dwords, to);
    else hipLaunchKernelGGL(mnb::regroup_kernel<4>, grid, dim3(256), 0, s, b, order, n, k, row_dwords, to);
    return static_cast<int>(hipGetLastError());
}

extern "C" int rocm_launch_gather_columns(const void* a, int a_dtype, const int32_t* order, int64_t m, int64_t k, void* out, rocm_stream_t stream)
{
    hipStream_t s = static_cast<hipStream_t>(stream);
    const bool wide = a_dtype == ROCM_DT_F32;
    for (int64_t row0 = 0; row0 < m; row0 += 65535) {                          // grid.y
        const int64_t rows = m - row0 < 65535 ? m - row0 : 65535;
        const dim3 grid(static_cast<unsigned>((k + 1023) / 1024), static_cast<unsigned>(rows));
        if (wide)
            hipLaunchKernelGGL(mnb::gather_columns_kernel<uint32_t>, grid, dim3(256), 0, s, static_cast<const uint32_t*>(a) + row0 * k, order, k, static_cast<uint32_t*>(out) + row0 * k);
        else
            hipLaunchKernelGGL(mnb::gather_columns_kernel<uint16_t>, grid, dim3(256), 0, s, static_cast<const uint16_t*>(a) + row0 * k, order, k, static_cast<uint16_t*>(out) + row0 * k);
    }
    return static_cast<int>(hipGetLastError());
}
