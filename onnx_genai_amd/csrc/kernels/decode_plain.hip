// The decode kernels over the repacked 4-bit stream with plain sums (decode_packed.hiph says which weights they serve and why; decode_packed.hip
// plans the launches as those of the builds that carry the offset).
#include "decode_plain.hiph"

namespace mnb {

template <bool BF16, int BS, int MR, typename ST>
__global__ __launch_bounds__((BS == 128 && sizeof(ST) == 2 && (MR != 16 || BF16)) ? 1024 : 512)
void decode_plain_kernel(PackedParams p)
{
    decode_packed_body<BF16, BS, MR, ST, 1, false, false, 4, true>(p);
}

template <bool BF16, int BS, typename ST, int RB, bool PF, bool DEEP>
__global__ __launch_bounds__(kWideWaves * 64)
void decode_plain_wide_kernel(PackedParams p)
{
    decode_wide_body<BF16, BS, ST, RB, false, PF, DEEP, false, kWideWaves, 4, true>(p);
}

template <bool BF16, int BS, int MR, typename ST>
static int launch_plain_mr(const PackedParams& p, int waves, hipStream_t stream)
{
    const unsigned grid = static_cast<unsigned>((p.n + 15) / 16);
    const size_t stage = static_cast<size_t>(waves) * 2 * (MR == 1 ? 1024 : MR * kRowPitchP);
    const size_t red = static_cast<size_t>(waves) * 1024;
    const size_t lds = stage > red ? stage : red;
    auto kernel = decode_plain_kernel<BF16, BS, MR, ST>;
    if (lds > 65536) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds));
        if (e != hipSuccess) return static_cast<int>(e);
    }
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(waves * 64), lds, stream, p);
    return static_cast<int>(hipGetLastError());
}

template <bool BF16, int BS, typename ST>
static int launch_plain_bs(const PackedParams& p, int waves, hipStream_t stream)
{
    if (p.m <= 1) return launch_plain_mr<BF16, BS, 1, ST>(p, waves, stream);
    if (p.m <= 4) return launch_plain_mr<BF16, BS, 4, ST>(p, waves, stream);
    if (p.m <= 8) return launch_plain_mr<BF16, BS, 8, ST>(p, waves, stream);
    return launch_plain_mr<BF16, BS, 16, ST>(p, waves, stream);
}

template <bool BF16, int BS, typename ST, int RB, bool PF, bool DEEP>
static int launch_plain_wide_cfg(const PackedParams& p, hipStream_t stream)
{
    constexpr size_t lds = 2 * RB * 16 * (4 * 256 + 16);           // two windows of four tiles
    const int64_t col_groups = (p.n + 15) / 16;
    auto kernel = decode_plain_wide_kernel<BF16, BS, ST, RB, PF, DEEP>;
    if (lds > 65536) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds));
        if (e != hipSuccess) return static_cast<int>(e);
    }
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>((col_groups + kWideWaves - 1) / kWideWaves)), dim3(kWideWaves * 64), lds, stream, p);
    return static_cast<int>(hipGetLastError());
}

template <bool BF16, int BS, typename ST>
static int launch_plain_wide_bs(const PackedParams& p, bool few_workgroups, hipStream_t stream)
{
    if (p.m <= 16) return few_workgroups ? launch_plain_wide_cfg<BF16, BS, ST, 1, true, true>(p, stream) : launch_plain_wide_cfg<BF16, BS, ST, 1, false, true>(p, stream);
    if constexpr (BS != 32) {
        if (p.m <= 32) return launch_plain_wide_cfg<BF16, BS, ST, 2, false, false>(p, stream);
    }
    return -1;
}

// `go`: called with the element type, the block size and the scales' storage type as compile-time values
template <typename Go>
static int by_build(bool bf16, bool f32_scales, int block_size, Go go)
{
    auto by_block = [&](auto bf, auto st) {
        switch (block_size) {
            case 32: return go(bf, std::integral_constant<int, 32>{}, st);
            case 64: return go(bf, std::integral_constant<int, 64>{}, st);
            default: return go(bf, std::integral_constant<int, 128>{}, st);
        }
    };
    if (bf16) return f32_scales ? by_block(std::true_type{}, float{}) : by_block(std::true_type{}, uint16_t{});
    return f32_scales ? by_block(std::false_type{}, float{}) : by_block(std::false_type{}, uint16_t{});
}

int launch_plain(const PackedParams& p, bool bf16, bool f32_scales, int block_size, int waves, hipStream_t stream)
{
    return by_build(bf16, f32_scales, block_size, [&](auto bf, auto bs, auto st) { return launch_plain_bs<decltype(bf)::value, decltype(bs)::value, decltype(st)>(p, waves, stream); });
}

int launch_plain_wide(const PackedParams& p, bool bf16, bool f32_scales, int block_size, bool few_workgroups, hipStream_t stream)
{
    return by_build(bf16, f32_scales, block_size,
                    [&](auto bf, auto bs, auto st) { return launch_plain_wide_bs<decltype(bf)::value, decltype(bs)::value, decltype(st)>(p, few_workgroups, stream); });
}

}  // namespace mnb
