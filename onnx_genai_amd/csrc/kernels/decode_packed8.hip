// The decode kernels over repacked 8-bit weights (two planes of nibbles per tile; decode_packed.hip plans the launches as those of the
// 4-bit call with twice the tiles). A plane's tile is unpacked and multiplied exactly like a 4-bit one, the activations staged once for both;
// what is streamed is 1.01 bytes per weight and the bound is HBM as for 4 bits: 3584 -> 152064, bf16, block 128, 1 / 4 / 16 rows 144 / 344 /
// 5535 -> 99 / 102 / 111 us (5.5 TB/s at one row), 3584 -> 37888 39.6 / 90 / 255 -> 29 / 37 / 38 us, 18944 -> 3584 29 / 47 / 180 -> 17 / 18 / 23 us.
// Before: a GEMV of one wave per column up to four rows, which reads every activation row again for each column, and from five rows
// the weights expanded to 16 bits on every call.
#include "decode_packed.hiph"
#include "decode_packed8.hiph"

namespace mnb {

template <bool BF16, int BS, int MR>
static int launch_packed8_mr(const PackedParams& p, int waves, hipStream_t stream)
{
    const unsigned grid = static_cast<unsigned>((p.n + 15) / 16);
    const size_t stage = static_cast<size_t>(waves) * 2 * (MR == 1 ? 1024 : MR * kRowPitchP);
    const size_t red = static_cast<size_t>(waves) * 1024;
    const size_t lds = stage > red ? stage : red;
    auto kernel = decode_packed8_kernel<BF16, BS, MR>;
    if (lds > 65536) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds));
        if (e != hipSuccess) return static_cast<int>(e);
    }
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(waves * 64), lds, stream, p);
    return static_cast<int>(hipGetLastError());
}

template <bool BF16, int BS>
static int launch_packed8_bs(const PackedParams& p, int waves, hipStream_t stream)
{
    if (p.m <= 1) return launch_packed8_mr<BF16, BS, 1>(p, waves, stream);
    if (p.m <= 4) return launch_packed8_mr<BF16, BS, 4>(p, waves, stream);
    if (p.m <= 8) return launch_packed8_mr<BF16, BS, 8>(p, waves, stream);
    return launch_packed8_mr<BF16, BS, 16>(p, waves, stream);
}

int launch_packed8(const PackedParams& p, bool bf16, int block_size, int waves, hipStream_t stream)
{
    switch (block_size) {
        case 32: return bf16 ? launch_packed8_bs<true, 32>(p, waves, stream) : launch_packed8_bs<false, 32>(p, waves, stream);
        case 64: return bf16 ? launch_packed8_bs<true, 64>(p, waves, stream) : launch_packed8_bs<false, 64>(p, waves, stream);
        default: return bf16 ? launch_packed8_bs<true, 128>(p, waves, stream) : launch_packed8_bs<false, 128>(p, waves, stream);
    }
}

template <bool BF16, int BS, int RB, bool SUMS, bool PF, bool DEEP>
static int launch_wide8_cfg(const PackedParams& p, hipStream_t stream)
{
    constexpr int AT = 2, NBT = 128 / BS, kRows = RB * 16;
    const size_t lds = 2 * kRows * (AT * 256 + 16) + (SUMS ? 2 * AT * NBT * kRows * 4 : 0);
    const int64_t col_groups = (p.n + 15) / 16;
    hipLaunchKernelGGL((decode_wide8_kernel<BF16, BS, RB, SUMS, PF, DEEP>), dim3(static_cast<unsigned>((col_groups + kWideWaves - 1) / kWideWaves)), dim3(kWideWaves * 64), lds,
                       stream, p);
    return static_cast<int>(hipGetLastError());
}

template <bool BF16, int BS>
static int launch_wide8_bs(const PackedParams& p, bool few_workgroups, hipStream_t stream)
{
    if (p.m <= 16) {
        // block 32 through the second MFMA (the sums build would take twice the registers), the others through the block sums
        if constexpr (BS == 32) return few_workgroups ? launch_wide8_cfg<BF16, BS, 1, false, true, true>(p, stream) : launch_wide8_cfg<BF16, BS, 1, false, false, true>(p, stream);
        else return few_workgroups ? launch_wide8_cfg<BF16, BS, 1, true, true, true>(p, stream) : launch_wide8_cfg<BF16, BS, 1, true, false, false>(p, stream);
    }
    if constexpr (BS != 32) {
        if (p.m <= 32) return launch_wide8_cfg<BF16, BS, 2, true, false, false>(p, stream);
    }
    return -1;
}

int launch_wide8(const PackedParams& p, bool bf16, int block_size, bool few_workgroups, hipStream_t stream)
{
    switch (block_size) {
        case 32: return bf16 ? launch_wide8_bs<true, 32>(p, few_workgroups, stream) : launch_wide8_bs<false, 32>(p, few_workgroups, stream);
        case 64: return bf16 ? launch_wide8_bs<true, 64>(p, few_workgroups, stream) : launch_wide8_bs<false, 64>(p, few_workgroups, stream);
        default: return bf16 ? launch_wide8_bs<true, 128>(p, few_workgroups, stream) : launch_wide8_bs<false, 128>(p, few_workgroups, stream);
    }
}

}  // namespace mnb
