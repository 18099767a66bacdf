// The decode kernels over the repacked stream with plain sums (decode_packed.hiph says which weights they serve and why; decode_packed.hip
// plans the launches as those of the builds that carry the offset, an 8-bit one's as those of the 4-bit call with twice the tiles).
//
// 8 bits: what is streamed is 1.01 bytes per weight and the bound is HBM. bf16, block 128, 1 / 4 / 16 rows, against a GEMV of one wave per column up to four
// rows and weights expanded to 16 bits on every call from five: 3584 -> 152064 144 / 344 / 5535 -> 104 / 102 / 113 us, 3584 -> 37888 39.6 / 90 / 255
// -> 28.4 / 31.4 / 31.5, 18944 -> 3584 29 / 47 / 180 -> 16.9 / 18.0 / 23.8. (As two planes of nibbles whose accumulators carried the offset: 106 / 108 / 115,
// 29.3 / 39.1 / 39.6, 17.1 / 18.6 / 24.4 - twice the matrix instructions.)
// 4 bits, act-order, gather included: HBM in f16 (3584 -> 37888, block 128, 1 / 16 rows 18.1 / 20.9 us, 17.8 / 20.1 with the offset), the vector ALU work of
// turning nibbles into bf16 integers otherwise (19.0 / 24.4 against 17.8 / 20.5).
#include "decode_plain.hiph"

namespace mnb {

// Waves per SIMD that the builds are held to: what the compiler reaches when it tries (left alone it takes a few registers more in a third of them).
constexpr int plain_waves_per_simd(bool bf16, int bs, int rows, bool f32_scales, int bits)
{
    // [f16 / bf16][4 bits, 4 bits with f32 scales, 8 bits][rows: 1, 2-4, 5-8, 9-16][block 32, 64, 128]
    constexpr unsigned char table[2][3][4][3] = {
        {{{7, 8, 8}, {6, 6, 7}, {5, 5, 5}, {4, 4, 4}}, {{7, 7, 8}, {5, 6, 7}, {5, 5, 5}, {4, 4, 4}}, {{8, 8, 8}, {6, 7, 7}, {6, 6, 8}, {5, 6, 6}}},
        {{{7, 8, 8}, {6, 7, 7}, {5, 5, 5}, {4, 4, 4}}, {{6, 7, 8}, {5, 6, 6}, {4, 5, 5}, {4, 4, 4}}, {{7, 8, 8}, {6, 7, 8}, {7, 6, 8}, {5, 6, 6}}},
    };
    return table[bf16][bits == 8 ? 2 : f32_scales ? 1 : 0][rows == 1 ? 0 : rows == 4 ? 1 : rows == 8 ? 2 : 3][bs == 32 ? 0 : bs == 64 ? 1 : 2];
}

// At most 80 scalar registers: with more, which only the rare second summation asks for, seven waves fit a SIMD instead of eight, and one workgroup of
// fourteen a CU instead of two (8 bits, bf16, one row, 3584 -> 37888: 28.6 -> 32.7 us).
template <bool BF16, int BS, int MR, typename ST, int BITS>
__global__ __launch_bounds__((BS == 128 && sizeof(ST) == 2 && (MR != 16 || BF16)) ? 1024 : 512)
__attribute__((amdgpu_num_sgpr(80), amdgpu_waves_per_eu(plain_waves_per_simd(BF16, BS, MR, sizeof(ST) == 4, BITS))))
void decode_plain_kernel(MNB_PACKED_ARGS)
{
    decode_packed_body<BF16, BS, MR, ST, 1, false, false, BITS, true>(MNB_PACKED_PARAMS);
}

// One row of activations that it gathers itself.
template <bool BF16, int BS, typename ST>
__global__ __launch_bounds__((BS == 128 && sizeof(ST) == 2) ? 1024 : 512)
__attribute__((amdgpu_num_sgpr(80), amdgpu_waves_per_eu(plain_waves_per_simd(BF16, BS, 1, sizeof(ST) == 4, 4))))
void decode_plain_gather_kernel(MNB_PACKED_ARGS)
{
    decode_packed_body<BF16, BS, 1, ST, 1, false, false, 4, true, true>(MNB_PACKED_PARAMS);
}

// One block of rows: weights and windows both ahead (8 bits, block 128, 16 rows, 3584 -> 152064: 112 us, windows alone 120, neither 114; act-order
// 4 bits 83 / 85 / 89); two: neither (registers).
template <bool BF16, int BS, typename ST, int RB, int WMAX, int BITS>
__global__ __launch_bounds__(WMAX * 64)
__attribute__((amdgpu_waves_per_eu(BF16 && BS == 128 && RB == 1 && WMAX == kWideWaves && BITS == 8 ? 6 : 1)))
void decode_plain_wide_kernel(MNB_PACKED_ARGS)
{
    decode_wide_body<BF16, BS, ST, RB, false, RB == 1, RB == 1, false, WMAX, BITS, true>(MNB_PACKED_PARAMS);
}

template <bool BF16, int BS, int MR, typename ST, int BITS>
static int launch_plain_mr(const PackedParams& p, int waves, hipStream_t stream)
{
    const unsigned grid = static_cast<unsigned>((static_cast<int64_t>(p.n) + 15) / 16);
    const size_t stage = static_cast<size_t>(waves) * 2 * (MR == 1 ? 1024 : MR * kRowPitchP);
    const size_t red = static_cast<size_t>(waves) * 1024;
    const size_t lds = stage > red ? stage : red;
    return launch_on(decode_plain_kernel<BF16, BS, MR, ST, BITS>, grid, waves, lds, stream, p);
}

template <bool BF16, int BS, typename ST, int BITS>
static int launch_plain_bs(const PackedParams& p, int waves, hipStream_t stream)
{
    if (p.m <= 1) return launch_plain_mr<BF16, BS, 1, ST, BITS>(p, waves, stream);
    if (p.m <= 4) return launch_plain_mr<BF16, BS, 4, ST, BITS>(p, waves, stream);
    if (p.m <= 8) return launch_plain_mr<BF16, BS, 8, ST, BITS>(p, waves, stream);
    return launch_plain_mr<BF16, BS, 16, ST, BITS>(p, waves, stream);
}

template <bool BF16, int BS, typename ST, int RB, int WMAX, int BITS>
static int launch_plain_wide_cfg(const PackedParams& p, int waves, hipStream_t stream)
{
    constexpr size_t lds = 2 * RB * 16 * (4 / (BITS / 4) * 256 + 16);      // two windows of the activations that four tiles of the stream meet
    const int64_t col_groups = (static_cast<int64_t>(p.n) + 15) / 16;
    return launch_on(decode_plain_wide_kernel<BF16, BS, ST, RB, WMAX, BITS>, static_cast<unsigned>((col_groups + waves - 1) / waves), waves, lds, stream, p);
}

template <bool BF16, int BS, typename ST, int BITS>
static int launch_plain_wide_bs(const PackedParams& p, int waves, hipStream_t stream)
{
    if (p.m <= 16) {
        if constexpr (BITS == 8 || BS != 32) {             // (sixteen scales a group: 4 bits at block 32 take more registers than twelve waves leave)
            if (waves > kWideWaves) return launch_plain_wide_cfg<BF16, BS, ST, 1, kWideWavesMax, BITS>(p, waves, stream);
        }
        return launch_plain_wide_cfg<BF16, BS, ST, 1, kWideWaves, BITS>(p, kWideWaves, stream);
    }
    if constexpr (BS != 32) {
        if (p.m <= 32) return launch_plain_wide_cfg<BF16, BS, ST, 2, kWideWaves, BITS>(p, kWideWaves, stream);
    }
    return -1;
}

// `go`: called with the element type, the block size, the scales' storage type and the bits as compile-time values
template <typename Go>
static int by_build(int bits, bool bf16, bool f32_scales, int block_size, Go go)
{
    auto by_block = [&](auto bf, auto st, auto bi) {
        switch (block_size) {
            case 32: return go(bf, std::integral_constant<int, 32>{}, st, bi);
            case 64: return go(bf, std::integral_constant<int, 64>{}, st, bi);
            default: return go(bf, std::integral_constant<int, 128>{}, st, bi);
        }
    };
    auto by_scales = [&](auto bf) {
        if (bits == 8) return f32_scales ? -1 : by_block(bf, uint16_t{}, std::integral_constant<int, 8>{});
        return f32_scales ? by_block(bf, float{}, std::integral_constant<int, 4>{}) : by_block(bf, uint16_t{}, std::integral_constant<int, 4>{});
    };
    return bf16 ? by_scales(std::true_type{}) : by_scales(std::false_type{});
}

int launch_plain(const PackedParams& p, int bits, bool bf16, bool f32_scales, int block_size, int waves, hipStream_t stream)
{
    return by_build(bits, bf16, f32_scales, block_size, [&](auto bf, auto bs, auto st, auto bi) {
        return launch_plain_bs<decltype(bf)::value, decltype(bs)::value, decltype(st), decltype(bi)::value>(p, waves, stream);
    });
}

int launch_plain_gather(const PackedParams& p, bool bf16, bool f32_scales, int block_size, int waves, hipStream_t stream)
{
    const unsigned grid = static_cast<unsigned>((static_cast<int64_t>(p.n) + 15) / 16);
    const size_t lds = plain_gather_lds(p.k, waves);
    return by_build(4, bf16, f32_scales, block_size, [&](auto bf, auto bs, auto st, auto bi) {
        if constexpr (decltype(bi)::value == 4) return launch_on(decode_plain_gather_kernel<decltype(bf)::value, decltype(bs)::value, decltype(st)>, grid, waves, lds, stream, p);
        else return -1;
    });
}

int launch_plain_wide(const PackedParams& p, int bits, bool bf16, bool f32_scales, int block_size, int waves, hipStream_t stream)
{
    return by_build(bits, bf16, f32_scales, block_size, [&](auto bf, auto bs, auto st, auto bi) {
        return launch_plain_wide_bs<decltype(bf)::value, decltype(bs)::value, decltype(st), decltype(bi)::value>(p, waves, stream);
    });
}

}  // namespace mnb

extern "C" int rocm_decode_plain_waves_per_simd(int block_size, int m, int f32_scales, int bf16, int bits)
{
    return mnb::plain_waves_per_simd(bf16 != 0, block_size, m <= 1 ? 1 : m <= 4 ? 4 : m <= 8 ? 8 : 16, f32_scales != 0, bits);
}
